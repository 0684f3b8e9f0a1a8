"""The attention work that a user of this package has it do, one case per way of using it.

A case is a dict of plain values; "kind" says which public entry points a pass goes through:

  block       the block operator on one (q chunk, kv chunk), layout [B,H,S,D]             _flash_attn_forward
  steps       one rank's ring by hand: the block operator per arriving chunk, merged      _flash_attn_forward, update_out_and_lse
  ring        ring attention, forward only (prefill, evaluation), layout [B,S,H,D]        sp_aurora_func
  train       ring attention, forward and backward                                        sp_aurora_func
  packed      the same on one packed qkv tensor                                           sp_aurora_qkvpacked_func
  ulysses     head-scatter / sequence-gather attention of all ranks, forward              ulysses_flash_attn_func
  hybrid      Ulysses inside groups, ring across them: the module, forward and backward   LongContextAttention
  varlen      a packed batch of sequences of different lengths, forward and backward      sp_aurora_varlen_func
  decode      a few new tokens against a KV cache of one length, 16-bit or e4m3           _flash_attn_forward
  serve       a decode step of a batch whose caches have different lengths                ops.flash_fwd_varlen
  e4m3        prefill with q, K and V quantised to e4m3                                   _flash_attn_forward
"""
import random

import torch

import sp_aurora_amd as sp

_DTYPE = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
_SIZE = {"float32": 4, "bfloat16": 2, "float16": 2, "e4m3": 1}


def listed():
    return [
        # The operator at the size its users try first and unit-test with: fp32, no mask, 0.5 GFLOP.  Latency.
        dict(name="block-fp32-512", kind="block", dtype="float32", batch=1, heads=8, rows=512, keys=512, dim=64, causal=False),
        # A training step of a small model, lengths that are no multiple of any tile: launches and host time.
        dict(name="train-fp16-250", kind="train", dtype="float16", batch=2, seq=250, heads=12, dim=64, causal=True, ring=1, zigzag=False),
        # Training on 64-wide heads over a ring of four: 1024 rows per rank.
        dict(name="train-ring4-4k-d64", kind="train", dtype="bfloat16", batch=2, seq=4096, heads=32, dim=64, causal=True, ring=4, zigzag=False),
        # The headline shape: a causal ring of eight over 8192 tokens, forward.
        dict(name="ring8-8k", kind="ring", dtype="bfloat16", batch=1, seq=8192, heads=32, dim=128, causal=True, ring=8, zigzag=False),
        # What each rank of that ring does when the communication is the caller's: the last rank's eight steps.
        dict(name="steps8-1k", kind="steps", dtype="bfloat16", batch=1, rows=1024, heads=32, dim=128, chunks=8),
        # Ulysses over eight ranks, 16384 tokens: the longest forward.
        dict(name="ulysses8-16k", kind="ulysses", dtype="bfloat16", batch=1, seq=16384, heads=32, dim=128, causal=True, ranks=8),
        # Long-context training on a packed qkv tensor, a ring of sixteen over 32768 tokens: the largest.
        dict(name="packed-ring16-32k", kind="packed", dtype="bfloat16", batch=1, seq=32768, heads=16, dim=128, causal=True, ring=16),
        # Two-dimensional sequence parallelism: Ulysses pairs in a ring of four, a training step of two sequences.
        dict(name="hybrid-2x4-4k", kind="hybrid", dtype="bfloat16", batch=2, seq=4096, heads=16, dim=128, causal=True, ulysses=2, ring=4),
        # Fine-tuning on documents of different lengths, packed without padding.
        dict(name="varlen-24x2k", kind="varlen", dtype="bfloat16", count=24, longest=2000, lens=1, heads=16, dim=128, causal=True, ring=1),
        # One new token of one sequence against a long cache.
        dict(name="decode-32k", kind="decode", dtype="bfloat16", cache="bfloat16", batch=1, heads=32, rows=1, keys=32768, dim=128),
        # A decode step of a server: 64 sequences, caches of 1024 to 4096 tokens held as e4m3.
        dict(name="serve-64x4k-e4m3", kind="serve", dtype="bfloat16", cache="e4m3", count=64, longest=4096, lens=2, heads=32, dim=128),
        # Prefill of a quantised model at the headline length.
        dict(name="e4m3-8k", kind="e4m3", dtype="bfloat16", batch=1, heads=32, rows=8192, dim=128, causal=True),
    ]


# ---------------------------------------------------------------- drawn cases
def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _length(rng, lo, hi, step=1):
    """A length spread over the logarithm of lo .. hi: every other one a multiple of 64, the rest as they fall."""
    n = _log(rng, lo, hi)
    if rng.random() < 0.5:
        n = (n + 63) // 64 * 64
    return max(step, n // step * step)


def _fit(n, flops_per_row2, limit):
    """The length, cut so that flops_per_row2 * n^2 stays below the limit."""
    return min(n, int((limit / flops_per_row2) ** 0.5))


def draw(rng):
    kind = rng.choice(["block", "steps", "ring", "train", "packed", "ulysses", "hybrid", "varlen", "decode", "serve", "e4m3"])
    dim = rng.choice([64, 128, 128])
    dtype = rng.choice(["bfloat16", "bfloat16", "float16"])
    causal = rng.random() < 0.75
    if kind == "block":
        # the operator's own benchmark range: 512 to 4096 rows, 8 to 32 heads, fp32 as often as 16 bits
        dtype = rng.choice(["float32", "float32", "bfloat16", "float16"])
        rows = _length(rng, 128, 4096)
        keys = rows if causal else _length(rng, 128, 4096)
        return dict(kind=kind, dtype=dtype, batch=rng.choice([1, 1, 2]), heads=rng.choice([8, 12, 16, 32]), rows=rows, keys=keys,
                    dim=rng.choice([32, 64, 128]), causal=causal)
    if kind == "steps":
        return dict(kind=kind, dtype=dtype, batch=rng.choice([1, 2]), rows=_length(rng, 128, 2048), heads=rng.choice([8, 16, 32]), dim=dim,
                    chunks=rng.choice([2, 4, 8]))
    if kind in ("ring", "train"):
        ring = rng.choice([1, 2, 4, 8])
        zigzag = causal and ring > 1 and rng.random() < 0.25
        batch, heads = rng.choice([1, 1, 2, 4]), rng.choice([8, 12, 16, 32])
        if kind == "train" and rng.random() < 0.25:
            dtype, batch, seq = "float32", 1, _length(rng, 128, 2048, 2 * ring)
        else:
            seq = _length(rng, 128, 16384, 2 * ring)
        seq = max(2 * ring, _fit(seq, 14.0 * batch * heads * dim, 2e12) // (2 * ring) * (2 * ring))
        return dict(kind=kind, dtype=dtype, batch=batch, seq=seq, heads=heads, dim=dim, causal=causal, ring=ring, zigzag=zigzag)
    if kind == "packed":
        ring, heads = rng.choice([1, 4, 16]), rng.choice([8, 16, 32])
        seq = _fit(_length(rng, 256, 32768, ring), 14.0 * heads * dim, 4e12) // ring * ring
        return dict(kind=kind, dtype=dtype, batch=1, seq=seq, heads=heads, dim=dim, causal=causal, ring=ring)
    if kind == "ulysses":
        ranks = rng.choice([2, 4, 8])
        return dict(kind=kind, dtype=dtype, batch=rng.choice([1, 2]), seq=_length(rng, 512, 16384, ranks), heads=rng.choice([16, 32]), dim=dim,
                    causal=causal, ranks=ranks)
    if kind == "hybrid":
        ulysses, ring = rng.choice([(2, 2), (2, 4), (4, 2)])
        return dict(kind=kind, dtype=dtype, batch=rng.choice([1, 2]), seq=_length(rng, 512, 8192, ulysses * ring), heads=rng.choice([8, 16]),
                    dim=dim, causal=causal, ulysses=ulysses, ring=ring)
    if kind == "varlen":
        return dict(kind=kind, dtype=dtype, count=rng.choice([3, 8, 24, 40]), longest=_length(rng, 200, 4096), lens=rng.randrange(1 << 20),
                    heads=rng.choice([8, 16]), dim=dim, causal=causal, ring=rng.choice([1, 1, 1, 4]))
    if kind == "decode":
        batch = rng.choice([1, 1, 4, 16])
        return dict(kind=kind, dtype=dtype, cache=rng.choice([dtype, "e4m3"]), batch=batch, heads=rng.choice([8, 32]),
                    rows=rng.choice([1, 1, 2, 8]), keys=_length(rng, 512, 65536 // batch), dim=dim)
    if kind == "serve":
        return dict(kind=kind, dtype=dtype, cache=rng.choice([dtype, "e4m3"]), count=rng.choice([8, 32, 64]), longest=_length(rng, 512, 8192),
                    lens=rng.randrange(1 << 20), heads=rng.choice([8, 32]), dim=dim)
    return dict(kind="e4m3", dtype="bfloat16", batch=rng.choice([1, 1, 2]), heads=rng.choice([8, 16, 32]), rows=_length(rng, 256, 8192), dim=128,
                causal=causal)


# ---------------------------------------------------------------- inputs
def _lengths(case):
    """The sequences' lengths of a ragged batch (per rank, with a ring): a quarter of the longest up to the longest."""
    r = random.Random(case["lens"])
    top = max(1, case["longest"] // case.get("ring", 1))
    lens = [r.randint(max(1, top // 4), top) for _ in range(case["count"])]
    lens[r.randrange(len(lens))] = top
    return lens


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype, D, H = case["kind"], _DTYPE[case["dtype"]], case["dim"], case["heads"]

    def normal(*shape, grad=False):
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype).requires_grad_(grad)

    def offsets(lens):
        at = [0]
        for n in lens:
            at.append(at[-1] + n)
        return torch.tensor(at, dtype=torch.int32, device="cuda")

    s = {"case": case}
    if kind == "block":
        B = case["batch"]
        s["q"] = normal(B, H, case["rows"], D)
        s["k"], s["v"] = (normal(B, H, case["keys"], D) for _ in range(2))
    elif kind == "steps":
        # the chunks in the order in which they arrive: the rank's own first
        s["q"] = normal(case["batch"], H, case["rows"], D)
        s["chunks"] = [(normal(*s["q"].shape), normal(*s["q"].shape)) for _ in range(case["chunks"])]
    elif kind in ("ring", "train"):
        shape, grad = (case["batch"], case["seq"], H, D), kind == "train"
        s["q"], s["k"], s["v"] = (normal(*shape, grad=grad) for _ in range(3))
        s["dout"] = normal(*shape) if grad else None
    elif kind == "packed":
        s["qkv"] = normal(case["batch"], case["seq"], 3, H, D, grad=True)
        s["dout"] = normal(case["batch"], case["seq"], H, D)
    elif kind == "ulysses":
        P = case["ranks"]
        s["q"], s["k"], s["v"] = (normal(P, case["batch"], case["seq"] // P, H, D) for _ in range(3))
    elif kind == "hybrid":
        W = case["ulysses"] * case["ring"]
        shape = (W, case["batch"], case["seq"] // W, H, D)
        s["q"], s["k"], s["v"] = (normal(*shape, grad=True) for _ in range(3))
        s["dout"] = normal(*shape)
        s["attention"] = sp.LongContextAttention(sp_ulysses_degree=case["ulysses"], sp_ring_degree=case["ring"])
    elif kind == "varlen":
        lens = _lengths(case)
        s["cu"], s["longest"] = offsets(lens), max(lens)
        total = sum(lens) * case["ring"]
        s["q"], s["k"], s["v"] = (normal(total, H, D, grad=True) for _ in range(3))
        s["dout"] = normal(total, H, D)
    elif kind == "decode":
        B = case["batch"]
        s["q"] = normal(B, H, case["rows"], D)
        s["k"], s["v"] = (normal(B, H, case["keys"], D) for _ in range(2))
        s["scales"] = {}
        if case["cache"] == "e4m3":
            s["k"], ks = sp.ops.quantize_fp8_per_head(s["k"], layout="bhsd")
            s["v"], vs = sp.ops.quantize_fp8_per_head(s["v"], layout="bhsd")
            s["scales"] = {"k_scale": ks, "v_scale": vs}
    elif kind == "serve":
        lens = _lengths(case)
        n, total = len(lens), sum(lens)
        s["cu_q"], s["cu_k"], s["longest"] = offsets([1] * n), offsets(lens), max(lens)
        s["q"] = normal(n, H, D)
        s["k"], s["v"] = (normal(total, H, D) for _ in range(2))
        s["scales"] = {}
        if case["cache"] == "e4m3":
            # one scale per (sequence, head): 448 is the largest e4m3 value, 5.6 bounds these normal values
            s["scales"] = {name: torch.rand(n, H, generator=gen, device="cuda") * 0.005 + 0.0125 for name in ("k_scale", "v_scale")}
            owner = torch.repeat_interleave(torch.arange(n, device="cuda"), torch.tensor(lens, device="cuda"))
            for t, name in (("k", "k_scale"), ("v", "v_scale")):
                s[t] = (s[t].float() / s["scales"][name][owner][:, :, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    elif kind == "e4m3":
        quantised = [sp.ops.quantize_fp8_per_head(normal(case["batch"], H, case["rows"], D), layout="bhsd") for _ in range(3)]
        (s["q"], qs), (s["k"], ks), (s["v"], vs) = quantised
        s["scales"] = {"q_scale": qs, "k_scale": ks, "v_scale": vs}
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    kind, causal = case["kind"], case.get("causal", False)
    if kind == "block":
        return sp._flash_attn_forward(s["q"], s["k"], s["v"], causal=causal)
    if kind == "steps":
        out = lse = None
        for i, (k, v) in enumerate(s["chunks"]):
            block_out, block_lse = sp._flash_attn_forward(s["q"], k, v, causal=i == 0)
            out, lse = sp.update_out_and_lse(out, lse, block_out, block_lse)
        return out.to(s["q"].dtype), lse.squeeze(-1).transpose(1, 2)
    if kind in ("ring", "train"):
        sharding = "zigzag" if case["zigzag"] else "contiguous"
        out = sp.sp_aurora_func(s["q"], s["k"], s["v"], causal=causal, ring_size=case["ring"], sharding=sharding)
        if kind == "ring":
            return out
        return (out, *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"]))
    if kind == "packed":
        out = sp.sp_aurora_qkvpacked_func(s["qkv"], causal=causal, ring_size=case["ring"])
        return (out, *torch.autograd.grad(out, (s["qkv"],), s["dout"]))
    if kind == "ulysses":
        return sp.ulysses_flash_attn_func(s["q"], s["k"], s["v"], causal=causal)
    if kind == "hybrid":
        out = s["attention"](s["q"], s["k"], s["v"], causal=causal)
        return (out, *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"]))
    if kind == "varlen":
        out = sp.sp_aurora_varlen_func(s["q"], s["k"], s["v"], s["cu"], max_seqlen=s["longest"], causal=causal, ring_size=case["ring"])
        return (out, *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"]))
    if kind == "serve":
        return sp.ops.flash_fwd_varlen(s["q"], s["k"], s["v"], s["cu_q"], s["cu_k"], 1, s["longest"], **s["scales"])
    return sp._flash_attn_forward(s["q"], s["k"], s["v"], causal=causal, **s["scales"])  # decode, e4m3


# ---------------------------------------------------------------- what a pass cannot do without
def _pairs(rows, keys, causal):
    """(query, key) pairs that see each other."""
    if not causal:
        return rows * keys
    n = min(rows, keys)
    return n * (n + 1) // 2 + (rows - n) * keys


def work(case):
    """flops: 4 D per visible (query, key) pair and head forward, 10 D backward (its five products); bytes: inputs read
    once, outputs written once (lse included where it is returned, and, with a backward, saved and read)."""
    kind, D, H, e = case["kind"], case["dim"], case["heads"], _SIZE[case["dtype"]]
    causal = case.get("causal", False)
    if kind in ("block", "decode", "e4m3"):
        B, rows, keys = case["batch"], case["rows"], case.get("keys", case["rows"])
        qe, ke = (1, 1) if kind == "e4m3" else (e, _SIZE[case.get("cache", case["dtype"])])
        return {"flops": 4 * B * H * D * _pairs(rows, keys, causal), "bytes": B * H * (rows * (D * (qe + e) + 4) + 2 * keys * D * ke)}
    if kind == "steps":
        B, n = case["batch"], case["rows"]
        pairs = _pairs(n, n, True) + (case["chunks"] - 1) * n * n
        return {"flops": 4 * B * H * D * pairs, "bytes": B * H * n * (2 * D * e + 4 + 2 * case["chunks"] * D * e)}
    if kind == "serve":
        lens = _lengths(case)
        return {"flops": 4 * H * D * sum(lens), "bytes": H * (len(lens) * (2 * D * e + 4) + 2 * sum(lens) * D * _SIZE[case["cache"]])}
    if kind == "varlen":
        lens = [n * case["ring"] for n in _lengths(case)]
        rows, pairs = sum(lens), sum(_pairs(n, n, causal) for n in lens)
    else:
        rows = case["batch"] * case["seq"]
        pairs = case["batch"] * _pairs(case["seq"], case["seq"], causal)
    if kind in ("ring", "ulysses"):
        return {"flops": 4 * H * D * pairs, "bytes": H * rows * 4 * D * e}
    # forward: q, k, v in, out and lse written; backward: q, k, v, out, dout, lse in, dq, dk, dv written
    return {"flops": 14 * H * D * pairs, "bytes": H * rows * ((4 + 8) * D * e + 8)}


def tolerance(case):
    """Sums in fp32 everywhere.  fp32 operands: the sums' rounding.  16-bit operands: P and dS are rounded to the type
    before they are multiplied, results and gradients once more."""
    return {"rel": {"float32": 2e-5, "float16": 3e-3, "bfloat16": 1e-2}[case["dtype"]]}
