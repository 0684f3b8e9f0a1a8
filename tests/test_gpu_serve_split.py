"""Decode over ragged caches with the keys cut into chunks, and with neighbouring heads taken together: chunk edges, sequences without rows or
keys, a longest sequence past the last chunk's even share, strides under which heads cannot be taken together; against the kernels that
do neither (spa_tune few_rows), and these against float64 on the host."""
import pytest
import torch

from conftest import rand_qkv
from oracle import attn_oracle as O
from sp_aurora_amd import _lib, ops
from test_gpu_parity import DEV

pytestmark = pytest.mark.gpu
# both sides round P or the result to the type: as test_gpu_parity's bounds against the oracle, once per side
TOL = {torch.bfloat16: 2e-2, torch.float16: 4e-3}


def caches(lens, H, D, dtype, fp8, seed):
    q, = rand_qkv((max(1, sum(n for _, n in lens)), H, D), seed, dtype, n=1)
    k, v = rand_qkv((max(1, sum(n for n, _ in lens)), H, D), seed + 1, dtype, n=2)
    cu = lambda x: torch.tensor([0] + torch.tensor(x).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    scales = {}
    if fp8:
        scales = {n: torch.rand(len(lens), H, device=DEV) * 0.01 + 0.01 for n in ("k_scale", "v_scale")}
        k, v = ((t.float() * 40).clamp(-448, 448).to(torch.float8_e4m3fn) for t in (k, v))
    return q.to(DEV), k.to(DEV), v.to(DEV), cu([n for _, n in lens]), cu([n for n, _ in lens]), scales


def split(q, k, v, cu_q, cu_k, max_q, max_k, chunk, k_scale=None, v_scale=None):
    lib, (T, H, D), nseq = _lib.load(), q.shape, cu_q.numel() - 1
    out, lse = torch.full_like(q, float("nan")), torch.full((H, T), float("nan"), device=DEV)
    n = lib.spa_flash_fwd_varlen_splitkv_workspace_bytes(nseq, H, k.shape[0], max_q, max_k, D, chunk)
    ws = torch.full((n,), 255, dtype=torch.uint8, device=DEV)
    st = lambda t: _lib.strides2((t.stride(1), t.stride(0)))
    scale = lambda t: 0 if t is None else t.data_ptr()
    _lib.check(lib.spa_flash_fwd_varlen_splitkv(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), scale(k_scale), scale(v_scale), out.data_ptr(), lse.data_ptr(), ws.data_ptr(), cu_q.data_ptr(),
        cu_k.data_ptr(), nseq, H, T, k.shape[0], max_q, max_k, D, chunk, st(q), st(k), st(v), st(out), D ** -0.5,
        _lib.SPA_BF16 if q.dtype == torch.bfloat16 else _lib.SPA_F16, torch.cuda.current_stream().cuda_stream))
    return out, lse


def reference(*args, **kw):
    _lib.tune("few_rows", 1)
    try:
        return ops.flash_fwd_varlen(*args, **kw)
    finally:
        _lib.tune("few_rows", 0)


def check(got, want, dtype):
    torch.testing.assert_close(got[0], want[0], atol=TOL[dtype], rtol=TOL[dtype])
    torch.testing.assert_close(got[1], want[1], atol=1e-3, rtol=1e-5)


def exact(q, k, v, cu_q, cu_k, k_scale=None, v_scale=None):
    """Every sequence by itself in float64; rows without keys: zeros and -inf."""
    q, k, v = (t.cpu().double() for t in (q, k, v))
    out, lse = torch.zeros_like(q), torch.full((q.shape[1], q.shape[0]), -float("inf"), dtype=torch.float64)
    bounds = lambda cu: list(zip(cu.tolist(), cu.tolist()[1:]))
    for i, ((a, b), (c, d)) in enumerate(zip(bounds(cu_q), bounds(cu_k))):
        if a == b or c == d:
            continue
        x, y, z = (t.transpose(0, 1) for t in (q[a:b], k[c:d], v[c:d]))
        y = y if k_scale is None else y * k_scale[i].cpu().double()[:, None, None]
        z = z if v_scale is None else z * v_scale[i].cpu().double()[:, None, None]
        s = x @ y.transpose(-1, -2) * q.shape[-1] ** -0.5
        out[a:b], lse[:, a:b] = (torch.softmax(s, -1) @ z).transpose(0, 1), torch.logsumexp(s, -1)
    return out, lse


def check_exact(got, want, dtype):
    check([t.cpu().double() for t in got], want, dtype)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("chunk", [1, 64, 257, 512])
@pytest.mark.parametrize("H,reps", [(3, 1), (4, 1), (4, 30)])
def test_chunks_of_ragged_caches(H, reps, chunk, D, dtype, fp8):
    # (keys, rows): around the chunk's length, without keys, without rows, one far longer than the mean
    lens = [(chunk, 1), (chunk + 1, 2), (0, 1), (7, 0), (max(1, chunk - 1), 3), (5 * chunk + 3, 1), (2 * chunk, 2)] * reps + [(2000, 1)]
    q, k, v, cu_q, cu_k, scales = caches(lens, H, D, dtype, fp8, 1000 + chunk)
    max_k = max(n for n, _ in lens)
    want = reference(q, k, v, cu_q, cu_k, 3, max_k, **scales)
    check_exact(want, exact(q, k, v, cu_q, cu_k, **scales), dtype)
    check(split(q, k, v, cu_q, cu_k, 3, max_k, chunk, **scales), want, dtype)
    check(ops.flash_fwd_varlen(q, k, v, cu_q, cu_k, 3, max_k, **scales), want, dtype)  # (not split: heads together where there are enough)


@pytest.mark.parametrize("dtype,fp8", [(torch.bfloat16, False), (torch.float16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("H", [32, 30])  # (30: a count that four does not divide)
def test_many_small_chunks(H, dtype, fp8):
    """Eight workgroups and more per CU with 512 bytes of heads each, D = 128."""
    lens = [(1 + (i * 37) % 130, 1 + i % 3) for i in range(34)] + [(0, 1), (130, 0), (144, 3)]
    q, k, v, cu_q, cu_k, scales = caches(lens, H, 128, dtype, fp8, 1300 + H)
    want = reference(q, k, v, cu_q, cu_k, 3, 144, **scales)
    check_exact(want, exact(q, k, v, cu_q, cu_k, **scales), dtype)
    check(split(q, k, v, cu_q, cu_k, 3, 144, 16, **scales), want, dtype)


@pytest.mark.parametrize("nseq,longest", [(3, 900), (70, 2300)])
def test_suggested_chunks_and_capture(nseq, longest):
    H, D, dtype = 4, 128, torch.bfloat16
    lens = [(1 + (i * 997) % 700, 1) for i in range(nseq - 1)] + [(longest, 1)]
    q, k, v, cu_q, cu_k, _ = caches(lens, H, D, dtype, False, 1100)
    assert _lib.load().spa_flash_fwd_varlen_splitkv_suggest(nseq, H, k.shape[0], 1, longest, D, _lib.SPA_BF16) > 0
    want = reference(q, k, v, cu_q, cu_k, 1, longest)
    check_exact(want, exact(q, k, v, cu_q, cu_k), dtype)
    check(ops.flash_fwd_varlen(q, k, v, cu_q, cu_k, 1, longest), want, dtype)
    check(ops.flash_fwd_varlen(q, k, v, cu_q, cu_k, 1, k.shape[0]), want, dtype)  # a bound that no sequence is near
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        res = ops.flash_fwd_varlen(q, k, v, cu_q, cu_k, 1, longest)
    for _ in range(3):
        res[0].fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        check(res, want, dtype)


@pytest.mark.parametrize("D,fp8", [(64, False), (64, True), (128, True)])
@pytest.mark.parametrize("rows", [1, 2, 3])
def test_heads_taken_together_at_a_fixed_length(rows, D, fp8):
    B, H, S, dtype = 65, 16, 193, torch.bfloat16
    q, = rand_qkv((B, rows, H, D), 1200, dtype, n=1)
    k, v = rand_qkv((B, S, H, D), 1201, dtype, n=2)
    q, k, v = q.to(DEV), k.to(DEV), v.to(DEV)
    scales = {}
    if fp8:
        (k, ks), (v, vs) = (ops.quantize_fp8_per_head(t, layout="bshd") for t in (k, v))
        scales = {"k_scale": ks, "v_scale": vs}
    apart = lambda t: t.transpose(1, 2).contiguous().transpose(1, 2)  # heads before rows: not side by side
    got = ops.flash_fwd(q, k, v, layout="bshd", **scales)
    single = ops.flash_fwd(q, apart(k), apart(v), layout="bshd", **scales)
    mixed = ops.flash_fwd(q, k, apart(v), layout="bshd", **scales)
    _lib.tune("few_rows", 1)
    try:
        want = ops.flash_fwd(q, k, v, layout="bshd", **scales)
    finally:
        _lib.tune("few_rows", 0)
    scale = lambda t: 1.0 if t is None else t[:, None, :, None].cpu().double()
    y, z = k.cpu().double() * scale(scales.get("k_scale")), v.cpu().double() * scale(scales.get("v_scale"))
    check_exact(want, O.full_attention(q.cpu(), y, z, None, False), dtype)
    for x in (got, single, mixed):
        check(x, want, dtype)


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
def test_chunks_whose_keys_are_all_hidden(D, dtype):
    """Keys hidden through the inputs (a head dim that is 1 in q and -inf in those keys): whole chunks without a finite score, first, last
    and in between, beside chunks with some; against float64."""
    H = 4
    hide = [(300, 0, 130), (300, 60, 300), (200, 64, 128), (700, 0, 699)]  # (keys, the hidden ones)
    lens = [(n, 2) for n, _, _ in hide]
    q, k, v, cu_q, cu_k, _ = caches(lens, H, D, dtype, False, 1300)
    q[..., 0], k[..., 0] = 1.0, 0.0
    at, wants = 0, []
    for i, (n, lo, hi) in enumerate(hide):
        k[at + lo:at + hi, :, 0] = -float("inf")
        s = torch.einsum("qhd,khd->hqk", q[2 * i:2 * i + 2].cpu().double(), k[at:at + n].cpu().double()) * D ** -0.5
        out = torch.einsum("hqk,khd->qhd", torch.softmax(s, -1), v[at:at + n].cpu().double())
        wants.append((out, torch.logsumexp(s, -1)))
        at += n
    want = torch.cat([o for o, _ in wants]), torch.cat([l for _, l in wants], 1)
    for got in (split(q, k, v, cu_q, cu_k, 2, 700, 64), ops.flash_fwd_varlen(q, k, v, cu_q, cu_k, 2, 700)):
        check([t.cpu().double() for t in got], want, dtype)
    # one length: the chunks' results merged by their lse
    n = 4096
    q, = rand_qkv((1, 2, H, D), 1301, dtype, n=1)
    k, v = rand_qkv((1, n, H, D), 1302, dtype, n=2)
    q[..., 0], k[..., 0] = 1.0, 0.0
    for lo, hi in ((0, 1500), (1000, n), (600, 3000)):
        kk = k.clone()
        kk[:, lo:hi, :, 0] = -float("inf")
        s = torch.einsum("bqhd,bkhd->bhqk", q.double(), kk.double()) * D ** -0.5
        want = torch.einsum("bhqk,bkhd->bqhd", torch.softmax(s, -1), v.double()), torch.logsumexp(s, -1)
        got = ops.flash_fwd(q.to(DEV), kk.to(DEV), v.to(DEV), layout="bshd")
        check([t.cpu().double() for t in got], want, dtype)


@pytest.mark.parametrize("nseq", [1, 2, 63, 64, 65, 129, 4095, 4097, 4200])
@pytest.mark.parametrize("chunk", [1, 16, 100])
def test_chunks_are_found_in_long_lists(nseq, chunk):
    """The chunks of all sequences are numbered through: one far longer than the others (up to 1500 chunks), sequences without keys, lists
    around the 64 sequences and the 64 * 64 that a step of the search takes, and offsets that do not begin at the first row."""
    H, D, dtype, at = 2, 64, torch.float16, 150
    lens = [((i * 37) % 41 if i % 5 else 0, 1) for i in range(nseq)]
    lens[nseq // 3] = (1500, 2)
    q, k, v, cu_q, cu_k, _ = caches(lens, H, D, dtype, False, 1400 + nseq)
    want = reference(q, k, v, cu_q, cu_k, 2, 1500)
    check_exact(want, exact(q, k, v, cu_q, cu_k), dtype)
    check(split(q, k, v, cu_q, cu_k, 2, 1500, chunk), want, dtype)
    behind = lambda t: torch.cat([torch.full_like(t[:1], float("nan")).expand(at, -1, -1), t])
    check(split(q, behind(k), behind(v), cu_q, cu_k + at, 2, 1500, chunk), want, dtype)


@pytest.mark.parametrize("H,fp8", [(8, False), (32, True)])
def test_one_long_cache_beside_short_ones(H, fp8):
    """The library's own choice of chunks, at D = 128: chunks of the one cache go to workgroups of their own, also with 512 bytes of heads each."""
    lens = [(300, 1)] * 70 + [(20000, 1)] + [(257, 1)] * 20
    q, k, v, cu_q, cu_k, scales = caches(lens, H, 128, torch.bfloat16, fp8, 1500)
    want = reference(q, k, v, cu_q, cu_k, 1, 20000, **scales)
    check_exact(want, exact(q, k, v, cu_q, cu_k, **scales), torch.bfloat16)
    check(ops.flash_fwd_varlen(q, k, v, cu_q, cu_k, 1, 20000, **scales), want, torch.bfloat16)


@pytest.mark.parametrize("D,dtype,fp8", [(64, torch.float16, False), (64, torch.bfloat16, True), (128, torch.bfloat16, False), (128, torch.bfloat16, True)])
@pytest.mark.parametrize("H,count,longest", [(8, 9, 9000), (32, 12, 2500)])  # (fewer workgroups than CUs, and more)
def test_one_row_in_chunks_of_the_librarys_choice(H, count, longest, D, dtype, fp8):
    lens = [(1 + (i * 1997) % longest, 1) for i in range(count - 1)] + [(longest, 1)]
    q, k, v, cu_q, cu_k, scales = caches(lens, H, D, dtype, fp8, 1500 + H + count)
    assert _lib.load().spa_flash_fwd_varlen_splitkv_suggest(count, H, k.shape[0], 1, longest, D, _lib.SPA_BF16 if dtype == torch.bfloat16 else _lib.SPA_F16) == 256
    want = reference(q, k, v, cu_q, cu_k, 1, longest, **scales)
    check_exact(want, exact(q, k, v, cu_q, cu_k, **scales), dtype)
    check(ops.flash_fwd_varlen(q, k, v, cu_q, cu_k, 1, longest, **scales), want, dtype)


@pytest.mark.parametrize("dtype,fp8", [(torch.float16, False), (torch.bfloat16, True)])
def test_one_row_of_many_heads_together(dtype, fp8):
    """Six workgroups and more per CU with 512 bytes of heads each and eight loads in flight."""
    lens = [(1 + (i * 37) % 330, 1) for i in range(60)] + [(0, 1), (344, 1)]
    q, k, v, cu_q, cu_k, scales = caches(lens, 32, 128, dtype, fp8, 1600)
    want = reference(q, k, v, cu_q, cu_k, 1, 344, **scales)
    check_exact(want, exact(q, k, v, cu_q, cu_k, **scales), dtype)
    check(split(q, k, v, cu_q, cu_k, 1, 344, 16, **scales), want, dtype)
