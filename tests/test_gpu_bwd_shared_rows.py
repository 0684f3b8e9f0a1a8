"""The forms of the backward's workgroups, among them those whose waves share rows (dq) or keys (dk/dv) and add their sums through LDS: sizes
around a half-tile, a tile and a workgroup, odd and even numbers of tiles, against float64 autograd on the host."""
import pytest
import torch

from conftest import rand_qkv
from oracle import attn_oracle as O
import sp_aurora_amd as spa
from sp_aurora_amd import _lib
from test_gpu_many_sequences import reference as packed_reference
from test_gpu_parity import DEV, check_grad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,dq,dkdv", [(128, 20, 2), (128, 24, 2), (64, 20, 2), (128, 4, 3), (128, 8, 3), (64, 4, 3)])
def test_forms_with_shared_rows(D, dq, dkdv, dtype):
    try:
        _lib.tune("bwd_dq_waves", dq)
        _lib.tune("bwd_dkdv_form", dkdv)
        for S in (2, 31, 33, 64, 65, 96, 127, 129, 192, 257, 320, 449, 575):
            for causal in (True, False):
                q, k, v, dout = rand_qkv((1, S, 2, D), 700 + S, dtype, n=4)
                want = O.attn_backward_autograd(q, k, v, dout, None, causal)
                xs = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
                spa.ring_flash_attn_func(*xs, causal=causal).backward(dout.to(DEV))
                for x, w, name in zip(xs, want, "qkv"):
                    check_grad(x.grad, w, dtype, f"d{name}, {S} rows, causal {causal}")
        # fp32 accumulators that are added to, more keys than queries and the reverse
        for Sq, Sk in ((65, 200), (200, 65), (64, 640), (575, 300), (300, 575)):
            q, _, _, dout = rand_qkv((1, Sq, 2, D), 720, dtype, n=4)
            k, v, _, _ = rand_qkv((1, Sk, 2, D), 721, dtype, n=4)
            for causal in (True, False):
                out, lse = spa.ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), causal=causal)
                want = O.attn_backward_autograd(q, k, v, dout, None, causal)
                base = [torch.randn(t.shape, device=DEV) for t in (q, k, v)]
                acc = [t.clone() for t in base]
                delta = spa.ops.bwd_delta(out, dout.to(DEV))
                spa.ops.flash_bwd(q.to(DEV), k.to(DEV), v.to(DEV), dout.to(DEV), lse, delta, *acc, causal=causal)
                for a, b, w, name in zip(acc, base, want, "qkv"):
                    check_grad((a - b).to(dtype), w, dtype, f"d{name} added, {Sq} rows {Sk} keys, causal {causal}")
    finally:
        _lib.tune("bwd_dq_waves", 0)
        _lib.tune("bwd_dkdv_form", 0)


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16)])
@pytest.mark.parametrize("S", [64, 128, 192])  # odd and even numbers of tiles, all of them full
def test_a_key_that_holds_an_infinity(S, D, dtype):
    """A key hidden by -inf in one head dim has no weight: its gradients are zero, not NaN, also where passes come in pairs and one lies behind
    the last tile (dq, 0 * inf, is NaN)."""
    q, k, v, dout = rand_qkv((1, S, 2, D), 740 + S, dtype, n=4)
    q[..., 0], k[..., 0] = 1.0, 0.0
    k[:, S // 2, :, 0] = -float("inf")
    _, want_dk, want_dv = O.attn_backward_autograd(q, k, v, dout, None, False)
    assert want_dk.isfinite().all() and want_dv.isfinite().all()
    stack = lambda t, P: torch.stack(t.to(DEV).chunk(P, 1)).contiguous()
    try:
        for form in (2, 3):
            _lib.tune("bwd_dkdv_form", form)
            for P in (1, 2):
                xs = [stack(t, P).requires_grad_(True) for t in (q, k, v)]
                spa.LongContextAttention(sp_ulysses_degree=1, sp_ring_degree=P)(*xs, causal=False).backward(stack(dout, P))
                for x, w, name in zip(xs[1:], (want_dk, want_dv), "kv"):
                    check_grad(torch.cat(list(x.grad), 1), w, dtype, f"d{name}, form {form}, {P} shards")
    finally:
        _lib.tune("bwd_dkdv_form", 0)


def packed_step(lens, q, k, v, dout, causal, longest=None):
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    xs = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    out = spa.sp_aurora_varlen_func(*xs, cu, max_seqlen=longest or max(lens), causal=causal)
    return torch.autograd.grad(out, xs, dout.to(DEV))


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (128, torch.float16), (64, torch.bfloat16)])
@pytest.mark.parametrize("lens", [[1, 16, 0, 31, 33, 2], [64, 65, 96, 127, 128], [129, 3, 161, 200, 257]])
def test_short_sequences_in_every_form(lens, D, dtype):
    """Sequences that leave waves of a workgroup without rows or keys: those take part in loads and barriers only."""
    q, k, v, dout = rand_qkv((sum(lens), 2, D), 760, dtype, n=4)
    want = packed_reference(q, k, v, dout, lens)[1]
    try:
        for dq, dkdv in ((0, 0), (4, 3), (8, 1), (20, 2), (24, 3)):
            _lib.tune("bwd_dq_waves", dq)
            _lib.tune("bwd_dkdv_form", dkdv)
            for g, w, name in zip(packed_step(lens, q, k, v, dout, True), want, "qkv"):
                check_grad(g, w, dtype, f"d{name}, forms {dq} and {dkdv}")
    finally:
        _lib.tune("bwd_dq_waves", 0)
        _lib.tune("bwd_dkdv_form", 0)


def test_a_long_sequence_among_short_ones_decides_the_forms():
    """Most of the work of such a batch is the one sequence's: 256 rows and 128 keys a workgroup, whose sums differ in their last bits from
    those of 64."""
    lens = [64] * 50 + [6000] + [128] * 50
    q, k, v, dout = rand_qkv((sum(lens), 16, 128), 770, torch.bfloat16, n=4)
    got = packed_step(lens, q, k, v, dout, True)
    try:
        grads = {}
        for dq, dkdv in ((8, 3), (20, 2)):
            _lib.tune("bwd_dq_waves", dq)
            _lib.tune("bwd_dkdv_form", dkdv)
            grads[dq] = packed_step(lens, q, k, v, dout, True)
    finally:
        _lib.tune("bwd_dq_waves", 0)
        _lib.tune("bwd_dkdv_form", 0)
    for g, a, b in zip(got, grads[8], grads[20]):
        assert torch.equal(g, a) and not torch.equal(g, b)
