"""Attention over sequences whose rows lie in shards (rank-stacked tensors, zigzag rings, packed batches of shards): segments
shorter and longer than a tile and around its size, every form of the kernels, against the call on the rows in order, which is itself
compared with float64 on the host."""
import pytest
import torch

from conftest import rand_qkv
from oracle import attn_oracle as O
import sp_aurora_amd as spa
from sp_aurora_amd import _lib
from test_gpu_many_sequences import reference as packed_reference
from test_gpu_parity import DEV, check_grad, check_out

pytestmark = pytest.mark.gpu
TOL = {torch.bfloat16: 2e-2, torch.float16: 4e-3, torch.float32: 1e-5}
FORMS = [dict(fwd_groups=1, bwd_dq_waves=4, bwd_dkdv_form=3), dict(fwd_groups=2, fwd_share=1, bwd_dq_waves=20, bwd_dkdv_form=2),
         dict(fwd_groups=2, fwd_share=2, bwd_dq_waves=8, bwd_dkdv_form=3), dict(bwd_dq_waves=24, bwd_dkdv_form=3)]


def close(got, want, tol):
    torch.testing.assert_close(got, want, atol=tol, rtol=tol)


def step(fn, leaves, dout):
    out = fn(*leaves)
    return (out.detach(), *torch.autograd.grad(out, leaves, dout))


def check_step(got, out, grads, dtype):
    check_out(got[0], out, dtype)
    for name, g, w in zip("qkv", got[1:], grads):
        check_grad(g, w, dtype, "d" + name)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 64), (torch.float32, 32)])
@pytest.mark.parametrize("P,seg", [(2, 1), (8, 17), (3, 63), (4, 64), (5, 65), (2, 200)])
def test_segments_around_the_tile_size(P, seg, dtype, D):
    B, H, S = 2, 3, P * seg
    q, k, v, dout = (t.to(DEV) for t in rand_qkv((B, S, H, D), 900 + S, dtype, n=4))
    stack = lambda t: torch.stack(t.chunk(P, 1)).contiguous()
    unstack = lambda t: torch.cat(list(t), 1)
    layer = spa.LongContextAttention(sp_ulysses_degree=1, sp_ring_degree=P)
    host = [t.cpu() for t in (q, k, v, dout)]
    exact = {c: (O.full_attention(*host[:3], None, c)[0], O.attn_backward_autograd(*host, None, c)) for c in (True, False)}
    for form in FORMS if dtype != torch.float32 else FORMS[:1]:
        try:
            for knob, value in form.items():
                _lib.tune(knob, value)
            for causal in (True, False):
                want = step(lambda *x: spa.sp_aurora_func(*x, causal=causal), [t.clone().requires_grad_() for t in (q, k, v)], dout)
                check_step(want, *exact[causal], dtype)
                got = step(lambda *x: layer(*x, causal=causal), [stack(t).requires_grad_() for t in (q, k, v)], stack(dout))
                for g, w in zip(got, want):
                    close(unstack(g), w, 2 * TOL[dtype])
            if S % (2 * P) == 0:  # the same rows as zigzag shards
                idx = spa.ring.zigzag_order(S, P, DEV)
                zig = lambda t: t.index_select(1, idx)
                want = step(lambda *x: spa.sp_aurora_func(*x, causal=True), [t.clone().requires_grad_() for t in (q, k, v)], dout)
                out, lse, _ = spa.sp_aurora_func(zig(q), zig(k), zig(v), causal=True, return_attn_probs=True, ring_size=P, sharding="zigzag")
                _, want_lse, _ = spa.sp_aurora_func(q, k, v, causal=True, return_attn_probs=True)
                close(out, zig(want[0]), TOL[dtype])
                torch.testing.assert_close(lse, want_lse.index_select(2, idx), atol=1e-4, rtol=1e-5)
                got = step(lambda *x: spa.sp_aurora_func(*x, causal=True, ring_size=P, sharding="zigzag"),
                           [zig(t).requires_grad_() for t in (q, k, v)], zig(dout))
                for g, w in zip(got, want):
                    close(g, zig(w), 2 * TOL[dtype])
        finally:
            for knob in form:
                _lib.tune(knob, 0)


@pytest.mark.parametrize("zigzag", [False, True])
@pytest.mark.parametrize("dtype,D,form", [(torch.bfloat16, 64, {}), (torch.float32, 64, {})] + [(torch.bfloat16, 128, form) for form in FORMS])
def test_packed_batches_of_shards(dtype, D, form, zigzag):
    try:
        for knob, value in form.items():
            _lib.tune(knob, value)
        packed_batch_of_shards(dtype, D, zigzag)
    finally:
        for knob in form:
            _lib.tune(knob, 0)


def packed_batch_of_shards(dtype, D, zigzag):
    P, local, H = 3, [2, 0, 64, 130, 36], 2
    T = sum(local)
    cu = torch.tensor([0] + torch.tensor(local).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    lens = [n * P for n in local]
    q, k, v, dout = (t.to(DEV) for t in rand_qkv((T * P, H, D), 930, dtype, n=4))  # rows in the sequences' own order
    if zigzag:
        idx = spa.zigzag_varlen_order(lens, P).to(DEV)
    else:
        starts = torch.tensor([0] + lens).cumsum(0).tolist()
        idx = torch.cat([torch.arange(starts[i] + r * n, starts[i] + (r + 1) * n) for r in range(P) for i, n in enumerate(local)]).to(DEV)
    cu_all = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    want = step(lambda *x: spa.sp_aurora_varlen_func(*x, cu_all, max_seqlen=max(lens), causal=True), [t.clone().requires_grad_() for t in (q, k, v)], dout)
    got = step(lambda *x: spa.sp_aurora_varlen_func(*x, cu, max_seqlen=max(local), causal=True, ring_size=P, sharding="zigzag" if zigzag else "contiguous"),
               [t[idx].requires_grad_() for t in (q, k, v)], dout[idx])
    check_step(want, *packed_reference(*(t.cpu() for t in (q, k, v, dout)), lens), dtype)
    for g, w in zip(got, want):
        close(g, w[idx], 2 * TOL[dtype])
