"""Rank-stacked operands with several batch entries that are views of [B,S,H,D] tensors, x.view(B, P, s, H, D).transpose(0, 1): their
rows follow each other, while those of a compact stacked result do not.  All of q, k, v so, and mixed with stacked copies, against
float64 attention over the whole sequences."""
import pytest
import torch

from conftest import rand_qkv
from oracle import attn_oracle as O
import sp_aurora_amd as spa
from test_gpu_parity import DEV, check_grad, check_out

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views", ["qkv", "q", "kv", ""])
@pytest.mark.parametrize("P,B,s,H,D,dtype", [(2, 2, 5, 2, 32, torch.float32), (4, 2, 16, 4, 64, torch.bfloat16), (2, 3, 70, 2, 128, torch.float16),
                                             (3, 1, 20, 3, 64, torch.bfloat16), (1, 2, 33, 2, 64, torch.bfloat16)])
def test_stacked_views(P, B, s, H, D, dtype, views):
    S = P * s
    q, k, v, dout = rand_qkv((B, S, H, D), 1300 + S, dtype, n=4)
    view = lambda t: t.view(B, P, s, H, D).transpose(0, 1)
    whole = lambda t: t.transpose(0, 1).reshape(B, S, H, D)
    layer = spa.LongContextAttention(sp_ulysses_degree=1, sp_ring_degree=P)
    want, _ = O.full_attention(q, k, v, None, True)
    grads = O.attn_backward_autograd(q, k, v, dout, None, True)
    for fn in (lambda *x: spa.ulysses_flash_attn_func(*x, causal=True), lambda *x: layer(*x, causal=True)):
        leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
        operands = [view(t) if n in views else view(t).contiguous() for n, t in zip("qkv", leaves)]
        with torch.no_grad():
            check_out(whole(fn(*operands)), want, dtype)
        out = fn(*operands)
        check_out(whole(out.detach()), want, dtype)
        for name, got, ref in zip("qkv", torch.autograd.grad(out, leaves, view(dout.to(DEV))), grads):
            check_grad(got, ref, dtype, "d" + name)
