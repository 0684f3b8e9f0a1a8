"""The fp32 backward in both forms of its workgroups (128 rows, or 32 rows whose tiles the waves share out): one tile, fewer tiles than
waves, a last tile with one row, more keys than queries and the reverse, packed batches; against the oracle's autograd."""
import pytest
import torch

from conftest import rand_qkv
from oracle import attn_oracle as O
import sp_aurora_amd as spa
from sp_aurora_amd import _lib, ops
from test_gpu_parity import DEV, check_grad

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[1, 2])
def form(request):
    _lib.tune("fwd32_split", request.param)
    yield request.param
    _lib.tune("fwd32_split", 0)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Sq,Sk,causal", [(1, 5, False), (32, 32, True), (33, 129, True), (129, 33, True), (160, 97, False), (257, 257, True)])
def test_both_forms(form, D, Sq, Sk, causal):
    q, dout = rand_qkv((2, Sq, 3, D), 1300, torch.float32, n=2)
    k, v = rand_qkv((2, Sk, 3, D), 1301, torch.float32, n=2)
    want = O.attn_backward_autograd(q, k, v, dout, None, causal)
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out = spa.sp_aurora_func(*leaves, causal=causal)
    grads = torch.autograd.grad(out, leaves, dout.to(DEV))
    for g, w, name in zip(grads, want, "qkv"):
        check_grad(g, w, torch.float32, "d" + name)
    # into accumulators that hold something
    qd, kd, vd, dd = (t.to(DEV) for t in (q, k, v, dout))
    o, lse = ops.flash_fwd(qd, kd, vd, None, causal)
    acc = [torch.ones_like(t) for t in (qd, kd, vd)]
    ops.flash_bwd(qd, kd, vd, dd, lse, ops.bwd_delta(o, dd), *acc, None, causal)
    for g, w, name in zip(acc, want, "qkv"):
        check_grad(g - 1, w, torch.float32, "d" + name)


def test_a_packed_batch(form):
    lens, H, D = [0, 3, 33, 0, 200, 64], 2, 64
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    q, k, v, dout = rand_qkv((sum(lens), H, D), 1310, torch.float32, n=4)
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    grads = torch.autograd.grad(spa.sp_aurora_varlen_func(*leaves, cu, max_seqlen=max(lens), causal=True), leaves, dout.to(DEV))
    at = 0
    for n in lens:
        if n:
            rows = slice(at, at + n)
            want = O.attn_backward_autograd(*(t[rows].unsqueeze(0) for t in (q, k, v, dout)), None, True)
            for g, w, name in zip(grads, want, "qkv"):
                check_grad(g[rows].unsqueeze(0), w, torch.float32, "d" + name)
        at += n
