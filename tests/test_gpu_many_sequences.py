"""Packed batches of many sequences: the search of a numbered grid at the edges of its blocks of 64 and groups of 512 sequences, and the
grid of sequences x tiles, forward and backward, against float64 attention of every sequence."""
import random

import pytest
import torch

from conftest import rand_qkv
import sp_aurora_amd as spa
from test_gpu_parity import DEV, check_grad, check_out

pytestmark = pytest.mark.gpu


def reference(q, k, v, dout, lens):
    """Causal attention and gradients of sequences packed back to back, float64: sequences of one length together."""
    leaves = [t.double().requires_grad_() for t in (q, k, v)]
    out = torch.zeros_like(leaves[0].detach())
    starts = torch.tensor([0] + lens).cumsum(0)
    for n in set(lens) - {0}:
        idx = torch.stack([torch.arange(int(s), int(s) + n) for s, m in zip(starts, lens) if m == n])
        x, y, z = (t[idx].transpose(1, 2) for t in leaves)
        s = (x @ y.transpose(-1, -2)) * q.shape[-1] ** -0.5
        p = torch.softmax(s.masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), -float("inf")), -1)
        out = out.index_put((idx,), (p @ z).transpose(1, 2))
    return out.detach(), torch.autograd.grad(out, leaves, dout.double())


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 64), (torch.float32, 32)])
@pytest.mark.parametrize("longest", [40, 3000])  # of one tile each: sequences x tiles; one far longer than the others: numbered
@pytest.mark.parametrize("nseq", [1, 63, 64, 65, 128, 511, 512, 513, 1100])
def test_many_sequences(nseq, longest, dtype, D):
    H, r = 2, random.Random(nseq)
    lens = [r.choice([0, 1, 2, 7, 33, 40]) for _ in range(nseq)]
    lens[nseq // 2] = longest
    lens[-1] = max(lens[-1], 3)
    total = sum(lens)
    q, k, v, dout = rand_qkv((total, H, D), 1400 + nseq, dtype, n=4)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    out = spa.sp_aurora_varlen_func(*leaves, cu, max_seqlen=longest, causal=True)
    got = torch.autograd.grad(out, leaves, dout.to(DEV))
    want, grads = reference(q, k, v, dout, lens)
    check_out(out, want, dtype)
    for name, g, w in zip("qkv", got, grads):
        check_grad(g, w, dtype, "d" + name)
