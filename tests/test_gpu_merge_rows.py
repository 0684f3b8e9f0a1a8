"""Merge of a block's result into the running sums: row counts below, at and past what a workgroup takes of a head, every head dim and type,
against float64.  Bounds: the sums' rounding (fp32, a few operations on values of size 4)."""
import pytest
import torch

import sp_aurora_amd as spa
from test_gpu_parity import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["bshd", "bhsd"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,S,H,D", [(2, 1, 5, 128), (1, 15, 3, 128), (2, 16, 3, 128), (1, 33, 8, 128), (1, 31, 3, 64), (2, 65, 4, 64), (1, 63, 2, 32),
                                     (1, 130, 3, 32), (1, 7, 3, 512), (2, 300, 2, 8)])
def test_merge_rows(B, S, H, D, dtype, layout):
    g = torch.Generator().manual_seed(S * 1000 + D)
    shape = (B, S, H, D) if layout == "bshd" else (B, H, S, D)
    acc, blk = torch.randn(shape, generator=g), torch.randn(shape, generator=g).to(dtype)
    la, lb = (torch.randn((B, H, S), generator=g) * 3 for _ in range(2))
    la[:, :, 0] = -float("inf")                    # nothing accumulated yet
    got, got_lse = acc.to(DEV), la.to(DEV)
    spa.ops.merge(got, got_lse, blk.to(DEV), lb.to(DEV), layout=layout)
    w = torch.sigmoid(lb.double() - la.double())[..., None]
    if layout == "bshd":
        w = w.transpose(1, 2)
    want = acc.double() + w * (blk.double() - acc.double())
    # the sums' three roundings of values up to 10, and the weight (a hardware exponential and a division)
    assert (got.cpu().double() - want).abs().max().item() < 1e-5
    assert (got_lse.cpu().double() - torch.logaddexp(la.double(), lb.double())).abs().max().item() < 4e-6
    first, first_lse = torch.empty_like(got), torch.empty_like(got_lse)
    spa.ops.merge(first, first_lse, blk.to(DEV), lb.to(DEV), layout=layout, init=True)
    assert torch.equal(first.cpu(), blk.float()) and torch.equal(first_lse.cpu(), lb)
