"""Queries whose rows are not back to back ([B,S,H,D], a packed qkv tensor) pass through LDS in the form with two wave groups: row
counts around a wave's rows and a workgroup's, a negative scale, keys fewer and more than rows, against the oracle."""
import pytest
import torch

from conftest import rand_qkv
from oracle import attn_oracle as O
import sp_aurora_amd as spa
from sp_aurora_amd import _lib
from test_gpu_parity import DEV, check_lse, check_out

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Sq,Sk,causal,scale", [(1, 65, False, None), (31, 130, False, -0.1), (33, 200, True, None), (127, 127, True, None),
                                                (129, 65, False, None), (200, 300, True, -0.05), (257, 257, True, None)])
def test_rows_through_lds(Sq, Sk, causal, scale, dtype):
    B, H, D = 2, 3, 128
    wide, = rand_qkv((B, Sq, 3 * H, D), 900, dtype, n=1)
    q = wide[:, :, H:2 * H]                       # rows 3 H D apart
    k, v = rand_qkv((B, Sk, H, D), 901, dtype, n=2)
    want, want_lse = O.attn_block(*(t.transpose(1, 2) for t in (q, k, v)), scale, causal)
    try:
        _lib.tune("fwd_groups", 2)
        _lib.tune("fwd_share", 1)
        _lib.tune("few_rows", 1)
        out, lse = spa.ops.flash_fwd(wide.to(DEV)[:, :, H:2 * H], k.to(DEV), v.to(DEV), softmax_scale=scale, causal=causal, split_kv=None)
    finally:
        for knob in ("fwd_groups", "fwd_share", "few_rows"):
            _lib.tune(knob, 0)
    check_out(out.transpose(1, 2), want, dtype)
    check_lse(lse, want_lse)
