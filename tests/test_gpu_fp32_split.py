"""The fp32 forward for launches with few query rows (32-row workgroups whose eight waves share the key tiles and
combine through LDS): forced on and off through spa_tune, both forms against the oracle on the same inputs, and the
library's own choice at the benchmark's config 1."""
import pytest
import torch

from conftest import rand_qkv
from oracle import attn_oracle as O
import sp_aurora_amd as sp
from sp_aurora_amd import _lib, ops
from test_gpu_parity import DEV, check_lse, check_out

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Sq, Sk, D, causal
    (1, 8, 512, 512, 64, False),    # benchmark config 1
    (1, 8, 512, 512, 64, True),
    (2, 3, 100, 333, 64, False),    # ragged rows and keys
    (1, 2, 257, 257, 32, True),     # one row in the last tile
    (1, 1, 31, 1000, 32, False),    # fewer rows than a tile, more key tiles than waves
    (1, 2, 300, 70, 64, True),      # more rows than keys: the last tiles see every key
    (1, 1, 64, 17, 64, False),      # fewer key tiles than waves
]


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal", CASES)
def test_both_fp32_forms_match_the_oracle(form, B, H, Sq, Sk, D, causal):
    g = torch.Generator().manual_seed(1234 + Sq + Sk)
    q = torch.randn((B, Sq, H, D), generator=g)
    k = torch.randn((B, Sk, H, D), generator=g)
    v = torch.randn((B, Sk, H, D), generator=g)
    want_o, want_l = O.full_attention(q, k, v, None, causal)
    _lib.tune("fwd32_split", form)
    try:
        for scale in (None, -0.2):
            out, lse = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), scale, causal, layout="bshd")
            if scale is None:
                check_out(out.cpu(), want_o, torch.float32, f"form {form}")
                check_lse(lse.cpu(), want_l)
            else:
                wo, wl = O.full_attention(q, k, v, scale, causal)
                check_out(out.cpu(), wo, torch.float32, f"form {form} negative scale")
                check_lse(lse.cpu(), wl)
    finally:
        _lib.tune("fwd32_split", 0)


def test_strided_views_and_the_librarys_choice():
    """config 1 as the packed tensor's views (the public qkv-packed call), no knob: the result is the oracle's; the two
    forms agree to rounding."""
    B, S, H, D = 1, 512, 8, 64
    (qkv,) = rand_qkv((B, S, 3, H, D), 77, torch.float32, n=1)
    q, k, v = (qkv[:, :, i] for i in range(3))
    want_o, want_l = O.full_attention(q, k, v, None, True)
    qd = qkv.to(DEV)
    res = {}
    for form in (0, 1, 2):
        _lib.tune("fwd32_split", form)
        try:
            res[form] = ops.flash_fwd(qd[:, :, 0], qd[:, :, 1], qd[:, :, 2], None, True, layout="bshd")
        finally:
            _lib.tune("fwd32_split", 0)
        check_out(res[form][0].cpu(), want_o, torch.float32, f"form {form}")
        check_lse(res[form][1].cpu(), want_l)
    assert torch.equal(res[0][0], res[2][0]), "32 workgroups of 128 rows on this device: the library takes the 32-row form"
    assert (res[1][0] - res[2][0]).abs().max().item() < 1e-5


# One, two and four workgroups to 32 rows, by how many tiles of 32 rows there are for the CUs (256): 10 to 13, 96, 120 and 200.
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal", [(1, 3, 100, 333, 128, False), (1, 2, 161, 161, 128, True), (1, 24, 100, 333, 128, False),
                                                (1, 24, 129, 200, 128, True), (1, 40, 129, 333, 128, False), (2, 20, 129, 100, 128, True),
                                                (1, 24, 129, 333, 64, True), (1, 40, 130, 97, 64, False), (1, 2, 33, 31, 128, False)])
def test_workgroups_that_share_rows(B, H, Sq, Sk, D, causal):
    """Results of the forms whose workgroups take a part of the head dims each against the oracle, and, with an infinity in one value,
    infinite and NaN where those of 128-row workgroups are (rows in shards as well)."""
    g = torch.Generator().manual_seed(Sq * D + H)
    q, k, v = (torch.randn((B, s, H, D), generator=g) for s in (Sq, Sk, Sk))
    want_o, want_l = O.full_attention(q, k, v, None, causal)
    bad = v.clone()
    bad[0, Sk // 2, 1, D - 3] = float("inf")
    bad[0, 0, 0, 5] = float("nan")
    dev = [t.to(DEV) for t in (q, k, v, bad)]
    res = {}
    for form in (1, 2):
        _lib.tune("fwd32_split", form)
        try:
            out, lse = ops.flash_fwd(*dev[:3], None, causal, layout="bshd")
            res[form] = ops.flash_fwd(dev[0], dev[1], dev[3], None, causal, layout="bshd")[0]
        finally:
            _lib.tune("fwd32_split", 0)
        check_out(out.cpu(), want_o, torch.float32, f"form {form}")
        check_lse(lse.cpu(), want_l)
    assert torch.equal(res[1].isnan(), res[2].isnan()) and torch.equal(res[1].isinf(), res[2].isinf())
    finite = res[1].isfinite()
    assert finite.any() and not finite.all()
    # (fp32 sums of Sk weighted values of size 1 in another order)
    assert (res[1] - res[2])[finite].abs().max().item() < 1e-5


@pytest.mark.parametrize("B,H,D", [(1, 2, 128), (1, 12, 128), (1, 12, 64), (2, 12, 128)])
def test_workgroups_that_share_rows_of_shards(B, H, D):
    S, P = 4 * 66, 4
    q, k, v = rand_qkv((B, S, H, D), 5 + H, torch.float32)
    want_o, _ = O.full_attention(q, k, v, None, True)
    order = torch.as_tensor(sp.ring.zigzag_order(S, P))
    for sharding in ("contiguous", "zigzag"):
        if sharding == "zigzag":
            x, want = [t[:, order].to(DEV) for t in (q, k, v)], want_o[:, order]
        else:
            x, want = [t.to(DEV) for t in (q, k, v)], want_o
        _lib.tune("fwd32_split", 2)
        try:
            out = sp.sp_aurora_func(*x, causal=True, ring_size=P, sharding=sharding)
        finally:
            _lib.tune("fwd32_split", 0)
        check_out(out.cpu(), want, torch.float32, sharding)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D,Sk", [(128, 256), (128, 300), (64, 300)])
def test_workgroups_that_share_head_dims_sum_in_the_same_order(D, Sk, causal):
    """8, 16 and 32 heads of 256 rows leave four, two and one workgroup for the head dims of a row (at D = 64 two at most): the small terms of a tile's
    products come first in each, so the bits are the same however many there are."""
    q, k, v = (torch.randn((1, 32, s, D), generator=torch.Generator().manual_seed(160 + i)).to(DEV) for i, s in enumerate((256, Sk, Sk)))
    _lib.tune("fwd32_split", 2)
    try:
        whole, lse = ops.flash_fwd(q, k, v, None, causal, layout="bhsd")
        for heads in (8, 16):
            out, l = ops.flash_fwd(q[:, :heads], k[:, :heads], v[:, :heads], None, causal, layout="bhsd")
            assert torch.equal(out, whole[:, :heads]) and torch.equal(l, lse[:, :heads]), f"{heads} heads"
    finally:
        _lib.tune("fwd32_split", 0)


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,form", [(1, 5, 79, 386, 64, True, 2), (4, 16, 70, 390, 128, True, 2), (1, 16, 114, 69, 32, False, 2), (4, 8, 409, 3565, 128, False, 2),
                                                     (4, 8, 2964, 1299, 128, False, 1)])
def test_the_librarys_choice_by_size(B, H, Sq, Sk, D, causal, form):
    """Short calls, and those whose longest chain of tiles decides, run on the kernel of few rows, large ones on the other: the bits tell."""
    q, k, v = (torch.randn((B, s, H, D), generator=torch.Generator().manual_seed(180 + i)).to(DEV) for i, s in enumerate((Sq, Sk, Sk)))
    own, got = ops.flash_fwd(q, k, v, None, causal)[0], {}
    for knob in (1, 2):
        _lib.tune("fwd32_split", knob)
        try:
            got[knob] = ops.flash_fwd(q, k, v, None, causal)[0]
        finally:
            _lib.tune("fwd32_split", 0)
    assert torch.equal(own, got[form]) and not torch.equal(own, got[3 - form])
