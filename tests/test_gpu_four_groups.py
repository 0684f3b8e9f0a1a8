"""The 16-bit forward's form of 64 query rows by four wave groups (taken where a launch leaves CUs idle; forced here by spa_tune fwd_groups = 4): edges of
its row tiles, of a step's 128 (D = 128) or 256 keys and of a group's share of them, rows staged through LDS and not, rows in shards, e4m3."""
import pytest
import torch

from conftest import rand
from oracle import attn_oracle as O
import sp_aurora_amd as spa
from sp_aurora_amd import _lib, ops
from test_gpu_fp8kv import quantised
from test_gpu_parity import DEV, check_lse, check_out

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (63, 64), (64, 65), (65, 33), (100, 257), (128, 128), (129, 129), (200, 511), (257, 300), (320, 513)]


@pytest.fixture
def four():
    _lib.tune("fwd_groups", 4)
    yield
    _lib.tune("fwd_groups", 0)


@pytest.mark.parametrize("layout", ["bhsd", "bshd"])  # (whole rows of q in a line: straight into the operands; the others through LDS)
@pytest.mark.parametrize("D,dtype", [(32, torch.bfloat16), (64, torch.bfloat16), (64, torch.float16), (128, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("Sq,Sk", SIZES)
def test_edges_against_the_oracle(four, layout, D, dtype, Sq, Sk):
    B, H = 2, 3
    q, k, v = (rand((B, s, H, D), 70 + Sk + i, dtype) for i, s in enumerate((Sq, Sk, Sk)))
    place = (lambda t: t.transpose(1, 2).contiguous().to(DEV)) if layout == "bhsd" else (lambda t: t.to(DEV))
    back = (lambda t: t.transpose(1, 2)) if layout == "bhsd" else (lambda t: t)
    for causal in (False, True):
        for scale in (None, -0.3):
            want_o, want_l = O.full_attention(q, k, v, scale, causal)
            out, lse = ops.flash_fwd(place(q), place(k), place(v), scale, causal, layout=layout, split_kv=1)
            check_out(back(out), want_o, dtype, f"causal {causal} scale {scale}")
            check_lse(lse, want_l)


@pytest.mark.parametrize("q8", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Sk", SIZES[1:])
def test_e4m3(four, D, q8, Sq, Sk):
    if q8 and D == 64:
        pytest.skip("8-bit scores: head dim 128")
    B, H, dtype = 1, 3, torch.bfloat16
    k8, ks, k = quantised((B, Sk, H, D), 90 + Sk, "bshd")
    v8, vs, v = quantised((B, Sk, H, D), 91 + Sk, "bshd")
    kw = {"k_scale": ks.to(DEV), "v_scale": vs.to(DEV)}
    if q8:
        q, qs, q_deq = quantised((B, Sq, H, D), 92 + Sk, "bshd")
        kw["q_scale"] = qs.to(DEV)
    else:
        q = q_deq = rand((B, Sq, H, D), 92 + Sk, dtype)
    for causal in (False, True):
        want_o, want_l = O.full_attention(q_deq, k, v, None, causal)
        out, lse = ops.flash_fwd(q.to(DEV), k8.to(DEV), v8.to(DEV), None, causal, split_kv=1, **kw)
        check_out(out, want_o, dtype, f"causal {causal}")
        check_lse(lse, want_l)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("P,half", [(2, 64), (4, 20), (3, 50)])  # (shards' halves of a sub-tile's rows and more, and of fewer)
def test_rows_in_shards(four, D, P, half):
    dtype, shape = torch.bfloat16, (1, 2 * P * half, 3, D)
    q, k, v = (rand(shape, 110 + i, dtype) for i in range(3))
    idx = O.zigzag_order(shape[1], P)
    want_o, want_l = O.full_attention(q, k, v, None, True)
    out, lse, _ = spa.sp_aurora_func(*(t[:, idx].contiguous().to(DEV) for t in (q, k, v)), causal=True, ring_size=P, sharding="zigzag", return_attn_probs=True)
    got_o, got_l = torch.empty_like(out.cpu()), torch.empty_like(lse.cpu())
    got_o[:, idx], got_l[:, :, idx] = out.cpu(), lse.cpu()
    check_out(got_o, want_o, dtype)
    check_lse(got_l, want_l)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bad", [65, 130, 200])
def test_an_infinite_value_stays_behind_its_tile(four, D, bad):
    """Causal: the rows of earlier tiles of 64 do not meet it, also where a step on the diagonal reaches further."""
    q, k, v = (rand((1, 256, 2, D), 130 + i, torch.bfloat16) for i in range(3))
    want_o, want_l = O.full_attention(q, k, v, None, True)
    v[0, bad] = float("inf")
    out, lse = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), None, True)
    before = bad // 64 * 64
    check_out(out[:, :before], want_o[:, :before], torch.bfloat16)
    check_lse(lse, want_l)
    assert not torch.isfinite(out[:, bad]).any()


@pytest.mark.parametrize("D,e4m3", [(32, False), (64, False), (64, True), (128, False)])
@pytest.mark.parametrize("Sk", [65, 100, 127])
def test_rows_far_apart(four, Sk, D, e4m3):
    """Rows 17 MB apart, all that lies between them infinite: a step of 256 keys would reach rows whose 32-bit offsets come round to the tensor again."""
    Sq, pitch = 70, 17 << 20
    if (Sk - 1) * pitch >= 2 ** 31:
        pitch = (2 ** 31 // (Sk - 1) - 1) // 256 * 256
    q, k, v = (rand((1, s, 1, D), 150 + i, torch.bfloat16) for i, s in enumerate((Sq, Sk, Sk)))
    kw, dtype, gap = {}, torch.bfloat16, float("inf")
    k_in, v_in, k_deq, v_deq = k, v, k, v
    if e4m3:
        (k_in, ks, k_deq), (v_in, vs, v_deq) = quantised((1, Sk, 1, D), 151, "bshd"), quantised((1, Sk, 1, D), 152, "bshd")
        kw, dtype, gap = dict(k_scale=ks.to(DEV), v_scale=vs.to(DEV)), torch.float8_e4m3fn, float("nan")

    def far(t):
        step = pitch // t.element_size()
        wide = torch.full(((Sk - 1) * step + D,), gap, device=DEV, dtype=torch.bfloat16).to(dtype)
        wide = wide.as_strided((1, Sk, 1, D), (0, step, D, 1))
        wide.copy_(t)
        return wide
    want_o, want_l = O.full_attention(q, k_deq, v_deq, None, False)
    out, lse = ops.flash_fwd(q.to(DEV), far(k_in), far(v_in), None, False, split_kv=1, **kw)
    check_out(out, want_o, torch.bfloat16)
    check_lse(lse, want_l)


@pytest.mark.parametrize("H,S", [(8, 700), (5, 1300)])
def test_the_form_is_taken_for_small_launches(H, S):
    """Bits tell the forms apart: the library's choice is this one."""
    q, k, v = (rand((1, S, H, 128), 140 + i, torch.bfloat16).to(DEV) for i in range(3))
    own = ops.flash_fwd(q, k, v, None, True)
    got = {}
    for groups in (2, 4):
        _lib.tune("fwd_groups", groups)
        try:
            got[groups] = ops.flash_fwd(q, k, v, None, True)
        finally:
            _lib.tune("fwd_groups", 0)
    assert torch.equal(own[0], got[4][0]) and not torch.equal(own[0], got[2][0])


@pytest.mark.parametrize("B,H,Sq,Sk,D", [(1, 100, 128, 2048, 128), (2, 128, 164, 8645, 32), (16, 8, 379, 22380, 64)])
def test_the_form_is_left_out_where_its_reads_decide(B, H, Sq, Sk, D):
    """Launches that fit its work but read K and V once a tile: the bits are another form's."""
    g = torch.Generator(device=DEV).manual_seed(170)
    q, k, v = (torch.randn((B, s, H, D), generator=g, device=DEV).bfloat16() for s in (Sq, Sk, Sk))
    own = ops.flash_fwd(q, k, v, None, False, split_kv=1)[0]
    _lib.tune("fwd_groups", 4)
    try:
        four = ops.flash_fwd(q, k, v, None, False, split_kv=1)[0]
    finally:
        _lib.tune("fwd_groups", 0)
    assert not torch.equal(own, four)
    # (weights rounded beside another reference maximum, sums in another order, rounded to bf16)
    assert (own.float() - four.float()).norm().item() <= 2.0 ** -7 * own.float().norm().item()
