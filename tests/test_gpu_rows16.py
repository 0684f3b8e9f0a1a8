"""Calls of up to 16 query rows without a mask, for the kernel that streams K and V through matrix instructions (rows of a head back to back, layout
[B, H, S, D], two rows and more or e4m3 K and V; more than three rows also with other heads in between) and those beside it: edges of its tiles of
32 keys and of a workgroup's pass, chunks, both element types and e4m3, the values a weight of several terms has to get right."""
import math

import pytest
import torch

from conftest import rand
from oracle import attn_oracle as O
from sp_aurora_amd import _lib, ops
from test_gpu_fp8kv import quantised
from test_gpu_parity import DEV, check_lse, check_out

pytestmark = pytest.mark.gpu


def both(q, k, v, scale=None, layout="bhsd", **kw):
    """The call on this kernel and on the others (spa_tune few_rows = 1)."""
    res = []
    for knob in (0, 1):
        _lib.tune("few_rows", knob)
        try:
            res.append(ops.flash_fwd(q, k, v, scale, False, layout=layout, **kw))
        finally:
            _lib.tune("few_rows", 0)
    return res


@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("Sq,Sk,nsplit", [(1, 1, 1), (3, 31, 1), (4, 32, 1), (16, 33, 1), (2, 255, 2), (9, 256, 1), (1, 257, 1), (16, 257, 2), (5, 1300, 4), (15, 777, 6),
                                          (3, 2049, 5)])
def test_edges_against_the_oracle(layout, D, dtype, Sq, Sk, nsplit):
    B, H = 2, 3
    q, k, v = (rand((B, s, H, D), 40 + Sk + i, dtype) for i, s in enumerate((Sq, Sk, Sk)))
    place = (lambda t: t.transpose(1, 2).contiguous().to(DEV)) if layout == "bhsd" else (lambda t: t.to(DEV))
    for scale in (None, -0.4):
        want_o, want_l = O.full_attention(q, k, v, scale, False)
        out, lse = ops.flash_fwd(place(q), place(k), place(v), scale, False, layout=layout, split_kv=nsplit)
        check_out(out.transpose(1, 2) if layout == "bhsd" else out, want_o, dtype, f"scale {scale}")
        check_lse(lse, want_l)
    k8, ks, k_deq = quantised((B, Sk, H, D), 50 + Sk, "bshd", spread=1.3)
    v8, vs, v_deq = quantised((B, Sk, H, D), 51 + Sk, "bshd")
    ks, vs = ks.to(DEV).clone(), vs.to(DEV)
    ks[0, 1] = 0.0  # every key counts alike
    k_deq = k_deq.clone()
    k_deq[0, :, 1] = 0.0
    want_o, want_l = O.full_attention(q, k_deq, v_deq, None, False)
    out, lse = ops.flash_fwd(place(q), place(k8), place(v8), None, False, layout=layout, k_scale=ks, v_scale=vs, split_kv=nsplit)
    check_out(out.transpose(1, 2) if layout == "bhsd" else out, want_o, dtype, "e4m3")
    check_lse(lse, want_l)


@pytest.mark.parametrize("e4m3", [False, True])
@pytest.mark.parametrize("Sq", [1, 2, 8])
def test_more_keys_than_the_memory_side_cache_holds(e4m3, Sq):
    """Above 64 MiB of K and V the loads carry the non-temporal hint (16-bit: four waves): the same results as for the heads' halves, which are below."""
    B, H, Sk, D = 2, 32, 6200 if e4m3 else 3100, 128
    q, k, v = (rand((B, H, s, D), 60 + i, torch.bfloat16).to(DEV) for i, s in enumerate((Sq, Sk, Sk)))
    kw = [{}, {}, {}]
    if e4m3:
        (k, ks), (v, vs) = (ops.quantize_fp8_per_head(t, layout="bhsd") for t in (k, v))
        kw = [dict(k_scale=a, v_scale=b) for a, b in ((ks, vs), (ks[:1], vs[:1]), (ks[1:], vs[1:]))]
    assert k.numel() * k.element_size() * 2 > 64 << 20 >= k.numel() * k.element_size()
    out, lse = ops.flash_fwd(q, k, v, None, False, layout="bhsd", split_kv=2, **kw[0])
    for i in range(2):
        o, l = ops.flash_fwd(q[i:i + 1], k[i:i + 1], v[i:i + 1], None, False, layout="bhsd", split_kv=2, **kw[1 + i])
        # sums over another number of waves, results (of chunks as well) rounded to bf16
        assert (o.float() - out[i:i + 1].float()).abs().max().item() <= 2.0 ** -6 * out.float().abs().max().item()
        assert (l - lse[i:i + 1]).abs().max().item() < 1e-5


@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (64, torch.float16), (128, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("e4m3,Sq", [(False, 2), (False, 8), (True, 1), (True, 3), (True, 16)])
def test_large_caches_of_each_type(e4m3, Sq, D, dtype, layout):
    """Above 64 MiB of K and V, in one piece and in two: every variant of the loads, and the kernels that take what this one leaves (16-bit rows of other heads in
    between), against one another and, for two heads, against float64."""
    B, H, Sk = 2, 32, (7000 if e4m3 else 3500) * 128 // D
    q, k, v = (rand((B, H, s, D), 62 + i, dtype).to(DEV) for i, s in enumerate((Sq, Sk, Sk)))
    kw, scales = {}, (None, None)
    if e4m3:
        (k, ks), (v, vs) = (ops.quantize_fp8_per_head(t, layout="bhsd") for t in (k, v))
        kw, scales = dict(k_scale=ks, v_scale=vs), (ks, vs)
    assert k.numel() * k.element_size() * 2 > 64 << 20
    place = (lambda t: t) if layout == "bhsd" else (lambda t: t.transpose(1, 2).contiguous())
    whole, cut = (ops.flash_fwd(place(q), place(k), place(v), None, False, layout=layout, split_kv=n, **kw) for n in (1, 2))
    if layout == "bshd":
        whole, cut = ((o.transpose(1, 2), l) for o, l in (whole, cut))
    for b, h in ((0, 0), (1, 31)):
        one = [q[b, h].double().cpu()] + [t[b, h].double().cpu() * (sc[b, h].double().cpu() if e4m3 else 1) for t, sc in zip((k, v), scales)]
        want_o, want_l = O.full_attention(*(t[None, :, None] for t in one), None, False)
        for o, l in (whole, cut):
            check_out(o[b, h][None, :, None], want_o, dtype)
            check_lse(l[b, h][None, None], want_l)
    # (results of chunks and of the call rounded to the type)
    assert (whole[0].float() - cut[0].float()).abs().max().item() <= 2.0 ** -6 * whole[0].float().abs().max().item()
    assert (whole[1] - cut[1]).abs().max().item() < 1e-5


@pytest.mark.parametrize("B,H", [(1, 8), (2, 8), (1, 16)])
@pytest.mark.parametrize("Sq,Sk,nsplit", [(1, 300, 1), (3, 700, 3), (8, 1300, 1), (16, 1300, 4)])
def test_neighbouring_e4m3_heads_that_share_lines(B, H, Sq, Sk, nsplit):
    """64 e4m3 elements are half a line: with a multiple of 8 heads, workgroups are renumbered so that neighbours run on one XCD.  Every head has its own scales."""
    D = 64
    q = rand((B, Sq, H, D), 64, torch.bfloat16)
    k8, ks, k = quantised((B, Sk, H, D), 65, "bshd")
    v8, vs, v = quantised((B, Sk, H, D), 66, "bshd")
    grow = torch.linspace(0.25, 2.0, B * H).reshape(B, H)
    ks, vs = ks.cpu() * grow, vs.cpu() * grow.flip(1)
    k, v = (t.cpu() * g[:, None, :, None] for t, g in ((k, grow.double()), (v, grow.flip(1).double())))
    want_o, want_l = O.full_attention(q, k, v, None, False)
    place = lambda t: t.transpose(1, 2).contiguous().to(DEV)
    out, lse = ops.flash_fwd(place(q), place(k8), place(v8), None, False, layout="bhsd", k_scale=ks.to(DEV), v_scale=vs.to(DEV), split_kv=nsplit)
    check_out(out.transpose(1, 2), want_o, torch.bfloat16)
    check_lse(lse, want_l)


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("Sq", [1, 3, 8])
def test_infinities_and_nan(Sq, D, dtype):
    """An infinity or a NaN in V reaches the dims that hold it and no others; a NaN in K reaches every row."""
    B, H, Sk = 1, 2, 300
    q, k, v = (rand((B, H, s, D), 70 + i, dtype) for i, s in enumerate((Sq, Sk, Sk)))
    v[0, 0, 7, 3] = float("inf")
    v[0, 0, 200, 5] = -float("inf")
    v[0, 1, 33, D - 1] = float("nan")
    out = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), None, False, layout="bhsd")[0].float().cpu()
    assert (out[0, 0, :, 3] == float("inf")).all() and (out[0, 0, :, 5] == -float("inf")).all() and out[0, 1, :, D - 1].isnan().all()
    clean = torch.ones_like(out, dtype=torch.bool)
    clean[0, 0, :, 3] = clean[0, 0, :, 5] = clean[0, 1, :, D - 1] = False
    assert out[clean].isfinite().all()
    k[0, 0, 10, 0] = float("nan")
    out = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), None, False, layout="bhsd")[0]
    assert out[0, 0].isnan().all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Sq", [1, 3])
def test_many_small_weights_beside_a_large_one(Sq, dtype):
    """One key of weight 1 and value 0, thousands of weight 2^-23.1 and value 2^12: the result, about 3.8, is the sum of what the element type alone
    would round away in fp16 (2^-24 is its smallest step)."""
    D, Sk = 64, 8192
    q = torch.zeros((1, 1, Sq, D), dtype=dtype)
    k = torch.zeros((1, 1, Sk, D), dtype=dtype)
    v = torch.full((1, 1, Sk, D), 4096.0, dtype=dtype)
    q[..., 0] = 4.0
    k[:, :, 1:, 0] = -4.0
    v[:, :, 0] = 0.0
    want, want_l = O.full_attention(*(t.transpose(1, 2) for t in (q, k, v)), 1.0, False)
    out, lse = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), 1.0, False, layout="bhsd", split_kv=None)
    # rounded once to the element type, weights off by 2^-22 at most
    assert (out.cpu().double() / want.transpose(1, 2) - 1).abs().max().item() < (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -10)
    check_lse(lse, want_l)


@pytest.mark.parametrize("e4m3", [False, True])
@pytest.mark.parametrize("Sq", [1, 2, 3])
def test_weights_far_below_the_largest(Sq, e4m3):
    """fp16: one key of weight 1 and value 0, 1023 of weight e^-30 = 2^-43.3 and value 57344: 5.5e-6 of a result whose steps are 2^-24 = 6e-8, half a step
    of error, and of weights in steps of 2^-50 half of 1023 * 57344 * 2^-50 at most."""
    D, Sk = 64, 1024
    q, k = torch.zeros((1, 1, Sq, D)), torch.zeros((1, 1, Sk, D))
    q[..., 0], k[:, :, 1:, 0] = 7.5, -4.0
    v = torch.full((1, 1, Sk, D), 448.0 if e4m3 else 57344.0)
    v[:, :, 0] = 0.0
    kw = {}
    if e4m3:
        kw = dict(k_scale=torch.ones((1, 1), device=DEV), v_scale=torch.full((1, 1), 128.0, device=DEV))
    place = lambda t: (t.to(torch.float8_e4m3fn) if e4m3 else t.half()).to(DEV)
    out, _ = ops.flash_fwd(q.half().to(DEV), place(k), place(v), 1.0, False, layout="bhsd", split_kv=None, **kw)
    want = 1023 * math.exp(-30.0) * 57344
    assert (out.double() - want).abs().max().item() <= 2.0 ** -25 + 0.5 * 1023 * 57344 * 2.0 ** -50


@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Sq", [1, 2, 3])
@pytest.mark.parametrize("nats", [10, 20, 40, 80])
def test_an_infinity_under_a_small_weight(nats, Sq, dtype, layout):
    """Up to three rows: a weight that fp32 holds (e^-80 = 2^-115) makes an infinity of V one in the result, however small it is; one of a score of
    -infinity is 0, and 0 times infinity no number."""
    D, Sk, H = 64, 700, 2
    q, k, v = torch.zeros((1, Sq, H, D)), torch.zeros((1, Sk, H, D)), rand((1, Sk, H, D), 75, torch.float32)
    q[..., 0], k[:, 333, :, 0] = 8.0, -nats / 8.0
    v[:, 333, 0, 3], v[:, 333, 1, 5] = float("inf"), -float("inf")
    place = (lambda t: t.to(dtype).transpose(1, 2).contiguous().to(DEV)) if layout == "bhsd" else (lambda t: t.to(dtype).to(DEV))
    run = lambda: ops.flash_fwd(place(q), place(k), place(v), 1.0, False, layout=layout, split_kv=None)[0].float().cpu()
    out = run() if layout == "bshd" else run().transpose(1, 2)
    assert (out[:, :, 0, 3] == float("inf")).all() and (out[:, :, 1, 5] == -float("inf")).all()
    out[:, :, 0, 3] = out[:, :, 1, 5] = 0.0
    assert out.isfinite().all()
    k[:, 333, :, 0] = -float("inf")
    out = run() if layout == "bshd" else run().transpose(1, 2)
    assert out[:, :, 0, 3].isnan().all() and out[:, :, 1, 5].isnan().all() and out[:, :, 0, 4].isfinite().all()


@pytest.mark.parametrize("Sq", [1, 3, 4, 16])
def test_large_values_do_not_overflow(Sq):
    """bf16 values near the largest number under weights that grow along the keys: finite, as on the other kernels."""
    B, H, Sk, D = 1, 2, 400, 128
    q = torch.ones((B, H, Sq, D), dtype=torch.bfloat16)
    k = (torch.arange(Sk).float()[None, None, :, None] * (0.05 if Sq <= 3 else 1.0) / D).expand(B, H, Sk, D).to(torch.bfloat16).contiguous()
    v = torch.full((B, H, Sk, D), 1e36, dtype=torch.bfloat16)
    (out, lse), (out2, lse2) = both(q.to(DEV), k.to(DEV), v.to(DEV), 1.0)
    assert out.isfinite().all() and (out / 1e36 - 1).abs().max().item() < 2.0 ** -6
    assert (lse - lse2).abs().max().item() < 1e-4
