"""The fp32 forward on three bf16 terms per value: both forms, every head dim, at the edges of their tiles (one key tile, two, a last
one that is whole, workgroups whose later waves have no rows), against float64."""
import pytest
import torch

from sp_aurora_amd import _lib, ops
from test_gpu_parity import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Sq,Sk,causal", [(1, 1, False), (32, 32, True), (64, 64, False), (96, 128, False), (128, 128, True), (129, 160, False),
                                          (33, 257, False), (300, 300, True), (200, 40, True)])
def test_fp32_against_float64(form, D, Sq, Sk, causal):
    g = torch.Generator().manual_seed(D + Sq + 7 * Sk)
    H = 3
    # values over six powers of ten: every term of a split value counts somewhere
    q, k, v = (torch.randn((1, S, H, D), generator=g) * 10 ** (torch.rand((1, S, H, D), generator=g) * 6 - 5) for S in (Sq, Sk, Sk))
    qh, kh, vh = (t.double().transpose(1, 2) for t in (q, k, v))
    s, mass = qh @ kh.transpose(-1, -2) * D ** -0.5, qh.abs() @ kh.abs().transpose(-1, -2) * D ** -0.5
    if causal:
        hidden = torch.ones(Sq, Sk, dtype=torch.bool).triu(1)
        s, mass = s.masked_fill(hidden, -float("inf")), mass.masked_fill(hidden, 0.0)
    p = torch.softmax(s, -1)
    want, lse = (p @ vh).transpose(1, 2), torch.logsumexp(s, -1)
    # A score is off by at most 2^-23 of the sum of its products' sizes for the terms left out, and D / 16 + 6 roundings of 2^-24 for
    # the sums, the exponent's argument and the exponential itself by 2^-22 more: a weight is off by that much of itself, an output
    # by twice that and the roundings of its own sum, times what the weights and |v| add up to.
    ds = mass * (2 + D / 16 + 6) * 2.0 ** -24 + (1 + s.abs().masked_fill(s.isinf(), 0.0)) * 2.0 ** -22
    worst = ds.amax(-1)
    bound = (2 * worst + (Sk / 16 + 8) * 2.0 ** -24)[..., None] * (p @ vh.abs())
    _lib.tune("fwd32_split", form)
    try:
        out, got_lse = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), None, causal, layout="bshd")
    finally:
        _lib.tune("fwd32_split", 0)
    err = (out.cpu().double() - want).abs().transpose(1, 2)
    assert (err <= bound + 1e-30).all(), float((err / bound).max())
    assert ((got_lse.cpu().double() - lse).abs() <= 2 * worst + 2.0 ** -22 * (1 + lse.abs())).all()


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("D,S,causal", [(32, 70, True), (64, 129, False), (128, 97, True)])
def test_fp32_values_that_have_no_three_terms(form, D, S, causal):
    """Infinities, a NaN and values above the largest bf16 number: they reach the results that they reach in plain arithmetic."""
    g = torch.Generator().manual_seed(S)
    H = 2
    q, k, v = (torch.randn((1, S, H, D), generator=g) for _ in range(3))
    v[0, 5, 0, 3], v[0, 20, 0, 9], v[0, 40, 1, 7] = float("inf"), -float("inf"), 3.4e38
    k[0, S - 2, 1, 1] = float("nan")
    s = (q.double().transpose(1, 2) @ k.double().transpose(1, 2).transpose(-1, -2)) * D ** -0.5
    seen = torch.ones(S, S, dtype=torch.bool).tril() if causal else torch.ones(S, S, dtype=torch.bool)
    p = torch.softmax(s.masked_fill(~seen, -float("inf")), -1)
    terms = p[..., None] * v.double().transpose(1, 2)[:, :, None]
    want = torch.where(seen[None, None, :, :, None], terms, torch.zeros(())).sum(3).transpose(1, 2)
    _lib.tune("fwd32_split", form)
    try:
        out, lse = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), None, causal, layout="bshd")
    finally:
        _lib.tune("fwd32_split", 0)
    # plain sums of at most 130 terms: a score is off by D and a weight by 2^-22 |score| roundings, the sum by one rounding a key
    torch.testing.assert_close(out.cpu().double(), want, rtol=1e-4, atol=1e-5, equal_nan=True)
    want_lse = torch.logsumexp(s.masked_fill(~seen, -float("inf")), -1)
    torch.testing.assert_close(lse.cpu().double(), want_lse, rtol=1e-5, atol=1e-5, equal_nan=True)


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("q_size,k_size,v_size,scale", [(1.0, 1.0, 1e-33, 0.1), (1.0, 1.0, 1e-36, 0.1), (1.0, 1.0, 1e-38, 0.1), (1e-36, 1e30, 1.0, 1e5),
                                                        (1e30, 1e-37, 1.0, 1e6), (1e-38, 1e-5, 1.0, 1e38), (1e15, 1e14, 1.0, 1e-30), (1e14, 1e13, 1e-37, 1e-28)])
def test_fp32_small_and_large_values(form, D, q_size, k_size, v_size, scale):
    """Values at which a term of a split value would leave the bf16 range: the results are as exact as those of values around one."""
    g = torch.Generator().manual_seed(D)
    S, H = 130, 2
    q, k, v = (torch.randn((1, S, H, D), generator=g) * x for x in (q_size, k_size, v_size))
    qh, kh, vh = (t.double().transpose(1, 2) for t in (q, k, v))
    s, mass = qh @ kh.transpose(-1, -2) * scale, qh.abs() @ kh.abs().transpose(-1, -2) * scale
    p = torch.softmax(s, -1)
    _lib.tune("fwd32_split", form)
    try:
        out, lse = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), scale, False, layout="bshd")
    finally:
        _lib.tune("fwd32_split", 0)
    # the bound of test_fp32_against_float64, and the smallest fp32 number, 2^-149, once for a result and once for its sum
    ds = mass * (2 + D / 16 + 6) * 2.0 ** -24 + (1 + s.abs()) * 2.0 ** -22
    bound = (2 * ds.amax(-1) + (S / 16 + 8) * 2.0 ** -24)[..., None] * (p @ vh.abs()) + 2.0 ** -148
    err = (out.cpu().double() - (p @ vh).transpose(1, 2)).abs().transpose(1, 2)
    assert (err <= bound).all(), float((err / bound).max())
    assert ((lse.cpu().double() - torch.logsumexp(s, -1)).abs() <= 2 * ds.amax(-1) + 2.0 ** -22 * (1 + s.abs().amax(-1))).all()


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("size", [1e16, 1e20, 1e25, 1e31, 3e36])
def test_fp32_large_values_under_weights_above_one(form, D, size):
    """Scores that rise along the keys by less than what moves the reference maximum: sums of 2^8 times the values, means that are finite."""
    g = torch.Generator().manual_seed(D)
    S, H = 300, 2
    q, k = torch.zeros(1, S, H, D), torch.zeros(1, S, H, D)
    q[..., 0], k[..., 0] = 1.0, torch.linspace(0.0, 5.4, S)[None, :, None]  # (times log2 e: 7.8)
    # (the weights below 1 add up to 300 / 5.4 = 56, times a mean value of 1.5 * 3e36: 2.5e38, less than the largest fp32 number)
    v = (1 + torch.rand((1, S, H, D), generator=g)) * size
    p = torch.softmax(q.double().transpose(1, 2) @ k.double().transpose(1, 2).transpose(-1, -2), -1)
    _lib.tune("fwd32_split", form)
    try:
        out, lse = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), 1.0, False, layout="bshd")
    finally:
        _lib.tune("fwd32_split", 0)
    # exponents are off by 2^-23 of at most 8, weights by 2^-22 more, sums by a rounding a key at most (all of one sign)
    torch.testing.assert_close(out.cpu().double(), (p @ v.double().transpose(1, 2)).transpose(1, 2), rtol=(S + 32) * 2.0 ** -24, atol=0.0)


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_score_of_one_product_is_rounded_once(form, D):
    """q with one value per row against one key: the score is that product, as plain fp32 rounds it."""
    g = torch.Generator().manual_seed(D)
    S, at = 4096, D - 3
    q, k, v = torch.zeros(1, S, 2, D), torch.randn((1, 1, 2, D), generator=g), torch.randn((1, 1, 2, D), generator=g)
    q[..., at] = torch.randn((1, S, 2), generator=g)
    _lib.tune("fwd32_split", form)
    try:
        # (a scale of ln 2: scores in units of log 2, whose factor is 1; one key: lse = score * ln 2)
        lse = ops.flash_fwd(q.to(DEV), k.to(DEV), v.to(DEV), 0.6931471805599453, False, layout="bshd")[1].cpu()
    finally:
        _lib.tune("fwd32_split", 0)
    want = ((q[..., at] * k[..., at]) * 0.6931471805599453).transpose(1, 2)
    # The terms left out, 2 * 2^-8 * 2^-17 of the product at most and 2^-27 as a rule, move the rounding of a few per cent of the products (simulated:
    # 4 %); a second rounding would move 21 %.
    assert (lse != want).float().mean() < 0.1
    assert ((lse - want).abs() <= 2.0 ** -22 * want.abs()).all()


@pytest.mark.parametrize("D,S,H", [(128, 1024, 32), (64, 1024, 16), (64, 512, 8), (32, 1000, 4)])
@pytest.mark.parametrize("of,value", [("q", float("nan")), ("k", float("nan")), ("v", float("nan")), ("v", float("inf")), ("v", 3.4e38)])
def test_fp32_rows_that_are_computed_again_cost_a_few_calls(D, S, H, of, value):
    """A value that reaches every row: as many results again as the call has, at a few times its time (by one row after another: 80 to 250 times)."""
    g = torch.Generator().manual_seed(D)
    t = {n: torch.randn((1, S, H, D), generator=g) for n in "qkv"}
    dev = {n: x.to(DEV) for n, x in t.items()}
    bad = dev[of].clone()
    bad[:, 3 if of != "q" else slice(None), :, 5] = value
    seen = 3 if of != "q" else 0

    def us(args):
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            out, lse = ops.flash_fwd(*args, None, True, layout="bshd")
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3)
        return best, out, lse
    base, want, want_lse = us([dev[n] for n in "qkv"])
    again, out, lse = us([bad if n == of else dev[n] for n in "qkv"])
    assert again < 10 * base + 100, (base, again)
    torch.testing.assert_close(out[:, :seen], want[:, :seen], rtol=1e-5, atol=1e-5)
    if of == "v":
        # the other columns are those of the finite value, to two of the bounds of test_fp32_against_float64 (a generous 1e-5 at values around 1)
        keep = [d for d in range(D) if d != 5]
        torch.testing.assert_close(out[..., keep], want[..., keep], rtol=1e-5, atol=1e-5)
        torch.testing.assert_close(lse, want_lse, rtol=1e-5, atol=1e-5)
        assert (out[:, 3:, :, 5].isnan() if value != value else out[:, 3:, :, 5] > 1e30).all()
    else:
        assert out[:, seen:].isnan().all() and lse[:, :, seen:].isnan().all()
