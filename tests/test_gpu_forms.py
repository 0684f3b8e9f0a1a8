"""The forms of a forward workgroup, the tile numbering of packed batches and the softmax that forms a row maximum only when one
is needed: each at the sizes where it can go wrong, against the oracle (tolerances of test_gpu_parity) or, for long lists of
sequences, against the fixed-length call on each sequence."""
import pytest
import torch

from conftest import rand, rand_qkv
from oracle import attn_oracle as O
import sp_aurora_amd as spa
from sp_aurora_amd import _lib, ops
from test_gpu_parity import DEV, check_grad, check_lse, check_out

pytestmark = pytest.mark.gpu


@pytest.fixture
def tuned():
    """Sets kernel-variant overrides for one test."""
    used = []

    def tune(**knobs):
        for k, v in knobs.items():
            _lib.tune(k, v)
            used.append(k)
    yield tune
    for k in used:
        _lib.tune(k, 0)


FORMS = {"one group": dict(fwd_groups=1), "split": dict(fwd_groups=2, fwd_share=1), "shared": dict(fwd_groups=2, fwd_share=2)}


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16)])
@pytest.mark.parametrize("Sq,Sk,causal", [(1, 65, False), (63, 63, True), (128, 129, False), (129, 127, True), (257, 257, True), (300, 640, False)])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_every_form_of_a_workgroup(tuned, form, Sq, Sk, causal, D, dtype):
    q, = rand_qkv((2, 3, Sq, D), 800, dtype, n=1)
    k, v = rand_qkv((2, 3, Sk, D), 801, dtype, n=2)
    want, want_lse = O.attn_block(q, k, v, None, causal)
    tuned(**FORMS[form], few_rows=1)
    out, lse = spa._flash_attn_forward(q.to(DEV), k.to(DEV), v.to(DEV), causal=causal)
    check_out(out, want, dtype)
    check_lse(lse, want_lse)


@pytest.mark.parametrize("growth", [0.5, 6.0, -6.0])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_scores_that_outgrow_the_first_keys(tuned, form, causal, growth):
    """Scores that rise (or fall) along the keys by many powers of two, in some rows only: the reference maximum of the first
    tile overflows P there and has to be replaced, and must not be elsewhere."""
    B, H, S, D, dtype = 1, 2, 512, 64, torch.bfloat16
    q, k, v = rand_qkv((B, H, S, D), 810, dtype)
    ramp = torch.linspace(0.0, 1.0, S)[None, None, :, None] * growth
    u = rand((1, 1, 1, D), 811)
    u = u / u.norm()
    q = (q.float() + 16.0 * (torch.arange(S) % 3 == 0)[None, None, :, None] * u).to(dtype)  # every third row looks along u
    k = (k.float() + ramp * 16.0 * u).to(dtype)
    want, want_lse = O.attn_block(q, k, v, None, causal)
    tuned(**FORMS[form])
    out, lse = spa._flash_attn_forward(q.to(DEV), k.to(DEV), v.to(DEV), causal=causal)
    check_out(out, want, dtype)
    # the lse grows to a few hundred here: one part in 2^20 of it beside the usual bound
    err = (lse.cpu().double() - want_lse).abs()
    assert bool((err <= 1e-3 + want_lse.abs() * 2.0 ** -20).all()), err.max()


@pytest.mark.parametrize("dtype,D,causal", [(torch.bfloat16, 128, True), (torch.float16, 64, False), (torch.float32, 32, True)])
@pytest.mark.parametrize("lengths", [[1], [257], [0, 5, 0, 128, 129], [127, 128, 129, 255, 256, 257, 3, 0], list(range(64)), list(range(65)),
                                     [7, 130, 0, 64] * 33])
def test_tiles_of_a_packed_batch(lengths, dtype, D, causal):
    """Every row of every sequence is computed once: 1 to 132 sequences, empty ones among them, lengths around the tile sizes."""
    H = 3
    T = sum(lengths)
    cu = torch.tensor([0] + torch.tensor(lengths).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
    q, k, v, dout = (t.to(DEV) for t in rand_qkv((T, H, D), 820 + len(lengths), dtype, n=4))
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    out, lse, _ = spa.sp_aurora_varlen_func(*leaves, cu, max_seqlen=max(lengths), causal=causal, return_attn_probs=True)
    grads = torch.autograd.grad(out, leaves, dout)
    tol = {torch.bfloat16: 2e-2, torch.float16: 4e-3, torch.float32: 1e-5}[dtype]
    at = 0
    for n in lengths:
        if n:
            rows = slice(at, at + n)
            one = [t[rows].unsqueeze(0).clone().requires_grad_() for t in (q, k, v)]
            want, want_lse, _ = spa.sp_aurora_func(*one, causal=causal, return_attn_probs=True)
            want_grads = torch.autograd.grad(want, one, dout[rows].unsqueeze(0))
            # the same arithmetic per row in another workgroup form: roundings of P and of the results apart
            torch.testing.assert_close(out[rows], want[0], atol=tol, rtol=tol)
            torch.testing.assert_close(lse[:, rows], want_lse[0], atol=1e-4, rtol=1e-5)
            for g, w in zip(grads, want_grads):
                torch.testing.assert_close(g[rows], w[0], atol=2 * tol, rtol=2 * tol)
        at += n
