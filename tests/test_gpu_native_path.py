"""The host path of the public calls (_native): every way of packing the operands, rings as one block call, what it hands on to
the Python path.  Against the oracle's full attention, tolerances of test_gpu_parity."""
import pytest
import torch

from conftest import rand_qkv
from oracle import attn_oracle as O
import sp_aurora_amd as spa
from sp_aurora_amd import _lib, ops
from test_gpu_parity import DEV, check_grad, check_lse, check_out

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ring,S,D,dtype,causal", [(1, 67, 64, torch.float16, True), (3, 99, 128, torch.bfloat16, True),
                                                   (4, 148, 64, torch.bfloat16, False), (2, 130, 32, torch.float32, True)])
@pytest.mark.parametrize("packing", ["q,k,v", "q,kv", "qkv"])
def test_every_packing_of_the_operands(packing, ring, S, D, dtype, causal):
    B, H = 2, 3
    q, k, v, dout = rand_qkv((B, S, H, D), 700 + S, dtype, n=4)
    want, want_lse = O.full_attention(q, k, v, None, causal)
    want_grads = O.attn_backward_autograd(q, k, v, dout, None, causal)
    if packing == "q,k,v":
        leaves = [t.to(DEV).requires_grad_() for t in (q, k, v)]
        fn, split = spa.sp_aurora_func, lambda g: g
    elif packing == "q,kv":
        leaves = [q.to(DEV).requires_grad_(), torch.stack([k, v], 2).to(DEV).requires_grad_()]
        fn, split = spa.sp_aurora_kvpacked_func, lambda g: (g[0], g[1][:, :, 0], g[1][:, :, 1])
    else:
        leaves = [torch.stack([q, k, v], 2).to(DEV).requires_grad_()]
        fn, split = spa.sp_aurora_qkvpacked_func, lambda g: tuple(g[0][:, :, i] for i in range(3))
    assert _lib.native().attention(*leaves, None, causal, 0) is not None  # a call this path takes
    out, lse, _ = fn(*leaves, causal=causal, return_attn_probs=True, ring_size=ring)
    assert not lse.requires_grad
    check_out(out, want, dtype)
    check_lse(lse, want_lse)
    for g in (dout.to(DEV), dout.to(DEV).transpose(1, 3).contiguous().transpose(1, 3)):  # a dout the kernels cannot read as it is, too
        grads = split(torch.autograd.grad(out, leaves, g, retain_graph=True))
        for got, w, name in zip(grads, want_grads, "qkv"):
            check_grad(got, w, dtype, "d" + name)
    with torch.no_grad():
        assert torch.equal(fn(*leaves, causal=causal, ring_size=ring), out)


def test_calls_that_need_more_than_the_native_path_still_run():
    q, k, v = rand_qkv((1, 40, 2, 64), 710, torch.bfloat16)
    want, _ = O.full_attention(q, k, v, 0.3, True)
    wide = torch.zeros(1, 40, 2, 67, dtype=torch.bfloat16, device=DEV)
    wide[..., 3:] = q.to(DEV)
    odd = wide[..., 3:]  # rows that are not 16-byte aligned: copied by the Python path
    assert _lib.native().attention(odd, k.to(DEV), v.to(DEV), 0.3, True, 0) is None
    check_out(spa.sp_aurora_func(odd, k.to(DEV), v.to(DEV), softmax_scale=0.3, causal=True), want, torch.bfloat16)
    with pytest.raises(ValueError):
        spa.sp_aurora_func(q, k, v)  # CPU tensors
    with pytest.raises((TypeError, ValueError)):
        spa._flash_attn_forward(q.to(DEV), k.to(DEV), v.to(DEV).float())
    with pytest.raises(ValueError):
        spa.sp_aurora_func(q.to(DEV), k.to(DEV), v.to(DEV), ring_size=3)  # does not divide the sequence
    with pytest.raises(ValueError):
        spa.sp_aurora_func(q.to(DEV), k.to(DEV), v.to(DEV), sharding="striped")


@pytest.mark.parametrize("S,H", [(33, 3), (4, 4)])  # (4, 4): a block whose two layouts have one shape is taken as [B,S,H,D]
def test_merge_of_two_blocks(S, H):
    B, D, dtype = 2, 64, torch.bfloat16
    q, = rand_qkv((B, H, S, D), 720, dtype, n=1)
    k, v = rand_qkv((B, H, 2 * S, D), 721, dtype, n=2)
    want, want_lse = O.attn_block(q, k, v, None, False)
    out = lse = None
    for i in range(2):
        part = slice(i * S, (i + 1) * S)
        blk, blk_lse = spa._flash_attn_forward(q.to(DEV), k[:, :, part].to(DEV), v[:, :, part].to(DEV))
        if i == 0:
            out, lse = spa.update_out_and_lse(None, None, blk, blk_lse)
            assert out.shape == (B, S, H, D) and lse.shape == (B, S, H, 1) and out.dtype == lse.dtype == torch.float32
        else:
            o2, l2 = spa.update_out_and_lse(out, lse, blk if S != H else blk.transpose(1, 2), blk_lse)
            assert o2 is out and l2 is lse
    check_out(out.transpose(1, 2), want, dtype)
    check_lse(lse.squeeze(-1).transpose(1, 2), want_lse)


def test_rank_stacked_tensors_are_no_operands_of_a_ring():
    q = torch.zeros(2, 2, 16, 2, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError):
        spa.sp_aurora_func(q, q, q, ring_size=2)
    with pytest.raises(ValueError):
        spa.sp_aurora_kvpacked_func(q, q)


def _leaves(seed, dtype=torch.bfloat16):
    return [t.to(DEV).requires_grad_() for t in rand_qkv((2, 40, 2, 64), seed, dtype)]


def test_forward_mode_and_transforms_are_refused():
    import torch.autograd.forward_ad as fwd_ad
    q, k, v = (t.detach() for t in _leaves(730))
    with fwd_ad.dual_level(), pytest.raises(RuntimeError):
        spa.sp_aurora_func(fwd_ad.make_dual(q, torch.ones_like(q)), k, v)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda x: spa.sp_aurora_func(x, k, v))(torch.stack([q, q]))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: spa.sp_aurora_func(x, k, v).float().sum())(q)


@pytest.mark.parametrize("unpack", [lambda t: t.to(DEV), lambda t: t.to(DEV).transpose(-1, -2).contiguous().transpose(-1, -2)])
def test_saved_tensors_that_went_through_a_hook(unpack):
    """Tensors offloaded to the host between forward and backward, and handed back in a layout that the kernels cannot read."""
    leaves = _leaves(731)
    dout = rand_qkv((2, 40, 2, 64), 732, torch.bfloat16, n=1)[0].to(DEV)
    want = torch.autograd.grad(spa.sp_aurora_func(*leaves, causal=True), leaves, dout)
    stays = lambda t: t.dim() == 4
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu() if stays(t) else t, lambda t: unpack(t) if stays(t) else t):
        out = spa.sp_aurora_func(*leaves, causal=True)
    for g, w in zip(torch.autograd.grad(out, leaves, dout), want):
        assert torch.equal(g, w)


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.float16), (32, torch.float32)])
def test_strides_of_operands_and_gradients(D, dtype):
    """Broadcast heads, batch entries and rows (stride 0), rows inside a wider tensor, heads before rows: the same as compact copies."""
    B, S, H = 2, 150, 3
    tol = {torch.bfloat16: 2e-2, torch.float16: 4e-3, torch.float32: 1e-5}[dtype]
    base = [t.to(DEV) for t in rand_qkv((B, S, H, D), 733, dtype, n=4)]
    forms = [lambda t: t[:, :, :1].expand(B, S, H, D), lambda t: t[:1].expand(B, S, H, D), lambda t: torch.cat([t, t], -1)[..., D:],
             lambda t: t.transpose(1, 2).contiguous().transpose(1, 2), lambda t: torch.cat([t, t], 1)[:, 1:S + 1], lambda t: t[:, :1].expand(B, S, H, D)]
    for f in forms:
        for which in range(4):
            x = [f(t) if i == which else t for i, t in enumerate(base)]
            got, want = [], []
            for ops_, res in ((x, got), ([t.contiguous() for t in x], want)):
                leaves = [t.detach().requires_grad_() for t in ops_[:3]]
                out = spa.sp_aurora_func(*leaves, causal=True)
                res += [out, *torch.autograd.grad(out, leaves, ops_[3])]
            for i, (g, w) in enumerate(zip(got, want)):
                if f is forms[-1] and which == 0:  # the Python path, whose delta is summed in another order: a rounding of the type here and there
                    torch.testing.assert_close(g, w, atol=tol, rtol=tol)
                else:
                    assert torch.equal(g, w), (forms.index(f), which, i)
            if which == 3 and f is forms[-1]:  # the Python path's kernels, and a packed batch
                out, lse = want[0].detach(), spa.sp_aurora_func(*[t.detach() for t in base[:3]], causal=True, return_attn_probs=True)[1]
                for g, w in zip(spa.ring.ring_flash_attn_backward(x[3], *base[:3], out, lse, None, True), want[1:]):
                    torch.testing.assert_close(g, w, atol=tol, rtol=tol)
                cu = torch.tensor([0, S, B * S], dtype=torch.int32, device=DEV)
                grads = []
                packed_dout = base[3][:1, :1].expand(B, S, H, D).reshape(B * S, H, D)
                for d in (base[3][0, :1].expand(B * S, H, D), packed_dout):
                    leaves = [t.reshape(B * S, H, D).clone().requires_grad_() for t in base[:3]]
                    grads.append(torch.autograd.grad(spa.sp_aurora_varlen_func(*leaves, cu, max_seqlen=S, causal=True), leaves, d))
                for g, w in zip(*grads):
                    assert torch.equal(g, w)


def test_a_gradient_that_never_comes_is_zero():
    class NoGrad(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.clone()

        @staticmethod
        def backward(ctx, g):
            return None

    leaves = _leaves(740)
    out = spa.sp_aurora_func(*leaves, causal=True)
    for g in torch.autograd.grad(NoGrad.apply(out).float().sum() + sum(t.sum() * 0 for t in leaves), leaves):
        assert not g.any()
    cu = torch.tensor([0, 40, 80], dtype=torch.int32, device=DEV)
    packed = [t.detach().reshape(80, 2, 64).requires_grad_() for t in leaves]
    out = spa.sp_aurora_varlen_func(*packed, cu, max_seqlen=40, causal=True)
    for g in torch.autograd.grad(NoGrad.apply(out).float().sum() + sum(t.sum() * 0 for t in packed), packed):
        assert not g.any()


@pytest.mark.parametrize("B,Sq,Sk,H,D,dtype", [(1, 1, 4096, 4, 128, torch.bfloat16), (2, 3, 3000, 4, 64, torch.float16), (1, 40, 5000, 4, 128, torch.bfloat16)])
def test_few_rows_of_a_differentiable_call_split_the_keys(B, Sq, Sk, H, D, dtype):
    """The differentiable functions take the same route as the operator: the same bits, and with gradients the same result."""
    q, = rand_qkv((B, Sq, H, D), 640, dtype, n=1)
    k, v = rand_qkv((B, Sk, H, D), 641, dtype, n=2)
    dout, = rand_qkv((B, Sq, H, D), 642, dtype, n=1)
    want, want_lse = O.full_attention(q, k, v, None, False)
    grads = O.attn_backward_autograd(q, k, v, dout, None, False)
    x, y, z = (t.to(DEV) for t in (q, k, v))
    op, op_lse = ops.flash_fwd(x, y, z, layout="bshd")
    assert _lib.load().spa_flash_fwd_splitkv_suggest(B, H, Sq, Sk, D, _lib.SPA_MASK_NONE, ops._DT[dtype]) > 1
    for fn in (lambda *t: spa.sp_aurora_func(*t), lambda a, b, c: spa.sp_aurora_kvpacked_func(a, torch.stack([b, c], 2)),
               lambda *t: spa.ulysses_flash_attn_func(*t), lambda *t: spa.LongContextAttention()(*t)):
        assert torch.equal(fn(x, y, z), op)
        leaves = [t.detach().clone().requires_grad_() for t in (x, y, z)]
        out = fn(*leaves)
        assert torch.equal(out, op)
        for name, g, w in zip("qkv", torch.autograd.grad(out, leaves, dout.to(DEV)), grads):
            check_grad(g, w, dtype, "d" + name)
    out, lse, _ = spa.sp_aurora_func(x, y, z, return_attn_probs=True)
    assert torch.equal(lse, op_lse)
    check_out(out, want, dtype)
    check_lse(lse, want_lse)


def test_every_function_works_without_the_native_module(monkeypatch):
    q, k, v, dout = (t.to(DEV) for t in rand_qkv((2, 96, 4, 64), 650, torch.bfloat16, n=4))
    cu = torch.tensor([0, 50, 192], dtype=torch.int32, device=DEV)
    rows, stacked = lambda t: t.reshape(192, 4, 64), lambda t: t.view(2, 2, 48, 4, 64).transpose(0, 1).contiguous()
    calls = [(lambda *t: spa.sp_aurora_func(*t, causal=True, ring_size=2), lambda t: t),
             (lambda *t: spa.sp_aurora_func(*t, causal=True, ring_size=2, sharding="zigzag"), lambda t: t),
             (lambda *t: spa.sp_aurora_varlen_func(*t, cu, max_seqlen=142, causal=True), rows),
             (lambda *t: spa.ulysses_flash_attn_func(*t, causal=True), stacked),
             (lambda *t: spa.LongContextAttention(sp_ulysses_degree=2, sp_ring_degree=1)(*t, causal=True), stacked)]
    results = []
    for module in (_lib.native(), False):
        monkeypatch.setattr(_lib, "_native", module)
        for fn, shape in calls:
            leaves = [shape(t).detach().clone().requires_grad_() for t in (q, k, v)]
            out = fn(*leaves)
            results.append((out.detach(), *torch.autograd.grad(out, leaves, shape(dout))))
        out, lse = ops.flash_fwd(q, k, v, None, True, layout="bshd")
        acc = spa.update_out_and_lse(None, None, out.transpose(1, 2).contiguous(), lse)
        results.append((out, lse, *spa.update_out_and_lse(*acc, out.transpose(1, 2).contiguous(), lse)))
    for one, other in zip(results[:len(calls) + 1], results[len(calls) + 1:]):
        for a, b in zip(one, other):  # (both round to bf16, at most once per ring step)
            torch.testing.assert_close(a, b, atol=4e-2, rtol=2e-2)


@pytest.mark.parametrize("grad", [False, True])
def test_a_forward_that_the_entry_point_refuses_is_the_python_paths_error(grad):
    """Rows 8 MiB apart, more than the kernels can re-base (2 GiB a head, 1 GiB in 128 rows): SpaError from every function, with and
    without gradients."""
    S, D, stride = 260, 64, (1 << 22) + 8
    base = torch.zeros(S * stride, dtype=torch.bfloat16, device=DEV)
    x = base.as_strided((1, S, 1, D), (S * stride, stride, D, 1)).requires_grad_(grad)
    cu = torch.tensor([0, S], dtype=torch.int32, device=DEV)
    for call in (lambda: spa.sp_aurora_func(x, x, x, causal=True), lambda: spa.ulysses_flash_attn_func(x, x, x),
                 lambda: spa.sp_aurora_varlen_func(x[0], x[0], x[0], cu, max_seqlen=S, causal=True),
                 lambda: spa._flash_attn_forward(*[x.transpose(1, 2)] * 3)):
        with pytest.raises(_lib.SpaError, match="1 GiB or more"):
            call()
