"""Training calls record a plain autograd.Function in eager mode and the registered torch.library op
where calls are traced, transformed or intercepted. Both routes: the same bits, results and gradients."""
import pytest
import torch

from titans_core.kernels import _lib
from titans_core.kernels import block_ell as kb
from titans_core.kernels.conv import causal_dwconv
from titans_core.kernels.norm import rms_norm
from titans_core.kernels.window_attn import windowed_attention


def _block_ell(activation):
    pat = kb.BlockELLPattern.sample(1, 3, 5, 2)
    return (lambda x, v, b: kb.block_ell_mm(x, v, pat, b, activation)), [(90, 192), (3, 2, 64, 64), (320,)]


def _attention(**kw):
    return (lambda q, k, v: windowed_attention(q, k, v, 40, 4, **kw)), [(2, 2, 100, 64)] * 3


CASES = {
    "norm": (lambda x, s: rms_norm(x, s), [(70, 128), (128,)]),
    "conv": (causal_dwconv, [(2, 75, 128), (128, 4)]),
    "linear": _block_ell(None),
    "linear_gelu": _block_ell("gelu"),
    "attention": _attention(),
    "attention_dropout": _attention(dropout_p=0.25, seed=11),
}


def _grads(fn, shapes, dtype, dev):
    g = torch.Generator().manual_seed(5)
    xs = [(torch.randn(*s, generator=g) * 0.3).to(dev, dtype).requires_grad_() for s in shapes]
    y = fn(*xs)
    y.backward(torch.randn(y.shape, generator=g).to(dev, dtype))
    return [y.detach()] + [x.grad for x in xs]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", list(CASES))
def test_routes_agree(dev, name, dtype, monkeypatch):
    fn, shapes = CASES[name]
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t) or t, lambda t: t):
        native = _grads(fn, shapes, dtype, dev)
    assert seen  # saved-tensor hooks see what the node keeps
    monkeypatch.setattr(_lib, "eager_native", lambda *a: False)
    for a, b in zip(native, _grads(fn, shapes, dtype, dev)):
        assert a.dtype == b.dtype and torch.equal(a, b)


def _mlp(dev, dtype):
    from titans_core.blocks.mlp import MLPBlock
    torch.manual_seed(4)
    m = MLPBlock(128, 256, block_ell=True, density=0.5).to(dev, dtype)
    ps = dict(m.named_parameters())
    return (lambda x, *p: torch.func.functional_call(m, dict(zip(ps, p)), (x,))), [(30, 128)] + [p.shape for p in ps.values()]


def _projection():
    from titans_core.kernels.linear import projection
    return projection, [(12010, 192), (640, 192)]


def _fused_qkv(dropout_p=0.0):
    from titans_core.kernels.window_attn import windowed_attention_qkv
    return (lambda qkv: windowed_attention_qkv(qkv, 2, 40, 4, dropout_p=dropout_p)), [(2, 90, 384)]


@pytest.mark.gpu
@pytest.mark.parametrize("name", [*CASES, "mlp", "projection", "fused_qkv", "fused_qkv_dropout"])
def test_batched_gradients(dev, name):
    """is_grads_batched: the backward meets batched tensors; each row's gradients are those of a backward
    by itself (up to the order of a bias gradient's sum)."""
    fn, shapes = {"mlp": lambda: _mlp(dev, torch.bfloat16), "projection": _projection, "fused_qkv": _fused_qkv,
                  "fused_qkv_dropout": lambda: _fused_qkv(0.25)}.get(name, lambda: CASES[name])()
    g = torch.Generator().manual_seed(6)
    xs = [(torch.randn(*s, generator=g) * 0.3).to(dev, torch.bfloat16).requires_grad_() for s in shapes]
    y = fn(*xs)
    gys = torch.randn(3, *y.shape, generator=g).to(dev, torch.bfloat16)
    batched = torch.autograd.grad(y, xs, gys, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for b, w in zip(batched, torch.autograd.grad(y, xs, gys[i], retain_graph=True)):
            if w.dim() == 1:  # fp32 sums of up to 90 terms, rounded or not, rounded to bfloat16
                assert torch.allclose(b[i].float(), w.float(), rtol=2.0 ** -7, atol=90 * 2.0 ** -8), name
            elif name == "projection":  # the library's product: fp32 sums in another order, then rounded
                scale = w.float().abs().max()
                assert torch.allclose(b[i].float(), w.float(), rtol=2.0 ** -7, atol=2.0 ** -10 * scale), name
            else:
                assert torch.equal(b[i], w), name


@pytest.mark.gpu
def test_changed_input_is_noticed(dev):
    """An input changed in place between forward and backward raises, as for the registered op."""
    x = torch.randn(8, 64, device=dev)
    s = torch.ones(64, device=dev, requires_grad=True)
    y = rms_norm(x, s)
    x.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


def test_eager_native_only_in_plain_eager_mode():
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class FM(TorchFunctionMode):
        def __torch_function__(self, f, types, args=(), kwargs=None):
            return f(*args, **(kwargs or {}))

    class DM(TorchDispatchMode):
        def __torch_dispatch__(self, f, types, args=(), kwargs=None):
            return f(*args, **(kwargs or {}))

    t, p = torch.zeros(2), torch.nn.Parameter(torch.zeros(2))
    assert _lib.eager_native(t, p, None)
    for mode in (FM(), DM()):
        with mode:
            assert not _lib.eager_native(t)
    with torch.autograd.forward_ad.dual_level():
        assert not _lib.eager_native(t)
    got = []
    torch.func.vmap(lambda v: got.append(_lib.eager_native(t)) or v)(t)
    torch.jit.trace(lambda v: got.append(_lib.eager_native(v)) or v + 1, t, check_trace=False)
    torch.func.grad(lambda v: got.append(_lib.eager_native(t)) or v.sum())(t)
    assert got == [False, False, False]

    class Sub(torch.Tensor):
        pass
    assert not _lib.eager_native(t.as_subclass(Sub))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,dh", [(2, 64), (3, 32), (1, 128), (2, 80)])
@pytest.mark.parametrize("kw", [{}, {"pattern": "blockwin", "causal": False}, {"dropout_p": 0.2}, {"mask": "bool"},
                                {"mask": "float"}])
def test_fused_qkv_gradient(dev, dtype, H, dh, kw, monkeypatch):
    """The fused projection's gradient written in place equals the one autograd joins from q, k and v
    (head dimension 80, padded to 128, takes that general route itself)."""
    from titans_core.kernels import window_attn as wa
    kw = dict(kw)
    g = torch.Generator().manual_seed(H * dh)
    B, S = 2, 150
    qkv = torch.randn(B, S, 3 * H * dh, generator=g).to(dev, dtype)
    go = torch.randn(B, S, H * dh, generator=g).to(dev, dtype)
    mask = kw.pop("mask", None)
    if mask is not None:
        keep = (torch.rand(S, S, generator=g) > 0.4) | torch.eye(S, dtype=torch.bool)
        bias = torch.randn(S, S, generator=g).masked_fill(~keep, float("-inf"))
        mask = {"bool": keep, "float": bias}[mask].to(dev)
    a, b = (qkv.clone().requires_grad_() for _ in range(2))
    calls = []
    fused = wa._FusedQKV.apply
    monkeypatch.setattr(wa._FusedQKV, "apply", lambda *args: calls.append(1) or fused(*args))
    torch.manual_seed(7)
    ya = wa.windowed_attention_qkv(a, H, 40, 4, attn_mask=mask, **kw)
    assert len(calls) == (dh in wa.HEAD_DIMS)
    ya.backward(go)
    torch.manual_seed(7)
    yb = windowed_attention(*wa._split_heads(b, H), 40, 4, attn_mask=mask, **kw).transpose(1, 2).reshape(B, S, -1)
    yb.backward(go)
    assert torch.equal(ya, yb) and torch.equal(a.grad, b.grad)
    assert torch.isfinite(a.grad).all()
    # an additive mask that needs its own gradient takes the general route
    if mask is not None and mask.is_floating_point():
        m = mask.clone().requires_grad_()
        del calls[:]
        wa.windowed_attention_qkv(a, H, 40, 4, attn_mask=m).backward(go)
        assert m.grad is not None and not calls
