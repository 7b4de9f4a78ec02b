"""The Block-ELL MLP's training step as one node (fc2's dX kernel forms the hidden gradient) against the
layers one after the other: the same bits but for fc1's bias gradient, whose fp32 sum has another order."""
import pytest
import torch

from titans_core.blocks.mlp import MLPBlock
from titans_core.kernels import _lib
from titans_core.kernels import block_ell as kb


def _step(mlp, x, gy):
    x = x.clone().requires_grad_()
    mlp.zero_grad(set_to_none=True)
    y = mlp(x)
    y.backward(gy)
    return [y.detach(), x.grad] + [p.grad for p in mlp.parameters()]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 63, 65, 255, 256, 257, 700])
def test_fused_step_equals_the_layers(dev, M, dtype, monkeypatch):
    torch.manual_seed(M)
    mlp = MLPBlock(192, 448, block_ell=True, density=0.5, seed=3).to(dev, dtype)
    x, gy = (torch.randn(M, 192, device=dev).to(dtype) for _ in range(2))
    calls = []
    fused = kb._bell_dx_gelu
    monkeypatch.setattr(kb, "_bell_dx_gelu", lambda *a: calls.append(1) or fused(*a))
    got = _step(mlp, x, gy)
    assert calls == [1]
    hook = mlp.fc1.register_forward_hook(lambda *a: None)  # observed layers run one after the other
    want = _step(mlp, x, gy)
    hook.remove()
    assert calls == [1]
    names = ["y", "dx"] + [n for n, _ in mlp.named_parameters()]
    for n, a, b in zip(names, got, want):
        if n != "fc1.bias":
            assert torch.equal(a, b), n
    # fc1.bias: sums of the M terms before their rounding (half an ulp each against the stored ones), in
    # another order, then one rounding to the 16-bit type
    i = names.index("fc1.bias")
    with torch.no_grad():
        z = kb.block_ell_mm(x, mlp.fc1.values, mlp.fc1.pattern, mlp.fc1.bias)
        ga = kb._bell_dx(gy, mlp.fc2.values, mlp.fc2.col_idx.reshape(-1), mlp.fc2.pattern.n_bcol)
        gz = kb._bell_gelu_bwd(ga, z, False)[0].double()
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    bound = (M * 2.0 ** -23 + ulp / 2 * (1 + ulp)) * gz.abs().sum(0) + ulp * gz.sum(0).abs() + M * 2.0 ** -25 + 2.0 ** -24
    assert torch.all((got[i].double() - gz.sum(0)).abs() <= bound)


@pytest.mark.gpu
def test_fused_step_partial_gradients(dev):
    """Frozen parameters, no biases' gradient, autocast and an input without gradient."""
    torch.manual_seed(0)
    mlp = MLPBlock(128, 256, block_ell=True, density=0.5).to(dev)
    x = torch.randn(3, 50, 128, device=dev)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = mlp(x)
    assert y.dtype == torch.bfloat16
    y.float().sum().backward()
    assert all(p.grad is not None and p.grad.dtype == torch.float32 for p in mlp.parameters())
    half = MLPBlock(128, 256, block_ell=True, density=0.5).to(dev, torch.bfloat16)
    half.fc1.bias.requires_grad_(False)
    half.fc2.values.requires_grad_(False)
    half(x.bfloat16()).sum().backward()
    assert half.fc1.bias.grad is None and half.fc2.values.grad is None
    assert half.fc1.values.grad is not None and half.fc2.bias.grad is not None


@pytest.mark.gpu
def test_training_fc2_alone_keeps_no_pre_activation(dev):
    """With fc1 frozen and an input without gradient, fc1 runs as in inference: nothing of it is kept."""
    mlp = MLPBlock(128, 256, block_ell=True, density=0.5).to(dev, torch.bfloat16)
    mlp.fc1.requires_grad_(False)
    x, gy = (torch.randn(70, 128, device=dev).bfloat16() for _ in range(2))
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(tuple(t.shape)) or t, lambda t: t):
        y = mlp(x)
    assert sorted(seen) == sorted([(70, 256), tuple(mlp.fc2.values.shape), tuple(mlp.fc2.pattern.device_index(dev)["col_idx"].shape)])
    y.backward(gy)
    with torch.no_grad():
        a = mlp.fc1(x, activation="gelu")
        assert torch.equal(y, mlp.fc2(a))
    want = kb._bell_sddmm(a, gy, mlp.fc2.pattern.device_index(dev)["col_idx"], *mlp.fc2.values.shape[:2], torch.bfloat16)
    assert torch.equal(mlp.fc2.values.grad, want) and mlp.fc1.bias.grad is None


@pytest.mark.gpu
@pytest.mark.parametrize("frozen", [(), ("fc1.values", "fc2.values", "x"), ("fc1.values", "fc1.bias", "fc2.values", "fc2.bias")])
def test_second_derivatives_are_not_dropped(dev, frozen):
    """create_graph: the same first gradients, and what is built on them raises or is right (fc2's bias
    gradient is a sum of the incoming one), whatever else requires grad: no gradient counts as a constant."""
    torch.manual_seed(1)
    mlp = MLPBlock(128, 256, block_ell=True, density=0.5).to(dev, torch.bfloat16)
    x = torch.randn(40, 128, device=dev).bfloat16().requires_grad_("x" not in frozen)
    ts = {"x": x, **dict(mlp.named_parameters())}
    for n in frozen:
        ts[n].requires_grad_(False)
    ts = {n: t for n, t in ts.items() if t.requires_grad}
    want = torch.autograd.grad(mlp(x).sum(), list(ts.values()))
    got = torch.autograd.grad(mlp(x).sum(), list(ts.values()), create_graph=True)
    for (n, g), w in zip(zip(ts, got), want):
        if n == "fc1.bias":  # the recorded route sums the rounded terms: 40 of them
            assert torch.allclose(g.float(), w.float(), rtol=2.0 ** -7, atol=40 * 2.0 ** -8), n
        else:
            assert torch.equal(g, w), n
        assert g.requires_grad == (n != "fc2.bias"), n
        if g.requires_grad:
            with pytest.raises(RuntimeError):
                torch.autograd.grad(g.float().pow(2).sum(), list(ts.values()), retain_graph=True, allow_unused=True)
    if "fc2.bias" in ts:
        gy = torch.randn(40, 128, device=dev).bfloat16().requires_grad_()
        (gb,) = torch.autograd.grad(mlp(x), ts["fc2.bias"], gy, create_graph=True)
        c = torch.randn(128, device=dev).bfloat16()
        (gg,) = torch.autograd.grad(gb, gy, c)
        assert torch.equal(gg, c.expand(40, 128))


@pytest.mark.gpu
def test_second_derivatives_of_single_layers(dev):
    """As above for the layers by themselves: a GELU layer whose only tracked input is its bias, and a
    plain layer's bias gradient."""
    torch.manual_seed(2)
    fc1, fc2 = (kb.BlockELLLinear(i, o, density=0.5).to(dev, torch.bfloat16) for i, o in ((128, 256), (256, 128)))
    fc1.values.requires_grad_(False)
    x = torch.randn(9, 128, device=dev).bfloat16()
    (g,) = torch.autograd.grad(fc1(x, activation="gelu").sum(), fc1.bias, create_graph=True)
    assert g.requires_grad
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g.sum(), fc1.bias)
    gy = torch.randn(9, 128, device=dev).bfloat16().requires_grad_()
    (gb,) = torch.autograd.grad(fc2(torch.randn(9, 256, device=dev).bfloat16()), fc2.bias, gy, create_graph=True)
    (gg,) = torch.autograd.grad(gb.sum(), gy)
    assert torch.equal(gg, torch.ones_like(gy))


def test_dx_gelu_argument_errors():
    import ctypes
    L, p = _lib.lib(), 4096  # an aligned address; nothing is launched
    nb = ctypes.c_size_t(0)
    assert L.tmac_bell_dx_gelu_workspace(0, 2, ctypes.byref(nb)) == -2
    assert L.tmac_bell_dx_gelu_workspace(257, 2, ctypes.byref(nb)) == 0 and nb.value == 2 * 128 * 4
    ok = [p, 192, p, p, p, 128, p, 128, p, p, nb.value, 257, 2, 3, 2, _lib.BF16, None]

    def call(**kw):
        a = list(ok)
        for k, v in kw.items():
            a[int(k[1:])] = v
        return L.tmac_bell_dx_gelu(*a)
    assert call(_4=None) == -1 and call(_9=None) == -1
    assert call(_5=64) == -2 and call(_15=_lib.F32) == -4
    assert call(_4=p + 2) == -5 and call(_10=nb.value - 4) == -6
