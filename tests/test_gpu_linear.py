"""Dense projections (kernels/linear.py): the HIP kernels against fp64 products of the same inputs, at
the edges of their tiles, and the calls that stay with torch."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from titans_core.kernels import _lib
from titans_core.kernels import linear as ln

HALF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}  # unit roundoff of the stored result


def _close(got, a, b):
    """got = a @ b up to the rounding of the stored value and of fp32 sums in any order: (K + 1) 2^-24
    times the sum of magnitudes bounds them; fp16 results below its normal range add 2^-25."""
    ref, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    bound = HALF[got.dtype] * ref.abs() + (a.shape[1] + 1) * 2.0 ** -24 * mag * (1 + HALF[got.dtype]) + 2.0 ** -24
    err = (got.double() - ref).abs()
    assert torch.all(err <= bound), f"max excess {(err - bound).max().item():.3g}"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (31, 64, 128), (64, 128, 64), (191, 192, 320),
                                   (193, 320, 192), (385, 256, 640), (515, 576, 128), (1000, 640, 192)])
def test_kernels_at_tile_edges(dev, M, N, K, dtype):
    g = torch.Generator().manual_seed(M + N + K)
    wide = torch.randn(M, K + 72, generator=g).to(dev, dtype)
    x = wide[:, 8:K + 8]  # a column slice: pitch K + 72, 16-byte aligned
    w = torch.randn(N, K, generator=g).to(dev, dtype)
    gy = torch.randn(M, N, generator=g).to(dev, dtype)
    _close(ln._fwd(x, w), x, w.t())
    _close(ln._dx(gy, w), gy, w)
    _close(ln._wgrad(gy, x), gy.t(), x)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(4099, 64, 64), (9001, 192, 640), (9001, 640, 192)])
def test_wgrad_split_over_rows(dev, M, N, K):
    nb = ctypes.c_size_t(0)
    assert _lib.lib().tmac_linear_wgrad_workspace(M, N, K, ctypes.byref(nb)) == 0 and nb.value > 0
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).to(dev, torch.bfloat16)
    gy = torch.randn(M, N, generator=g).to(dev, torch.bfloat16)
    a = ln._wgrad(gy, x)
    _close(a, gy.t(), x)
    assert torch.equal(a, ln._wgrad(gy, x))


@pytest.mark.gpu
def test_rows_past_the_end_do_not_leak(dev):
    """Infinities in the last row reach only what that row contributes to, and the last row counts once."""
    x = torch.ones(200, 64, device=dev, dtype=torch.bfloat16)
    x[-1] = float("inf")
    w = torch.ones(64, 64, device=dev, dtype=torch.bfloat16)
    y = ln._fwd(x, w)
    assert torch.all(y[:-1] == 64) and torch.all(torch.isinf(y[-1]))
    gy = torch.ones(200, 64, device=dev, dtype=torch.bfloat16)
    x[-1] = 3  # the rows copied past the end repeat the last one: each would add 3
    assert torch.all(ln._wgrad(gy, x) == 199 + 3)


@pytest.mark.gpu
def test_projection_gradients_and_modes(dev):
    g = torch.Generator().manual_seed(3)
    p = ln.Projection(192, 640).to(dev, torch.bfloat16)
    x = torch.randn(10, 1201, 192, generator=g).to(dev, torch.bfloat16).requires_grad_()
    gy = torch.randn(10, 1201, 640, generator=g).to(dev, torch.bfloat16)
    y = p(x)
    _close(y.detach().reshape(-1, 640), x.detach().reshape(-1, 192), p.weight.detach().t())
    y.backward(gy)
    _close(x.grad.reshape(-1, 192), gy.reshape(-1, 640), p.weight.detach())
    _close(p.weight.grad, gy.reshape(-1, 640).t(), x.detach().reshape(-1, 192))
    # an expanded gradient (stride 0) and a hook on the saved tensors
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(1) or t, lambda t: t):
        y = p(x)
    assert seen
    x.grad = p.weight.grad = None
    y.sum().backward()
    ones = torch.ones(12010, 640, device=dev, dtype=torch.bfloat16)
    _close(x.grad.reshape(-1, 192), ones, p.weight.detach())
    # double backward, functorch and forward-mode AD stay with torch's products
    (gx,) = torch.autograd.grad(p(x).float().pow(2).sum(), x, create_graph=True)
    gx.float().sum().backward()
    out = torch.func.vmap(p)(x.detach())
    assert out.shape == (10, 1201, 640)
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x))
        assert torch.autograd.forward_ad.unpack_dual(p(d)).tangent is not None
    # autocast: fp32 module, 16-bit product
    q = ln.Projection(192, 640).to(dev)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = q(x.detach().float())
    assert y.dtype == torch.bfloat16
    _close(y.detach().reshape(-1, 640), x.detach().reshape(-1, 192), q.weight.detach().bfloat16().t())


@pytest.mark.gpu
def test_result_changed_in_place(dev):
    """A projection's result may be changed in place, as nn.Linear's: y += residual, in training."""
    p = ln.Projection(192, 640).to(dev, torch.bfloat16)
    x = torch.randn(10, 1201, 192, device=dev).bfloat16().requires_grad_()
    gy = torch.randn(10, 1201, 640, device=dev).bfloat16()
    want = torch.autograd.grad(p(x), [x, p.weight], gy)
    y = p(x)
    y += torch.ones_like(gy)
    for a, b in zip(torch.autograd.grad(y, [x, p.weight], gy), want):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [3, 12010])
@pytest.mark.parametrize("leaf_x", [False, True])
def test_autocast_casts_the_weight_once(dev, rows, leaf_x):
    """Eight calls in one autocast context keep one cast copy of the fp32 weight, as nn.Linear's do, both
    where the kernels run and where the library does; the next context casts the changed weight again."""
    p = ln.Projection(192, 640).to(dev)
    x = torch.randn(rows, 192, device=dev).requires_grad_()
    gy = torch.randn(rows, 640, device=dev)

    def casts(fn):
        kept = []
        def pack(t):
            if t.dtype == torch.bfloat16 and t.shape in (p.weight.shape, p.weight.t().shape):
                kept.append(t)
            return t
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t), torch.autocast("cuda", dtype=torch.bfloat16):
            ys = [fn(x if leaf_x else x * (1 + 0 * i)) for i in range(8)]
            assert all(y.dtype == torch.bfloat16 for y in ys)
        (gw,) = torch.autograd.grad(sum(ys), p.weight, gy.bfloat16())
        assert gw.dtype == torch.float32
        return len({t.untyped_storage().data_ptr() for t in kept}), ys[0].detach(), gw
    n, y, gw = casts(p)
    n_ref, y_ref, gw_ref = casts(lambda t: F.linear(t, p.weight))
    assert n == n_ref == 1
    scale = gw_ref.abs().max()
    assert torch.allclose(y.float(), y_ref.float(), rtol=2.0 ** -7, atol=2.0 ** -7)
    assert torch.allclose(gw, gw_ref, rtol=2.0 ** -6, atol=2.0 ** -6 * scale)
    with torch.no_grad():
        p.weight.mul_(2)
    _, y2, _ = casts(p)
    assert torch.equal(y2, 2 * y)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(p(x), y2)


@pytest.mark.gpu
def test_only_what_a_gradient_needs_is_kept(dev):
    """As nn.Linear: with a frozen weight the input is not kept (and may change before the backward), for
    an input without gradient the weight is not."""
    p = ln.Projection(192, 640).to(dev, torch.bfloat16)
    x = torch.randn(12010, 192, device=dev).bfloat16()
    gy = torch.randn(12010, 640, device=dev).bfloat16()

    def kept(x):
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t, lambda t: t):
            y = p(x)
        return y, seen
    y, seen = kept(x)
    assert seen == [x.shape]
    with torch.no_grad():
        p.weight.add_(1)
    (gw,) = torch.autograd.grad(y, p.weight, gy)
    _close(gw, gy.t(), x)
    p.weight.requires_grad_(False)
    leaf = x.clone().requires_grad_()
    h = leaf * 1
    y, seen = kept(h)
    assert seen == [p.weight.shape]
    h.add_(1)
    (gx,) = torch.autograd.grad(y, leaf, gy)
    _close(gx, gy, p.weight.detach())


def test_rules_stay_within_what_was_measured():
    """(M, N, K) of each rule's edges: taken where the kernel measured faster, left to the library where it
    measured slower (more than 5 %) or nothing was measured."""
    for rule, taken, left in (
            (ln._fwd_applies, [(17920, 1920, 640), (2240, 1920, 640), (17920, 640, 640), (12000, 768, 768), (32768, 384, 384)],
             [(4480, 640, 640), (3000, 2304, 768), (17920, 768, 768), (6000, 2304, 768), (9000, 1536, 512), (9000, 1024, 1024)]),
            (ln._dx_applies, [(17920, 1920, 640), (4480, 640, 640), (12000, 1536, 1536), (17920, 2048, 2048)],
             [(9000, 1536, 1536), (17920, 2304, 768), (32768, 6144, 2048), (17920, 4096, 4096), (4480, 3072, 3072),
              (32768, 3072, 1024), (12000, 1280, 1280)]),
            (ln._wgrad_applies, [(17920, 1920, 640), (2240, 640, 640), (9000, 2048, 2048)],
             [(512, 640, 640), (1100, 1024, 1024), (17920, 4608, 1536), (9000, 6144, 2048), (17920, 4096, 4096),
              (4480, 12288, 4096), (1 << 20, 1 << 14, 1 << 14)])):
        assert all(rule(*s) for s in taken), rule.__name__
        assert not any(rule(*s) for s in left), rule.__name__


def test_projection_on_the_cpu_is_nn_linear():
    p = ln.Projection(64, 128)
    x = torch.randn(3, 5, 64, requires_grad=True)
    assert isinstance(p, torch.nn.Linear) and p.bias is None
    assert torch.equal(p(x), F.linear(x, p.weight))


def test_argument_errors():
    L, p = _lib.lib(), 4096  # an aligned address; nothing is launched
    nb = ctypes.c_size_t(0)
    assert L.tmac_linear_fwd(0, 64, p, 64, p, 64, 8, 64, 64, _lib.BF16, None) == -1
    assert L.tmac_linear_fwd(p, 64, p, 64, p, 64, 8, 63, 64, _lib.BF16, None) == -2
    assert L.tmac_linear_fwd(p, 32, p, 64, p, 64, 8, 64, 64, _lib.BF16, None) == -2
    assert L.tmac_linear_fwd(p, 64, p, 64, p, 64, 8, 64, 64, _lib.F32, None) == -4
    assert L.tmac_linear_dx(p + 2, 64, p, 64, p, 64, 8, 64, 64, _lib.BF16, None) == -5
    assert L.tmac_linear_dx(p, 1 << 23, p, 64, p, 64, 8, 64, 64, _lib.BF16, None) == -2
    assert L.tmac_linear_wgrad_workspace(0, 64, 64, ctypes.byref(nb)) == -2
    assert L.tmac_linear_wgrad(p, 64, p, 64, p, None, 0, 1 << 16, 64, 64, _lib.BF16, None) == -6
