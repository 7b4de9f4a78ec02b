"""RMSNorm at the edges of the backward's row split (64 rows a workgroup, 8 or 16 a wave) and of the
register counts, against fp64."""
import pytest
import torch

from titans_core.kernels import norm as kn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [8, 640, 2048, 2056, 4096])
@pytest.mark.parametrize("M", [1, 7, 8, 9, 63, 65, 200])
def test_rms_norm_rows(dev, M, D, dtype):
    g = torch.Generator().manual_seed(M + D)
    x, gy = (torch.randn(M, D, generator=g).to(dev, dtype) for _ in range(2))
    s = (torch.rand(D, generator=g) + 0.5).to(dev, dtype)
    y, rstd = kn._rmsnorm_fwd(x, s, 1e-5)
    dx, ds = kn._rmsnorm_bwd(gy, x, s, rstd)
    assert torch.equal(ds, kn._rmsnorm_bwd(gy, x, s, rstd)[1])
    xd, gd, sd = x.double(), gy.double(), s.double()
    r = 1 / torch.sqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-5)
    want_dx = r * gd * sd - xd * r ** 3 * (gd * sd * xd).mean(-1, keepdim=True)
    # one rounding of the result (bfloat16 has 8 significant bits, half an ulp 2^-8); fp32 sums of D (rows) or M (columns) terms and a few products before it
    u = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype] * 1.01
    n = (D + 16) * 2.0 ** -24
    mag = r * (gd * sd).abs() + xd.abs() * r ** 3 * (gd * sd * xd).abs().mean(-1, keepdim=True)
    assert torch.all((y.double() - xd * r * sd).abs() <= (u + n) * (xd * r * sd).abs() + 2.0 ** -24)
    assert torch.all((dx.double() - want_dx).abs() <= u * want_dx.abs() + n * mag + 2.0 ** -24)
    terms = gd * xd * r
    assert torch.all((ds.double() - terms.sum(0)).abs() <= (M + D + 16) * 2.0 ** -24 * terms.abs().sum(0))
