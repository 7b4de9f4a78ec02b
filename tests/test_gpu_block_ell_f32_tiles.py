"""fp32 Block-ELL products at the edges of both tile heights (64 rows for small grids, 128 for large ones and
where long lists fill the CUs evenly)."""
import pytest
import torch

from titans_core.kernels import block_ell as kb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,n_brow,n_bcol,width", [(1, 2, 3, 1), (63, 3, 5, 2), (64, 3, 5, 5), (65, 1, 4, 4), (127, 3, 2, 2),
                                                   (129, 3, 5, 3), (6529, 3, 40, 10), (6528, 40, 3, 2), (6401, 40, 10, 5),
                                                   (4090, 16, 64, 32)])
def test_f32_products(dev, M, n_brow, n_bcol, width):
    g = torch.Generator().manual_seed(M)
    pat = kb.BlockELLPattern.sample(2, n_brow, n_bcol, width)
    x = torch.randn(M, 64 * n_brow, generator=g).to(dev)
    gy = torch.randn(M, 64 * n_bcol, generator=g).to(dev)
    v = torch.randn(n_brow, width, 64, 64, generator=g).to(dev)
    b = torch.randn(64 * n_bcol, generator=g).to(dev)
    ci = torch.from_numpy(pat.col_idx).to(dev)
    W = torch.zeros(n_brow, n_bcol, 64, 64, dtype=torch.float64, device=dev)
    W[torch.arange(n_brow, device=dev)[:, None], ci.long()] = v.double()
    W = W.permute(0, 2, 1, 3).reshape(64 * n_brow, 64 * n_bcol)

    def close(got, a, w, add=None):
        """fp32 sums in any order: (K + 2) 2^-24 times the sum of magnitudes."""
        ref, mag = a.double() @ w, a.double().abs() @ w.abs()
        if add is not None:
            ref, mag = ref + add.double(), mag + add.double().abs()
        assert torch.all((got.double() - ref).abs() <= (w.shape[0] + 2) * 2.0 ** -24 * mag)
    close(kb.block_ell_mm(x, v, pat, b), x, W, b)
    close(kb._bell_dx(gy, v, ci.reshape(-1), n_bcol), gy, W.t())
    dv = kb._bell_sddmm(x, gy, ci.reshape(-1), n_brow, width, torch.float32)
    ref = (x.double().t() @ gy.double()).reshape(n_brow, 64, n_bcol, 64).permute(0, 2, 1, 3)
    mag = (x.double().abs().t() @ gy.double().abs()).reshape(n_brow, 64, n_bcol, 64).permute(0, 2, 1, 3)
    rows = torch.arange(n_brow, device=dev)[:, None]
    err = (dv.double() - ref[rows, ci.long()]).abs()
    assert torch.all(err <= (M + 2) * 2.0 ** -24 * mag[rows, ci.long()])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n_brow,n_bcol,width", [(40, 10, 5), (7, 4, 3), (16, 8, 6), (9, 16, 9), (1, 8, 5)])
@pytest.mark.parametrize("M", [1, 33, 700, 2100])
def test_sddmm_blocks_across_rows(dev, M, n_brow, n_bcol, width, dtype):
    """Widths whose blocks fp32 takes four at a time across block-rows, from 256 rows on: every block of dW,
    twice the same."""
    _sddmm(dev, M, n_brow, n_bcol, width, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [8191, 8192, 8225])
@pytest.mark.parametrize("n_brow", [31, 32, 41])
def test_sddmm_blocks_across_rows_16_bit(dev, M, n_brow, dtype):
    """The same in 16 bit: width 5, at least 40 groups (32 block-rows) and 8192 rows."""
    _sddmm(dev, M, n_brow, 6, 5, dtype)


def _sddmm(dev, M, n_brow, n_bcol, width, dtype):
    g = torch.Generator().manual_seed(M + width)
    pat = kb.BlockELLPattern.sample(3, n_brow, n_bcol, width)
    x = torch.randn(M, 64 * n_brow, generator=g).to(dev, dtype)
    gy = torch.randn(M, 64 * n_bcol, generator=g).to(dev, dtype)
    ci = torch.from_numpy(pat.col_idx).to(dev)
    dv = kb._bell_sddmm(x, gy, ci.reshape(-1), n_brow, width, torch.float32)
    assert torch.equal(dv, kb._bell_sddmm(x, gy, ci.reshape(-1), n_brow, width, torch.float32))

    def blocks(a, b):
        full = (a.double().t() @ b.double()).reshape(n_brow, 64, n_bcol, 64).permute(0, 2, 1, 3)
        return full[torch.arange(n_brow, device=dev)[:, None], ci.long()]
    # fp32 sums of exact products in any order (16-bit) or of rounded ones (fp32)
    err = (dv.double() - blocks(x, gy)).abs()
    assert torch.all(err <= (M + 2) * 2.0 ** -24 * blocks(x.abs(), gy.abs()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [40, 700])
@pytest.mark.parametrize("width", [2, 5])
def test_sddmm_infinity_in_the_last_row(dev, M, width, dtype):
    """An infinite gradient in the last row gives infinities of the right sign: rows past the range add nothing."""
    pat = kb.BlockELLPattern.sample(1, 3, 6, width)
    x = torch.ones(M, 192, device=dev, dtype=dtype)
    x[-1, ::2] = -1
    gy = torch.ones(M, 384, device=dev, dtype=dtype)
    gy[-1] = float("inf")
    dv = kb._bell_sddmm(x, gy, torch.from_numpy(pat.col_idx).to(dev).reshape(-1), 3, width, torch.float32)
    assert torch.all(dv[:, :, ::2] == float("-inf")) and torch.all(dv[:, :, 1::2] == float("inf"))
