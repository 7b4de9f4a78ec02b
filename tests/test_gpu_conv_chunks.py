"""Causal depthwise conv at sizes of every chunk length (8, 16, 32 and 64 positions per thread), with ragged
last chunks and chunk edges, against the fp64 oracle.

Bars: a 16-bit output is an fp32 sum of k exact products, rounded once: 2^-8 (bfloat16) of the value
plus the fp32 sum's error, k 2^-23 of its terms' sizes. The weight gradient, an fp32 sum of B T products
of unit-variance numbers in chunks of at most 64 (then of the partial sums): 1e-5 of its largest entry.
"""
import numpy as np
import pytest
import torch

from oracle import attention as oa
from titans_core.kernels.conv import causal_dwconv, dwconv_causal_bwd

pytestmark = pytest.mark.gpu


# (chunk of the forward, of the backward) in 16 bit
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,C,k", [
    (1, 8, 64, 4), (2, 9, 64, 4),  # 8, 8: one chunk, one row more
    (1, 17, 64, 8), (1, 16, 64, 8),  # 16, 16: eight taps
    (2, 521, 2048, 4),  # 8, 16
    (3, 1505, 2048, 4),  # 8, 32
    (3, 3009, 2048, 3),  # 16, 64
    (40, 257, 512, 4),  # 8, 32: more than 512 partial rows of 16
    (40, 400, 512, 4),  # 8, 64: more than 512 partial rows of 32
    (2, 8001, 2048, 4),  # 32, 64
    (17, 257, 512, 8),  # 16, 32: six taps and more in 16 bit, one round of 256 workgroups (fp32 16)
    (40, 257, 512, 7),  # 16, 64 (fp32 32)
])
def test_chunk_lengths(dev, dtype, B, T, C, k):
    g = torch.Generator().manual_seed(T + C + k)
    x, dy = (torch.randn(B, T, C, generator=g).to(dtype) for _ in range(2))
    w = (torch.randn(C, k, generator=g) * 0.5).to(dtype)
    xd, wd, dyd = x.to(dev), w.to(dev), dy.to(dev)
    with torch.no_grad():
        y = causal_dwconv(xd, wd)
        dx, dw = dwconv_causal_bwd(dyd, xd, wd)
    xn, wn, dyn = x.float().numpy(), w.float().numpy(), dy.float().numpy()
    want_dx, want_dw = oa.causal_dwconv_grads(xn, wn, dyn)
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    for got, want in ((y, oa.causal_dwconv(xn, wn)), (dx, want_dx)):
        err = np.abs(got.float().cpu().numpy() - want)
        # |terms| <= 6 sigma * 6 sigma * 0.5 = 18 each
        assert (err <= rel * np.abs(want) + k * k * 18 * 2.0 ** -23).all(), err.max()
    assert np.abs(dw.cpu().numpy() - want_dw).max() <= 1e-5 * np.abs(want_dw).max()
