"""dK/dV of the persistent keys at head dimension 64: their key block's list ends in a tail of query
tiles that the waves share (one slice up to 32 persistent tokens, two up to 64, none past that, none in lists
of less than 16 tiles or with a tail of less than 8). All gradients against the fp64 oracle, deterministic, at
the edges of those ranges."""
import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle import masks as om
from titans_core.kernels.window_attn import windowed_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dropout", [0.0, 0.2])
@pytest.mark.parametrize("S,w,Np", [(900, 64, 1), (1300, 96, 16), (1301, 64, 32), (1100, 64, 33),
                                    (1283, 100, 64), (1150, 64, 65), (576, 0, 5), (1217, 64, 128),
                                    (1000, 340, 16), (1000, 340, 48), (1000, 400, 16)])
def test_persistent_key_tail(dev, S, w, Np, dropout):
    g = torch.Generator().manual_seed(S + Np)
    B, H, D = 1, 2, 64
    q, k, v, do = (torch.randn(B, H, S, D, generator=g).to(torch.bfloat16) for _ in range(4))

    def grads():
        ts = [t.to(dev).requires_grad_() for t in (q, k, v)]
        windowed_attention(*ts, w, Np, True, dropout_p=dropout, seed=9).backward(do.to(dev))
        return [t.grad for t in ts]

    got = grads()
    assert all(torch.equal(a, b) for a, b in zip(got, grads()))
    args = [t.double().numpy() for t in (q, k, v, do)]
    mask = om.band_mask(S, w, Np)
    if dropout:
        from oracle import dropout as od
        bias = np.where(mask, 0.0, -np.inf)
        want = oa.biased_attention_grads(*args, bias, drop=od.drop_factors(B, H, S, 9, dropout))
    else:
        want = oa.masked_attention_grads(*args, mask)
    for t, r in zip(got, want):
        sc = max(1.0, float(np.abs(r).max()))  # rounding scales with the largest entries
        err = np.abs(t.double().cpu().numpy() - r) / sc
        assert np.all(err <= 2e-2 + 1e-2 * np.abs(r) / sc), err.max()
