"""Bias-free dense projections on the GPU (HIP kernels for gfx950).

The attention modules' qkv and output projections are ``nn.Linear(..., bias=False)``
(attn/windowed_attention.py:229-230, attn/block_sparse_attention.py:84, :101). ``projection``
computes ``F.linear(x, weight)``: 16-bit GPU inputs run the MFMA kernels of
``csrc/linear_kernels.hip`` (forward, input and weight gradient), everything else torch's own.
``Projection`` is an ``nn.Linear`` whose forward calls it.
"""
from __future__ import annotations

import ctypes

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib

_HALF = (torch.bfloat16, torch.float16)
_MAX_PITCH = 1 << 22  # the kernels address a tile's rows with 32-bit offsets
_MAX_WEIGHT, _MAX_ROWS = 1 << 30, 1 << 30


def _rows(t: torch.Tensor) -> torch.Tensor:
    """t as [M, features] rows the kernels can read: unit column stride, a row pitch of a multiple of
    8 elements, a 16-byte aligned start (copied if it has not got that)."""
    t2 = t.reshape(-1, t.shape[-1])
    if (t2.stride(1) != 1 or t2.stride(0) < t2.shape[1] or t2.stride(0) % 8
            or t2.stride(0) > _MAX_PITCH or t2.data_ptr() % 16):
        t2 = t2.clone(memory_format=torch.contiguous_format)
    return t2


def _fwd(x2: torch.Tensor, w: torch.Tensor, lead=None) -> torch.Tensor:
    """x2 [M, K] · wᵀ as [M, N], or [*lead, N]: not a view of it, which an autograd node may not return
    to a caller that changes it in place."""
    (M, K), N = x2.shape, w.shape[0]
    y = torch.empty((M, N) if lead is None else (*lead, N), dtype=x2.dtype, device=x2.device)
    with _lib.device_guard(x2.device):
        rc = _lib.lib().tmac_linear_fwd(x2.data_ptr(), x2.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(), N,
                                        M, N, K, _lib.dtype_code(x2.dtype), _lib.stream_ptr(x2.device))
    _lib.check(rc, "tmac_linear_fwd")
    return y


def _dx(g2: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    (M, N), K = g2.shape, w.shape[1]
    dx = torch.empty((M, K), dtype=g2.dtype, device=g2.device)
    with _lib.device_guard(g2.device):
        rc = _lib.lib().tmac_linear_dx(g2.data_ptr(), g2.stride(0), w.data_ptr(), w.stride(0), dx.data_ptr(), K,
                                       M, N, K, _lib.dtype_code(g2.dtype), _lib.stream_ptr(g2.device))
    _lib.check(rc, "tmac_linear_dx")
    return dx


def _wgrad(g2: torch.Tensor, x2: torch.Tensor) -> torch.Tensor:
    (M, N), K = g2.shape, x2.shape[1]
    L = _lib.lib()
    nb = ctypes.c_size_t(0)
    _lib.check(L.tmac_linear_wgrad_workspace(M, N, K, ctypes.byref(nb)), "tmac_linear_wgrad_workspace")
    ws = torch.empty(nb.value, dtype=torch.uint8, device=g2.device)
    dw = torch.empty((N, K), dtype=g2.dtype, device=g2.device)
    with _lib.device_guard(g2.device):
        rc = L.tmac_linear_wgrad(g2.data_ptr(), g2.stride(0), x2.data_ptr(), x2.stride(0), dw.data_ptr(),
                                 ws.data_ptr(), nb.value, M, N, K, _lib.dtype_code(g2.dtype),
                                 _lib.stream_ptr(g2.device))
    _lib.check(rc, "tmac_linear_wgrad")
    return dw


# Where each kernel replaces the library's GEMM: where it measured faster or as fast (us, this kernel /
# library, GPU time of [M, K] x [N, K] in bf16; fp16 gives the same ratios to 9 %), over model widths 256 to
# 4096, N = K and 3 K, and 512 to 32768 rows (of 315 sizes so taken, 9 are 3 to 7 % slower). Forward and dX walk 192 x 128 output tiles, two workgroups per CU: few
# tiles, or a nearly empty last round of 512, leave the chip idle, and long walks and wide outputs are the
# library's, whose larger tiles read less through LDS.

def _tiles(rows: int, cols: int) -> int:
    return -(-rows // 192) * -(-cols // 128)


def _fill(tiles: int) -> float:
    """The share of the rounds of 512 workgroups that the tiles fill."""
    return tiles / (512 * -(-tiles // 512))


def _fwd_applies(M: int, N: int, K: int) -> bool:
    """(17920, 640, 1920), as (M, K, N): 46 / 82; (17920, 640, 640): 18.5 / 35; (2240, 640, 1920), 180 tiles:
    11.6 / 13.8; (12000, 768, 768), 378: 18.6 / 19.0; at K < 512 also rounds half empty: (32768, 384, 384),
    fill 0.50: 18.9 / 24.9. Left to the library: (4480, 640, 640), 120 tiles: 10.8 / 8.7; (3000, 768, 2304),
    288: 17.5 / 15.6; (17920, 768, 768), fill 0.55: 28.8 / 23.3; (4480, 1024, 3072): 34 / 26."""
    if K > 768:
        return False
    t = _tiles(M, N)
    return t >= (150 if K <= 512 else 180 if K <= 640 else 300) and (K < 512 or t <= 512 or _fill(t) >= 0.6)


def _dx_applies(M: int, N: int, K: int) -> bool:
    """(17920, 640, 640): 18.5 / 38; (4480, 640, 640), 120 tiles: 11.2 / 13.2; (12000, 768, 768): 19.6 / 31;
    (17920, 640, 1920), fill 0.92: 43 / 67; (12000, 1536, 1536), 0.74: 57 / 83. Left to the library:
    (4480, 768, 768), 144 tiles: 12.9 / 12.2; (17920, 768, 768), fill 0.55: 31 / 27; (12000, 640, 1920), 0.62:
    38 / 34; (9000, 1536, 1536), 0.55: 51 / 40; (32768, 1024, 3072): 196 / 165; (17920, 4096, 4096): 546 / 486."""
    t = _tiles(M, K)
    if N <= 640:
        return t >= 100
    if N <= 1024:
        return t >= 180 and (t <= 512 or _fill(t) >= 0.6)
    return N < 3072 and t <= 1536 and _fill(t) >= 0.7


def _wgrad_applies(M: int, N: int, K: int) -> bool:
    """The kernel splits the rows over the chip, which pays while the output has few tiles (of 256 x 128) and
    the rows are many: (17920, 640, 1920): 63 / 145; (17920, 640, 640): 30 / 105; (2240, 640, 1920): 19.9 /
    20.5; (17920, 2048, 2048), 128 tiles: 164 / 271. Left to the library: (1100, 1024, 1024): 14.8 / 13.2;
    (512, 640, 640): 9.4 / 8.2; (17920, 1536, 4608), 216 tiles: 281 / 258; (4480, 3072, 3072): 131 / 92."""
    return M >= 2048 and -(-N // 256) * -(-K // 128) <= 128


def _forward(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    N, K = weight.shape
    if not _fwd_applies(x.numel() // K, N, K):
        return F.linear(x, weight)
    return _fwd(_rows(x), _rows(weight), x.shape[:-1])


class _Projection(torch.autograd.Function):
    """F.linear(x, weight) with its gradients on the kernels. A backward that is itself differentiated
    (create_graph) uses torch's products, as nn.Linear's own double backward does."""

    @staticmethod
    def forward(ctx, x, weight):
        # what a gradient needs, as nn.Linear keeps: frozen weights hold no activations, and the other
        # operand may change before the backward
        ctx.save_for_backward(x if ctx.needs_input_grad[1] else None, weight if ctx.needs_input_grad[0] else None)
        return _forward(x, weight)

    @staticmethod
    def backward(ctx, gy):
        x, weight = ctx.saved_tensors
        gx = gw = None
        if torch.is_grad_enabled() or not _lib.direct_backward(gy, x, weight):
            if ctx.needs_input_grad[0]:
                gx = gy @ weight
            if ctx.needs_input_grad[1]:
                gw = gy.reshape(-1, gy.shape[-1]).t() @ x.reshape(-1, x.shape[-1])
            return gx, gw
        g2 = _rows(gy)
        M, N = g2.shape
        if ctx.needs_input_grad[0]:
            gx = _dx(g2, _rows(weight)) if _dx_applies(M, N, weight.shape[1]) else g2 @ weight
            gx = gx.view(*gy.shape[:-1], weight.shape[1])
        if ctx.needs_input_grad[1]:
            x2 = x.reshape(-1, x.shape[-1])
            gw = _wgrad(g2, _rows(x2)) if _wgrad_applies(M, N, x2.shape[1]) else g2.t() @ x2
        return gx, gw


def _applies(x: torch.Tensor, weight: torch.Tensor, grad: bool) -> bool:
    """Whether a kernel takes a part of this call (of plain GPU tensors whose types it takes): by shape
    alone, so that all other calls reach F.linear as they are."""
    if weight.device != x.device or weight.dim() != 2 or x.dim() < 1 or x.shape[-1] != weight.shape[1] or x.numel() == 0:
        return False
    (N, K), M = weight.shape, x.numel() // x.shape[-1]
    if N == 0 or N % 64 or K % 64 or max(N, K) > _MAX_PITCH or N * K > _MAX_WEIGHT or M > _MAX_ROWS:
        return False
    return _fwd_applies(M, N, K) or grad and (_dx_applies(M, N, K) or _wgrad_applies(M, N, K))


def _autocast(t: torch.Tensor, dt: torch.dtype) -> torch.Tensor:
    """t in the autocast type dt. A leaf that requires grad is cast through autocast's own cache, once per
    autocast context, as for F.linear: a one-operand einsum returns the cast tensor itself."""
    if t.dtype == dt or not (t.requires_grad and t.is_leaf):
        return t.to(dt)
    c = torch._VF.einsum("...->...", [t])
    return c if c.dtype == dt else t.to(dt)


def projection(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """F.linear(x, weight): [..., K] x [N, K] -> [..., N]. The kernels take bfloat16 and float16 (inside
    torch.autocast the inputs are cast to its dtype, as F.linear's are) with N and K multiples of 64."""
    ac = torch.is_autocast_enabled("cuda")
    if not (ac or x.dtype in _HALF) or not (x.is_cuda and weight.is_cuda and _lib.eager_native(x, weight)):
        return F.linear(x, weight)
    grad = torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad)
    if not _applies(x, weight, grad):
        return F.linear(x, weight)
    if ac:
        dt = torch.get_autocast_dtype("cuda")
        if dt not in _HALF or not all(t.dtype in (torch.float32, *_HALF) for t in (x, weight)):
            return F.linear(x, weight)
        x, weight = _autocast(x, dt), _autocast(weight, dt)
        with torch.autocast("cuda", enabled=False):
            return _run(x, weight, grad)
    if weight.dtype != x.dtype:
        return F.linear(x, weight)
    return _run(x, weight, grad)


def _run(x: torch.Tensor, weight: torch.Tensor, grad: bool) -> torch.Tensor:
    return _Projection.apply(x, weight) if grad else _forward(x, weight)


class Projection(nn.Linear):
    """nn.Linear(in_features, out_features, bias=False) on ``projection``."""

    def __init__(self, in_features: int, out_features: int):
        super().__init__(in_features, out_features, bias=False)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return projection(x, self.weight)
