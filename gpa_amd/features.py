"""The quadratic Q/K feature map on the device (`gpa_quad_features_forward`,
`gpa_quad_features_backward`): reference src/gpa/features.py:17-25.

One kernel launch forward (unit(x), the two products on the MFMA, the
normalised output) and one backward (dx, plus u and d(a)|d(b) for the weight
gradients u^T da, u^T db: `gpa_quad_weight_grads` in bfloat16, one batched
product in float32).  The weights are passed as two zero-padded copies in the
activation type (transposed for the forward products, row-major for the
backward's); they are parameters of a few hundred KB, rebuilt per call in one
launch (`gpa_quad_pack_weights`).
"""
from __future__ import annotations

import math

import torch
from torch import Tensor

from . import _lib


def _pad(d: int) -> int:
    return -(-d // 32) * 32


def _check_parameters(x: Tensor, left: Tensor, right: Tensor, gain: Tensor) -> None:
    """The kernels address both matrices and the gain by x's [.., heads, dim]."""
    heads, dim, device = x.shape[-2], x.shape[-1], x.device
    for name, w in (("left", left), ("right", right)):
        if w.shape != (heads, dim, dim) or w.device != device:
            raise _lib.HipBackendError(f"quadratic features: {name} must be [{heads}, {dim}, {dim}] on {x.device}, "
                                       f"got {list(w.shape)} on {w.device}")
    if gain.numel() != heads or gain.device != device:
        raise _lib.HipBackendError(f"quadratic features: one gain per head ({heads}) on {x.device} needed, "
                                   f"got {gain.numel()} on {gain.device}")


def _weights(left: Tensor, right: Tensor, dtype: torch.dtype, backward: bool):
    """wt [H][2][DP][DP] (wt[h][p][n][k] = W_p[h][k][n]) and, for the backward, w
    [H][DP][2DP] (w[h][k][p*DP + n] = W_p[h][k][n]), zero-padded, in `dtype`."""
    h, d, _ = left.shape
    dp = _pad(d)
    left, right = left.float().contiguous(), right.float().contiguous()
    wt = torch.empty(h, 2, dp, dp, device=left.device, dtype=dtype)
    w = torch.empty(h, dp, 2 * dp, device=left.device, dtype=dtype) if backward else None
    _lib.check(_lib.load().gpa_quad_pack_weights(left.data_ptr(), right.data_ptr(), h, d, _lib.DTYPE_CODES[dtype],
                                                 wt.data_ptr(), w.data_ptr() if backward else None,
                                                 _lib.stream_handle(left.device)), "gpa_quad_pack_weights")
    return wt, w


def _problem(x: Tensor, wt: Tensor, w: Tensor | None, gain: Tensor, out: Tensor | None) -> _lib.QuadProblem:
    rows, heads, dim = x.shape
    p = _lib.QuadProblem()
    p.rows, p.heads, p.dim, p.dtype = rows, heads, dim, _lib.DTYPE_CODES[x.dtype]
    p.x, p.row_stride = x.data_ptr(), x.stride(0)
    # (the forward reads wt alone)
    p.wt, p.w, p.gain = wt.data_ptr(), (w if w is not None else wt).data_ptr(), gain.data_ptr()
    p.out = out.data_ptr() if out is not None else None
    return p


class _QuadFeatures(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, left, right, gain):
        _check_parameters(x, left, right, gain)
        lib = _lib.load()
        wt, w = _weights(left, right, x.dtype, False)
        gain = gain.float().contiguous()
        out = torch.empty_like(x)
        _lib.check(lib.gpa_quad_features_forward(_problem(x, wt, w, gain, out), _lib.stream_handle(x.device)),
                   "gpa_quad_features_forward")
        ctx.save_for_backward(x, left, right, gain)
        return out

    @staticmethod
    def backward(ctx, dout):
        lib = _lib.load()
        x, left, right, gain = ctx.saved_tensors
        rows, heads, dim = x.shape
        dp = _pad(dim)
        wt, w = _weights(left, right, x.dtype, True)
        dout = dout.to(x.dtype).contiguous()
        dx = torch.empty_like(x)
        u = torch.empty(heads, rows, dp, device=x.device, dtype=x.dtype)
        dab = torch.empty(heads, rows, 2 * dp, device=x.device, dtype=x.dtype)
        dgain = torch.empty(-(-rows // 32), heads, device=x.device, dtype=torch.float32)
        grads = _lib.QuadGrads(dout.data_ptr(), dx.data_ptr(), u.data_ptr(), dab.data_ptr(), dgain.data_ptr())
        prob = _problem(x, wt, w, gain, None)
        _lib.check(lib.gpa_quad_features_backward(prob, grads, _lib.stream_handle(x.device)),
                   "gpa_quad_features_backward")
        # dW_p = u^T d(u W_p), in the activation type
        if x.dtype == torch.bfloat16:
            f32 = dict(device=x.device, dtype=torch.float32)
            partials = torch.empty(lib.gpa_quad_grad_partials(prob), **f32)
            dw = torch.empty(2, heads, dp, dp, **f32)
            _lib.check(lib.gpa_quad_weight_grads(prob, u.data_ptr(), dab.data_ptr(), partials.data_ptr(), dw.data_ptr(),
                                                 dw.data_ptr() + 4 * heads * dp * dp, _lib.stream_handle(x.device)),
                       "gpa_quad_weight_grads")
            dleft, dright = dw[0, :, :dim, :dim], dw[1, :, :dim, :dim]
        else:
            dw = torch.bmm(u.transpose(1, 2).contiguous(), dab)           # [H, DP, 2DP], contiguous operands
            dleft, dright = dw[:, :dim, :dim], dw[:, :dim, dp:dp + dim]
        return dx, dleft.to(left.dtype), dright.to(right.dtype), dgain.sum(0)


def supported(x: Tensor) -> bool:
    return x.is_cuda and x.dtype in _lib.DTYPE_CODES and 1 <= x.shape[-1] <= _lib.QUAD_MAX_DIM


def quadratic_features(x: Tensor, left: Tensor, right: Tensor, gain_raw: Tensor) -> Tensor:
    """x [..., H, D] -> the feature map of x (same shape and dtype)."""
    _lib.require_device(x)
    if not supported(x):
        raise _lib.HipBackendError("quadratic features: float32/bfloat16 with dim 1..256")
    heads, dim = x.shape[-2:]
    gain = 2 * gain_raw.sigmoid() * math.sqrt(dim)
    flat = x.reshape(-1, heads, dim).contiguous()
    if flat.shape[0] == 0:
        return x.clone()
    return _QuadFeatures.apply(flat, left, right, gain).reshape(x.shape)
