"""fxlm.norm: fused RMSNorm (bf16 I/O, fp32 math) on gfx950.

y = x * rsqrt(mean(x^2) + eps) * w.  The forward stores rstd (fp32, one per
row); the backward produces dx and dw from a single pass over x and dy
(fx_rms_norm_bwd).  Surface and checks follow ml/fxlm/norm.py:30-90.  ``pre_norm``
returns the residual stream with the normed input so that the GPT block's two
gradients of x are summed inside that pass (fx_rms_norm_bwd_add).
"""
import torch

from fxgpu.abi import call, host, lib, ptr, stream_of


def _check(x, w):
    if x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16:
        raise TypeError(f"x and weight must be bfloat16 ({x.dtype}, {w.dtype})")
    if not (x.is_cuda and w.is_cuda):
        raise TypeError("x and weight must be cuda tensors")
    D = x.shape[-1]
    if w.shape != (D,):
        raise ValueError(f"weight must have shape ({D},), got {tuple(w.shape)}")
    if D % 8 != 0 or D > 8192:
        raise ValueError(f"D={D}: needs D % 8 == 0 and D <= 8192")
    if not x.is_contiguous() or not w.is_contiguous():
        raise ValueError("x and weight must be contiguous")
    return D


def _al(t):
    """t itself when its data is 16-byte aligned (the kernels read 16-byte vectors), else
    an aligned copy: a contiguous view at an odd storage offset is accepted, as the
    reference accepts any contiguous tensor."""
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _fwd(x, w, eps):
    """(y, rstd, x, w): x and w as the kernels read them (an aligned copy where needed)."""
    r = host.norm_fwd(x, w, eps)
    if r is None:
        _check(x, w)
        x, w = _al(x), _al(w)
        r = host.norm_fwd(x, w, eps)
    return r[0], r[1], x, w


class _RMSNorm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, eps):
        y, rstd, x, w = _fwd(x, w, eps)
        ctx.save_for_backward(x, w, rstd)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, w, rstd = ctx.saved_tensors
        dx, dw = host.norm_bwd(x, dy, w, rstd, None)
        return dx, dw, None


def rms_norm(x, weight, eps=1e-6):
    """x (..., D) bf16, weight (D,) bf16 -> y (..., D) bf16."""
    return _RMSNorm.apply(x, weight, float(eps))


class _PreNorm(torch.autograd.Function):
    """(x, rms_norm(x)) for a pre-norm residual block, whose input feeds both the norm
    and the residual sum: the backward gets both gradients and forms
    dx = dres + d(norm)/dx in the norm kernel's pass (fx_rms_norm_bwd_add) instead of the
    separate add autograd would run for ml/fxlm/model.py:69,71."""

    @staticmethod
    def forward(ctx, x, w, eps):
        y, rstd, xa, w = _fwd(x, w, eps)
        ctx.save_for_backward(xa, w, rstd)
        ctx.set_materialize_grads(False)
        return x, y

    @staticmethod
    def backward(ctx, dres, dy):
        x, w, rstd = ctx.saved_tensors
        if dy is None:
            return dres, None, None
        dx, dw = host.norm_bwd(x, dy, w, rstd, dres)
        return dx, dw, None


def pre_norm(x, weight, eps=1e-6):
    """(x, rms_norm(x, weight, eps)): the residual stream and the block's normed input,
    with the two gradients of x summed inside the norm's backward kernel."""
    return _PreNorm.apply(x, weight, float(eps))


class _AddPreNorm(torch.autograd.Function):
    """(s, rms_norm(s)) for s = x + r: the residual sum of ml/fxlm/model.py:69,71 done in
    the pass of the norm that reads it (fx_rms_norm_fwd_add; s, y and rstd are bit for
    bit those of the bf16 add followed by the norm).  Both inputs get the gradient of s,
    formed as in _PreNorm."""

    @staticmethod
    def forward(ctx, x, r, w, eps):
        got = host.norm_add_fwd(x, r, w, eps)
        if got is None:
            _check(x, w)
            if r.shape != x.shape or r.dtype != x.dtype or not r.is_contiguous():
                raise ValueError(f"r must be a contiguous {tuple(x.shape)} {x.dtype} tensor")
            w = _al(w)
            got = host.norm_add_fwd(_al(x), _al(r), w, eps)
        s, y, rstd = got
        ctx.save_for_backward(s, w, rstd)
        ctx.set_materialize_grads(False)
        return s, y

    @staticmethod
    def backward(ctx, ds, dy):
        s, w, rstd = ctx.saved_tensors
        if dy is None:
            return ds, ds, None, None
        dx, dw = host.norm_bwd(s, dy, w, rstd, ds)
        return dx, dx, dw, None


def add_pre_norm(x, r, weight, eps=1e-6):
    """(x + r, rms_norm(x + r, weight, eps)) in one pass over x and r; the backward is
    pre_norm's, with the gradient of the sum going to both x and r."""
    return _AddPreNorm.apply(x, r, weight, float(eps))


def rms_norm_fwd_stats(x, weight, eps=1e-6):
    """Forward only, returning (y, rstd): the fp32 per-row rstd for parity checks."""
    D = _check(x, weight)
    weight = _al(weight)
    N = x.numel() // D
    x2 = _al(x.view(N, D))
    y = torch.empty_like(x2)
    rstd = torch.empty(N, device=x.device, dtype=torch.float32)
    call("fx_rms_norm_fwd", ptr(x2), ptr(weight), ptr(y), ptr(rstd), N, D, float(eps),
         stream_of(x))
    return y.view(x.shape), rstd


def rms_norm_bwd_raw(x, dy, weight, rstd):
    """Backward only, returning (dx, dw_f32, dw_bf16) for parity checks."""
    D = _check(x, weight)
    weight = _al(weight)
    N = x.numel() // D
    x2, dy2 = _al(x.view(N, D)), _al(dy.contiguous().view(N, D))
    dx = torch.empty_like(x2)
    dw32 = torch.empty(D, device=x.device, dtype=torch.float32)
    dw = torch.empty(D, device=x.device, dtype=torch.bfloat16)
    work = torch.empty(max(1, lib().fx_rms_norm_bwd_workspace(N, D) // 4), device=x.device,
                       dtype=torch.float32)
    call("fx_rms_norm_bwd", ptr(x2), ptr(dy2), ptr(weight), ptr(rstd), ptr(dx), ptr(dw32),
         ptr(dw), ptr(work), N, D, stream_of(x))
    return dx.view(x.shape), dw32, dw
