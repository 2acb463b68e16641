"""Gated residual + AdaLN modulation of the FLUX blocks in one HIP pass (csrc/adaln.hip).

``adaln_modulate(x, shift, scale, y=y, gate=gate, x_out=x)`` computes, per token row,

    r = x + gate * y;  x_out = r;  out = shift + LayerNorm(r) * (1 + scale)

which the FLUX blocks (diffusers 0.36.0 FluxTransformerBlock / FluxSingleTransformerBlock with
AdaLayerNormZero / AdaLayerNormZeroSingle / AdaLayerNormContinuous) run as separate torch passes:
``torch.addcmul`` for the gated residual, ``layer_norm``, ``1 + scale`` and another ``addcmul``.
"""

from __future__ import annotations

import ctypes

import torch

from . import _lib

_DTYPES = {torch.bfloat16: 0, torch.float16: 1}


def _strides(t, name, shape, dtype, device):
    """(batch, row) strides of one [B, rows, hidden] operand, and whether it is of x's kind."""
    st = t.stride()
    if t.shape != shape or st[2] != 1:
        raise ValueError(f"{name} must be [B, rows, hidden] with a contiguous last dimension")
    return st[0], st[1], t.dtype == dtype and t.device == device


def _operands(x, shift, scale, y, gate, x_out, out):
    """Checked operands of one row set: seven pointers and ten strides in the order of
    hb_adaln_modulate_pair, the sizes, and the output.  (A short call is as long as these checks, so
    each tensor attribute is read once.)"""
    if not (isinstance(x, torch.Tensor) and x.is_cuda):
        _lib.require_gpu(x)
    dtype, device, shape = x.dtype, x.device, x.shape
    if dtype not in _DTYPES:
        raise ValueError("adaln_modulate takes bf16 or fp16 rows")
    if len(shape) != 3:
        raise ValueError("x must be [B, rows, hidden] with a contiguous last dimension")
    xb, xn, same = _strides(x, "x", shape, dtype, device)
    yb = yn = gate_b = ob = on = 0
    py = pg = po = None
    if (y is None) != (gate is None):
        raise ValueError("y and gate are given together")
    if x_out is not None and y is None:
        raise ValueError("x_out is written only with a residual update")
    row = (shape[0], shape[2])
    for m in (shift, scale) if gate is None else (shift, scale, gate):
        if m.shape != row or m.stride(1) != 1 or m.dtype != dtype:
            raise ValueError("shift/scale/gate must be [B, hidden] views with a contiguous last dim")
        same = same and m.device == device
    mod_b = shift.stride(0)
    if scale.stride(0) != mod_b:
        raise ValueError("shift and scale must share one batch stride")
    if y is not None:
        yb, yn, ok = _strides(y, "y", shape, dtype, device)
        same, py, pg, gate_b = same and ok, y.data_ptr(), gate.data_ptr(), gate.stride(0)
    if x_out is not None:
        ob, on, ok = _strides(x_out, "x_out", shape, dtype, device)
        same, po = same and ok, x_out.data_ptr()
    if out is None:
        out = torch.empty(shape, dtype=dtype, device=device)
        pb, pn = shape[1] * shape[2], shape[2]
    else:
        pb, pn, ok = _strides(out, "out", shape, dtype, device)
        same = same and ok
    if not same:
        raise ValueError("all tensors must share x's device and dtype")
    return ((x.data_ptr(), py, pg, po, shift.data_ptr(), scale.data_ptr(), out.data_ptr()),
            (xb, xn, yb, yn, gate_b, ob, on, mod_b, pb, pn), (*shape, _DTYPES[dtype], device), out)


def adaln_modulate(x, shift, scale, *, y=None, gate=None, x_out=None, out=None, eps=1e-6):
    """x [B, rows, hidden]; shift / scale / gate [B, hidden] (views with a contiguous last dim,
    e.g. chunks of one modulation projection); y like x.  Returns out [B, rows, hidden]."""
    (px, py, pg, po, psh, psc, pout), (xb, xn, yb, yn, gb, ob, on, mb, pb, pn), (B, R, C, code, device), out = \
        _operands(x, shift, scale, y, gate, x_out, out)
    rc = _lib.load().hb_adaln_modulate(
        B, R, C, code, float(eps), px, xb, xn, py, yb, yn, pg, gb, po, ob, on, psh, psc, mb, pout, pb, pn,
        _lib.stream_ptr(device))
    _lib.check(rc, "hb_adaln_modulate")
    return out


def adaln_modulate_pair(first, second, *, eps=1e-6):
    """adaln_modulate of two row sets in one launch (the image and text streams of a double block):
    ``first`` and ``second`` are its arguments as dicts, of one batch, hidden size, dtype and device.
    Returns both outputs."""
    sets = [_operands(s["x"], s["shift"], s["scale"], s.get("y"), s.get("gate"), s.get("x_out"),
                      s.get("out")) for s in (first, second)]
    (pa, sa, (B, ra, C, code, device), out_a), (pb, sb, (Bb, rb, Cb, codeb, deviceb), out_b) = sets
    if (B, C, code, device) != (Bb, Cb, codeb, deviceb):
        raise ValueError("both row sets must share batch, hidden size, dtype and device")
    rc = _lib.load().hb_adaln_modulate_pair(
        B, (ctypes.c_int32 * 2)(ra, rb), C, code, float(eps), (ctypes.c_void_p * 14)(*pa, *pb),
        (ctypes.c_int64 * 20)(*sa, *sb), _lib.stream_ptr(device))
    _lib.check(rc, "hb_adaln_modulate_pair")
    return out_a, out_b
