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


def _rows(t, name, B, R, C):
    if t.ndim != 3 or t.shape != (B, R, C) or t.stride(-1) != 1:
        raise ValueError(f"{name} must be [B, rows, hidden] with a contiguous last dimension")
    return t.stride(0), t.stride(1)


def _operands(x, shift, scale, y, gate, x_out, out):
    """Checked (pointers, strides, out) of one row set, in the order of hb_adaln_modulate_pair."""
    _lib.require_gpu(x)
    if x.dtype not in _DTYPES:
        raise ValueError("adaln_modulate takes bf16 or fp16 rows")
    B, R, C = x.shape if x.ndim == 3 else (0, 0, 0)
    xb, xn = _rows(x, "x", B, R, C)
    yb = yn = ob = on = 0
    if (y is None) != (gate is None):
        raise ValueError("y and gate are given together")
    if x_out is not None and y is None:
        raise ValueError("x_out is written only with a residual update")
    mods = [shift, scale] + ([gate] if gate is not None else [])
    for m in mods:
        if m.ndim != 2 or m.shape != (B, C) or m.stride(-1) != 1 or m.dtype != x.dtype:
            raise ValueError("shift/scale/gate must be [B, hidden] views with a contiguous last dim")
    mod_b = shift.stride(0)
    if scale.stride(0) != mod_b:
        raise ValueError("shift and scale must share one batch stride")
    tensors = [x] + mods
    if y is not None:
        yb, yn = _rows(y, "y", B, R, C)
        tensors.append(y)
    if x_out is not None:
        ob, on = _rows(x_out, "x_out", B, R, C)
        tensors.append(x_out)
    if out is None:
        out = torch.empty(B, R, C, dtype=x.dtype, device=x.device)
    pb, pn = _rows(out, "out", B, R, C)
    tensors.append(out)
    if any(t.device != x.device or t.dtype != x.dtype for t in tensors):
        raise ValueError("all tensors must share x's device and dtype")
    pointers = [None if t is None else t.data_ptr() for t in (x, y, gate, x_out, shift, scale, out)]
    gate_b = gate.stride(0) if gate is not None else 0
    return pointers, [xb, xn, yb, yn, gate_b, ob, on, mod_b, pb, pn], out


def adaln_modulate(x, shift, scale, *, y=None, gate=None, x_out=None, out=None, eps=1e-6):
    """x [B, rows, hidden]; shift / scale / gate [B, hidden] (views with a contiguous last dim,
    e.g. chunks of one modulation projection); y like x.  Returns out [B, rows, hidden]."""
    (px, py, pg, po, psh, psc, pout), (xb, xn, yb, yn, gb, ob, on, mb, pb, pn), out = _operands(
        x, shift, scale, y, gate, x_out, out)
    B, R, C = x.shape
    rc = _lib.load().hb_adaln_modulate(
        B, R, C, _DTYPES[x.dtype], float(eps), px, xb, xn, py, yb, yn, pg, gb, po, ob, on, psh, psc,
        mb, pout, pb, pn, _lib.stream_ptr(x.device),
    )
    _lib.check(rc, "hb_adaln_modulate")
    return out


def adaln_modulate_pair(first, second, *, eps=1e-6):
    """adaln_modulate of two row sets in one launch (the image and text streams of a double block):
    ``first`` and ``second`` are its arguments as dicts, of one batch, hidden size, dtype and device.
    Returns both outputs."""
    sets = [_operands(s["x"], s["shift"], s["scale"], s.get("y"), s.get("gate"), s.get("x_out"),
                      s.get("out")) for s in (first, second)]
    a, b = first["x"], second["x"]
    if a.shape[0] != b.shape[0] or a.shape[2] != b.shape[2] or a.dtype != b.dtype or a.device != b.device:
        raise ValueError("both row sets must share batch, hidden size, dtype and device")
    rc = _lib.load().hb_adaln_modulate_pair(
        a.shape[0], (ctypes.c_int32 * 2)(a.shape[1], b.shape[1]), a.shape[2], _DTYPES[a.dtype], float(eps),
        (ctypes.c_void_p * 14)(*sets[0][0], *sets[1][0]), (ctypes.c_int64 * 20)(*sets[0][1], *sets[1][1]),
        _lib.stream_ptr(a.device))
    _lib.check(rc, "hb_adaln_modulate_pair")
    return sets[0][2], sets[1][2]
