"""Linear layers of a few rows: the FLUX conditioning path in streamed HIP launches (csrc/cond.hip).

``linear_layers`` applies many layers to the same rows (every block's AdaLN modulation, diffusers
0.36.0 AdaLayerNormZero and its kin); ``embed`` is CombinedTimestepGuidanceTextProjEmbeddings: the
sinusoidal timestep and guidance embeddings and the pooled text, each through a SiLU MLP, summed.
Both return what the separate torch calls return up to the order of each fp32 sum.  Rows, sizes or
types the kernels do not take (more than eight rows, depths that are no multiple of 8, other than
bf16 / fp16, traced or differentiated inputs, autocast to another type) run as those torch calls, and
so do the layers of ``linear_layers`` that are too deep for their rows (``_pays``).
"""

from __future__ import annotations

import ctypes
import math

import torch
import torch.nn.functional as F

from . import _lib

MAX_ROWS = 8       # input rows per launch (hb_linear_rows)
MAX_LAYERS = 64    # layers per launch
_DTYPES = {torch.bfloat16: 0, torch.float16: 1}


def _takes(x, layers):
    """Whether hb_linear_rows takes rows ``x`` through each (weight, bias) of ``layers``."""
    # (first: a traced or transformed tensor has no address to look at)
    if not _lib.is_plain(x, *(t for layer in layers for t in layer if t is not None)):
        return False
    # (under autocast the torch calls compute in its type, whatever the layer's)
    if torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != x.dtype:
        return False
    if x.ndim != 2 or not 1 <= x.shape[0] <= MAX_ROWS or x.dtype not in _DTYPES or x.shape[1] % 8:
        return False
    if x.shape[1] == 0 or x.stride(1) != 1 or x.stride(0) % 8 or not 0 <= x.stride(0) < 2**31 or x.data_ptr() % 16:
        return False
    for w, b in layers:
        if w.ndim != 2 or w.shape[1] != x.shape[1] or not w.shape[0] or not w.is_contiguous() or w.data_ptr() % 16:
            return False
        if b is not None and (b.shape != w.shape[:1] or not b.is_contiguous()):
            return False
        if any(t is not None and (t.dtype != x.dtype or t.device != x.device) for t in (w, b)):
            return False
    return True


def _launch(xs, layers, outs, *, sum=1, silu=False):
    """outs[o] = sum over s of layers[o * sum + s] applied to xs[o * sum + s], in few launches."""
    x0 = xs[0]
    per = MAX_LAYERS // sum
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    with torch.cuda.device(x0.device):
        for lo in range(0, len(outs), per):
            o = outs[lo:lo + per]
            x, la = xs[lo * sum:(lo + per) * sum], layers[lo * sum:(lo + per) * sum]
            m, pointers = len(x), ctypes.c_void_p * len(x)
            rc = _lib.load().hb_linear_rows(
                len(o), sum, x0.shape[0], _DTYPES[x0.dtype], int(silu), pointers(*[t.data_ptr() for t in x]),
                (ctypes.c_int64 * m)(*[t.stride(0) for t in x]), pointers(*[w.data_ptr() for w, _ in la]),
                pointers(*[ptr(b) for _, b in la]), (ctypes.c_void_p * len(o))(*[t.data_ptr() for t in o]),
                (ctypes.c_int32 * len(o))(*[t.shape[1] for t in o]),
                (ctypes.c_int32 * m)(*[t.shape[1] for t in x]), _lib.stream_ptr(x0.device))
            _lib.check(rc, "hb_linear_rows")
    return outs


def _pays(rows, depth, columns, layers):
    """Whether one launch for ``layers`` layers of ``columns`` outputs in all beats a library call for each.

    With one or two rows it is bound by the read of the weights and always does; with more, by its
    products, and the library's matrix instructions win past a depth, sooner where fewer columns leave
    CUs idle (hb_linear_rows' line between one and four columns per wave).  One layer, kernel / library
    us on MI355X: 18432 columns, 8 rows of depth 6144 75 / 102, of 8192 91 / 71 (of 1024 24 / 20, where a
    library call is as long as its launch and a second layer turns it); 9216 columns, 8 rows of
    depth 1024 20 / 20, of 2048 33 / 20, 4 rows of 3072 25 / 20; 3072 columns, 8 rows of depth 3072
    17 / 20, of 4096 22 / 20.  All modulations of a two-block 3072-wide model, 8 rows: 101 / 160."""
    if rows <= 2:
        return True
    if columns >= 16384:
        return depth <= 6144
    return depth <= 4096 and columns * depth <= 3072 * 3072 * layers


def linear_layers(x, layers):
    """[F.linear(x, weight, bias) for weight, bias in layers] for rows x [B, K]."""
    if not layers or not _takes(x, layers) or not _pays(*x.shape, sum(w.shape[0] for w, _ in layers), len(layers)):
        return [F.linear(x, w, b) for w, b in layers]
    return _launch([x] * len(layers), layers, [x.new_empty(x.shape[0], w.shape[0]) for w, _ in layers])


def timestep_projection(t, dim=256):
    """diffusers get_timestep_embedding(flip_sin_to_cos=True, downscale_freq_shift=0): [cos | sin]
    of t * 10000^(-j/half)."""
    half = dim // 2
    freqs = torch.exp(-math.log(10000) * torch.arange(half, dtype=torch.float32, device=t.device) / half)
    angles = t[:, None].float() * freqs[None, :]
    return torch.cat([angles.cos(), angles.sin()], dim=-1)


def _mlp(x, layers):
    (w1, b1), (w2, b2) = layers
    return F.linear(F.silu(F.linear(x, w1, b1)), w2, b2)


def embed(scalars, scalar_mlps, pooled, pooled_mlp, dim, *, silu=False):
    """Sum over ``scalars`` (timestep, guidance: [B] in the model's type) of their MLP applied to
    the [cos | sin] embedding of 1000 times the scalar, plus ``pooled_mlp`` of ``pooled`` [B, K];
    its SiLU with ``silu``.  An MLP is two (weight, bias) layers with a SiLU between."""
    mlps = [*scalar_mlps, pooled_mlp]
    B = pooled.shape[0] if pooled.ndim == 2 else 0
    first, second = [m[0] for m in mlps], [m[1] for m in mlps]
    hidden = [w.shape[0] for w, _ in first]
    if (1 <= len(scalars) <= 2 and dim % 8 == 0 and _takes(pooled, first[-1:]) and _lib.is_plain(*scalars)
            and all(t.shape == (B,) and t.is_contiguous() and t.dtype == pooled.dtype
                    and t.device == pooled.device for t in scalars)):
        waves = pooled.new_empty(len(scalars), B, dim)
        h = [pooled.new_empty(B, n) for n in hidden]
        if (all(_takes(x, [layer]) for x, layer in zip(waves, first)) and
                all(_takes(x, [layer]) for x, layer in zip(h, second)) and
                len({w.shape[0] for w, _ in second}) == 1):
            with torch.cuda.device(pooled.device):
                rc = _lib.load().hb_sinusoid_rows(
                    scalars[0].data_ptr(), scalars[1].data_ptr() if len(scalars) == 2 else None, B, dim,
                    _DTYPES[pooled.dtype], waves.data_ptr(), _lib.stream_ptr(pooled.device))
            _lib.check(rc, "hb_sinusoid_rows")
            _launch([*waves, pooled], first, h, silu=True)
            out = pooled.new_empty(B, second[0][0].shape[0])
            return _launch(h, second, [out], sum=len(mlps), silu=silu)[0]
    total = None
    for t, mlp in zip(scalars, scalar_mlps):
        y = _mlp(timestep_projection(t * 1000, dim).to(pooled.dtype), mlp)
        total = y if total is None else total + y
    total = total + _mlp(pooled, pooled_mlp)
    return F.silu(total) if silu else total
