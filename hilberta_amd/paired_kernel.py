"""Exact 128-query paired block-sparse attention: the default inference entry point.

Drop-in for the reference module hilberta/paired_kernel.py: ``paired_attention`` keeps its
signature, host-side checks and error messages (paired_kernel.py:97-172) and launches the gfx950
HIP kernel ``hb_paired_fwd`` in place of the Triton ``_paired_fwd``.  Query halves of a paired row
share K/V loads but keep their own masks and softmax denominators (flag bit half + 2*key_half).
"""

from __future__ import annotations

import math
from numbers import Integral, Real

import torch

from .sparse_kernel import (
    LOG2E,
    _check_lse,
    _check_vector_layout,
    _non_overlapping_strides,
    _tensor_byte_span,
)


# Persistent workgroup count for hb_paired_fwd; 0 lets the library choose (2 per compute unit; 3
# for D = 64 calls with at least two items per workgroup).
NUM_GROUPS = 0


def _paired_fwd(q, k, v, out, lse, metadata, scale_log2, all_queries):
    """Launch through the operator hilberta_hip::paired_fwd on the current stream (module-level so
    tests can patch it)."""
    from . import ops

    ops.paired_fwd(q, k, v, out, lse, metadata.kv_indices, metadata.kv_flags, metadata.kv_counts,
                   int(metadata.global_tokens), int(metadata.key_block_size), float(scale_log2),
                   bool(all_queries), int(NUM_GROUPS))


def paired_attention(
    q, k, v, metadata, *, global_strategy="flash", num_warps=4, num_stages=2, scale=None, out=None,
    lse=None,
):
    """Exact inference attention over paired tables; metadata validated on CPU before transfer.

    Input checks inspect host-side tensor properties only: no device values are read, nothing
    synchronises, no mask is built and Q/K/V are not packed.  Both ``global_strategy`` values run
    the single HIP kernel (global query rows attend every key block in the same launch); the
    tuning keywords are validated as in the reference but select no code path.  ``lse`` may be a
    contiguous float32 [B,H,N] tensor that receives the natural-log row logsumexp.
    """
    # (sizes, strides and dtypes are read once: each read of a tensor attribute costs the host about as
    # much as a comparison, and a short call is as long as its checks)
    shape, dtype, device = q.shape, q.dtype, q.device
    if q.ndim != 4 or k.shape != shape or v.shape != shape or min(shape) <= 0:
        raise ValueError("Equal nonempty B,H,N,D Q/K/V required")
    strides = q.stride(), k.stride(), v.stride()
    if shape[-1] not in (64, 128) or any([s[-1] != 1 for s in strides]):
        raise ValueError("D64 or128 must be contiguous")
    if dtype not in (torch.float16, torch.bfloat16) or k.dtype != dtype or v.dtype != dtype:
        raise TypeError("Q/K/V must share BF16/FP16 dtype")
    if not q.is_cuda or k.device != device or v.device != device:
        raise ValueError("Q/K/V must be on the same CUDA device")
    if any([min(s[:3]) <= 0 for s in strides]):
        raise ValueError("Positive Q/K/V outer strides required")
    if torch.is_grad_enabled() and (q.requires_grad or k.requires_grad or v.requires_grad):
        raise ValueError("Inference only; disable autograd")
    N, G, key_block = metadata.tokens, metadata.global_tokens, metadata.key_block_size
    for value in (N, G, key_block):
        if type(value) is not int and (isinstance(value, bool) or not isinstance(value, Integral)):
            raise TypeError("Integer metadata shape fields required")
    if shape[-2] != N or G % 128 or N % 128 or not 0 <= G < N or key_block not in (64, 128):
        raise ValueError("Metadata/token shape mismatch or invalid128-token alignment")
    rows = (N - G) // 128
    ids, flags, counts = metadata.kv_indices, metadata.kv_flags, metadata.kv_counts
    table = ids.shape
    if ids.ndim != 2 or table[0] != rows or table[1] < 1:
        raise ValueError("Paired index shape must match ordinary query pairs")
    if flags.shape != table or counts.shape != (rows,):
        raise ValueError("Paired flag/count shape mismatch")
    for x in (ids, flags, counts):
        if x.device != device or x.dtype != torch.int32 or not x.is_contiguous():
            raise ValueError("Cached CUDA contiguous int32 metadata required")
    if global_strategy not in ("flash", "triton"):
        raise ValueError("Invalid global strategy")
    if any([isinstance(x, bool) or not isinstance(x, Integral) for x in (num_warps, num_stages)]):
        raise TypeError("Integer launch tuning required")
    if num_warps not in (4, 8) or num_stages not in (1, 2, 3, 4):
        raise ValueError("Invalid launch tuning")
    if scale is not None and (isinstance(scale, bool) or not isinstance(scale, Real)):
        raise TypeError("scale must be a real scalar, never a tensor")
    scale = shape[-1] ** -0.5 if scale is None else float(scale)
    if not math.isfinite(scale) or scale <= 0:
        raise ValueError("Positive finite scale required")
    if out is not None:
        out_strides = out.stride()
        if out.shape != shape or out.dtype != dtype or out.device != device or out_strides[-1] != 1:
            raise ValueError("Output must match Q shape/dtype/device with contiguous D")
        if min(out_strides) <= 0 or not _non_overlapping_strides(out):
            raise ValueError("Positive non-overlapping output strides required")
        if torch.is_grad_enabled() and out.requires_grad:
            raise ValueError("Inference output cannot require gradients")
        begin, end = _tensor_byte_span(out)
        for x in (q, k, v, ids, flags, counts):
            first, last = _tensor_byte_span(x)
            if begin < last and first < end:
                raise ValueError("Output cannot alias inputs or metadata")
    else:
        out = torch.empty_like(q)
    _check_lse(lse, q)
    _check_vector_layout((q, k, v, out))
    _paired_fwd(q, k, v, out, lse, metadata, scale * LOG2E, True)
    return out
