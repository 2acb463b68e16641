"""Per-(device, stream) workspaces for the attention kernels (csrc/torch_ops.cpp holds them).

A workspace holds the persistent kernel's work-queue counters (zero-filled once at allocation;
every launch leaves them at zero) and the partial results of split global query tiles.  Keying
by stream keeps launches that may overlap in time from sharing one; threads of one stream take turns
in the operators, each until both kernels of its call are enqueued.

A launch captured into a HIP graph gets a workspace of its own, made during the capture with a
fill kernel (so every replay zero-fills it before the attention kernel runs) and released when the
launch returns: it comes from the capture's private memory pool, which the graph keeps alive, and
later allocations of the same capture may reuse it only in stream order, after this launch's
kernels.  Captured launches therefore hold no memory beyond their graph's lifetime.
"""

from __future__ import annotations

import torch

from . import _lib, ops


class _Cache:
    """The (device, stream) keys of the cached eager workspaces."""

    def __iter__(self):
        keys = ops.workspace_keys()
        return iter(list(zip(keys[::2], keys[1::2])))


_CACHE = _Cache()


def attention_workspace(device, batch, heads, tokens, head_dim, global_tokens, width,
                        key_block_size, *, paired, all_queries):
    need = _lib.load().hb_attention_workspace_bytes(
        batch, heads, tokens, head_dim, global_tokens, width, key_block_size, int(paired),
        int(all_queries))
    if need < 0:
        _lib.check(1, "hb_attention_workspace_bytes")
    return ops.attention_workspace(torch.device(device), need)


def clear() -> None:
    """Drop the cached eager workspaces."""
    ops.clear_workspaces()
