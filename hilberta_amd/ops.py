"""torch operators over the C ABI (namespace ``hilberta_hip``).

The reference launches its kernels as framework-visible Triton launches (paired_kernel.py:181-204,
sparse_kernel.py:315-339) and gathers with ``index_select`` (flux_adapter.py:209-212, :243).
Here each HIP entry point of include/hilberta_hip.h is a registered operator with a schema and a HIP
implementation (csrc/torch_ops.cpp, libhilberta_torch.so, loaded below), a fake (shape-only)
implementation for tracing and, for pair_rows alone, a CPU one:

  hilberta_hip::paired_fwd(q, k, v, out!, lse!?, kv_indices, kv_flags, kv_counts, global_tokens,
                           key_block_size, scale_log2, all_queries, num_groups) -> ()
  hilberta_hip::sparse_fwd(q, k, v, out!, lse!?, kv_indices, kv_counts, global_tokens,
                           scale_log2, all_queries, num_groups) -> ()
  hilberta_hip::gather_rows(x, dim, index) -> Tensor
  hilberta_hip::pair_rows(kv_indices, kv_counts, total_blocks, key_block_size, paired_width)
                           -> (ids, flags, counts)

The attention ops write into caller-provided outputs (declared mutated), as the reference's
launches write into ``out``.  Argument checks with the reference's messages stay in the Python
entry points (paired_attention, sparse_attention) and run before the op; the library repeats the
cheap ones and reports them as ValueError.  The attention and gather ops have no CPU kernel: on
CPU tensors they raise.  pair_rows is plan setup and also runs on CPU tensors, through the
library's host table builder (hb_pair_rows_host, bit-identical to the device kernel).  Without the
built library the operators do not exist and every use of one raises.
"""

import torch
from torch import Tensor

from ._lib import LIB_PATH, header_abi_version, load

_NS = "hilberta_hip"
TORCH_LIB_PATH = LIB_PATH.with_name("libhilberta_torch.so")
# key blocks per row hb_pair_rows pairs (include/hilberta_hip.h)
PAIR_MAX_BLOCKS = 16384


def _fake_none(*args):
    return None


def _fake_pair_rows(kv_indices, kv_counts, total_blocks, key_block_size, paired_width):
    prows = (kv_indices.shape[0] + 1) // 2
    ids = kv_indices.new_empty((prows, paired_width))
    return ids, torch.empty_like(ids), kv_indices.new_empty((prows,))


def _fake_gather_rows(x, dim, index):
    shape = list(x.shape)
    shape[dim % x.ndim] = index.shape[0]
    return x.new_empty(shape)


def _pair_rows_cpu(kv_indices: Tensor, kv_counts: Tensor, total_blocks: int, key_block_size: int,
                   paired_width: int) -> tuple[Tensor, Tensor, Tensor]:
    """pair_rows of CPU tensors by hb_pair_rows_host."""
    from ._tables import pair_rows_device

    return pair_rows_device(kv_indices, kv_counts, total_blocks, key_block_size=key_block_size,
                            paired_width=paired_width)


class _Missing:
    """An operator whose library could not be loaded: calling it raises."""

    def __init__(self, name, reason):
        self.name, self.reason = name, reason

    def __call__(self, *args, **kwargs):
        raise RuntimeError(f"{_NS}::{self.name}: {self.reason}")


def _load():
    """The operators of libhilberta_torch.so, in the order they are bound below."""
    if not TORCH_LIB_PATH.exists():
        raise RuntimeError(f"{TORCH_LIB_PATH} is missing: build the library first "
                           "(python -m hilberta_amd.build); there is no CPU fallback")
    load()  # the C ABI library, its version checked, before the operators bind to it
    torch.ops.load_library(str(TORCH_LIB_PATH))
    version = getattr(getattr(torch.ops, _NS), "_abi_version", None)  # (absent in the oldest ones)
    built, declared = version() if version else 0, header_abi_version()
    if built != declared:
        raise RuntimeError(f"{TORCH_LIB_PATH} was built for {f'ABI {built}' if built else 'an older ABI'} but "
                           f"include/hilberta_hip.h declares ABI {declared}: rebuild the libraries "
                           "(python -m hilberta_amd.build)")
    fakes = dict(paired_fwd=_fake_none, sparse_fwd=_fake_none, pair_rows=_fake_pair_rows,
                 gather_rows=_fake_gather_rows)
    for name, fake in fakes.items():
        torch.library.register_fake(f"{_NS}::{name}", fake)
    torch.library.impl(f"{_NS}::pair_rows", "cpu", _pair_rows_cpu)
    return [getattr(getattr(torch.ops, _NS), name).default for name in _NAMES]


_NAMES = ("paired_fwd", "sparse_fwd", "pair_rows", "gather_rows", "_attention_workspace",
          "_workspace_keys", "_clear_workspaces")
try:
    _bound = _load()
except (RuntimeError, OSError) as e:  # the package still imports, so that it can be (re)built
    _bound = [_Missing(name, str(e)) for name in _NAMES]
paired_fwd, sparse_fwd, pair_rows, gather_rows, attention_workspace, workspace_keys, clear_workspaces = _bound
