"""The transformer's linear layers over row ranges of a batch (CPU): the values of F.linear, and never as
a batched product, whose transposed right operand has faulted MI355X in bf16."""

import pytest
import torch
import torch.nn.functional as F
from torch.utils._python_dispatch import TorchDispatchMode

from hilberta_amd.flux_model import _linear


class _Products(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names += [name for name in ("baddbmm", "bmm", "addmm") if name in str(func)][:1]
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("batch", [1, 2, 3])
@pytest.mark.parametrize("lo,hi", [(0, 7), (0, 3), (3, 7)])
def test_row_ranges(batch, lo, hi):
    gen = torch.Generator().manual_seed(batch)
    x = torch.randn(batch, 7, 16, generator=gen)[:, lo:hi]
    w, b = torch.randn(8, 16, generator=gen), torch.randn(8, generator=gen)
    with _Products() as products:
        got = _linear(x, w, b)
    assert products.names and set(products.names) == {"addmm"}
    # sums of 16 fp32 products in another order: 16 units of 2^-24 of sums below 2^5
    assert got.is_contiguous() and (got - F.linear(x, w, b)).abs().max() <= 2 ** -14


def test_other_orders():
    """A transposed batch of rows (no contiguous last dimension) gives the same values."""
    x = torch.randn(2, 16, 5, generator=torch.Generator().manual_seed(0)).transpose(1, 2)
    w, b = torch.randn(8, 16), torch.randn(8)
    with _Products() as products:
        got = _linear(x, w, b)
    assert set(products.names) == {"addmm"} and (got - F.linear(x, w, b)).abs().max() <= 2 ** -14
