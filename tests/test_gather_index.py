"""What gather_into hands to the kernel (CPU, with a stand-in for the launch)."""

import ctypes
from types import SimpleNamespace
from unittest.mock import patch

import pytest
import torch

from hilberta_amd import _lib, layout


@pytest.mark.parametrize("index", [torch.arange(12)[::3], torch.tensor([2]).expand(5), torch.arange(4)])
def test_index_strides(index):
    seen = []

    def launch(src, dst, pointer, rows, *rest):
        seen.extend((ctypes.c_int64 * rows).from_address(pointer))
        return 0

    x = torch.zeros(12, 3)
    with patch.object(_lib, "load", lambda: SimpleNamespace(hb_gather_rows=launch)), \
            patch.object(_lib, "stream_ptr", lambda device: 0):
        assert layout.gather_into(x, 0, index).shape == (index.numel(), 3)
    assert seen == index.tolist()


def test_written_tensors_on_the_device():
    """The kernel writes through these addresses: host memory under a device call would fault."""
    x, index = torch.zeros(12, 3), torch.arange(4)
    with patch.object(_lib, "load", side_effect=AssertionError("launched")):
        for kw in (dict(out=torch.empty(4, 3, device="meta")), dict(error=torch.zeros(1, dtype=torch.int8)),
                   dict(error=torch.zeros(1, dtype=torch.int32, device="meta")),
                   dict(error=torch.zeros(0, dtype=torch.int32))):
            with pytest.raises(ValueError):
                layout.gather_into(x, 0, index, **kw)
