"""A stale operator library is refused before its operators are bound (CPU)."""

import pytest
import torch

from hilberta_amd import _lib, ops


def test_built_for_this_abi():
    assert torch.ops.hilberta_hip._abi_version() == _lib.header_abi_version() == _lib.load().hb_version()


def test_stale_operator_library(monkeypatch):
    monkeypatch.setattr(ops, "header_abi_version", lambda: _lib.header_abi_version() + 1)
    with pytest.raises(RuntimeError, match="rebuild the libraries"):
        ops._load()
