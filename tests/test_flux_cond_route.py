"""Which layers hb_linear_rows takes, by the route alone (CPU)."""

import pytest
import torch

from hilberta_amd import _lib, flux_cond


@pytest.fixture(autouse=True)
def as_on_a_device(monkeypatch):
    monkeypatch.setattr(_lib, "is_plain", lambda *tensors: True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_autocast_to_another_type(dtype):
    """F.linear computes and returns autocast's type; the kernel keeps the layer's."""
    x, layers = torch.zeros(2, 16, dtype=dtype), [(torch.zeros(8, 16, dtype=dtype), torch.zeros(8, dtype=dtype))]
    was = torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")
    try:
        for cast in (torch.bfloat16, torch.float16):
            torch.set_autocast_enabled("cuda", True)
            torch.set_autocast_dtype("cuda", cast)
            assert flux_cond._takes(x, layers) == (cast == dtype)
            torch.set_autocast_enabled("cuda", False)
            assert flux_cond._takes(x, layers)
    finally:
        torch.set_autocast_enabled("cuda", was[0])
        torch.set_autocast_dtype("cuda", was[1])


@pytest.mark.parametrize("rows,depth,columns,layers,kernel", [
    (1, 12288, 9216, 1, True), (2, 8192, 3072, 1, True),                       # bound by the weights
    (8, 3072, 3072, 1, True), (8, 4096, 3072, 1, False), (3, 12288, 1024, 1, False),
    (4, 3072, 9216, 1, False), (8, 1024, 9216, 1, True), (8, 3072, 9216, 3, True),
    (8, 3072, 52224, 4, True), (5, 6144, 18432, 1, True), (5, 8192, 18432, 1, False)])
def test_where_the_library_is_faster(monkeypatch, rows, depth, columns, layers, kernel):
    """More than two rows of a deep layer go to the library, as measured."""
    taken = []
    monkeypatch.setattr(flux_cond, "_takes", lambda x, layers: True)
    monkeypatch.setattr(flux_cond, "_launch", lambda xs, layers, outs: taken.append(1) or outs)
    x = torch.empty(rows, depth, device="meta")
    ws = [(torch.empty(columns // layers, depth, device="meta"), None) for _ in range(layers)]
    assert [t.shape for t in flux_cond.linear_layers(x, ws)] == [(rows, columns // layers)] * layers
    assert bool(taken) == kernel
