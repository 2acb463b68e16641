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
