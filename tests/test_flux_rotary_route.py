"""Which calls of rotary_tables the one-launch kernel serves, by the route alone (CPU).

The kernel reads three ids a token: any other number of axes has to be composed."""

import pytest
import torch

from hilberta_amd import _lib, flux_inputs
from oracle import flux_ops as F


@pytest.mark.parametrize("axes,kernel", [((128,), False), ((64, 64), False), ((16, 56, 56), True), ((0, 64, 64), True),
                                         ((32, 32, 32, 32), False), ((16, 16, 32, 32, 32), False)])
def test_axes(monkeypatch, axes, kernel):
    taken = []

    def hip(ids, theta, axes_dim):
        taken.append(axes_dim)
        return F.rotary_tables(ids, theta, axes_dim)

    monkeypatch.setattr(_lib, "is_plain", lambda *tensors: True)   # as device ids are
    monkeypatch.setattr(flux_inputs, "_rotary_tables_hip", hip)
    ids = torch.rand(9, len(axes), generator=torch.Generator().manual_seed(0)) * 100
    got = flux_inputs.rotary_tables(ids, axes_dim=axes)
    assert bool(taken) == kernel
    for g, r in zip(got, F.rotary_tables(ids, axes_dim=axes)):
        assert g.shape == (9, 128) and torch.equal(g, r)
