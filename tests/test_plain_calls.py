"""Which calls the fused passes leave to the torch operations they replace, and that those still run
under tracing and transforms (CPU)."""

import pytest
import torch

from hilberta_amd import flux_inputs, sampling_layout


def _rows(gen, *shape):
    return torch.randn(*shape, generator=gen).bfloat16()


def _calls():
    """(name, function of its tensors, tensors) of each entry that has a fused pass."""
    gen = torch.Generator().manual_seed(0)
    x = _rows(gen, 2, 16)
    return {
        "rotary": (flux_inputs.rotary_tables, (torch.rand(5, 3, generator=gen) * 50,)),
        "euler": (lambda a, b: sampling_layout.euler_step(a, b, 0.5), (x, _rows(gen, 2, 16))),
    }


def _flat(out):
    return [out] if isinstance(out, torch.Tensor) else list(out)


@pytest.mark.parametrize("name", list(_calls()))
def test_compiled_whole(name):
    call, tensors = _calls()[name]
    torch._dynamo.reset()
    got = torch.compile(call, fullgraph=True, backend="eager")(*tensors)
    for g, r in zip(_flat(got), _flat(call(*tensors)), strict=True):
        assert torch.equal(g, r)
