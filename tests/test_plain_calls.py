"""Which calls the fused passes leave to the torch operations they replace, and that those still run
under tracing and transforms (CPU)."""

import warnings

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from hilberta_amd import _lib, flux_cond, flux_inputs, sampling_layout


def _rows(gen, *shape):
    return torch.randn(*shape, generator=gen).bfloat16()


def _calls():
    """(name, function of its tensors, tensors) of each entry that has a fused pass."""
    gen = torch.Generator().manual_seed(0)
    x = _rows(gen, 2, 16)
    weight = lambda n, k: _rows(gen, n, k) * k ** -0.5  # noqa: E731
    layers = [(weight(8, 16), _rows(gen, 8)), (weight(4, 16), None)]
    mlp = lambda: ((weight(24, 16), _rows(gen, 24)), (weight(8, 24), None))  # noqa: E731
    timestep, mlps, pooled_mlp = torch.rand(2, generator=gen).bfloat16(), [mlp()], mlp()
    return {
        "linear_layers": (lambda a: flux_cond.linear_layers(a, layers), (x,)),
        "embed": (lambda t, a: flux_cond.embed([t], mlps, a, pooled_mlp, 16, silu=True), (timestep, x)),
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


@pytest.mark.parametrize("name", ["linear_layers", "embed", "euler"])
def test_under_vmap(name):
    call, tensors = _calls()[name]
    got = torch.func.vmap(call)(*(torch.stack([t, 2 * t]) for t in tensors))
    for i in (0, 1):
        for g, r in zip(_flat(got), _flat(call(*((1 + i) * t for t in tensors))), strict=True):
            # A batched product may sum in another order, so a value may round to the next bf16, 2^-7 of
            # it: each of up to four roundings of an output, and each hidden value of an embedding, which
            # moves an output by 2^-7 |w| |h| <= 2^-7 * 1.5 * 4 in each of the two MLPs.
            torch.testing.assert_close(g[i], r, rtol=2 ** -5, atol=0.1)


@pytest.mark.parametrize("name", ["linear_layers", "embed", "euler", "rotary"])
def test_fake_tensors(name):
    """Shapes of device tensors without a device, and no look at an address (which would warn)."""
    call, tensors = _calls()[name]
    want = [t.shape for t in _flat(call(*tensors))]
    with FakeTensorMode(allow_non_fake_inputs=True), warnings.catch_warnings():
        warnings.simplefilter("error")
        got = call(*(torch.empty(t.shape, dtype=t.dtype) for t in tensors))
    assert [t.shape for t in _flat(got)] == want


class _Device(torch.Tensor):
    """(stands for a device tensor where there is none)"""

    is_cuda = True


def test_default_device_is_plain(monkeypatch):
    """torch.set_default_device is a function mode, and the fused passes are taken under it; under any
    other, alone or beside it, they are not."""
    monkeypatch.setattr(_lib, "_PLAIN_TYPES", (_Device,))
    t = torch.zeros(2).as_subclass(_Device)
    assert _lib.is_plain(t)
    with torch.device("cpu"):
        assert torch._C._len_torch_function_stack() == 1 and _lib.is_plain(t)
        with torch.overrides.BaseTorchFunctionMode():
            assert not _lib.is_plain(t)
    try:
        torch.set_default_device("cpu")
        assert _lib.is_plain(t)
    finally:
        torch.set_default_device(None)
    with torch.overrides.BaseTorchFunctionMode(), torch.device("cpu"):
        assert not _lib.is_plain(t)
