"""The conditioning launches (csrc/cond.hip) against fp32 torch on the same device.

An output is an fp32 sum of K products of 16-bit values, rounded once to 16 bits (half a unit in
the last place, u = 2^-8 for bf16 and 2^-11 for fp16 relative); sums taken in another order differ by
far less than that, so a value may fall on the other side of one rounding boundary: one unit, 2u of
the larger value.  A sum of layers rounds every partial, a SiLU once more: one more unit each, of a
magnitude the partials bound.
"""

import pytest
import torch

from hilberta_amd import flux_cond as C
from tests.helpers import say

pytestmark = pytest.mark.gpu

UNIT = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}


def _normal(gen, shape, dtype, std=1.0):
    return (torch.randn(shape, generator=gen) * std).to(dtype).cuda()


def _layer(gen, n, k, dtype):
    return _normal(gen, (n, k), dtype, k ** -0.5), _normal(gen, (n,), dtype, 0.5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 2, 3, 5, 8])
def test_linear_layers(hip_device, rows, dtype):
    gen = torch.Generator().manual_seed(rows)
    # column counts around a wave's and a workgroup's; depths around a wave's 512
    for k in (8, 256, 504, 512, 520, 3072):
        x = _normal(gen, (rows, k + 8), dtype)[:, :k]   # a row stride of its own
        layers = [_layer(gen, n, k, dtype) for n in (1, 3, 4, 5, 16, 17, 130)]
        layers.append((layers[-1][0], None))
        say(f"case linear_layers rows={rows} k={k} {dtype}")
        assert C._takes(x, layers)
        for y, (w, b) in zip(C.linear_layers(x, layers), layers):
            ref = x.float() @ w.float().t() + (0 if b is None else b.float())
            assert y.shape == ref.shape and y.dtype == dtype
            assert ((y.float() - ref).abs() <= UNIT[dtype] * ref.abs() + 1e-5).all()


def test_wide_layers(hip_device):
    """Enough columns in all for four columns per wave, ragged ones among them."""
    gen = torch.Generator().manual_seed(4)
    for rows in (1, 2, 4, 8):
        x = _normal(gen, (rows, 72), torch.bfloat16)
        layers = [_layer(gen, n, 72, torch.bfloat16) for n in (16384, 1, 6, 3)]
        say(f"case linear_layers wide rows={rows}")
        for y, (w, b) in zip(C.linear_layers(x, layers), layers):
            ref = x.float() @ w.float().t() + b.float()
            assert ((y.float() - ref).abs() <= UNIT[x.dtype] * ref.abs() + 1e-5).all()


def test_more_layers_than_a_launch(hip_device):
    gen = torch.Generator().manual_seed(3)
    x = _normal(gen, (2, 64), torch.bfloat16)
    layers = [_layer(gen, 1 + i % 7, 64, torch.bfloat16) for i in range(C.MAX_LAYERS + 3)]
    say("case linear_layers beyond one launch")
    for y, (w, b) in zip(C.linear_layers(x, layers), layers, strict=True):
        ref = x.float() @ w.float().t() + b.float()
        assert ((y.float() - ref).abs() <= UNIT[x.dtype] * ref.abs() + 1e-5).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,scalars", [(1, 2), (3, 1), (8, 2)])
def test_embed(hip_device, rows, scalars, dtype):
    gen = torch.Generator().manual_seed(rows)
    mlp = lambda k: (_layer(gen, 96, k, dtype), _layer(gen, 41, 96, dtype))  # noqa: E731
    mlps, pooled_mlp = [mlp(256) for _ in range(scalars)], mlp(72)
    # (1000 t below fp16's 65504 for guidance, too)
    ts = [torch.rand(rows, generator=gen).mul(3.5).to(dtype).cuda() for _ in range(scalars)]
    pooled = _normal(gen, (rows, 72), dtype)
    say(f"case embed rows={rows} scalars={scalars} {dtype}")
    got = C.embed(ts, mlps, pooled, pooled_mlp, 256)
    act = C.embed(ts, mlps, pooled, pooled_mlp, 256, silu=True)
    parts = [C._mlp(C.timestep_projection(t * 1000).to(dtype), m) for t, m in zip(ts, mlps)]
    parts.append(C._mlp(pooled, pooled_mlp))
    ref = sum(p.float() for p in parts)
    # hidden values a unit apart move an output by about a unit of its terms' norm, |h| |w| <= 4
    bound = UNIT[dtype] * (2 * sum(p.float().abs() for p in parts) + 4)
    assert ((got.float() - ref).abs() <= bound).all()
    assert ((act.float() - torch.nn.functional.silu(got.float())).abs() <= UNIT[dtype] * got.float().abs() + 1e-6).all()


def test_other_rows_run_as_torch_calls(hip_device):
    gen = torch.Generator().manual_seed(9)
    w, b = _layer(gen, 16, 24, torch.bfloat16)
    x = _normal(gen, (9, 24), torch.bfloat16)
    for rows in (x, x[:2].requires_grad_(), x[:, :20]):
        layer = (w[:, :rows.shape[1]], b)
        assert not C._takes(rows, [layer])
        assert torch.equal(C.linear_layers(rows, [layer])[0], torch.nn.functional.linear(rows, *layer))
