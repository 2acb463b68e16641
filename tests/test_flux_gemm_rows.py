"""How the single blocks' GEMMs walk the joint rows: whole, or text and image apart (CPU)."""

import pytest
import torch

from hilberta_amd.flux_model import _gemm_rounds, _linear_rows, _row_parts


def test_rounds():
    assert [_gemm_rounds(r, 9216) for r in (0, 1, 1792, 1793, 16384, 16385)] == [0, 1, 1, 2, 9, 10]


@pytest.mark.parametrize("image,whole", [(1024, {9216, 3072}), (4096, {9216, 3072}), (16384, set())])
def test_parts_of_the_measured_shapes(image, whole):
    for columns in (9216, 12288, 3072):
        assert (_row_parts(512, (1, 512 + image), columns) is None) == (columns in whole)


@pytest.mark.parametrize("batch,T,N,columns", [(1, 512, 16896, 8), (2, 3, 7, 8), (3, 512, 16896, 256), (1, 0, 5, 8)])
def test_every_row_once(batch, T, N, columns):
    gen = torch.Generator().manual_seed(N)
    x, y = torch.randn(batch, N, 4, generator=gen), torch.randn(batch, N, 2, generator=gen)
    w, b, w2 = (torch.randn(s, generator=gen) for s in ((columns, 4), (columns,), (columns, 2)))
    out = torch.full((batch, N, columns), float("nan"))
    _linear_rows(x, w, b, out, T, add=(y, w2))
    assert torch.allclose(out, x @ w.t() + b + y @ w2.t(), atol=1e-5)


@pytest.mark.parametrize("batch,T,N,columns,parts", [
    (1, 512, 1536, 8, None), (3, 512, 1536, 8, None), (11, 256, 512, 8, [(0, 512)]), (2, 512, 4608, 8, [(0, 4608)]),
    (1, 512, 1408, 8, [(0, 512), (512, 1408)]),
    (2, 1024, 6144, 8, [(0, 1024), (1024, 6144)]), (2, 512, 512, 8, None)])
@pytest.mark.parametrize("gelu", [False, True])
def test_every_walk(batch, T, N, columns, parts, gelu):
    """All rows at once, one element at a time, and text and image apart, each with more than one part and
    with text; the second product and the activation on every one."""
    assert _row_parts(T, (batch, N), columns) == (
        None if parts is None else [(b, lo, hi) for b in range(batch) for lo, hi in parts])
    gen = torch.Generator().manual_seed(N)
    x, y = torch.randn(batch, N, 2, generator=gen), torch.randn(batch, N, 1, generator=gen)
    w, b, w2 = (torch.randn(s, generator=gen) for s in ((columns, 2), (columns,), (columns, 1)))
    out = torch.full((batch, N, columns), float("nan"))
    _linear_rows(x, w, b, out, T, gelu=gelu, add=None if gelu else (y, w2))
    ref = x @ w.t() + b
    ref = torch.nn.functional.gelu(ref, approximate="tanh") if gelu else ref + y @ w2.t()
    # sums of two or three fp32 products in another order; the CPU epilogue of _addmm_activation may be
    # the exact GELU, which the tanh form follows to 5e-4
    assert (out - ref).abs().max() <= (5e-4 if gelu else 1e-5)


def test_batches_of_the_measured_shapes():
    """Batch 2: 1024 px joins each element's rows, never both at once; 2048 px stays apart."""
    for columns in (9216, 3072):
        assert _row_parts(512, (2, 4608), columns) == [(0, 0, 4608), (1, 0, 4608)]
    for columns in (9216, 12288, 3072):
        assert _row_parts(512, (2, 16896), columns) == [(b, *r) for b in (0, 1) for r in ((0, 512), (512, 16896))]
