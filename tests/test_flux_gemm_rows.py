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
