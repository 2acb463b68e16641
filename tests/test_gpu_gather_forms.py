"""The native gather operator over every form its stride walk accepts, against index_select bit for
bit (a copy), and what it refuses."""

import itertools

import pytest
import torch

import hilberta_amd  # noqa: F401  (registers the operators)
from tests.helpers import say

pytestmark = pytest.mark.gpu

OPS = torch.ops.hilberta_hip


@pytest.mark.parametrize("sizes", [(3, 2, 5, 4), (1, 4, 1, 3), (2, 1, 6, 1), (4, 1, 1, 2)])
def test_orders_and_strides(hip_device, sizes):
    say(f"case gather forms {sizes}")
    for order in itertools.permutations(range(3)):
        # storage order of the first three dims, the last one contiguous; and a sliced, expanded copy
        base = torch.randn([sizes[i] for i in order] + [sizes[3] + 3], device=hip_device)
        x = base[..., :sizes[3]].permute(*[order.index(i) for i in range(3)], 3)
        for view in (x, x.contiguous(), x[:1].expand(3, -1, -1, -1), x.bfloat16()):
            for dim in range(-1, 4):
                index = torch.randint(0, view.shape[dim], (14,), device=hip_device)[::2]
                inner = torch.empty(view.shape[dim:][1:], device="meta")
                strides = zip(view.shape[dim:][1:], view.stride()[dim:][1:], inner.stride())
                if any(n > 1 and got != dense for n, got, dense in strides):
                    with pytest.raises(ValueError, match="contiguous"):
                        OPS.gather_rows(view, dim, index)
                    continue
                got = OPS.gather_rows(view, dim, index)
                assert got.is_contiguous() and torch.equal(got, view.index_select(dim, index))


def test_refusals(hip_device):
    x, index = torch.zeros(4, 8, device=hip_device), torch.arange(2, device=hip_device)
    for bad in (index.int(), index[None], index.cpu()):
        with pytest.raises(ValueError):
            OPS.gather_rows(x, 0, bad)
    with pytest.raises(IndexError):
        OPS.gather_rows(x, 2, index)
    q = torch.zeros(1, 1, 256, 128, device=hip_device, dtype=torch.bfloat16)
    table = torch.zeros(1, 1, device=hip_device, dtype=torch.int32)
    args = (table, table, table[0], 128, 64, 0.1, True, 0)
    with pytest.raises(ValueError):
        OPS.paired_fwd(q, q[:, :, :128], q, torch.empty_like(q), None, *args)
    with pytest.raises(ValueError):
        OPS.paired_fwd(q.float(), q.float(), q.float(), torch.empty_like(q.float()), None, *args)


def test_streams_keep_workspaces_apart(hip_device):
    from hilberta_amd import _workspace

    side = torch.cuda.Stream()
    args = (hip_device, 1, 24, 4608, 128, 512, 40, 64)
    main = _workspace.attention_workspace(*args, paired=1, all_queries=1)
    with torch.cuda.stream(side):
        other = _workspace.attention_workspace(*args, paired=1, all_queries=1)
        assert _workspace.attention_workspace(*args, paired=1, all_queries=1).data_ptr() == other.data_ptr()
    assert main.data_ptr() != other.data_ptr()
    assert len(set(_workspace._CACHE)) >= 2
    torch.cuda.synchronize()
    _workspace.clear()
    assert set(_workspace._CACHE) == set()


@pytest.mark.parametrize("row_bytes", [1, 3, 8, 15, 16, 17, 18, 24, 31, 33, 48, 63, 130, 4097])
def test_row_sizes_and_alignments(hip_device, row_bytes):
    """Rows around the 16-byte vector, at every kind of start: bytes, and bytes past the rows stay."""
    from hilberta_amd.layout import gather_into

    say(f"case gather rows of {row_bytes} bytes")
    gen = torch.Generator().manual_seed(row_bytes)
    for offset, gap in ((0, 0), (1, 0), (2, 5), (4, 12), (8, 8), (16, 32)):
        flat = torch.randint(-128, 128, (offset + 300 * (row_bytes + gap),), dtype=torch.int8, generator=gen)
        x = flat.to(hip_device)[offset:].view(300, row_bytes + gap)[:, :row_bytes]
        index = torch.randint(0, 300, (77,), generator=gen).to(hip_device)
        buf = torch.full((77 * row_bytes + 64 + offset,), 99, dtype=torch.int8, device=hip_device)
        out = buf[32 + offset:32 + offset + 77 * row_bytes].view(77, row_bytes)
        assert torch.equal(gather_into(x, 0, index, out=out), x.index_select(0, index))
        assert (buf[:32 + offset] == 99).all() and (buf[32 + offset + 77 * row_bytes:] == 99).all()
