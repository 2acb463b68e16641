"""The HBM passes on both sides of the cache-size line, where their loads change policy: the same values.

Each call past the line is compared with the same rows in calls below it: rows are independent, so
the results are equal bit for bit."""

import pytest
import torch

from tests.helpers import say

pytestmark = pytest.mark.gpu

CACHE = 256 << 20


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("residual", [True, False])
def test_adaln(hip_device, dtype, residual):
    from hilberta_amd.flux_norm import adaln_modulate

    C, passes = 512, 4 if residual else 2
    rows = CACHE // (2 * C * passes) + 37
    gen = torch.Generator(hip_device).manual_seed(1)
    x, y = (torch.randn(1, rows, C, device=hip_device, generator=gen).to(dtype) for _ in range(2))
    shift, scale, gate = torch.randn(1, 3 * C, device=hip_device, generator=gen).to(dtype).chunk(3, 1)
    say(f"case adaln past the cache size {dtype} residual={residual}")

    def call(lo, hi):
        if not residual:
            return (adaln_modulate(x[:, lo:hi], shift, scale),)
        r = torch.empty_like(x[:, lo:hi])
        return r, adaln_modulate(x[:, lo:hi], shift, scale, y=y[:, lo:hi], gate=gate, x_out=r)

    parts = [call(0, rows // 2), call(rows // 2, rows)]
    for i, whole in enumerate(call(0, rows)):
        assert torch.equal(whole, torch.cat([p[i] for p in parts], 1))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads", [5, 6, 8])
def test_qk_prep(hip_device, dtype, heads):
    from hilberta_amd.flux_inputs import qk_prep, qk_prep_pair

    n = CACHE // (heads * 512) + 29
    gen = torch.Generator(hip_device).manual_seed(2)
    x = torch.randn(1, n, 2 * heads * 128, device=hip_device, generator=gen).to(dtype)
    w = torch.rand(128, device=hip_device, generator=gen).to(dtype)
    cos, sin = torch.rand(2, n, 128, device=hip_device, generator=gen)
    say(f"case qk_prep past the cache size {dtype} heads={heads}")
    whole = qk_prep_pair(None, x, heads=heads, cos=cos, sin=sin, weights=((None, w), (None, w)))
    single = qk_prep(None, x[..., :heads * 128], heads=heads, weight_image=w, cos=cos, sin=sin)
    assert torch.equal(single, whole[0])
    for lo, hi in ((0, n // 3), (n // 3, 2 * n // 3), (2 * n // 3, n)):
        part = qk_prep_pair(None, x[:, lo:hi], heads=heads, cos=cos[lo:hi], sin=sin[lo:hi],
                            weights=((None, w), (None, w)))
        assert torch.equal(part, whole[:, :, lo:hi])


@pytest.mark.parametrize("row_bytes", [12, 130, 512, 6144])
def test_gather(hip_device, row_bytes):
    from hilberta_amd.layout import index_select_rows

    rows = CACHE // (2 * row_bytes) + 53
    x = torch.randint(-128, 128, (rows, row_bytes), dtype=torch.int8, device=hip_device)
    index = torch.randperm(rows, device=hip_device)
    say(f"case gather past the cache size, rows of {row_bytes} bytes")
    assert torch.equal(index_select_rows(x, 0, index), x.index_select(0, index))


def _us(call, n=10):
    """Shortest of five times a call, in microseconds."""
    best = float("inf")
    for _ in range(6):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for _ in range(n):
            call()
        end.record()
        torch.cuda.synchronize()
        best = min(best, begin.elapsed_time(end) / n * 1e3)
    return best


@pytest.mark.parametrize("unique", [1, 16, 16384])
def test_gather_of_repeated_rows(hip_device, unique):
    """More rows than the source has, past the line: the same bytes, and (from the caches) in less time
    than a copy takes that reads as much as it writes."""
    from hilberta_amd.layout import index_select_rows

    x = torch.randn(unique, 3072, device=hip_device).to(torch.bfloat16)
    index = torch.randint(0, unique, (65536,), device=hip_device)
    say(f"case gather of 65536 rows out of {unique}")
    out = index_select_rows(x, 0, index)
    assert torch.equal(out, x.index_select(0, index))
    if unique <= 16:
        source = torch.empty_like(out)
        took, copy = _us(lambda: index_select_rows(x, 0, index)), _us(lambda: out.copy_(source))
        say(f"gather {took:.1f} us, copy {copy:.1f} us")
        assert took < copy


def test_gather_of_one_image_for_a_batch(hip_device):
    from hilberta_amd.layout import index_select_rows

    x = torch.randn(1, 8192, 3072, device=hip_device).to(torch.bfloat16).expand(4, -1, -1)
    index = torch.randperm(8192, device=hip_device)
    say("case gather of an expanded batch")
    assert torch.equal(index_select_rows(x, 1, index), x.index_select(1, index))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_adaln_of_repeated_rows(hip_device, dtype):
    """One image for a batch and one row of y for an image, past the line: as with copies of them."""
    from hilberta_amd.flux_norm import adaln_modulate

    C, B = 1024, 4
    rows = CACHE // (2 * C * 4 * B) + 5
    gen = torch.Generator(hip_device).manual_seed(7)
    new = lambda *s: torch.randn(*s, device=hip_device, generator=gen).to(dtype)  # noqa: E731
    x, y = new(1, rows, C).expand(B, -1, -1), new(B, 1, C).expand(-1, rows, -1)
    shift, scale, gate = new(B, 3 * C).chunk(3, 1)
    say(f"case adaln of repeated rows past the cache size {dtype}")

    def call(x, y):
        r = torch.empty(B, rows, C, device=hip_device, dtype=dtype)
        return r, adaln_modulate(x, shift, scale, y=y, gate=gate, x_out=r)

    dense = call(x.contiguous(), y.contiguous())
    for pair in ((x, y), (x, y.contiguous()), (x.contiguous(), y)):
        for got, ref in zip(call(*pair), dense):
            assert torch.equal(got, ref)
    assert torch.equal(adaln_modulate(x, shift, scale), adaln_modulate(x.contiguous(), shift, scale))


@pytest.mark.parametrize("expand", [(4, -1, -1), (1, -1, -1)])
def test_qk_prep_of_one_image_for_a_batch(hip_device, expand):
    """A batch stride of zero past the line, and a single image at a row stride of its own."""
    from hilberta_amd.flux_inputs import qk_prep_pair

    heads = 8
    n = CACHE // (heads * 1024 * expand[0]) + 13
    gen = torch.Generator(hip_device).manual_seed(8)
    x = torch.randn(1, n, 3 * heads * 128, device=hip_device, generator=gen).to(torch.bfloat16)
    x = x[..., :2 * heads * 128].expand(*expand)
    w = torch.rand(128, device=hip_device, generator=gen).to(torch.bfloat16)
    cos, sin = torch.rand(2, n, 128, device=hip_device, generator=gen)
    say(f"case qk_prep of an expanded batch {expand[0]}")
    got = qk_prep_pair(None, x, heads=heads, cos=cos, sin=sin, weights=((None, w), (None, w)))
    one = qk_prep_pair(None, x[:1], heads=heads, cos=cos, sin=sin, weights=((None, w), (None, w)))
    for b in range(expand[0]):
        assert torch.equal(got[:, b], one[:, 0])
