"""The Euler update (csrc/euler.hip) rounds as the torch sequence does: bitwise equal, at ragged sizes
around a thread's eight values and a workgroup's 2048, infinities and NaN included."""

import pytest
import torch

from hilberta_amd.sampling_layout import euler_step
from tests.helpers import say

pytestmark = pytest.mark.gpu


def _torch(x, y, step):
    return (x.float() + step * y.float()).to(y.dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 2047, 2048, 2049, 262144])
def test_bitwise(hip_device, n, dtype):
    gen = torch.Generator().manual_seed(n)
    x, y = (torch.randn(n, generator=gen).mul(9).to(dtype).to(hip_device) for _ in range(2))
    if n > 8:
        x[:4] = torch.tensor([float("inf"), float("-inf"), float("nan"), 0.0], dtype=dtype)
        y[3:6] = torch.tensor([float("inf"), float("nan"), 0.0], dtype=dtype)
    say(f"case euler n={n} {dtype}")
    for step in (-0.0371, 1e-5, 3.0):
        got, ref = euler_step(x, y, step), _torch(x, y, step)
        assert got.dtype == dtype and torch.equal(got.isnan(), ref.isnan())
        assert torch.equal(got.nan_to_num(), ref.nan_to_num())


def test_other_forms(hip_device):
    x = torch.randn(4, 64, device=hip_device)
    for a, b in ((x, x.bfloat16()), (x.bfloat16().t(), x.bfloat16().t()), (x.bfloat16()[:, 1:], x.bfloat16()[:, 1:])):
        assert torch.equal(euler_step(a, b, 0.5), _torch(a, b, 0.5))
