"""rotary_tables on the device in one launch (csrc/rope.hip) against the oracle on the host.

Both take cos and sin of the same float64 angle up to 2 ulp of pow and one of the product: an angle
of at most 4096 then differs by at most 4096 * 2^-51 = 2e-12, far below half a unit of float32
(2^-25 = 3e-8 near one), so values differ only where a rounding boundary falls between: by one
float32 unit, 2^-24 at most below one.  Rows past a workgroup's 32 tokens, ragged ends, permuted and
strided ids and other axis splits are covered; sizes without a kernel keep the composed result.
"""

import pytest
import torch

from hilberta_amd.flux_inputs import rotary_tables
from oracle import flux_ops as F
from tests.helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 31, 32, 33, 255, 4608])
@pytest.mark.parametrize("axes", [(16, 56, 56), (0, 64, 64), (2, 126, 0)])
def test_against_oracle(hip_device, n, axes):
    gen = torch.Generator().manual_seed(n)
    ids = torch.randint(0, 257, (n, 3), generator=gen).float()
    ids[:, 0] = torch.rand(n, generator=gen) * 4096
    say(f"case rotary n={n} axes={axes}")
    got = rotary_tables(ids.to(hip_device), axes_dim=axes)
    for g, r in zip(got, F.rotary_tables(ids, axes_dim=axes)):
        assert g.shape == (n, 128) and g.dtype == torch.float32 and g.is_contiguous()
        assert (g.cpu() - r).abs().max() <= 2 ** -24


def test_other_forms(hip_device):
    ids = torch.randint(0, 200, (50, 6), generator=torch.Generator().manual_seed(1))
    ref = F.rotary_tables(ids[:, ::2].float())
    say("case rotary strided int64 and bf16 ids, no rows, gradients kept")
    for x in (ids.to(hip_device)[:, ::2], ids.to(hip_device, torch.bfloat16)[:, ::2]):
        for g, r in zip(rotary_tables(x), ref):
            assert (g.cpu() - r).abs().max() <= 2 ** -24
    assert [t.shape for t in rotary_tables(torch.zeros(0, 3, device=hip_device))] == [(0, 128)] * 2
    x = ids[:, :3].float().to(hip_device).requires_grad_()
    assert rotary_tables(x)[0].requires_grad   # the composed path serves differentiation


@pytest.mark.parametrize("axes", [(128,), (64, 64), (32, 32, 32, 32)])
def test_other_axis_counts(hip_device, axes):
    """Composed: the kernel reads rows of three ids."""
    gen = torch.Generator().manual_seed(len(axes))
    ids = torch.randint(0, 257, (77, len(axes)), generator=gen).float()
    say(f"case rotary axes={axes}")
    for g, r in zip(rotary_tables(ids.to(hip_device), axes_dim=axes), F.rotary_tables(ids, axes_dim=axes)):
        assert g.shape == (77, 128) and (g.cpu() - r).abs().max() <= 2 ** -24
