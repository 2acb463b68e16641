"""The fused device plan at the smallest grids, where the image has fewer blocks than a wave has
lanes and a workgroup's rows span phases, against the host builder: integers, bit for bit."""

import pytest

from tests.helpers import eq_exact, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,tiles", [(16, 1), (32, 1), (32, 4), (64, 1)])
@pytest.mark.parametrize("k,key_block", [(1, 64), (4, 128)])
def test_small_plans(hip_device, grid, tiles, k, key_block):
    from hilberta_amd.bridge_k import paired_plan_device

    say(f"case small plan grid={grid} tiles={tiles} K={k} KB{key_block}")
    args = dict(grid_size=grid, text_tokens=128, key_block_size=key_block)
    dev = paired_plan_device(tiles, k, False, device=hip_device, **args)
    host = paired_plan_device(tiles, k, False, device="cpu", **args)
    for f in ("original_order", "inverse_original", "image_order", "inverse_image_order",
              "physical_original_blocks", "original_to_physical"):
        eq_exact(getattr(dev.layout, f), getattr(host.layout, f).numpy(), f)
    for phase, (d, h) in enumerate(zip(dev.phases, host.phases)):
        for f in ("kv_indices", "kv_flags", "kv_counts"):
            eq_exact(getattr(d, f), getattr(h, f).numpy(), f"phase {phase} {f}")
