"""Launches with a lane for every ray hand the rays out without cursors, an
even number to each wave.  One block per CU makes the switch to cursors fall
at a known count: every ray must be traced exactly once on both sides of it,
at fewer rays than waves, and at counts that leave the last waves partly or
wholly empty."""
import numpy as np
import pytest
import torch

import oracle as O
from test_gpu_query import assert_equal_up_to_ties, oscene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def soup(rt, gpu_ctx):
    hs = rt.scene_soup(3000, 4)
    return hs, gpu_ctx.upload(hs)


# relative to the lanes of one block per CU ("lanes") and its waves
@pytest.mark.parametrize("base,off", [("zero", 1), ("zero", 3), ("zero", 64), ("zero", 257), ("waves", -1), ("waves", 0),
                                      ("waves", 1), ("lanes", -65), ("lanes", -1), ("lanes", 0), ("lanes", 1),
                                      ("lanes", 777)])
@pytest.mark.parametrize("steal", [0, 1, 65])
def test_rays_handed_out_once(rt, gpu_ctx, soup, base, off, steal):
    hs, scene = soup
    lanes = 256 * torch.cuda.get_device_properties(0).multi_processor_count
    n = {"zero": 0, "waves": lanes // 64, "lanes": lanes}[base] + off
    rays_np = rt.rays_box(n, 70 + n % 11, 1.0)
    rays = rt.rays_to_device(rays_np)
    print(f"case: {n} rays, steal {steal}", flush=True)
    want = O.closest_hit(oscene(hs), rays_np, O.TRAV_ORDERED, threads=8)
    hits = torch.full((n, 4), float("nan"), device="cuda")
    batched = torch.full((n, 4), float("nan"), device="cuda")
    gpu_ctx.set_tuning(blocks_per_cu=1, steal=steal)
    try:
        gpu_ctx.closest_hit(scene, rays, hits)
        b = rt.Batch(gpu_ctx, [(scene, rays, batched)], rt.batch_config(blocks_per_cu=1))
        b.launch()
        torch.cuda.synchronize()
        b.destroy()
    finally:
        gpu_ctx.set_tuning()
    for h in (hits, batched):
        got = rt.hits_from_device(h)
        assert not np.isnan(got["t"]).any()
        assert assert_equal_up_to_ties(oscene(hs), rays_np, got, want) <= 4
