"""Waves take their rays in short runs from all over a launch: two at a time
where every wave gets its rays at the start, eight where queries fetch them
from the cursors.  Every ray must be traced exactly once at odd and even
numbers of rays a wave, at counts that cut the last row or the last run short,
and on both sides of the counts where the runs change or end."""
import numpy as np
import pytest
import torch

import oracle as O
from test_gpu_query import assert_equal_up_to_ties, oscene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def soup(rt, gpu_ctx):
    hs = rt.scene_soup(500, 9)
    return hs, gpu_ctx.upload(hs)


# rays for each wave of a launch of one block per CU, and a few more or less
@pytest.mark.parametrize("each,off", [(1, 5), (2, -1), (2, 0), (2, 1), (3, 0), (5, -3), (63, 0), (64, -65), (64, -1), (64, 0),
                                      (64, 1), (65, 63), (100, 9), (128, 0), (192, -1), (192, 0)])
def test_every_ray_once(rt, gpu_ctx, soup, each, off):
    hs, scene = soup
    n = 4 * torch.cuda.get_device_properties(0).multi_processor_count * each + off
    rays_np = rt.rays_box(n, 40 + each, 1.0)
    rays = rt.rays_to_device(rays_np)
    print(f"case: {n} rays", flush=True)
    want = O.closest_hit(oscene(hs), rays_np, O.TRAV_ORDERED, threads=8)
    hits = torch.full((n, 4), float("nan"), device="cuda")
    gpu_ctx.set_tuning(blocks_per_cu=1)
    try:
        gpu_ctx.closest_hit(scene, rays, hits)
        torch.cuda.synchronize()
    finally:
        gpu_ctx.set_tuning()
    got = rt.hits_from_device(hits)
    assert not np.isnan(got["t"]).any()
    assert assert_equal_up_to_ties(oscene(hs), rays_np, got, want) <= 4
