"""Lanes whose ray has ended hold its hit until their wave refills or is
drained; rays that miss the scene's frame end before their first step.  Hits
must come out for all of them: in launches of nothing but such rays, where
they fall in runs or among others, and with refills at one idle lane and at 64."""
import numpy as np
import pytest
import torch

import oracle as O
from test_gpu_query import assert_equal_up_to_ties, oscene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def soup(rt, gpu_ctx):
    hs = rt.scene_soup(400, 21)
    return hs, gpu_ctx.upload(hs)


@pytest.mark.parametrize("n", [1, 64, 5000, 70001])
@pytest.mark.parametrize("away", ["all", "half", "third", "none"])
@pytest.mark.parametrize("refill,steal", [(1, 0), (64, 0), (0, 65), (0, 1)])
def test_rays_that_end_at_once(rt, gpu_ctx, soup, n, away, refill, steal):
    hs, scene = soup
    rays_np = rt.rays_box(n, 77, 1.0)
    gone = {"all": slice(None), "half": slice(0, n // 2), "third": slice(0, None, 3), "none": slice(0, 0)}[away]
    flat = rays_np.view(np.float32).reshape(n, 8)
    flat[gone, 0:3] += 50.0
    rays = rt.rays_to_device(rays_np)
    print(f"case: {n} rays, {away} away, refill {refill}, steal {steal}", flush=True)
    want = O.closest_hit(oscene(hs), rays_np, O.TRAV_ORDERED, threads=8)
    hits = torch.full((n, 4), float("nan"), device="cuda")
    gpu_ctx.set_tuning(blocks_per_cu=1, refill=refill, steal=steal)
    try:
        gpu_ctx.closest_hit(scene, rays, hits)
        torch.cuda.synchronize()
    finally:
        gpu_ctx.set_tuning()
    got = rt.hits_from_device(hits)
    assert not np.isnan(got["t"]).any()
    assert assert_equal_up_to_ties(oscene(hs), rays_np, got, want) <= 4
