"""Batches whose scenes need a little more stack than a work-group's 24
entries, under every stack setting, and the autotuner over them: the same hits
whatever part of the stacks is in LDS, also after a change of setting."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# stacks of 25 to 40 entries (three for each 4-wide level, and one), and of under 16
@pytest.mark.parametrize("tris", [500, 20000, 100000, 400000])
@pytest.mark.parametrize("block", [128, 256])
def test_batch_stacks(rt, gpu_ctx, tris, block):
    scene = gpu_ctx.upload(rt.scene_clusters(tris, 12))
    rays = rt.rays_to_device(rt.rays_box(30011, 4, 4.0))
    want = rt.hits_from_device(gpu_ctx.closest_hit(scene, rays))
    hits = torch.empty((30011, 4), device="cuda")
    b = rt.Batch(gpu_ctx, [(scene, rays, hits)], rt.batch_config(block=block, stack_lds=32))
    for lds in (32, 0, 8, 32, 16, 0):
        print(f"case: batch of {tris} triangles, block {block}, {lds} stack entries in LDS", flush=True)
        b.set_config(rt.batch_config(block=block, stack_lds=lds))
        hits.fill_(-7.0)
        b.launch()
        assert np.array_equal(rt.hits_from_device(hits).view(np.uint8), want.view(np.uint8)), lds
    if block == 256 and tris == 100000:
        b.autotune(trials=1)
        hits.fill_(-7.0)
        b.launch()
        assert np.array_equal(rt.hits_from_device(hits).view(np.uint8), want.view(np.uint8))
    b.destroy()
    scene.release()
