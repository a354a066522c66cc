"""The shading stage collects a tile's surviving rays in LDS before they enter
the next bounce's queue: images at path counts around its block, wave and
tile sizes, from a single pixel to several tiles a block, equal the oracle's."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,frames", [(1, 1, 1), (63, 1, 1), (64, 4, 1), (257, 1, 1), (511, 1, 1), (513, 3, 1),
                                        (640, 410, 1), (1024, 513, 2)])
def test_images_at_tile_edges(rt, gpu_ctx, w, h, frames):
    hs = rt.scene_soup(600, 9)
    scene = gpu_ctx.upload(hs)
    print(f"case: render {w}x{h}, {frames} frames, 4 bounces", flush=True)
    img, _ = gpu_ctx.render_frames(scene, [0.0, 3.0, 0.0], w, h, frames, vfov=60.0, bounces=4)
    torch.cuda.synchronize()
    osc = O.Scene(hs.triangles, hs.materials, hs.nodes, hs.lights, hs.spheres)
    ref, _ = O.render_frames(osc, [0.0, 3.0, 0.0], w, h, frames, vfov=60.0, bounces=4, traversal=O.TRAV_ORDERED,
                             threads=8)
    d = (img.cpu().numpy().astype(np.float64) - ref.astype(np.float64)) / 255.0
    assert np.sqrt((d * d).mean(axis=(0, 1))).max() <= 1e-3
    scene.release()
