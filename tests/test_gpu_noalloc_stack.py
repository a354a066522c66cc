"""rt_closest_hit_noalloc and stack_lds: a setting that asks for a part of the
stack is refused by the depth of the caller's tree alone, whatever tree the
traversal walks, and else the whole stack is in LDS."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tris,lds,refused", [(12, 8, True), (12, 16, True), (12, 32, False), (16000, 32, False),
                                              (40000, 32, True), (12, 0, False), (40000, 0, False)])
def test_partial_stacks(rt, gpu_ctx, tris, lds, refused):
    sc = gpu_ctx.upload(rt.scene_clusters(tris, 5))
    rays = rt.rays_to_device(rt.rays_box(5000, 6, 4.0))
    want = gpu_ctx.closest_hit(sc, rays)
    hits = torch.full((5000, 4), -3.0, device="cuda")
    p = rt.QueryParams(0, 0, 0, 0)
    print(f"case: noalloc query, {tris} triangles, stack_lds {lds}", flush=True)
    gpu_ctx.set_tuning(stack_lds=lds)
    try:
        rc = rt.lib().rt_closest_hit_noalloc(gpu_ctx._h, sc.handle, rt._dev_ptr(rays), 5000, rt._dev_ptr(hits),
                                             ctypes.byref(p), None)
    finally:
        gpu_ctx.set_tuning()
    torch.cuda.synchronize()
    assert rc == (rt.RT_ERR_UNSUPPORTED if refused else rt.RT_OK)
    assert bool((hits == -3.0).all()) if refused else torch.equal(hits.view(torch.int32), want.view(torch.int32))
    sc.release()
