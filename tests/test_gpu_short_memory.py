"""Calls while the device's memory is all but used up: what is only there for
speed (stack areas, the traversal tree) is done without, and the call succeeds."""
import contextlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@contextlib.contextmanager
def memory_left(mib):
    """All device memory taken but about `mib` MiB."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held = []
    for step in (1 << 36, 1 << 33, 1 << 30):
        while torch.cuda.mem_get_info()[0] >= step + mib * MIB:
            held.append(torch.empty(step, dtype=torch.uint8, device="cuda"))
    rest = (torch.cuda.mem_get_info()[0] // MIB - mib) & ~1
    if rest >= 10:                       # smaller tensors share a block of 20 MiB
        held.append(torch.empty(rest * MIB, dtype=torch.uint8, device="cuda"))
    try:
        yield
    finally:
        torch.cuda.synchronize()
        held.clear()
        torch.cuda.empty_cache()


def test_queries_without_room_for_a_stack_area(rt):
    """The smallest area takes 32 MiB, the batch's 35."""
    hs = rt.scene_clusters(600000, 12)
    n = 1 << 20
    rays_host = rt.rays_box(n, 9, 4.0)
    other = rt.Context(0)
    sc = other.upload(hs)
    rays = rt.rays_to_device(rays_host)
    want = rt.hits_from_device(other.closest_hit(sc, rays))
    ctx = rt.Context(0)
    scene = ctx.upload(hs)
    srv = rt.Server(ctx, slots=1, max_batch_rays=1 << 18)
    sid = srv.add_scene(hs)
    hits = torch.full((n, 4), -7.0, device="cuda")
    bhits = torch.full((n, 4), -7.0, device="cuda")
    pin_rays, pin_hits = rt.pinned_array(1 << 18, rt.RAY_DT), rt.pinned_array(1 << 18, rt.HIT_DT)
    pin_rays[:] = rays_host[:1 << 18]
    # (the batch's tables, and a first area of few blocks; the larger one finds no room)
    batch = rt.Batch(ctx, [(scene, rays, bhits)], rt.batch_config(blocks_per_cu=1, use_graph=0))
    print("case: plain, batched and served query of a new context with 24 MiB left", flush=True)
    with memory_left(24):
        ctx.closest_hit(scene, rays, hits)
        torch.cuda.synchronize()
        batch.set_config(rt.batch_config(stack_lds=8))
        batch.launch()
        torch.cuda.synchronize()
        status = srv.wait(srv.submit_query(sid, pin_rays, pin_hits))
    assert np.array_equal(rt.hits_from_device(hits).view(np.uint8), want.view(np.uint8))
    assert np.array_equal(rt.hits_from_device(bhits).view(np.uint8), want.view(np.uint8))
    assert status == rt.RT_OK
    assert np.array_equal(np.ascontiguousarray(pin_hits).view(np.uint8), want[:1 << 18].view(np.uint8))
    srv.close()
    batch.destroy()
    scene.release()
    sc.release()
    ctx.close()
    other.close()


def hits_of(rt, ctx, host, rays):
    scene = ctx.upload(host)
    out = rt.hits_from_device(ctx.closest_hit(scene, rays))
    scene.release()
    return out


# 262,144 triangles: scratch of 103 MiB that the context keeps, a scene of 63;
# 1,048,576: 350 MiB given back after the upload, a scene of 250
@pytest.mark.parametrize("tris,left", [(262144, 112), (1048576, 460)])
def test_upload_without_room_for_its_scratch_and_the_scene(rt, tris, left):
    hs = rt.scene_clusters(tris, 12)
    rays = rt.rays_to_device(rt.rays_box(5000, 9, 4.0))
    other = rt.Context(0)
    want = hits_of(rt, other, hs, rays)
    other.close()
    ctx = rt.Context(0)
    print(f"case: upload of {tris} triangles with {left} MiB left", flush=True)
    with memory_left(left):
        scene = ctx.upload(hs)
    got = rt.hits_from_device(ctx.closest_hit(scene, rays))
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    scene.release()
    ctx.close()


def test_server_frees_scratch_before_scenes(rt):
    """Adding a scene of about 60 MiB with 200 left, half of which its scratch takes:
    no idle scene need go."""
    hosts = [rt.scene_clusters(20000, 1), rt.scene_clusters(262144, 2)]
    ctx = rt.Context(0)
    srv = rt.Server(ctx, slots=1, max_batch_rays=1 << 16, max_render_pixels=1 << 16)
    first = srv.add_scene(hosts[0])
    print("case: server addition with 200 MiB left", flush=True)
    with memory_left(200):
        second = srv.add_scene(hosts[1])
        assert sorted(srv.scenes()) == sorted([first, second])
        assert srv.stats().scenes_evicted == 0
    rays = rt.rays_box(5000, 9, 4.0)
    hits = np.zeros(5000, rt.HIT_DT)
    assert srv.wait(srv.submit_query(second, rays, hits)) == rt.RT_OK
    want = hits_of(rt, ctx, hosts[1], rt.rays_to_device(rays))
    assert np.array_equal(hits.view(np.uint8), want.view(np.uint8))
    srv.close()
    ctx.close()
