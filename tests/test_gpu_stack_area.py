"""Traversal stacks deeper than their part in LDS: the entries past it live in
an area of the context made on first use.  Hits must not depend on how many
entries are in LDS, and a query captured into a graph by a context that has
no such area yet must run without one."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def overlapping(rt, n, seed):
    """Long thin triangles through one another: every box of a node overlaps
    the others, so rays defer nearly all children and stacks fill up."""
    rng = np.random.default_rng(seed)
    t = np.zeros(n, rt.TRI_DT)
    c = rng.uniform(-1, 1, (n, 3))
    for k, s in (("v0", 0.8), ("v1", 0.8), ("v2", 0.002)):
        t[k] = c + rng.uniform(-s, s, (n, 3))
    return rt.HostScene(t, np.zeros(1, rt.MAT_DT), rt.bvh_build(t, seed=1))


@pytest.mark.parametrize("tris", [3000, 40000])
def test_hits_do_not_depend_on_the_stack_in_lds(rt, gpu_ctx, tris):
    hs = overlapping(rt, tris, 5)
    scene = gpu_ctx.upload(hs)
    rays = rt.rays_to_device(rt.rays_box(20001, 8, 1.5))
    print(f"case: stacks in LDS 8, 16, 32, default; {tris} overlapping triangles", flush=True)
    ref = rt.hits_from_device(gpu_ctx.closest_hit(scene, rays, traversal=rt.TRAVERSE_PACKED))
    binary = None
    for kw in (dict(stack_lds=8), dict(stack_lds=16), dict(stack_lds=32), dict(stack_lds=8, steal=1),
               dict(stack_lds=8, steal=rt.STEAL_NEVER), dict(node_layout=rt.LAYOUT_Q16)):
        gpu_ctx.set_tuning(**kw)
        try:
            got = rt.hits_from_device(gpu_ctx.closest_hit(scene, rays))
        finally:
            gpu_ctx.set_tuning()
        if "node_layout" in kw:
            binary = got
            continue
        assert np.array_equal(got.view(np.uint8), ref.view(np.uint8)), kw
    assert np.array_equal(binary["t"].view(np.uint32), ref["t"].view(np.uint32))
    scene.release()


def test_captured_query_before_the_area_exists(rt):
    ctx = rt.Context(0)
    scene = ctx.upload(rt.scene_clusters(150000, 6))
    rays = rt.rays_to_device(rt.rays_box(400001, 9, 4.0))
    hits = torch.full((400001, 4), -7.0, device="cuda")
    print("case: query of 400,001 rays captured by a new context", flush=True)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ctx.closest_hit(scene, rays, hits)
    other = rt.Context(0)
    want = rt.hits_from_device(other.closest_hit(scene, rays))
    for _ in range(3):
        hits.fill_(-7.0)
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(rt.hits_from_device(hits).view(np.uint8), want.view(np.uint8))
        other.closest_hit(scene, rays)
    del g
    scene.release()
    ctx.close()
    other.close()
