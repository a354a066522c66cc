"""The server's batches read rays from and write hits to the callers' memory
in kernels: page-locked buffers in place, at any offset inside their
allocation, pageable ones by way of staging, and buffers that are not aligned
to 8 bytes by copies.  Requests that share a run of 64 rays, end inside one or
span several must each get their own hits and nothing beside them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = ["pinned", "inner", "pageable", "odd"]


def buffer(rt, kind, n, dt):
    """(array of n, what surrounds it)"""
    size = n * dt.itemsize
    if kind == "pageable":
        return np.zeros(n, dt), None
    pad = {"pinned": 0, "inner": 32, "odd": 4}[kind]
    raw = rt.pinned_array((size + 2 * pad,), np.uint8)
    raw[:] = 0xA5
    return raw[pad:pad + size].view(dt), (raw, pad)


@pytest.mark.parametrize("counts", [[1] * 150, [63, 64, 65, 1, 128, 4095, 2, 300], [1, 40001, 7]],
                         ids=["ones", "edges", "long"])
@pytest.mark.parametrize("kinds", [[k] for k in KINDS] + [KINDS], ids=KINDS + ["mixed"])
def test_each_request_gets_its_hits(rt, gpu_ctx, counts, kinds):
    print(f"case: {len(counts)} requests, {kinds}", flush=True)
    hs = [rt.scene_soup(700, 3), rt.scene_clusters(5000, 4)]
    srv = rt.Server(gpu_ctx, slots=2, max_batch_rays=1 << 16, max_render_pixels=64 * 64)
    try:
        ids = [srv.add_scene(h) for h in hs]
        alone = [gpu_ctx.upload(h) for h in hs]
        reqs = []
        for k, n in enumerate(counts):
            kind = kinds[k % len(kinds)]
            rays, _ = buffer(rt, kind, n, np.dtype(rt.RAY_DT))
            hits, around = buffer(rt, kind, n, np.dtype(rt.HIT_DT))
            reqs.append((k % 2, rays, hits, around))
        for turn in range(3):
            for k, (_, rays, hits, _) in enumerate(reqs):
                rays[:] = rt.rays_box(len(rays), 900 + k + 1000 * turn, 2.0)
            rids = [srv.submit_query(ids[s], rays, hits) for s, rays, hits, _ in reqs]
            for r in rids:
                assert srv.wait(r, 60000) == rt.RT_OK
            for s, rays, hits, around in reqs:
                ref = rt.hits_from_device(gpu_ctx.closest_hit(alone[s], rt.rays_to_device(np.array(rays))))
                assert np.array_equal(hits.copy().view(np.uint32), ref.view(np.uint32))
                if around is not None:
                    raw, pad = around
                    assert (raw[:pad] == 0xA5).all() and (raw[raw.size - pad:] == 0xA5).all()
                hits[:] = 0
    finally:
        srv.close()
