"""Servers of one context take scenes from several threads, beside the
context's own uploads: every scene's hits are those of the scene alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_uploads_of_one_context_from_several_threads(rt):
    sizes = [3000, 70000, 900, 200000, 20000, 1500, 120000, 5000]
    hosts = [rt.scene_clusters(n, 70 + i) for i, n in enumerate(sizes)]
    rays = rt.rays_box(20000, 8, 4.0)
    dev = rt.rays_to_device(rays)
    alone = rt.Context(0)
    want = []
    for h in hosts:
        s = alone.upload(h)
        want.append(rt.hits_from_device(alone.closest_hit(s, dev)))
        s.release()
    ctx = rt.Context(0)
    servers = [rt.Server(ctx, slots=1, max_batch_rays=1 << 15) for _ in range(2)]
    ids = [[None] * len(hosts) for _ in servers]
    scenes = [None] * len(hosts)
    print("case: two servers and uploads of one context, three threads", flush=True)

    def serve(k):
        order = range(len(hosts)) if k == 0 else reversed(range(len(hosts)))
        for i in order:
            ids[k][i] = servers[k].add_scene(hosts[i])

    def upload():
        for i in range(len(hosts)):
            scenes[i] = ctx.upload(hosts[(i + 3) % len(hosts)])

    threads = [threading.Thread(target=serve, args=(k,)) for k in range(2)] + [threading.Thread(target=upload)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, srv in enumerate(servers):
        for i in range(len(hosts)):
            hits = np.zeros(len(rays), rt.HIT_DT)
            assert srv.wait(srv.submit_query(ids[k][i], rays, hits)) == rt.RT_OK
            assert np.array_equal(hits.view(np.uint8), want[i].view(np.uint8)), (k, i)
    for i, s in enumerate(scenes):
        got = rt.hits_from_device(ctx.closest_hit(s, dev))
        assert np.array_equal(got.view(np.uint8), want[(i + 3) % len(hosts)].view(np.uint8)), i
        s.release()
    for srv in servers:
        srv.close()
    ctx.close()
    alone.close()
