"""The HBM budget counts what scenes need: traversal trees take what it has to
spare and are given up before a scene is refused or evicted."""
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bytes_without_tree(rt, hs):
    """The caller's arrays, triangle ids, 4-wide records (one for each inner
    node at even depth) and packed triangles."""
    n = hs.nodes
    level, depth, records = np.array([0]), 0, 0
    while len(level):
        inner = level[n["object"][level] < 0]
        records += len(inner) if depth % 2 == 0 else 0
        level = np.concatenate([n["left"][inner], n["right"][inner]])
        depth += 1
    t = len(hs.triangles)
    arrays = 48 * t + 32 * len(hs.materials) + 48 * len(n) + 8 * len(hs.lights) + 32 * len(hs.spheres)
    return arrays + 4 * t + (64 * records + 255) // 256 * 256 + 48 * t


def check(rt, srv, sid, rays, want):
    hits = np.zeros(len(rays), rt.HIT_DT)
    assert srv.wait(srv.submit_query(sid, rays, hits)) == rt.RT_OK
    assert np.array_equal(hits.view(np.uint8), want.view(np.uint8))


def test_trees_go_before_scenes(rt, gpu_ctx):
    sizes = [60000, 3000, 200000, 15001]
    hosts = [rt.scene_clusters(n, 40 + i) for i, n in enumerate(sizes)]
    rays = rt.rays_box(20000, 3, 4.0)
    dev = rt.rays_to_device(rays)
    want, full = [], []
    for h in hosts:
        s = gpu_ctx.upload(h)
        full.append(s.info.device_bytes)
        want.append(rt.hits_from_device(gpu_ctx.closest_hit(s, dev)))
        s.release()
    bare = [bytes_without_tree(rt, h) for h in hosts]
    assert all(b < f for b, f in zip(bare, full))
    print(f"case: budget of {sum(bare)} bytes, scenes of {sum(full)} with their trees", flush=True)
    srv = rt.Server(gpu_ctx, slots=2, hbm_budget=sum(bare))
    ids = []
    for k, h in enumerate(hosts):
        ids.append(srv.add_scene(h))
        st = srv.stats()
        assert st.scenes_evicted == 0 and st.resident_bytes <= sum(bare)
        if k == 0:
            assert st.resident_bytes == full[0]          # room to spare: with its tree
        for i in range(k + 1):
            check(rt, srv, ids[i], rays, want[i])
    assert srv.stats().resident_bytes == sum(bare)
    # one more: the least recently used goes, as it always has
    again = srv.add_scene(hosts[0])
    assert sorted(srv.scenes()) == sorted(ids[1:] + [again]) and srv.stats().scenes_evicted == 1
    check(rt, srv, again, rays, want[0])
    srv.close()
    # room for one scene without its tree
    srv = rt.Server(gpu_ctx, slots=1, hbm_budget=bare[2])
    check(rt, srv, srv.add_scene(hosts[2]), rays, want[2])
    srv.close()


def test_trees_are_given_up_under_load(rt, gpu_ctx):
    """Queries of the scene that loses its tree run all the while."""
    hosts = [rt.scene_clusters(150000, 50), rt.scene_clusters(100000, 51)]
    rays = rt.rays_box(30000, 3, 4.0)
    s = gpu_ctx.upload(hosts[0])
    want = rt.hits_from_device(gpu_ctx.closest_hit(s, rt.rays_to_device(rays)))
    s.release()
    budget = sum(bytes_without_tree(rt, h) for h in hosts)
    srv = rt.Server(gpu_ctx, slots=4, hbm_budget=budget)
    first = srv.add_scene(hosts[0])
    stop, failed, done = threading.Event(), [], []
    print("case: a tree given up while its scene is queried", flush=True)

    def load():
        hits = np.zeros(len(rays), rt.HIT_DT)
        while not stop.is_set() and not failed:
            hits[:] = np.zeros(1, rt.HIT_DT)
            try:
                check_hits = srv.wait(srv.submit_query(first, rays, hits)) == rt.RT_OK and \
                    np.array_equal(hits.view(np.uint8), want.view(np.uint8))
            except rt.RtError as e:
                check_hits = str(e)
            if check_hits is not True:
                failed.append((len(done), check_hits))
            done.append(1)

    def until(count):
        while len(done) < count and not failed:
            time.sleep(0.001)

    threads = [threading.Thread(target=load) for _ in range(4)]
    for t in threads:
        t.start()
    until(20)
    second = srv.add_scene(hosts[1])
    until(len(done) + 20)
    stop.set()
    for t in threads:
        t.join()
    assert not failed, failed
    assert sorted(srv.scenes()) == sorted([first, second]) and srv.stats().scenes_evicted == 0
    assert srv.stats().resident_bytes <= budget
    srv.close()
