"""Uploads pack ordinary scenes on the device and leave the others to the host
packer.  A context whose layout needs binary records always packs on the
host, so both ways are compared: the same scene facts, the same hits; and
what the device declines or the host rejects ends as it did."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def scene(rt, n, seed):
    hs = rt.scene_soup(max(n, 4), seed)
    t = hs.triangles[:n].copy()
    return rt.HostScene(t, hs.materials, rt.bvh_build(t, seed=seed) if n else None, rt.scene_lights(t, hs.materials))


def chain(rt, n, seed):
    """A tree as deep as it has leaves: inner node k holds leaf k and the rest."""
    hs = scene(rt, n, seed)
    t = hs.triangles
    v = np.stack([t["v0"], t["v1"], t["v2"]])
    lo, hi = v.min(0) - np.float32(1e-4), v.max(0) + np.float32(1e-4)
    nd = np.zeros(2 * n - 1, rt.NODE_DT)
    nd["left"] = nd["right"] = nd["object"] = -1
    for k in range(n):
        leaf = 2 * k if k == n - 1 else 2 * k + 1
        nd["object"][leaf], nd["min"][leaf], nd["max"][leaf] = k, lo[k], hi[k]
        if k < n - 1:
            nd["left"][2 * k], nd["right"][2 * k] = 2 * k + 1, 2 * k + 2
            nd["min"][2 * k], nd["max"][2 * k] = lo[k:].min(0), hi[k:].max(0)
    return rt.HostScene(t, hs.materials, nd, hs.lights)


def variant(rt, kind):
    hs = scene(rt, 500, 3)
    n = hs.nodes
    if kind == "unreached":                       # a subtree cut off: its nodes stay in the array
        inner = np.nonzero(n["object"] < 0)[0][5]
        leaf = np.nonzero(n["object"] >= 0)[0][0]
        n["left"][inner] = -1
        n["right"][inner] = -1
        n["object"][inner] = n["object"][leaf]
        t = hs.triangles[n["object"][leaf]]
        v = np.stack([t["v0"], t["v1"], t["v2"]])
        n["min"][inner] = np.minimum(n["min"][inner], v.min(0) - np.float32(1e-3))
        n["max"][inner] = np.maximum(n["max"][inner], v.max(0) + np.float32(1e-3))
        n["min"][:] = np.where((n["object"] < 0)[:, None], np.float32(-4), n["min"])
        n["max"][:] = np.where((n["object"] < 0)[:, None], np.float32(4), n["max"])
    elif kind == "one_child":                     # an inner node with a single child
        inner = np.nonzero(n["object"] < 0)[0][7]
        n["right"][inner] = -1
    elif kind == "loose":                         # a leaf box that does not hold its triangle
        leaf = np.nonzero(n["object"] >= 0)[0][9]
        n["max"][leaf] = n["min"][leaf]
    elif kind == "twice":                         # one triangle under two leaves, in a box that holds both
        a, b = np.nonzero(n["object"] >= 0)[0][[3, 4]]
        n["object"][b] = n["object"][a]
        n["min"][:], n["max"][:] = np.minimum(n["min"], -4), np.maximum(n["max"], 4)
    return hs


def facts(rt, sc):
    info = rt.SceneInfo()
    assert rt.lib().rt_scene_info_get(sc.handle, ctypes.byref(info)) == rt.RT_OK
    return {k: getattr(info, k) for k, _ in info._fields_ if k != "device_bytes"}


def both(rt, ctx, hs, rays):
    dev = rt.rays_to_device(rays)
    out = []
    for layout in (rt.LAYOUT_AUTO, rt.LAYOUT_F32):            # the upload's layout; both queries read 4-wide records
        ctx.set_tuning(node_layout=layout)
        try:
            sc = ctx.upload(hs)
        finally:
            ctx.set_tuning()
        out.append((facts(rt, sc), rt.hits_from_device(ctx.closest_hit(sc, dev))))
        sc.release()
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 63, 257, 4097, 20000])
def test_device_and_host_packing_agree(rt, gpu_ctx, n):
    hs = scene(rt, n, 11 + n)
    rays = rt.rays_box(5000, n, 1.0)
    print(f"case: {n} triangles packed on the device and on the host", flush=True)
    (fa, a), (fb, b) = both(rt, gpu_ctx, hs, rays)
    assert fa == fb and fa["reachable_leaves"] == n and fa["enclosing"] == 1
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("n", [2, 7, 30, 60, 64, 66, 140, 300])
def test_deep_trees(rt, gpu_ctx, n):
    """Chains: up to 64 levels take the packed traversal, deeper ones the
    shader's order, past 128 levels the device packer gives up first."""
    hs = chain(rt, n, 5)
    rays = rt.rays_box(3000, n, 1.0)
    print(f"case: chain of {n} leaves", flush=True)
    dev = rt.rays_to_device(rays)
    sc = gpu_ctx.upload(hs)
    assert facts(rt, sc)["tree_height"] == n - 1
    assert facts(rt, sc)["fast_path"] == (1 if n - 1 <= 64 else 0)
    want = rt.hits_from_device(gpu_ctx.closest_hit(sc, dev, traversal=rt.TRAVERSE_REFERENCE))
    try:
        got = rt.hits_from_device(gpu_ctx.closest_hit(sc, dev))
    except rt.RtError as e:                       # the caller's tree needs more stack than a kernel holds
        assert e.status == rt.RT_ERR_UNSUPPORTED and 3 * ((n - 2) // 2 + 1) + 1 > 96
    else:
        assert np.array_equal(got["t"].view(np.uint32), want["t"].view(np.uint32))
    sc.release()


@pytest.mark.parametrize("kind", ["unreached", "one_child", "loose", "twice"])
def test_trees_left_to_the_host(rt, gpu_ctx, kind):
    hs = variant(rt, kind)
    rays = rt.rays_box(4000, 2, 1.0)
    print(f"case: {kind}", flush=True)
    (fa, a), (fb, b) = both(rt, gpu_ctx, hs, rays)
    assert fa == fb
    status, info, _ = rt.scene_check(hs)
    assert status == rt.RT_OK and fa["fast_path"] == info.fast_path and fa["reachable_leaves"] == info.reachable_leaves
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("field,at,value", [("left", 3, 10 ** 6), ("right", 0, 0), ("object", 900, 10 ** 6),
                                            ("left", 0, 7), ("material", 5, 99)])
def test_invalid_scenes_keep_their_message(rt, gpu_ctx, field, at, value):
    hs = scene(rt, 500, 3)
    if field == "material":
        hs.triangles["materialIndex"][at] = value
    else:
        hs.nodes[field][at] = value
    status, _, reason = rt.scene_check(hs)
    print(f"case: {field}[{at}] = {value}: {reason}", flush=True)
    assert status == rt.RT_ERR_INVALID
    with pytest.raises(rt.RtError) as e:
        gpu_ctx.upload(hs)
    assert e.value.status == rt.RT_ERR_INVALID and reason in str(e.value)
