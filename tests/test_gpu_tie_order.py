"""Which of several hits at exactly equal t a query reports: the first one
that an ordered traversal of the caller's own tree, collapsed two levels at a
time into records of up to four children with 16-bit boxes, meets.  The
library walks another tree and settles ties afterwards (rt_trace_dev.hpp), so
the order is restated here from the caller's node array: frame, quantized
boxes, entry distances in binary32, the five-comparator sort, depth first.
On the tie grid the triangle test is exact, so ids must be equal."""
import numpy as np
import pytest
import torch

from test_gpu_query import tie_grid, tie_rays

pytestmark = pytest.mark.gpu
f32 = np.float32


class FourWide:
    def __init__(self, nodes, tris):
        self.tris = tris
        n = nodes
        inner = n["object"] < 0
        boxes = np.concatenate([np.concatenate([n["min"][k], n["max"][k]])[None] for k in
                                np.concatenate([n["left"][inner], n["right"][inner]])]).astype(np.float64)
        lo, hi = boxes[:, :3].min(0), boxes[:, 3:].max(0)
        self.scl, self.org = np.zeros(3), np.zeros(3)
        for a in range(3):
            ext = max(hi[a] - lo[a], 1e-30)
            s = f32(ext / 65000.0)
            if float(s) * 65000.0 < ext:
                s = np.nextafter(s, f32(np.inf))
            o = f32(lo[a] - 2.0 * float(s))
            if float(o) > lo[a] - 2.0 * float(s):
                o = np.nextafter(o, f32(-np.inf))
            self.scl[a], self.org[a] = float(s), float(o)
        self.n = n
        q = (n["min"].astype(np.float64) - self.org) / self.scl
        self.qlo = np.clip(np.floor(q) - 1.0, 0.0, 65535.0)
        q = (n["max"].astype(np.float64) - self.org) / self.scl
        self.qhi = np.clip(np.ceil(q) + 1.0, 0.0, 65535.0)

    def children(self, i):
        out = []
        for c in (self.n["left"][i], self.n["right"][i]):
            if self.n["object"][c] >= 0:
                out.append(c)
            else:
                out += [self.n["left"][c], self.n["right"][c]]
        return out

    def trace(self, o, d, tmin, tmax):
        tiny = f32(2.0 ** -80)              # a zero component's reciprocal stays finite
        inv = (f32(1.0) / np.where(np.abs(d) < tiny, np.copysign(tiny, d), d) * self.scl.astype(f32)).astype(f32)
        bo = (o.astype(np.float64) - self.org) / self.scl
        c = (-(2.0 ** 23 + bo) * inv.astype(np.float64)).astype(f32)
        best, best_t = -1, float(tmax)
        stack = [0]
        while stack:
            i = stack.pop()
            if self.n["object"][i] >= 0:
                t = self.meet(self.tris[self.n["object"][i]], o, d, tmin)
                if t is not None and t < best_t:
                    best, best_t = int(self.n["object"][i]), t
                continue
            kids = self.children(i)
            key, ref = [np.inf] * 4, kids + [-1] * (4 - len(kids))
            for k, ch in enumerate(kids):
                plo = ((2.0 ** 23 + self.qlo[ch]) * inv.astype(np.float64) + c).astype(f32)
                phi = ((2.0 ** 23 + self.qhi[ch]) * inv.astype(np.float64) + c).astype(f32)
                near = max(np.where(np.signbit(inv), phi, plo).max(), f32(tmin))
                far = min(np.where(np.signbit(inv), plo, phi).min(), f32(best_t))
                if f32(float(near) - abs(float(near)) * 2.0 ** -15) <= far:
                    key[k] = float(near)
            hits = sum(k < np.inf for k in key)
            for a, b in ((0, 1), (2, 3), (0, 2), (1, 3), (1, 2)):
                if key[b] < key[a]:
                    key[a], key[b], ref[a], ref[b] = key[b], key[a], ref[b], ref[a]
            stack += [ref[k] for k in range(hits - 1, -1, -1)]
        return best

    def meet(self, tr, o, d, tmin):
        v0, v1, v2 = (tr[k].astype(np.float64) for k in ("v0", "v1", "v2"))
        o, d = o.astype(np.float64), d.astype(np.float64)
        a, b, p = v0 - v1, v2 - v0, v0 - o
        n, q = np.cross(b, a), np.cross(p, d)
        det = d @ n
        u, v, t = q @ b / det, q @ a / det, n @ p / det
        return t if u >= 0 and u <= 1 and v >= 0 and u + v <= 1 and t > tmin else None


def grid_scene(rt, n, layers, copies):
    tris = np.concatenate([tie_grid(rt, n=n, layers=layers)] * copies)
    return rt.HostScene(tris, np.zeros(1, rt.MAT_DT), rt.bvh_build(tris, seed=1))


def grid_rays(rt, n, count, seed):
    if n > 2:
        return tie_rays(rt, count, n=n, seed=seed)
    rng = np.random.default_rng(seed)       # a grid without inner vertices: its border and diagonals
    r = np.zeros(count, rt.RAY_DT)
    o = np.stack([rng.integers(0, 8 * n, count) / 8.0, rng.integers(0, 8 * n, count) / 8.0, np.full(count, 4.0)], 1)
    to = np.stack([rng.integers(0, 4 * n + 1, count) / 4.0, rng.integers(0, 4 * n + 1, count) / 4.0,
                   np.zeros(count)], 1)
    r["o"], r["d"], r["tmin"], r["tmax"] = o, to - o, 0.001, 10000.0
    return r


# triangles: 2, 4, 6, 16, 54, 324, 9600: one record, a few levels, many; `copies` makes every hit a tie
@pytest.mark.parametrize("n,layers,copies", [(1, 1, 1), (1, 1, 2), (1, 3, 1), (2, 1, 2), (3, 3, 1), (9, 2, 1), (40, 3, 1)])
def test_equal_t_is_settled_by_the_callers_tree(rt, gpu_ctx, n, layers, copies):
    hs = grid_scene(rt, n, layers, copies)
    scene = gpu_ctx.upload(hs)
    rays = grid_rays(rt, n, 600, 51 + n)
    model = FourWide(hs.nodes, hs.triangles)
    want = np.array([model.trace(r["o"], r["d"], float(r["tmin"]), float(r["tmax"])) for r in rays])
    dev = rt.rays_to_device(rays)
    print(f"case: tie order, {len(hs.triangles)} triangles, {len(rays)} rays", flush=True)
    for steal in (0, 1, rt.STEAL_NEVER):
        gpu_ctx.set_tuning(steal=steal)
        try:
            got = rt.hits_from_device(gpu_ctx.closest_hit(scene, dev))
        finally:
            gpu_ctx.set_tuning()
        assert np.array_equal(got["id"], want), (steal, np.nonzero(got["id"] != want)[0][:8])
    out = torch.full((len(rays), 4), -7.0, device="cuda")
    b = rt.Batch(gpu_ctx, [(scene, dev, out)])
    b.launch()
    assert np.array_equal(rt.hits_from_device(out)["id"], want)
    b.destroy()
    scene.release()
