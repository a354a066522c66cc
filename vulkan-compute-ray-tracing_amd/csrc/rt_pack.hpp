// rt_pack.hpp -- an upload's packing on the device: the caller's arrays are
// copied as they are, and kernels validate them, walk the tree, and write
// the 4-wide records, packed triangles and leaf boxes that rt_wide.hpp builds
// from.  Part of rt_build.hip.
//
// It covers the ordinary scene: indices in range, a tree in which every
// reachable node is a leaf without children or has two, boxes that enclose
// their subtrees, and a traversal tree that beats the caller's.  Anything
// else -- an error to be named among them -- is left to the host packer,
// which sees the arrays as if nothing had been tried.  The results are the
// host packer's bit for bit, but for the order of the records and of the
// triangles, which follow the node array here.
//
// Uploading 262,144 triangles took 38 ms with the host packer (one thread
// walking the tree four times, then two copies of everything it made); the
// kernels take under 1 ms, and the copies of the caller's arrays the rest.
#pragma once

#include <cstring>

#include "rt_math.hpp"
#include "rt_wide.hpp"

#pragma clang fp contract(off)

namespace rtamd {
namespace {

constexpr uint32_t kUnreached = 0xffffffffu;

struct PackFacts {
    uint32_t bad;                 // left to the host packer
    uint32_t lo[3], hi[3];        // bounds of the boxes below the root (order_bits)
};

// Finite floats as unsigned integers in the same order.
__device__ __forceinline__ uint32_t order_bits(float x) {
    const uint32_t b = __float_as_uint(x);
    return b >> 31 ? ~b : b | 0x80000000u;
}

__global__ void k_pack_init(PackFacts* facts, uint32_t* level_count, uint32_t* list, uint32_t* depth, double* cost) {
    const uint32_t t = threadIdx.x;
    if (t < kMaxLevels + 1) level_count[t] = t == 0 ? 1u : 0u;
    if (t == 0) {
        facts->bad = 0u;
        list[0] = 0u;
        depth[0] = 0u;
        cost[1] = 0.0;
    }
    if (t < 3) {
        facts->lo[t] = 0xffffffffu;
        facts->hi[t] = 0u;
    }
}

// Index ranges of every triangle and node (check_scene's tests).
__global__ __launch_bounds__(256) void k_pack_ranges(const rt_triangle* __restrict__ tris, uint32_t nt, uint32_t nmat,
                                                     const rt_bvh_node* __restrict__ nodes, uint32_t m,
                                                     PackFacts* __restrict__ facts) {
    bool bad = false;
    const uint32_t stride = gridDim.x * blockDim.x, g = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t i = g; i < nt; i += stride) bad = bad || tris[i].materialIndex >= nmat;
    for (uint32_t i = g; i < m; i += stride) {
        const int32_t l = nodes[i].leftNodeIndex, r = nodes[i].rightNodeIndex, o = nodes[i].objectIndex;
        bad = bad || l < -1 || l >= (int32_t)m || r < -1 || r >= (int32_t)m || o < -1 || o >= (int32_t)nt;
    }
    if (bad) facts->bad = 1u;
}

__device__ __forceinline__ bool finite3(const float* v) { return isfinite(v[0]) && isfinite(v[1]) && isfinite(v[2]); }

// Nodes of depth `level`: the tests of check_scene's walk, and their children
// onto the next level's list.  Reading stops once anything is bad.
__global__ __launch_bounds__(256) void k_pack_level(const rt_triangle* __restrict__ tris,
                                                    const rt_bvh_node* __restrict__ nodes, uint32_t level,
                                                    uint32_t* __restrict__ list, uint32_t* __restrict__ level_count,
                                                    uint32_t* __restrict__ depth, PackFacts* __restrict__ facts) {
    if (facts->bad) return;
    uint32_t begin = 0;
    for (uint32_t l = 0; l < level; ++l) begin += level_count[l];
    const uint32_t count = level_count[level], next = begin + count;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t rounds = (count + 63u) / 64u, waves = gridDim.x * (blockDim.x / 64u);
    for (uint32_t w = blockIdx.x * (blockDim.x / 64u) + threadIdx.x / 64u; w < rounds; w += waves) {
        const uint32_t q = w * 64u + lane;
        bool bad = false, inner = false;
        int32_t l = -1, r = -1;
        if (q < count) {
            const rt_bvh_node n = nodes[list[begin + q]];
            l = n.leftNodeIndex;
            r = n.rightNodeIndex;
            if (n.objectIndex != -1) {
                bad = l != -1 || r != -1;
                const rt_triangle& t = tris[n.objectIndex];
                bad = bad || !finite3(n.min) || !finite3(n.max) || !finite3(t.v0) || !finite3(t.v1) || !finite3(t.v2);
                for (int k = 0; k < 3; ++k) {
                    const float lo = fminf(fminf(t.v0[k], t.v1[k]), t.v2[k]);
                    const float hi = fmaxf(fmaxf(t.v0[k], t.v1[k]), t.v2[k]);
                    bad = bad || !(n.min[k] < lo) || !(hi < n.max[k]);
                }
            } else {
                inner = l != -1 && r != -1;
                bad = !inner;
                if (inner) {
                    for (int32_t c : {l, r}) {
                        const rt_bvh_node& k = nodes[c];
                        bad = bad || !finite3(n.min) || !finite3(n.max) || !finite3(k.min) || !finite3(k.max);
                        for (int a = 0; a < 3; ++a) bad = bad || !(n.min[a] <= k.min[a]) || !(k.max[a] <= n.max[a]);
                        // a node reached twice is no tree
                        if (atomicExch(&depth[c], level + 1u) != kUnreached) bad = true;
                    }
                }
            }
        }
        if (__ballot(bad)) {
            if (lane == 0) facts->bad = 1u;
            return;
        }
        const uint64_t mask = __ballot(inner);
        if (mask == 0) continue;
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&level_count[level + 1u], 2u * (uint32_t)__popcll(mask));
        base = next + __builtin_amdgcn_readfirstlane(base) + 2u * (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
        if (inner) {
            list[base] = (uint32_t)l;
            list[base + 1u] = (uint32_t)r;
        }
    }
}

// Bounds of the boxes below the root, and each node's part in the output: a
// leaf (1) or an inner node at even depth, which becomes a record (1 << 32).
__global__ __launch_bounds__(256) void k_pack_bounds(const rt_bvh_node* __restrict__ nodes, uint32_t m,
                                                     const uint32_t* __restrict__ depth, uint64_t* __restrict__ part,
                                                     PackFacts* __restrict__ facts) {
    uint32_t lo[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, hi[3] = {0u, 0u, 0u};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) {
        uint64_t p = 0;
        if (depth[i] != kUnreached) {
            const rt_bvh_node& n = nodes[i];
            if (i != 0)
                for (int a = 0; a < 3; ++a) {
                    lo[a] = min(lo[a], order_bits(n.min[a]));
                    hi[a] = max(hi[a], order_bits(n.max[a]));
                }
            p = n.objectIndex != -1 ? 1ull : (depth[i] & 1u) == 0 ? 1ull << 32 : 0ull;
        }
        part[i] = p;
    }
    for (int a = 0; a < 3; ++a)
        for (int o = 32; o > 0; o >>= 1) {
            lo[a] = min(lo[a], (uint32_t)__shfl_xor((int)lo[a], o, 64));
            hi[a] = max(hi[a], (uint32_t)__shfl_xor((int)hi[a], o, 64));
        }
    if ((threadIdx.x & 63u) == 0)
        for (int a = 0; a < 3; ++a) {
            // few waves improve on what is there
            if (lo[a] < facts->lo[a]) atomicMin(&facts->lo[a], lo[a]);
            if (hi[a] > facts->hi[a]) atomicMax(&facts->hi[a], hi[a]);
        }
}

// A node's box in the frame: quantize_nodes' double arithmetic.
__device__ __forceinline__ uint4 pack_words(const rt_bvh_node& n, const QFrame& f) {
    const float org[3] = {f.ox, f.oy, f.oz}, scl[3] = {f.sx, f.sy, f.sz};
    uint32_t w[3];
    for (int k = 0; k < 3; ++k) {
        const double lo = floor(((double)n.min[k] - (double)org[k]) / (double)scl[k]) - 1.0;
        const double hi = ceil(((double)n.max[k] - (double)org[k]) / (double)scl[k]) + 1.0;
        w[k] = (uint32_t)fmin(65535.0, fmax(0.0, lo)) | (uint32_t)fmin(65535.0, fmax(0.0, hi)) << 16;
    }
    return make_uint4(w[0], w[1], w[2], 0u);
}

// Leaves: packed triangle, id, box words and sort key.  Inner nodes at even
// depth: the record of their grandchildren and leaf children.
__global__ __launch_bounds__(256) void k_pack_emit(const rt_triangle* __restrict__ tris,
                                                   const rt_bvh_node* __restrict__ nodes, uint32_t m,
                                                   const uint32_t* __restrict__ depth, const uint64_t* __restrict__ rank,
                                                   QFrame f, PTri* __restrict__ ptris, int32_t* __restrict__ ids,
                                                   uint4* __restrict__ words, uint64_t* __restrict__ keys,
                                                   uint32_t* __restrict__ vals, PNode4* __restrict__ given,
                                                   double* __restrict__ cost) {
    double sum = 0.0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) {
        if (depth[i] == kUnreached) continue;
        const rt_bvh_node n = nodes[i];
        if (n.objectIndex != -1) {
            const uint32_t slot = (uint32_t)rank[i];
            const rt_triangle& t = tris[n.objectIndex];
            const f3 v0 = ld3(t.v0), v1 = ld3(t.v1), v2 = ld3(t.v2);
            const f3 e = v0 - v1;        // triIntersect's a
            const f3 g = v2 - v0;        // triIntersect's b
            const f3 c = cross(g, e);
            ptris[slot] = PTri{make_float4(v0.x, v0.y, v0.z, e.x), make_float4(e.y, e.z, g.x, g.y),
                               make_float4(g.z, c.x, c.y, c.z)};
            ids[slot] = n.objectIndex;
            const uint4 w = pack_words(n, f);
            words[slot] = w;
            keys[slot] = wide_key(w);
            vals[slot] = slot;
        } else if ((depth[i] & 1u) == 0) {
            PNode4 out;
            int at = 0;
            auto put = [&](int32_t c) {
                const rt_bvh_node& k = nodes[c];
                const uint4 w = pack_words(k, f);
                out.w[3 * at] = w.x;
                out.w[3 * at + 1] = w.y;
                out.w[3 * at + 2] = w.z;
                if (k.objectIndex != -1) {
                    out.ref[at] = ~(int32_t)(uint32_t)rank[c];
                } else {
                    out.ref[at] = (int32_t)(rank[c] >> 32);
                    sum += (double)box_area(w.x, w.y, w.z, f);
                }
                ++at;
            };
            for (int32_t c : {n.leftNodeIndex, n.rightNodeIndex}) {
                const rt_bvh_node& k = nodes[c];
                if (k.objectIndex != -1) {
                    put(c);
                } else {
                    put(k.leftNodeIndex);
                    put(k.rightNodeIndex);
                }
            }
            for (; at < 4; ++at) {
                out.w[3 * at] = out.w[3 * at + 1] = out.w[3 * at + 2] = 0u;
                out.ref[at] = kNoChild;
            }
            given[(uint32_t)(rank[i] >> 32)] = out;
        }
    }
    block_add(sum, cost);
}

float from_order_bits(uint32_t b) {
    const uint32_t u = b >> 31 ? b & 0x7fffffffu : ~b;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

}  // namespace

// Packs `d` on the device into P (wide, frame, facts, bytes to come).  *done
// stays false, with nothing changed, where the host packer has to do it.
int device_pack(rt_ctx* ctx, const rt_scene_desc& d, PreparedScene& P, bool* done) {
    *done = false;
    const uint32_t nt = d.num_triangles, m = d.num_nodes;
    if (!d.triangles || !d.nodes || nt < 2 || m < 3 || nt > (1u << 30) || m > 0x7fffffffu) return RT_OK;
    hipStream_t s = nullptr;
    const uint32_t n_max = (m + 1u) / 2u;
    std::unique_ptr<WideTree, WideTreeDelete> t(new (std::nothrow) WideTree());
    if (!t) return RT_OK;
    size_t scan_bytes = 0;
    RT_HIP(ctx, rocprim::exclusive_scan(nullptr, scan_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr, (uint64_t)0, m,
                                        rocprim::plus<uint64_t>(), s));
    // the packing's temporaries are done when the tree build starts on the same memory
    WideLayout L;
    L.raw_tris = L.take(sizeof(rt_triangle) * (size_t)nt);
    L.raw_nodes = L.take(sizeof(rt_bvh_node) * (size_t)m);
    // inner nodes at even depth: at most two for each one at odd depth, and the root
    int rc = L.wide(ctx, n_max, (uint32_t)(((uint64_t)2u * n_max) / 3u + 1u), s);
    if (rc) return rc;
    size_t off = L.overlay;
    auto take = [&](size_t b) { const size_t o = off; off += align256(b); return o; };
    const size_t o_depth = take(4 * (size_t)m), o_list = take(4 * (size_t)m), o_part = take(8 * (size_t)m),
                 o_rank = take(8 * (size_t)m), o_scan = take(scan_bytes);
    const size_t total = std::max(off, L.bytes);
    if (!t->allocate(ctx, total)) return RT_OK;
    char* b = t->base;
    rt_triangle* tris = (rt_triangle*)(b + L.raw_tris);
    rt_bvh_node* nodes = (rt_bvh_node*)(b + L.raw_nodes);
    uint32_t *depth = (uint32_t*)(b + o_depth), *list = (uint32_t*)(b + o_list);
    uint64_t *part = (uint64_t*)(b + o_part), *rank = (uint64_t*)(b + o_rank);
    uint32_t* counts = (uint32_t*)(b + L.counts);
    double* cost = (double*)(b + L.cost);
    PackFacts* facts = (PackFacts*)(b + L.facts);
    RT_HIP(ctx, hipMemcpy(tris, d.triangles, sizeof(rt_triangle) * (size_t)nt, hipMemcpyHostToDevice));
    RT_HIP(ctx, hipMemcpy(nodes, d.nodes, sizeof(rt_bvh_node) * (size_t)m, hipMemcpyHostToDevice));
    const dim3 block(256);
    auto grid = [&](uint64_t work, uint32_t per_cu) {
        return dim3((uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((work + 255) / 256, (uint64_t)ctx->num_cus * per_cu)));
    };
    rc = launch_fill_u32(ctx, depth, kUnreached, m, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_pack_init, dim3(1), block, 0, s, facts, counts, list, depth, cost);
    hipLaunchKernelGGL(k_pack_ranges, grid(m, 16), block, 0, s, tris, nt, d.num_materials, nodes, m, facts);
    static_assert(sizeof(PackFacts) <= sizeof(WideProgress::facts), "facts end what is read back");
    WideProgress now{};
    const uint32_t* h = now.counts;
    uint32_t level = 0;
    for (;;) {
        const uint32_t end = std::min(level == 0 ? first_levels(n_max, 1) : level + 2u * kLevelsPerSync, kMaxLevels);
        for (; level < end; ++level)
            hipLaunchKernelGGL(k_pack_level, grid(n_max, 8), block, 0, s, tris, nodes, level, list, counts, depth, facts);
        RT_HIP(ctx, hipGetLastError());
        RT_HIP(ctx, hipMemcpyAsync(&now, counts, sizeof now, hipMemcpyDeviceToHost, s));
        RT_HIP(ctx, hipStreamSynchronize(s));
        const bool bad = reinterpret_cast<const PackFacts*>(now.facts)->bad != 0u;
        if (bad || h[level] != 0) {
            if (bad || level == kMaxLevels) return RT_OK;
            continue;
        }
        break;
    }
    uint64_t reached = 0;
    uint32_t height = 0;                           // depth of the deepest leaf
    for (uint32_t l = 0; l < level && h[l]; ++l) {
        reached += h[l];
        height = l;
    }
    // (unreached nodes are the host packer's business too)
    const uint32_t n = n_max;
    if (reached != m || height == 0) return RT_OK;
    hipLaunchKernelGGL(k_pack_bounds, grid(m, 4), block, 0, s, nodes, m, depth, part, facts);
    RT_HIP(ctx, hipGetLastError());
    RT_HIP(ctx, rocprim::exclusive_scan((void*)(b + o_scan), scan_bytes, part, rank, (uint64_t)0, m,
                                        rocprim::plus<uint64_t>(), s));
    PackFacts hf{};
    uint64_t last[2] = {0, 0};
    RT_HIP(ctx, hipMemcpyAsync(&hf, facts, sizeof hf, hipMemcpyDeviceToHost, s));
    RT_HIP(ctx, hipMemcpyAsync(&last[0], part + (m - 1u), 8, hipMemcpyDeviceToHost, s));
    RT_HIP(ctx, hipMemcpyAsync(&last[1], rank + (m - 1u), 8, hipMemcpyDeviceToHost, s));
    RT_HIP(ctx, hipStreamSynchronize(s));
    const uint64_t counted = last[0] + last[1];
    const uint32_t G = (uint32_t)(counted >> 32);
    if ((uint32_t)counted != n || G == 0 || G > 2u * n_max / 3u + 1u) return RT_OK;
    double lo[3], hi[3];
    for (int k = 0; k < 3; ++k) {
        lo[k] = (double)from_order_bits(hf.lo[k]);
        hi[k] = (double)from_order_bits(hf.hi[k]);
    }
    const QFrame f = quant_frame(lo, hi);
    t->bind(L, n, G);
    hipLaunchKernelGGL(k_pack_emit, grid(m, 8), block, 0, s, tris, nodes, m, depth, rank, f, t->tris, t->ids, t->words,
                       t->keys, t->vals, t->given, cost + 1);
    // (the packing's temporaries are read for the last time above)
    hipLaunchKernelGGL(k_wide_root, dim3(1), block, 0, s, t->recs, counts, counts + kMaxLevels + 1, cost, 0u);
    RT_HIP(ctx, hipGetLastError());
    uint32_t records = 0, need = 0;
    bool better = false;
    rc = wide_core(ctx, *t, L, f, s, records, need, &better);
    if (rc) return rc;
    const uint32_t inner_height = height;          // inner nodes on the longest path
    if (!better || inner_height > kMaxPackedHeight) return RT_OK;
    t->raw_tris = tris;
    t->raw_nodes = nodes;
    P.wide = std::move(t);
    P.wide_records = records;
    P.wide_need = need;
    P.device_packed = true;
    P.fast = true;
    P.chk = SceneCheck{};
    P.chk.height = height;
    P.chk.leaves = n;
    P.packed.frame = f;
    P.packed.root = 0;
    P.packed.root4 = 0;
    P.packed.height = inner_height;
    P.packed.stack4 = 3u * ((inner_height - 1u) / 2u + 1u) + 1u;
    P.given_records = G;
    P.leaf_slots = n;
    *done = true;
    return RT_OK;
}

}  // namespace rtamd
