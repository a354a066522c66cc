// rt_wide.hpp -- the tree the 4-wide traversal walks, built on the device at
// upload.  Part of rt_build.hip, whose radix tree it shares.
//
// The caller's tree decides which of two hits at exactly equal t is
// reported, and nothing else: a closest hit does not depend on the tree.
// The reference's builder splits medians along random axes (Bvh.h:141-209),
// a poor tree to traverse, so an upload builds a second one over the same
// leaves, with the same leaf boxes in the same 16-bit frame, and the
// traversal walks that.  A ray that meets its closest t twice is traced
// once more through the caller's records, which alone name the winner
// (trace_persistent).
//
// Steps, all on one stream, for n leaves:
//  1. leaf words (lo | hi << 16 per axis) from the caller's 4-wide records,
//     and 48-bit Morton codes of their centres
//  2. stable radix sort of (code, leaf)
//  3. radix tree over the sorted codes (Karras, HPG 2012), equal codes
//     ordered by position, as in rt_build.hip
//  4. boxes: a 64-ary pyramid of unions over the sorted leaves, then each
//     internal node unions the entries that tile its range
//  5. collapse to four children, top down, one launch per level: the child
//     with the largest box is opened next.  A child of two leaves counts
//     four times its area (opening it saves its whole record) and one of
//     three or four a quarter (it fills a record by itself): 0.42-0.43
//     records per leaf where plain largest-area has 0.46-0.50, with the
//     same number of records read per ray
//  6. records numbered in depth-first preorder.  A node covering the sorted
//     leaves [lo, hi] has preorder rank lo + (ancestors whose left subtree
//     holds it) among the binary tree's internal nodes: every split before
//     lo belongs to a node already left or to an ancestor, and of the splits
//     from lo on only those ancestors come first
//
// Records per ray on a CPU model of the traversal (caller's tree / this one;
// a 16-bin surface-area sweep in brackets): 4,194,304-triangle clustered
// soup 186 / 67 (63), 262,144 triangles 68 / 27 (25), 81,920-triangle
// icosphere 20.6 / 16.0 (15.0).  The longest ray of 100,000 on the first:
// 2,037 / 530 steps.
#pragma once

#include <algorithm>
#include <new>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "rt_common.hpp"

namespace rtamd {
namespace {

constexpr uint32_t kCodeBits = 48;
constexpr uint32_t kMaxLevels = 128;          // 4-wide levels of a collapse
constexpr uint32_t kLevelsPerSync = 12;

// A box in the 16-bit frame: lo | hi << 16 per axis (w unused).
__device__ __forceinline__ uint32_t axis_union(uint32_t a, uint32_t b) {
    return min(a & 0xffffu, b & 0xffffu) | (max(a >> 16, b >> 16) << 16);
}
__device__ __forceinline__ uint4 box_union(uint4 a, uint4 b) {
    return make_uint4(axis_union(a.x, b.x), axis_union(a.y, b.y), axis_union(a.z, b.z), 0u);
}
__device__ __forceinline__ uint4 empty_box() { return make_uint4(0xffffu, 0xffffu, 0xffffu, 0u); }

// Half the surface area, in the frame's scale.
__device__ __forceinline__ float box_area(uint32_t x, uint32_t y, uint32_t z, const QFrame& f) {
    const float dx = (float)((x >> 16) - (x & 0xffffu)) * f.sx, dy = (float)((y >> 16) - (y & 0xffffu)) * f.sy,
                dz = (float)((z >> 16) - (z & 0xffffu)) * f.sz;
    return dx * dy + dy * dz + dz * dx;
}

__device__ inline double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Adds every thread's v to *total, one atomic a block.  Called by whole blocks of 256.
__device__ inline void block_add(double v, double* total) {
    __shared__ double part[4];
    v = wave_sum(v);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double sum = (part[0] + part[1]) + (part[2] + part[3]);
        if (sum != 0.0) atomicAdd(total, sum);
    }
}

// Morton code of a box's centre, 16 bits an axis.
__device__ __forceinline__ uint64_t wide_key(uint4 w) {
    return (spread3(((w.x & 0xffffu) + (w.x >> 16)) >> 1) << 2) | (spread3(((w.y & 0xffffu) + (w.y >> 16)) >> 1) << 1) |
           spread3(((w.z & 0xffffu) + (w.z >> 16)) >> 1);
}

// One thread per child slot of the caller's records: the words and code of
// each leaf, and the summed area of the inner children (the records a ray
// reads, by the surface-area measure).
__global__ __launch_bounds__(256) void k_wide_leaves(const PNode4* __restrict__ given, uint32_t n_given, QFrame f,
                                                     uint4* __restrict__ words, uint64_t* __restrict__ keys,
                                                     uint32_t* __restrict__ vals, double* __restrict__ cost) {
    double sum = 0.0;
    const uint64_t total = (uint64_t)n_given * 4u;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (uint64_t)gridDim.x * blockDim.x) {
        const PNode4& r = given[i >> 2];
        const uint32_t k = (uint32_t)i & 3u;
        const int32_t ref = r.ref[k];
        if (ref == kNoChild) continue;
        const uint32_t x = r.w[3 * k], y = r.w[3 * k + 1], z = r.w[3 * k + 2];
        if (ref >= 0) {
            sum += (double)box_area(x, y, z, f);
            continue;
        }
        const uint32_t leaf = (uint32_t)~ref;
        words[leaf] = make_uint4(x, y, z, 0u);
        keys[leaf] = wide_key(words[leaf]);
        vals[leaf] = leaf;
    }
    block_add(sum, cost);
}

// Leaf words in sorted order.
__global__ __launch_bounds__(256) void k_wide_sorted(const uint4* __restrict__ words, const uint32_t* __restrict__ order,
                                                     uint32_t n, uint4* __restrict__ sorted) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) sorted[k] = words[order[k]];
}

// Internal node i: its children (>= 0 an internal node, < 0 the sorted leaf
// ~child) and the far end of its range [min(i, far), max(i, far)].
__global__ __launch_bounds__(256) void k_wide_tree(const uint64_t* __restrict__ keys, uint32_t n, int2* __restrict__ kids,
                                                   uint32_t* __restrict__ far) {
    const int64_t N = n;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N - 1; i += (int64_t)gridDim.x * blockDim.x) {
        int64_t j, g;
        radix_split(keys, N, i, j, g);
        const int64_t lo = i < j ? i : j, hi = i < j ? j : i;
        kids[i] = make_int2(lo == g ? ~(int32_t)g : (int32_t)g, hi == g + 1 ? ~(int32_t)(g + 1) : (int32_t)(g + 1));
        far[i] = (uint32_t)j;
    }
}

// 64-ary pyramid of unions over the sorted leaves (level 0).
struct WPyramid {
    const uint4* lvl[kPyramidLevels];
    uint32_t count[kPyramidLevels];
    uint32_t levels;
};

__device__ __forceinline__ uint32_t wave_axis(uint32_t v) {
    for (int o = 32; o > 0; o >>= 1) v = axis_union(v, (uint32_t)__shfl_xor((int)v, o, 64));
    return v;
}

// One wave per 64-entry block of level `level` -> entry of level + 1.
__global__ __launch_bounds__(256) void k_wide_pyramid(WPyramid p, uint32_t level, uint4* __restrict__ out) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t blocks = p.count[level + 1];
    for (uint32_t m = (blockIdx.x * blockDim.x + threadIdx.x) / 64u; m < blocks; m += gridDim.x * blockDim.x / 64u) {
        const uint32_t k = m * 64u + lane;
        uint4 b = k < p.count[level] ? p.lvl[level][k] : empty_box();
        b.x = wave_axis(b.x);
        b.y = wave_axis(b.y);
        b.z = wave_axis(b.z);
        if (lane == 0) out[m] = b;
    }
}

// Internal node i's box: the union over its sorted leaf range.
__global__ __launch_bounds__(256) void k_wide_boxes(WPyramid p, uint32_t n, const uint32_t* __restrict__ far,
                                                    uint4* __restrict__ boxes) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i + 1 < n; i += gridDim.x * blockDim.x) {
        const uint32_t j = far[i];
        uint32_t lo = i < j ? i : j, hi = (i < j ? j : i) + 1;    // [lo, hi) at level 0
        uint4 u = empty_box();
        for (uint32_t level = 0; lo < hi; ++level) {
            const uint4* q = p.lvl[level];
            if (level + 1 == p.levels || hi - lo <= 64u) {
                for (uint32_t k = lo; k < hi; ++k) u = box_union(u, q[k]);
                break;
            }
            const uint32_t a = min(hi, (lo + 63u) & ~63u);          // head up to a block boundary
            const uint32_t b = max(a, hi & ~63u);                    // tail from the last boundary
            for (uint32_t k = lo; k < a; ++k) u = box_union(u, q[k]);
            for (uint32_t k = b; k < hi; ++k) u = box_union(u, q[k]);
            lo = a / 64u;                                           // whole blocks [a, b) one level up
            hi = b / 64u;
        }
        boxes[i] = u;
    }
}

// A 4-wide record to be: its binary node, the first sorted leaf under it,
// the ancestors whose left subtree holds it, and the stack entries a ray can
// have deferred on its way to this record's children.
struct WideRec {
    int32_t node;
    uint32_t lo, left, need;
    int32_t child[4];            // internal node, ~leaf, or kNoChild
    uint32_t rank[4];            // preorder rank of an internal child
};

// The first level of the collapse, and its sums at zero (cost[1], the caller's
// tree's, only with zero_given).
__global__ void k_wide_root(WideRec* recs, uint32_t* level_count, uint32_t* need, double* cost, uint32_t zero_given) {
    const uint32_t t = threadIdx.x;
    if (t < kMaxLevels + 1) level_count[t] = t == 0 ? 1u : 0u;
    if (t == 0) {
        recs[0].node = 0;
        recs[0].lo = recs[0].left = recs[0].need = 0u;
        *need = 0u;
        cost[0] = 0.0;
        if (zero_given) cost[1] = 0.0;
    }
}

// Level `level` of the collapse: opens children until a record has four,
// appends its internal children to the next level.
__global__ __launch_bounds__(256) void k_wide_collapse(const int2* __restrict__ kids, const uint32_t* __restrict__ far,
                                                       const uint4* __restrict__ boxes, QFrame f, uint32_t level,
                                                       uint32_t cap, WideRec* __restrict__ recs,
                                                       uint32_t* __restrict__ level_count, uint32_t* __restrict__ flags,
                                                       uint32_t* __restrict__ need, double* __restrict__ cost) {
    uint32_t begin = 0;
    for (uint32_t l = 0; l < level; ++l) begin += level_count[l];
    const uint32_t count = level_count[level];
    const uint32_t next = begin + count;
    double sum = 0.0;
    for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < count; q += gridDim.x * blockDim.x) {
        if (begin + q >= cap) break;                 // more records than reserved: the host gives up on this tree
        const WideRec me = recs[begin + q];
        int32_t code[4];
        uint32_t lo[4], left[4], cnt[4];
        float area[4];
        uint32_t n = 0;
        auto put = [&](uint32_t at, int32_t c, uint32_t l, uint32_t a) {
            code[at] = c;
            lo[at] = l;
            left[at] = a;
            cnt[at] = 1;
            area[at] = 0.0f;
            if (c >= 0) {
                const uint32_t e = far[c];
                cnt[at] = (e > (uint32_t)c ? e - (uint32_t)c : (uint32_t)c - e) + 1u;
                const uint4 b = boxes[c];
                area[at] = box_area(b.x, b.y, b.z, f);
            }
        };
        auto open = [&](uint32_t at, int32_t node, uint32_t l, uint32_t a) {
            const int2 k = kids[node];
            put(at, k.x, l, a + 1u);
            put(n, k.y, l + cnt[at], a);
            ++n;
        };
        n = 1;
        open(0, me.node, me.lo, me.left);
        while (n < 4) {
            int best = -1;
            float bw = -1.0f;
            for (uint32_t k = 0; k < n; ++k) {
                if (code[k] < 0) continue;
                const float w = area[k] * (cnt[k] == 2 ? 4.0f : cnt[k] <= 4 ? 0.25f : 1.0f);
                if (w > bw) {
                    bw = w;
                    best = (int)k;
                }
            }
            if (best < 0) break;
            open((uint32_t)best, code[best], lo[best], left[best]);
        }
        WideRec r = me;
        r.need = me.need + n - 1u;
        uint32_t inner = 0;
        for (uint32_t k = 0; k < 4; ++k) {
            r.child[k] = k < n ? code[k] : kNoChild;
            r.rank[k] = k < n && code[k] >= 0 ? lo[k] + left[k] : 0u;
            if (k < n && code[k] >= 0) {
                ++inner;
                sum += (double)area[k];
            }
        }
        recs[begin + q] = r;
        flags[me.lo + me.left] = 1u;
        if (r.need > *need) atomicMax(need, r.need);
        if (inner) {
            uint32_t at = next + atomicAdd(&level_count[level + 1], inner);
            for (uint32_t k = 0; k < n; ++k) {
                if (code[k] < 0) continue;
                if (at < cap) {
                    recs[at].node = code[k];
                    recs[at].lo = lo[k];
                    recs[at].left = left[k];
                    recs[at].need = r.need;
                }
                ++at;
            }
        }
    }
    block_add(sum, cost);
}

// The records, numbered from `first` in preorder; leaf refs are ~(sorted position).
__global__ __launch_bounds__(256) void k_wide_emit(const WideRec* __restrict__ recs, uint32_t count,
                                                   const uint32_t* __restrict__ rank_to_index,
                                                   const uint4* __restrict__ boxes, const uint4* __restrict__ leaves,
                                                   uint32_t first, PNode4* __restrict__ out) {
    for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < count; q += gridDim.x * blockDim.x) {
        const WideRec r = recs[q];
        PNode4 o;
        for (int k = 0; k < 4; ++k) {
            const int32_t c = r.child[k];
            const uint4 b = c == kNoChild ? make_uint4(0u, 0u, 0u, 0u) : c >= 0 ? boxes[c] : leaves[~c];
            o.w[3 * k] = b.x;
            o.w[3 * k + 1] = b.y;
            o.w[3 * k + 2] = b.z;
            o.ref[k] = c >= 0 ? (int32_t)(first + rank_to_index[r.rank[k]]) : c;
        }
        out[first + rank_to_index[r.lo + r.left]] = o;
    }
}

// Triangles into sorted order, and where each of the caller's slots went.
__global__ __launch_bounds__(256) void k_wide_gather(const uint32_t* __restrict__ order, uint32_t n,
                                                     const PTri* __restrict__ tris, const int32_t* __restrict__ ids,
                                                     PTri* __restrict__ out_tris, int32_t* __restrict__ out_ids,
                                                     uint32_t* __restrict__ place) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const uint32_t s = order[k];
        out_tris[k] = tris[s];
        out_ids[k] = ids[s];
        place[s] = k;
    }
}

// The caller's records with their leaf refs at the triangles' new places.
__global__ __launch_bounds__(256) void k_wide_place(const PNode4* __restrict__ given, uint32_t n_given,
                                                    const uint32_t* __restrict__ place, PNode4* __restrict__ out) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n_given; i += gridDim.x * blockDim.x) {
        PNode4 r = given[i];
        for (int k = 0; k < 4; ++k)
            if (r.ref[k] < 0 && r.ref[k] != kNoChild) r.ref[k] = ~(int32_t)place[~r.ref[k]];
        out[i] = r;
    }
}

}  // namespace

// Where a build's arrays lie in its one device allocation: what packing makes
// for it, then what is only used by the build (from `overlay` on).
struct WideLayout {
    size_t bytes = 0, overlay = 0;
    size_t raw_tris = 0, raw_nodes = 0;
    size_t given = 0, tris = 0, ids = 0, words = 0, keys = 0, vals = 0, counts = 0, cost = 0, facts = 0;
    size_t sorted = 0, keys2 = 0, order = 0, kids = 0, far = 0, boxes = 0, recs = 0, rank = 0, tmp = 0;
    size_t lvl[kPyramidLevels] = {};
    size_t sort_bytes = 0, scan_bytes = 0;
    size_t take(size_t b) { const size_t o = bytes; bytes += align256(b); return o; }
    // n leaves and `records` of the caller's records, at most
    int wide(rt_ctx* ctx, uint32_t n, uint32_t records, hipStream_t s) {
        RT_HIP(ctx, rocprim::radix_sort_pairs(nullptr, sort_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                              (uint32_t*)nullptr, (uint32_t*)nullptr, n, 0u, kCodeBits, s));
        RT_HIP(ctx, rocprim::exclusive_scan(nullptr, scan_bytes, (uint32_t*)nullptr, (uint32_t*)nullptr, 0u, n,
                                            rocprim::plus<uint32_t>(), s));
        given = take(sizeof(PNode4) * (size_t)records);
        tris = take(sizeof(PTri) * (size_t)n);
        ids = take(4 * (size_t)n);
        words = take(16 * (size_t)n);
        keys = take(8 * (size_t)n);
        vals = take(4 * (size_t)n);
        counts = take(4 * (kMaxLevels + 2));
        cost = take(16);
        facts = take(64);
        overlay = bytes;
        sorted = take(16 * (size_t)n);
        keys2 = take(8 * (size_t)n);
        order = take(4 * (size_t)n);
        kids = take(8 * (size_t)n);
        far = take(4 * (size_t)n);
        boxes = take(16 * (size_t)n);
        recs = take(sizeof(WideRec) * (size_t)std::max(1u, n / 2u));
        rank = take(4 * (size_t)n);
        uint32_t count = n;
        for (int k = 1; k < kPyramidLevels; ++k) {
            count = (count + 63u) / 64u;
            lvl[k] = take(16 * (size_t)count);
        }
        tmp = take(std::max(sort_bytes, scan_bytes));
        return RT_OK;
    }
};

// Levels to launch before their sizes are first read back: as many as a
// balanced tree over n leaves has with `bits` of n's bits to a level, and two
// more.  An empty level's launch costs 4 us, most of a small scene's upload
// (256 triangles 0.43 -> 0.37 ms, 1,024 0.54 -> 0.47, with one copy for all that
// is read back);
// a deeper tree waits for kLevelsPerSync more at a time.
static uint32_t first_levels(uint32_t n, uint32_t bits) {
    uint32_t k = 2;
    while (n > 1u) { n >>= bits; ++k; }
    return k;
}

// What a build's host side reads back between passes: counts, cost and facts
// as they lie in the allocation.
struct WideProgress {
    uint32_t counts[align256(4 * (kMaxLevels + 2)) / 4];
    double cost[align256(16) / 8];
    uint32_t facts[16];
};

// A build between its two halves.  Its memory is the context's upload
// workspace where that is small, else an allocation of its own.
struct WideTree {
    char* base = nullptr;
    bool own = false;
    PNode4* given = nullptr;
    PTri* tris = nullptr;
    int32_t* ids = nullptr;
    uint4 *words = nullptr, *sorted = nullptr, *boxes = nullptr;
    uint64_t* keys = nullptr;
    uint32_t *vals = nullptr, *order = nullptr, *rank_to_index = nullptr, *place = nullptr;
    WideRec* recs = nullptr;
    uint32_t n = 0, n_given = 0;
    const rt_triangle* raw_tris = nullptr;    // the caller's arrays, when packed on the device
    const rt_bvh_node* raw_nodes = nullptr;
    ~WideTree() { if (own && base) (void)hipFree(base); }
    // false: no room.  (Leaves the context's error text alone: that belongs to
    // the thread that uses the context, which a server's additions need not be.)
    bool allocate(rt_ctx* ctx, size_t bytes) {
        void*& kept = ctx->ws[kWsUpload];
        size_t& kept_bytes = ctx->ws_bytes[kWsUpload];
        own = bytes > kUploadKept;
        if (!own && kept_bytes >= bytes) {
            base = (char*)kept;
            return true;
        }
        if (!own && kept) {
            // (waits for the kernels that use it)
            (void)hipFree(kept);
            kept = nullptr;
            kept_bytes = 0;
        }
        const size_t grown = own ? bytes : bytes + bytes / 8;
        if (hipMalloc((void**)&base, grown) != hipSuccess) {
            (void)hipGetLastError();
            base = nullptr;
            own = false;
            return false;
        }
        if (!own) {
            kept = base;
            kept_bytes = grown;
        }
        return true;
    }
    void bind(const WideLayout& L, uint32_t leaves, uint32_t records) {
        n = leaves;
        n_given = records;
        given = (PNode4*)(base + L.given);
        tris = (PTri*)(base + L.tris);
        ids = (int32_t*)(base + L.ids);
        words = (uint4*)(base + L.words);
        keys = (uint64_t*)(base + L.keys);
        vals = (uint32_t*)(base + L.vals);
        sorted = (uint4*)(base + L.sorted);
        boxes = (uint4*)(base + L.boxes);
        order = (uint32_t*)(base + L.order);
        rank_to_index = (uint32_t*)(base + L.rank);
        place = vals;                              // the sort's input indices, free by then
        recs = (WideRec*)(base + L.recs);
    }
};

void WideTreeDelete::operator()(WideTree* t) const { delete t; }

// The tree over t's leaves (words, keys, vals, and the caller's cost in
// cost[1] are set).  *better stays false where the caller's tree is to be
// traversed as it is.  Waits for the build.
static int wide_core(rt_ctx* ctx, WideTree& t, const WideLayout& L, const QFrame& f, hipStream_t s, uint32_t& records,
                     uint32_t& need, bool* better) {
    const uint32_t n = t.n;
    const uint32_t cap = std::max(1u, n / 2u);
    char* b = t.base;
    uint64_t* keys2 = (uint64_t*)(b + L.keys2);
    int2* kids = (int2*)(b + L.kids);
    uint32_t *far = (uint32_t*)(b + L.far), *counts = (uint32_t*)(b + L.counts);
    uint32_t* flags = (uint32_t*)t.words;         // the unsorted words are done when the collapse starts
    uint32_t* d_need = counts + kMaxLevels + 1;
    double* cost = (double*)(b + L.cost);
    WPyramid pyr{};
    pyr.count[0] = n;
    pyr.levels = 1;
    while (pyr.levels < (uint32_t)kPyramidLevels && pyr.count[pyr.levels - 1] > 1) {
        pyr.count[pyr.levels] = (pyr.count[pyr.levels - 1] + 63u) / 64u;
        ++pyr.levels;
    }
    auto grid = [&](uint64_t work) {
        return dim3((uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((work + 255) / 256, (uint64_t)ctx->num_cus * 16u)));
    };
    const dim3 block(256);
    size_t sort_bytes = L.sort_bytes, scan_bytes = L.scan_bytes;
    RT_HIP(ctx, rocprim::radix_sort_pairs((void*)(b + L.tmp), sort_bytes, t.keys, keys2, t.vals, t.order, n, 0u, kCodeBits, s));
    hipLaunchKernelGGL(k_wide_sorted, grid(n), block, 0, s, t.words, t.order, n, t.sorted);
    hipLaunchKernelGGL(k_wide_tree, grid(n - 1), block, 0, s, keys2, n, kids, far);
    pyr.lvl[0] = t.sorted;
    for (uint32_t k = 1; k < pyr.levels; ++k) pyr.lvl[k] = (uint4*)(b + L.lvl[k]);
    for (uint32_t k = 0; k + 1 < pyr.levels; ++k)
        hipLaunchKernelGGL(k_wide_pyramid, grid((uint64_t)pyr.count[k + 1] * 64u), block, 0, s, pyr, k,
                           (uint4*)(b + L.lvl[k + 1]));
    hipLaunchKernelGGL(k_wide_boxes, grid(n - 1), block, 0, s, pyr, n, far, t.boxes);
    RT_HIP(ctx, hipGetLastError());
    int rc = launch_fill_u32(ctx, flags, 0u, n, s);
    if (rc) return rc;
    // levels until one is empty; their sizes live on the device and are read
    // back every kLevelsPerSync levels
    WideProgress now{};
    const uint32_t* h = now.counts;
    const double* c = now.cost;
    uint32_t level = 0;
    for (;;) {
        // (more levels than for even records: boxes open unevenly)
        const uint32_t end = std::min(level == 0 ? first_levels(n, 2) + 4u : level + kLevelsPerSync, kMaxLevels);
        for (; level < end; ++level)
            hipLaunchKernelGGL(k_wide_collapse, grid(cap), block, 0, s, kids, far, t.boxes, f, level, cap, t.recs, counts,
                               flags, d_need, cost);
        RT_HIP(ctx, hipGetLastError());
        RT_HIP(ctx, hipMemcpyAsync(&now, counts, sizeof now, hipMemcpyDeviceToHost, s));
        RT_HIP(ctx, hipStreamSynchronize(s));
        if (h[level] == 0 || level == kMaxLevels) break;
    }
    if (h[level] != 0) return RT_OK;              // deeper than kMaxLevels levels
    uint64_t R = 0;
    for (uint32_t l = 0; l < level; ++l) R += h[l];
    // more records than reserved, a stack no kernel variant holds, or a
    // caller's tree that is the better one (its boxes' summed area smaller)
    if (R > cap || h[kMaxLevels + 1] + 1u > kMaxWideStack || !(c[0] < c[1])) return RT_OK;
    RT_HIP(ctx, rocprim::exclusive_scan((void*)(b + L.tmp), scan_bytes, flags, t.rank_to_index, 0u, n,
                                        rocprim::plus<uint32_t>(), s));
    records = (uint32_t)R;
    need = h[kMaxLevels + 1] + 1u;
    *better = true;
    return RT_OK;
}

int wide_build(rt_ctx* ctx, const PackedTree& packed, hipStream_t s, std::unique_ptr<WideTree, WideTreeDelete>& out,
               uint32_t& records, uint32_t& need) {
    out.reset();
    records = need = 0;
    const uint32_t n = (uint32_t)packed.tris.size(), G = (uint32_t)packed.w4nodes.size();
    if (n < 2 || G == 0 || packed.root4 != 0) return RT_OK;
    std::unique_ptr<WideTree, WideTreeDelete> t(new (std::nothrow) WideTree());
    if (!t) return RT_OK;
    WideLayout L;
    int rc = L.wide(ctx, n, G, s);
    if (rc) return rc;
    // no room for the scratch: the caller's tree is traversed as it is
    if (!t->allocate(ctx, L.bytes)) return RT_OK;
    t->bind(L, n, G);
    uint32_t* counts = (uint32_t*)(t->base + L.counts);
    double* cost = (double*)(t->base + L.cost);
    RT_HIP(ctx, hipMemcpyAsync(t->given, packed.w4nodes.data(), sizeof(PNode4) * (size_t)G, hipMemcpyHostToDevice, s));
    RT_HIP(ctx, hipMemcpyAsync(t->tris, packed.tris.data(), sizeof(PTri) * (size_t)n, hipMemcpyHostToDevice, s));
    RT_HIP(ctx, hipMemcpyAsync(t->ids, packed.tri_id.data(), 4 * (size_t)n, hipMemcpyHostToDevice, s));
    const dim3 block(256);
    const dim3 grid((uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((4ull * G + 255) / 256, (uint64_t)ctx->num_cus * 8u)));
    hipLaunchKernelGGL(k_wide_root, dim3(1), block, 0, s, t->recs, counts, counts + kMaxLevels + 1, cost,
                       1u);
    hipLaunchKernelGGL(k_wide_leaves, grid, block, 0, s, t->given, G, packed.frame, t->words, t->keys, t->vals, cost + 1);
    RT_HIP(ctx, hipGetLastError());
    bool better = false;
    rc = wide_core(ctx, *t, L, packed.frame, s, records, need, &better);
    if (rc) return rc;
    if (better) out = std::move(t);
    return RT_OK;
}

int wide_emit(rt_ctx* ctx, const WideTree& t, uint32_t records, PNode4* nodes, PTri* tris, int32_t* ids, hipStream_t s) {
    auto grid = [&](uint64_t work) {
        return dim3((uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((work + 255) / 256, (uint64_t)ctx->num_cus * 16u)));
    };
    const dim3 block(256);
    hipLaunchKernelGGL(k_wide_gather, grid(t.n), block, 0, s, t.order, t.n, t.tris, t.ids, tris, ids, t.place);
    hipLaunchKernelGGL(k_wide_place, grid(t.n_given), block, 0, s, t.given, t.n_given, t.place, nodes);
    hipLaunchKernelGGL(k_wide_emit, grid(records), block, 0, s, t.recs, records, t.rank_to_index, t.boxes, t.sorted,
                       t.n_given, nodes);
    RT_HIP(ctx, hipGetLastError());
    return RT_OK;
}

const rt_triangle* wide_triangles(const WideTree& t) { return t.raw_tris; }
const rt_bvh_node* wide_nodes(const WideTree& t) { return t.raw_nodes; }

}  // namespace rtamd
