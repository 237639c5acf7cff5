// GPU BVH construction: a linear BVH (Karras, "Maximizing parallelism in
// the construction of BVHs, octrees, and k-d trees", HPG 2012) over 63-bit
// Morton codes of triangle centroids, its boxes united from aligned runs of
// sorted leaves, then collapsed to the BVH4 layout the traversal kernels
// read, all on the device.
// Replaces the host BVHMesh::Compile (Shape/BVHMesh.cpp:78-107,203-269) where
// build time matters more than tree quality (many or large scenes).
//
// Steps (one stream; the host waits once per batch of collapse levels):
//   1. triangle boxes; centroid bounds by block reductions
//   2. Morton codes (21 bits per axis) and radix sort of (code, triangle)
//   3. unions of the sorted leaf boxes over aligned runs of 2, 4, 8, ... leaves
//   4. Karras hierarchy: n-1 internal nodes, n leaves; a node's box is the
//      union of the runs its range of leaves is made of
//   5. collapse, level by level: each wide node opens its largest-area
//      internal children until it has four; a subtree of at most max_leaf
//      triangles becomes one leaf (its triangles are contiguous in Morton order)
//   6. triangles packed in Morton order
#include <hip/hip_runtime.h>
#include <hipcub/device/device_radix_sort.hpp>

#include <algorithm>
#include <cfloat>
#include <cstring>
#include <vector>

#include "geom.hpp"
#include "internal.hpp"

namespace ilm {
namespace {

constexpr int kBlock = 256;

struct Box6 {
    float lo[3], hi[3];
};

__device__ __forceinline__ Box6 empty_box() {
    return Box6{{FLT_MAX, FLT_MAX, FLT_MAX}, {-FLT_MAX, -FLT_MAX, -FLT_MAX}};
}
__device__ __forceinline__ Box6 unite(const Box6& a, const Box6& b) {
    Box6 u;
    for (int c = 0; c < 3; ++c) {
        u.lo[c] = fminf(a.lo[c], b.lo[c]);
        u.hi[c] = fmaxf(a.hi[c], b.hi[c]);
    }
    return u;
}
// The union of the workgroup's boxes, in thread 0.
__device__ __forceinline__ Box6 block_unite(Box6 b) {
    __shared__ Box6 waves[kBlock / 64];
    for (int off = 32; off > 0; off >>= 1) {
        Box6 o;
        for (int c = 0; c < 3; ++c) {
            o.lo[c] = __shfl_xor(b.lo[c], off);
            o.hi[c] = __shfl_xor(b.hi[c], off);
        }
        b = unite(b, o);
    }
    if (__lane_id() == 0) waves[threadIdx.x / 64] = b;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < kBlock / 64; ++w) b = unite(b, waves[w]);
    return b;
}

// 1. triangle boxes, and per workgroup the bounds of their centroids. One
// set of bounds per workgroup of at most kBoundBlocks, reduced by one more
// workgroup: with six same-address atomics per 256 triangles this pass took
// 355 us at 1.31M triangles, against 19 us (and 4 us for the reduction).
constexpr int kBoundBlocks = 1024;
__global__ void __launch_bounds__(kBlock) k_tri_boxes(const float* __restrict__ pos, const int32_t* __restrict__ idx,
                                                      int64_t nt, Box6* __restrict__ boxes, Box6* __restrict__ partial) {
    Box6 all = empty_box();
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < nt; i += (int64_t)gridDim.x * kBlock) {
        Box6 b = empty_box();
        for (int v = 0; v < 3; ++v) {
            const float* p = pos + 3 * (int64_t)idx[3 * i + v];
            for (int k = 0; k < 3; ++k) { b.lo[k] = fminf(b.lo[k], p[k]); b.hi[k] = fmaxf(b.hi[k], p[k]); }
        }
        boxes[i] = b;
        Box6 c;
        for (int k = 0; k < 3; ++k) c.lo[k] = c.hi[k] = 0.5f * (b.lo[k] + b.hi[k]);
        all = unite(all, c);
    }
    all = block_unite(all);
    if (threadIdx.x == 0) partial[blockIdx.x] = all;
}
// One workgroup: the union of n boxes.
__global__ void __launch_bounds__(kBlock) k_unite(const Box6* __restrict__ boxes, int n, Box6* __restrict__ out) {
    Box6 all = empty_box();
    for (int i = threadIdx.x; i < n; i += kBlock) all = unite(all, boxes[i]);
    all = block_unite(all);
    if (threadIdx.x == 0) *out = all;
}

__device__ __forceinline__ uint64_t spread21(uint64_t x) {
    x &= 0x1FFFFFull;
    x = (x | (x << 32)) & 0x1F00000000FFFFull;
    x = (x | (x << 16)) & 0x1F0000FF0000FFull;
    x = (x | (x << 8)) & 0x100F00F00F00F00Full;
    x = (x | (x << 4)) & 0x10C30C30C30C30C3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

// 2. Morton codes of centroids in the centroid bounds
__global__ void __launch_bounds__(kBlock) k_morton(const Box6* __restrict__ boxes, int64_t nt,
                                                   const Box6* __restrict__ cbounds, uint64_t* __restrict__ codes,
                                                   int32_t* __restrict__ ids) {
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= nt) return;
    const Box6 b = boxes[i];
    uint64_t q[3];
    for (int k = 0; k < 3; ++k) {
        float lo = cbounds->lo[k], hi = cbounds->hi[k];
        float c = 0.5f * (b.lo[k] + b.hi[k]);
        float e = hi - lo;
        float u = e > 0.0f ? (c - lo) / e : 0.5f;
        u = fminf(fmaxf(u, 0.0f), 1.0f);
        q[k] = (uint64_t)fminf(u * 2097152.0f, 2097151.0f);
    }
    codes[i] = (spread21(q[0]) << 2) | (spread21(q[1]) << 1) | spread21(q[2]);
    ids[i] = (int32_t)i;
}

// common-prefix length of sorted keys i and j; equal codes are told apart by
// their positions (Karras, section 4)
__device__ __forceinline__ int delta(const uint64_t* __restrict__ k, int32_t n, int32_t i, int32_t j) {
    if (j < 0 || j >= n) return -1;
    uint64_t a = k[i], b = k[j];
    if (a != b) return __clzll((long long)(a ^ b));
    return 64 + __clz((int)((uint32_t)i ^ (uint32_t)j));
}

// 3. The union of every aligned run of 2^j of the n boxes `in`, j = 1 ..
// levels, written at out[j - 1]. The first pass gathers the leaf boxes (ids
// given) and stores them in sorted order. A workgroup covers 256 boxes and
// their eight levels in LDS.
constexpr int kRunLevels = 8;
struct RunArgs {
    const Box6* in;
    const int32_t* ids;  // first pass: in[ids[k]] is box k; null: in[k]
    Box6* sorted;        // first pass: box k to sorted[k]
    int32_t n, levels;
    Box6* out[kRunLevels];
};
__global__ void __launch_bounds__(kBlock) k_runs(RunArgs a) {
    __shared__ Box6 run[kBlock];
    const int32_t t = threadIdx.x, k = blockIdx.x * kBlock + t;
    Box6 b = empty_box();
    if (k < a.n) {
        b = a.in[a.ids ? a.ids[k] : k];
        if (a.ids) a.sorted[k] = b;
    }
    run[t] = b;
    int32_t count = a.n;
    for (int j = 0; j < a.levels; ++j) {
        const int32_t width = kBlock >> (j + 1), at = blockIdx.x * width + t;
        count = (count + 1) / 2;
        __syncthreads();
        if (t < width) b = unite(run[2 * t], run[2 * t + 1]);
        __syncthreads();
        if (t < width) {
            run[t] = b;
            if (at < count) a.out[j][at] = b;
        }
    }
}

// 4. Internal node i of n-1, its children, range of leaves and box; nodes
// 0..n-2 internal, n-1.. leaves (leaf k = n-1+k). A range is made of at most
// two runs per level (mostly few: half of the nodes hold two or three
// leaves). Climbing from the leaves instead, the second child to arrive
// uniting the boxes, needs an acquire and a release at device scope at every
// step, which write back and invalidate the caches of the eight XCDs: 5.1 ms
// at 1.31M triangles, against 30 us for the runs and 27 us more here.
constexpr int kMaxRunLevels = 27;  // fewer than 2^26 leaves
struct Runs {
    const Box6* level[kMaxRunLevels];  // [0] the sorted leaf boxes
};
__global__ void __launch_bounds__(kBlock) k_karras(const uint64_t* __restrict__ keys, int32_t n, Runs runs,
                                                   int32_t* __restrict__ left, int32_t* __restrict__ right,
                                                   int32_t* __restrict__ range_lo, int32_t* __restrict__ range_hi,
                                                   Box6* __restrict__ boxes) {
    int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n - 1) return;
    int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = delta(keys, n, i, i - d);
    int32_t lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax *= 2;
    int32_t l = 0;
    for (int32_t t = lmax / 2; t >= 1; t /= 2)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int32_t j = i + l * d;
    int dnode = delta(keys, n, i, j);
    // l >= 1 because keys extended by their positions are distinct; the loop
    // also ends for l == 0
    int32_t s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int32_t gamma = i + s * d + min(d, 0);
    int32_t lo = min(i, j), hi = max(i, j);
    left[i] = (lo == gamma) ? (n - 1 + gamma) : gamma;
    right[i] = (hi == gamma + 1) ? (n - 1 + gamma + 1) : (gamma + 1);
    range_lo[i] = lo;
    range_hi[i] = hi;
    Box6 box = empty_box();
    int32_t a = lo, b = hi + 1;
    for (int lv = 0; a < b; ++lv, a >>= 1, b >>= 1) {
        if (a & 1) box = unite(box, runs.level[lv][a++]);
        if (b & 1) box = unite(box, runs.level[lv][--b]);
    }
    boxes[i] = box;
}

__device__ __forceinline__ float area6(const Box6& b) {
    float dx = b.hi[0] - b.lo[0], dy = b.hi[1] - b.lo[1], dz = b.hi[2] - b.lo[2];
    return 2.0f * (dx * dy + dy * dz + dz * dx);
}

// Counters of the collapse, read back by the host after every few levels.
constexpr int kMaxLevels = 128;  // a Karras tree over 63 + 32 key bits is shallower
struct CollapseCounts {
    uint32_t items[kMaxLevels + 1];  // wide nodes of each level
    uint32_t max_leaf;
    double cost;
};

struct CollapseArgs {
    int32_t n, max_leaf, level;
    const int32_t *left, *right, *range_lo, *range_hi;
    const Box6* nodes;
    WideNode<4>* wide;
    const int32_t* qin;   // binary nodes of this level's wide nodes, in order
    int32_t* qout;        // and of the next level's
    CollapseCounts* counts;
};

__device__ __forceinline__ int32_t subtree_size(const CollapseArgs& a, int32_t node) {
    return node >= a.n - 1 ? 1 : a.range_hi[node] - a.range_lo[node] + 1;
}
__device__ __forceinline__ bool leafable(const CollapseArgs& a, int32_t node) {
    return node >= a.n - 1 || subtree_size(a, node) <= a.max_leaf;
}

// 5. one level of the collapse: one thread per wide node of this level. A
// level's wide nodes are numbered in queue order after those of the levels
// above, so a child's number follows from its place in the next queue, and a
// workgroup takes its places with one atomic (and adds to the cost and the
// largest leaf with one each at its end): one same-address atomic per child,
// node and leaf made the levels of 1.31M triangles 650 us, against 200 us.
// The grid does not depend on the level's size, which the host does not wait
// for: workgroups without work leave at once.
__global__ void __launch_bounds__(kBlock) k_collapse(CollapseArgs a) {
    __shared__ uint32_t s_sum[2][kBlock / 64], s_base[2];
    __shared__ double s_cost[kBlock / 64];
    __shared__ uint32_t s_leaf[kBlock / 64];
    const uint32_t items = a.counts->items[a.level];
    if (blockIdx.x * kBlock >= items) return;
    uint32_t first = 0;  // number of this level's first wide node
    for (int l = 0; l < a.level; ++l) first += a.counts->items[l];
    const Box6 root = a.nodes[0];
    const float ra = area6(root), inv_root_area = ra > 0 ? 1.0f / ra : 0.0f;
    const int lane = (int)__lane_id(), wave = threadIdx.x / 64;
    double cost = 0;
    uint32_t max_leaf = 0;
    int par = 0;
    for (uint32_t base = blockIdx.x * kBlock; base < items; base += gridDim.x * kBlock, par ^= 1) {
        const uint32_t t = base + threadIdx.x;
        const bool live = t < items;
        int32_t kids[4] = {-1, -1, -1, -1};
        int nk = 0;
        uint32_t inner = 0;  // bit k: child k is a wide node of the next level
        if (live) {
            const int32_t node = a.qin[t];
            kids[0] = a.left[node];
            kids[1] = a.right[node];
            nk = 2;
            while (nk < 4) {
                int best = -1;
                float best_a = -1.0f;
                for (int k = 0; k < nk; ++k) {
                    if (leafable(a, kids[k])) continue;
                    float ar = area6(a.nodes[kids[k]]);
                    if (ar > best_a) { best_a = ar; best = k; }
                }
                if (best < 0) break;
                int32_t open = kids[best];
                kids[best] = a.left[open];
                kids[nk++] = a.right[open];
            }
            for (int k = 0; k < nk; ++k) inner |= leafable(a, kids[k]) ? 0u : 1u << k;
            cost += (double)area6(a.nodes[node]) * inv_root_area;
        }
        // places in the next queue: within the wave, the workgroup, the level
        const uint32_t mine = (uint32_t)__popc(inner);
        uint32_t incl = mine;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t v = __shfl_up(incl, off);
            if (lane >= off) incl += v;
        }
        if (lane == 63) s_sum[par][wave] = incl;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t total = 0;
            for (int w = 0; w < kBlock / 64; ++w) total += s_sum[par][w];
            s_base[par] = total ? atomicAdd(&a.counts->items[a.level + 1], total) : 0u;
        }
        __syncthreads();
        uint32_t place = s_base[par] + incl - mine;
        for (int w = 0; w < wave; ++w) place += s_sum[par][w];
        if (!live) continue;
        WideNode<4> w;
        for (int k = 0; k < 4; ++k) {
            if (k >= nk) {
                w.lox[k] = w.loy[k] = w.loz[k] = w.hix[k] = w.hiy[k] = w.hiz[k] = FLT_MAX;
                w.child[k] = make_leaf(0, 0);
                continue;
            }
            const int32_t c = kids[k];
            const Box6 b = a.nodes[c];
            w.lox[k] = b.lo[0]; w.hix[k] = b.hi[0];
            w.loy[k] = b.lo[1]; w.hiy[k] = b.hi[1];
            w.loz[k] = b.lo[2]; w.hiz[k] = b.hi[2];
            if (inner >> k & 1u) {
                a.qout[place] = c;
                w.child[k] = first + items + place;
                ++place;
            } else {
                const int32_t at = c >= a.n - 1 ? c - (a.n - 1) : a.range_lo[c];
                const int32_t cnt = subtree_size(a, c);
                w.child[k] = make_leaf((uint32_t)at, (uint32_t)cnt);
                max_leaf = max(max_leaf, (uint32_t)cnt);
                cost += (double)area6(b) * inv_root_area * cnt;
            }
        }
        a.wide[first + t] = w;
    }
    for (int off = 32; off > 0; off >>= 1) {
        cost += __shfl_xor(cost, off);
        max_leaf = max(max_leaf, (uint32_t)__shfl_xor((int)max_leaf, off));
    }
    if (lane == 0) {
        s_cost[wave] = cost;
        s_leaf[wave] = max_leaf;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / 64; ++w) {
            cost += s_cost[w];
            max_leaf = max(max_leaf, s_leaf[w]);
        }
        atomicAdd(&a.counts->cost, cost);
        atomicMax(&a.counts->max_leaf, max_leaf);
    }
}

// Before the first level: one item, the root, nothing counted.
__global__ void k_collapse_begin(CollapseCounts* c, int32_t* q) {
    const int t = threadIdx.x;
    if (t <= kMaxLevels) c->items[t] = t == 0 ? 1u : 0u;
    if (t == 0) {
        c->max_leaf = 0u;
        c->cost = 0.0;
        q[0] = 0;
    }
}

// 6. triangles in Morton order: (v0, original index), (v1, 0), (v2, 0)
__global__ void __launch_bounds__(kBlock) k_pack(const float* __restrict__ pos, const int32_t* __restrict__ idx,
                                                 const int32_t* __restrict__ ids, int32_t n, float4* __restrict__ out) {
    int32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= n) return;
    int32_t t = ids[k];
    for (int v = 0; v < 3; ++v) {
        const float* p = pos + 3 * (int64_t)idx[3 * (int64_t)t + v];
        out[3 * (int64_t)k + v] = make_float4(p[0], p[1], p[2], v == 0 ? __int_as_float(t) : 0.0f);
    }
}

// float BVH4 nodes -> quantised nodes (same quantiser as the host builders)
__global__ void __launch_bounds__(kBlock) k_quantize(const WideNode<4>* __restrict__ in, int64_t n,
                                                     QNode4* __restrict__ out) {
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    QNode4 q;
    quantize_node(in[i], q);
    out[i] = q;
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

// Builds the BVH4 of m on its context's device. On success m->d_nodes,
// m->d_tris, m->info, m->h_nodes and m->h_order hold the result.
int build_lbvh(ilm_mesh* m, int max_leaf, int node_format) {
    ilm_ctx* ctx = m->ctx;
    const int64_t nt = m->nt, nv = m->nv;
    if (nt > (1 << 26) - 1) return fail(ILM_ERR_INVALID, "more than 2^26 - 1 triangles");
    max_leaf = std::max(1, std::min(max_leaf, kMaxLeafTris));
    const int32_t n = (int32_t)nt;
    hipStream_t st = ctx->stream;

    // Scratch: the context's build workspace where it is free (no other thread
    // builds) and large enough once grown, else an allocation of this call's.
    // One array per buffer, allocated and freed by every build, took 4.1 of
    // the 10.1 ms that a build and trace of 1.31M triangles take (0.6 MB to
    // 150 MB each: a hipFree of the large ones takes up to 2 ms).
    const int32_t ninner = std::max(n - 1, 1);
    size_t sort_bytes = 0;
    ILM_HIP(hipSetDevice(ctx->device));
    ILM_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                               (int32_t*)nullptr, (int32_t*)nullptr, n, 0, 63, st));
    size_t need = 0;
    auto place = [&](size_t bytes) {
        const size_t at = need;
        need += (std::max<size_t>(bytes, 16) + 255) / 256 * 256;
        return at;
    };
    const size_t o_pos = place(nv * 3 * sizeof(float)), o_idx = place(nt * 3 * sizeof(int32_t)),
                 o_tri_boxes = place(nt * sizeof(Box6)),
                 o_cb = place((kBoundBlocks + 1) * sizeof(Box6)),  // centroid bounds, then the workgroups'
                 o_codes_in = place(nt * sizeof(uint64_t)), o_codes = place(nt * sizeof(uint64_t)),
                 o_ids_in = place(nt * sizeof(int32_t)), o_ids = place(nt * sizeof(int32_t)),
                 o_left = place(ninner * sizeof(int32_t)), o_right = place(ninner * sizeof(int32_t)),
                 o_rlo = place(ninner * sizeof(int32_t)), o_rhi = place(ninner * sizeof(int32_t)),
                 o_nodes = place((2 * nt) * sizeof(Box6)), o_runs = place((nt + kMaxRunLevels) * sizeof(Box6)),
                 o_qa = place(ninner * sizeof(int32_t)), o_qb = place(ninner * sizeof(int32_t)),
                 o_counts = place(sizeof(CollapseCounts)), o_sort = place(sort_bytes),
                 o_wide = place((size_t)ninner * sizeof(WideNode<4>));  // at most one per internal node
    BuildWorkspace held(ctx, need <= kBuildKeep);
    void* own = nullptr;
    int rc = held.mine ? ensure_build_ws(ctx, need) : ilm_alloc(ctx, need, &own);
    if (rc) return rc;
    char* ws = held.mine ? (char*)ctx->build_ws : (char*)own;
    float* d_pos = (float*)(ws + o_pos);
    int32_t *d_idx = (int32_t*)(ws + o_idx), *ids_in = (int32_t*)(ws + o_ids_in), *ids = (int32_t*)(ws + o_ids),
            *left = (int32_t*)(ws + o_left), *right = (int32_t*)(ws + o_right), *rlo = (int32_t*)(ws + o_rlo),
            *rhi = (int32_t*)(ws + o_rhi), *qa = (int32_t*)(ws + o_qa), *qb = (int32_t*)(ws + o_qb);
    uint64_t *codes_in = (uint64_t*)(ws + o_codes_in), *codes = (uint64_t*)(ws + o_codes);
    Box6 *tri_boxes = (Box6*)(ws + o_tri_boxes), *nodes = (Box6*)(ws + o_nodes), *runs = (Box6*)(ws + o_runs),
         *cb = (Box6*)(ws + o_cb);
    CollapseCounts* counts = (CollapseCounts*)(ws + o_counts);
    WideNode<4>* wide = (WideNode<4>*)(ws + o_wide);
    void *sort_tmp = ws + o_sort, *d_nodes = nullptr;
    float* d_tris = nullptr;
    auto cleanup = [&]() {
        if (own) ilm_free(ctx, own);
    };
    if (ilm_alloc(ctx, (size_t)nt * 12 * sizeof(float), (void**)&d_tris) != ILM_OK) {
        cleanup();
        return fail(ILM_ERR_NOMEM, "LBVH output allocation failed");
    }
    auto fail_all = [&](int code, const char* what) {
        (void)hipStreamSynchronize(st);  // nothing of this build runs on when the workspace is free again
        if (d_nodes) ilm_free(ctx, d_nodes);
        ilm_free(ctx, d_tris);
        cleanup();
        return fail(code, what);
    };
#define LBVH_HIP(call)                                              \
    do {                                                            \
        hipError_t e_ = (call);                                     \
        if (e_ != hipSuccess) {                                     \
            fail_hip(e_, #call);                                    \
            std::string msg_ = ilm_last_error();                    \
            return fail_all(ILM_ERR_HIP, msg_.c_str());             \
        }                                                           \
    } while (0)

    hipEvent_t e0, e1;
    LBVH_HIP(hipEventCreate(&e0));
    LBVH_HIP(hipEventCreate(&e1));
    LBVH_HIP(hipMemcpyAsync(d_pos, m->pos.data(), nv * 3 * sizeof(float), hipMemcpyHostToDevice, st));
    LBVH_HIP(hipMemcpyAsync(d_idx, m->idx.data(), nt * 3 * sizeof(int32_t), hipMemcpyHostToDevice, st));
    LBVH_HIP(hipEventRecord(e0, st));
    const int bound_blocks = (int)std::min<int64_t>(blocks_for(nt), kBoundBlocks);
    hipLaunchKernelGGL(k_tri_boxes, dim3((unsigned)bound_blocks), dim3(kBlock), 0, st, d_pos, d_idx, nt, tri_boxes,
                       cb + 1);
    hipLaunchKernelGGL(k_unite, dim3(1), dim3(kBlock), 0, st, cb + 1, bound_blocks, cb);
    hipLaunchKernelGGL(k_morton, dim3(blocks_for(nt)), dim3(kBlock), 0, st, tri_boxes, nt, cb, codes_in, ids_in);
    LBVH_HIP(hipGetLastError());
    LBVH_HIP(hipcub::DeviceRadixSort::SortPairs(sort_tmp, sort_bytes, codes_in, codes, ids_in, ids, n, 0, 63, st));

    int levels = 0;
    int64_t nwide = 0;
    CollapseCounts h;
    h.max_leaf = 0;
    h.cost = 0;
    if (n <= max_leaf) {
        // a single leaf under the root
        WideNode<4> w;
        float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
        for (int64_t t = 0; t < nt; ++t)
            for (int v = 0; v < 3; ++v)
                for (int k = 0; k < 3; ++k) {
                    float c = m->pos[3 * (int64_t)m->idx[3 * t + v] + k];
                    lo[k] = std::min(lo[k], c);
                    hi[k] = std::max(hi[k], c);
                }
        for (int k = 0; k < 4; ++k) {
            w.lox[k] = w.loy[k] = w.loz[k] = w.hix[k] = w.hiy[k] = w.hiz[k] = FLT_MAX;
            w.child[k] = make_leaf(0, 0);
        }
        w.lox[0] = lo[0]; w.loy[0] = lo[1]; w.loz[0] = lo[2];
        w.hix[0] = hi[0]; w.hiy[0] = hi[1]; w.hiz[0] = hi[2];
        w.child[0] = make_leaf(0, (uint32_t)n);
        LBVH_HIP(hipMemcpyAsync(wide, &w, sizeof w, hipMemcpyHostToDevice, st));
        nwide = 1;
        h.max_leaf = (uint32_t)n;
        h.cost = (double)n;
        levels = 1;
    } else {
        // runs of 2, 4, ... leaves, eight levels per pass until one box is left
        Runs tree{};
        tree.level[0] = nodes + (n - 1);
        Box6* at = runs;
        int32_t count = n;
        for (int lv = 0; count > 1;) {
            RunArgs r{};
            r.in = lv == 0 ? tri_boxes : tree.level[lv];
            r.ids = lv == 0 ? ids : nullptr;
            r.sorted = nodes + (n - 1);
            r.n = count;
            const unsigned blocks = blocks_for(count);
            while (r.levels < kRunLevels && count > 1) {
                count = (count + 1) / 2;
                tree.level[++lv] = r.out[r.levels++] = at;
                at += count;
            }
            hipLaunchKernelGGL(k_runs, dim3(blocks), dim3(kBlock), 0, st, r);
        }
        hipLaunchKernelGGL(k_karras, dim3(blocks_for(n - 1)), dim3(kBlock), 0, st, codes, n, tree, left, right, rlo,
                           rhi, nodes);
        hipLaunchKernelGGL(k_collapse_begin, dim3(1), dim3(kBlock), 0, st, counts, qa);
        LBVH_HIP(hipGetLastError());
        CollapseArgs a;
        a.n = n;
        a.max_leaf = max_leaf;
        a.left = left; a.right = right; a.range_lo = rlo; a.range_hi = rhi;
        a.nodes = nodes;
        a.wide = wide;
        a.counts = counts;
        int32_t *qin = qa, *qout = qb;
        const unsigned grid = (unsigned)std::min<int64_t>(blocks_for(n), (int64_t)ctx->cu_count * 8);
        // a balanced tree's levels and a few more before the first wait
        int until = 4;
        for (int64_t m = n; m > max_leaf; m /= 4) ++until;
        for (;;) {
            for (; levels < until; ++levels) {
                a.level = levels;
                a.qin = qin; a.qout = qout;
                hipLaunchKernelGGL(k_collapse, dim3(grid), dim3(kBlock), 0, st, a);
                std::swap(qin, qout);
            }
            LBVH_HIP(hipGetLastError());
            LBVH_HIP(hipMemcpyAsync(&h, counts, sizeof h, hipMemcpyDeviceToHost, st));
            LBVH_HIP(hipStreamSynchronize(st));
            if (h.items[levels] == 0) break;
            if (levels == kMaxLevels) return fail_all(ILM_ERR_STATE, "LBVH collapse did not terminate");
            until = std::min(levels + 4, kMaxLevels);
        }
        while (levels > 0 && h.items[levels - 1] == 0) --levels;
        for (int l = 0; l < levels; ++l) nwide += h.items[l];
    }
    hipLaunchKernelGGL(k_pack, dim3(blocks_for(n)), dim3(kBlock), 0, st, d_pos, d_idx, ids, n,
                       reinterpret_cast<float4*>(d_tris));
    LBVH_HIP(hipGetLastError());
    const size_t stride = node_format == ILM_NODES_QUANTIZED ? sizeof(QNode4) : sizeof(WideNode<4>);
    if (ilm_alloc(ctx, (size_t)nwide * stride, &d_nodes) != ILM_OK) return fail_all(ILM_ERR_NOMEM, "LBVH nodes");
    if (node_format == ILM_NODES_QUANTIZED) {
        hipLaunchKernelGGL(k_quantize, dim3(blocks_for(nwide)), dim3(kBlock), 0, st, wide, nwide,
                           reinterpret_cast<QNode4*>(d_nodes));
        LBVH_HIP(hipGetLastError());
    } else {
        LBVH_HIP(hipMemcpyAsync(d_nodes, wide, (size_t)nwide * stride, hipMemcpyDeviceToDevice, st));
    }
    LBVH_HIP(hipEventRecord(e1, st));
    LBVH_HIP(hipStreamSynchronize(st));
    float gpu_ms = 0;
    LBVH_HIP(hipEventElapsedTime(&gpu_ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);

    // host copies for export and for hit-slot lookups
    m->h_nodes.resize((size_t)nwide * stride);
    m->h_order.resize(nt);
    LBVH_HIP(hipMemcpy(m->h_nodes.data(), d_nodes, m->h_nodes.size(), hipMemcpyDeviceToHost));
    LBVH_HIP(hipMemcpy(m->h_order.data(), ids, nt * sizeof(int32_t), hipMemcpyDeviceToHost));
    cleanup();
#undef LBVH_HIP

    if (m->d_nodes) ilm_free(ctx, m->d_nodes);
    if (m->d_tris) ilm_free(ctx, m->d_tris);
    if (m->d_slot_of) { ilm_free(ctx, m->d_slot_of); m->d_slot_of = nullptr; }
    m->d_nodes = d_nodes;
    m->d_tris = d_tris;
    m->width = 4;
    m->node_format = node_format;
    m->info.node_format = node_format;
    m->info.node_stride = (int32_t)stride;
    m->info.nodes = nwide;
    m->info.node_bytes = nwide * (int64_t)stride;
    m->info.tri_bytes = nt * 12 * (int64_t)sizeof(float);
    m->info.width = 4;
    m->info.depth = levels;
    m->info.max_leaf = (int32_t)h.max_leaf;
    m->info.stack_need = 3 * levels + 1;  // at most three deferred siblings per level
    m->info.build_ms = gpu_ms;
    m->info.sah_cost = h.cost;
    m->built = true;
    return ILM_OK;
}

}  // namespace ilm
