// GPU BVH build and ray-cast entry points of the lmgpu C ABI (gfx950).
//
// Replaces Accel_SAHBVH::build (src/accel/accel_sahbvh.cpp:127-267), a
// top-down full-sort SAH build on host threads, with a fully device-side
// pipeline:
//   1. per-triangle bounds + centroid bounds (ordered-int atomics),
//   2. 63-bit Morton codes of the centroids,
//   3. stable radix sort of (code, index) pairs (sort.hip), checked ordered,
//   4. binary LBVH topology (Karras, HPG 2012), ties broken by index, or
//      PLOC (ploc.hip),
//   5. triangles copied into traversal order (48 B each) and bottom-up bounds
//      refit, one block per 1024 or 4096 leaves and one block for the nodes
//      above, which also fills the SAH cost tables of the collapse
//      (sah_tables),
//   6. collapse into a W-wide tree (W = 2, 4, 8) of least SAH cost: the
//      dynamic program decides which binary subtrees become wide nodes and
//      which become leaves of at most `leaf_size` triangles (a contiguous
//      range of the sorted triangle array); the greedy alternative opens the
//      largest-area child until a node has W children.
// and Accel_SAHBVH::intersect (:269-299) with the ordered wide traversal of
// bvh.h.

#include <algorithm>
#include <type_traits>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "build.h"
#include "bvh.h"
#include "lmgpu_internal.h"

namespace lmgpu {

// Build defaults: leaves of at most 2 triangles, and a triangle test costing
// half a wide-node visit in the SAH collapse (the watertight test of a
// prefetched triangle is cheaper than a node's 4-8 slab tests plus the sort;
// 0.5 measured 2-3% more incoherent closest-hit rays than 1.0 on a 1.32M
// triangle mesh, with the same hits).
constexpr int kDefaultLeafSize = 2;
constexpr float kDefaultSahTriCost = 0.5f;
// Leaves per refit block, four for each thread. A large block leaves fewer
// nodes that span blocks to the single block that does those (1.3M triangles:
// 15560 for 1024 leaves, 4809 for 4096), a small one spreads a small mesh over
// more CUs. Build times, 1024 / 2048 / 4096 leaves: 50K triangles 513, 519,
// 531 us; 200K 566, 571, 583; 600K 750, 714, 695; 1.3M 1093, 997, 960; 4M 2847,
// 2362, 2100.
constexpr int kRefitSmall = 1024, kRefitLarge = 4096;
constexpr int64_t kRefitLargeFrom = 400000;
// Collapse levels launched between two reads of the level sizes; a level past
// the last one is a launch of blocks that find no item (4 us), a read back is
// a wait of some 40 us.
constexpr int kCollapseLevelsPerSync = 16;
constexpr int kCollapseMaxLevels = 4096;
constexpr unsigned kCollapseMaxBlocks = 2048;

// What the build kernels count, on the device; cleared when a build starts.
struct BuildHead {
    float4 root_lo, root_hi;   // bounds of the root
    double sah;                // summed half areas of the collapse (unnormalised SAH cost)
    int32_t leaves;            // wide-tree leaves
    int32_t unsorted;          // the sort's result was not in order
    int32_t frontier;          // nodes left to k_refit_top
    int32_t pad;
    // wide nodes of each level, and the slot of the first: level l holds the
    // slots [first[l], first[l] + count[l])
    int32_t count[kCollapseMaxLevels + kCollapseLevelsPerSync + 1];
    int32_t first[kCollapseMaxLevels + kCollapseLevelsPerSync + 1];
};

// ---------------------------------------------------------------------------
// build kernels
// ---------------------------------------------------------------------------

__device__ __forceinline__ void tri_bounds(const float* v, float4& lo, float4& hi) {
    lo = make_float4(fminf(v[0], fminf(v[3], v[6])), fminf(v[1], fminf(v[4], v[7])), fminf(v[2], fminf(v[5], v[8])),
                     0.f);
    hi = make_float4(fmaxf(v[0], fmaxf(v[3], v[6])), fmaxf(v[1], fmaxf(v[4], v[7])), fmaxf(v[2], fmaxf(v[5], v[8])),
                     0.f);
}

// Per-triangle AABB (float4 lo, hi); per-block centroid bounds into
// `partial` (6 floats per block), reduced by k_reduce_bounds.
__global__ __launch_bounds__(256) void k_prep(const float* __restrict__ verts, int64_t n, float4* __restrict__ tlo,
                                              float4* __restrict__ thi, float* __restrict__ partial) {
    __shared__ float red[6][4];
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    float cmin[3] = {3e38f, 3e38f, 3e38f}, cmax[3] = {-3e38f, -3e38f, -3e38f};
    if (i < n) {
        float4 lo, hi;
        tri_bounds(verts + 9 * i, lo, hi);
        cmin[0] = cmax[0] = (lo.x + hi.x) * 0.5f;
        cmin[1] = cmax[1] = (lo.y + hi.y) * 0.5f;
        cmin[2] = cmax[2] = (lo.z + hi.z) * 0.5f;
        tlo[i] = lo;
        thi[i] = hi;
    }
    const int w = threadIdx.x >> 6;
    for (int a = 0; a < 3; a++) {
        float mn = cmin[a], mx = cmax[a];
        for (int off = 32; off > 0; off >>= 1) {
            mn = fminf(mn, __shfl_xor(mn, off));
            mx = fmaxf(mx, __shfl_xor(mx, off));
        }
        if ((threadIdx.x & 63) == 0) {
            red[a][w] = mn;
            red[3 + a][w] = mx;
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        float x = red[a][0];
        for (int k = 1; k < 4; k++) x = a < 3 ? fminf(x, red[a][k]) : fmaxf(x, red[a][k]);
        partial[6 * int64_t(blockIdx.x) + a] = x;
    }
}

// One block reduces the per-block partial bounds into cb[6] (floats).
__global__ __launch_bounds__(256) void k_reduce_bounds(const float* __restrict__ partial, int nparts,
                                                       float* __restrict__ cb) {
    __shared__ float red[6][4];
    float v[6] = {3e38f, 3e38f, 3e38f, -3e38f, -3e38f, -3e38f};
    for (int b = threadIdx.x; b < nparts; b += blockDim.x)
        for (int a = 0; a < 6; a++)
            v[a] = a < 3 ? fminf(v[a], partial[6 * b + a]) : fmaxf(v[a], partial[6 * b + a]);
    const int w = threadIdx.x >> 6;
    for (int a = 0; a < 6; a++) {
        float x = v[a];
        for (int off = 32; off > 0; off >>= 1) x = a < 3 ? fminf(x, __shfl_xor(x, off)) : fmaxf(x, __shfl_xor(x, off));
        if ((threadIdx.x & 63) == 0) red[a][w] = x;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        float x = red[a][0];
        for (int k = 1; k < 4; k++) x = a < 3 ? fminf(x, red[a][k]) : fmaxf(x, red[a][k]);
        cb[a] = x;
    }
}

__device__ __forceinline__ uint64_t spread21(uint64_t x) {
    x &= 0x1fffffull;
    x = (x | x << 32) & 0x1f00000000ffffull;
    x = (x | x << 16) & 0x1f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}

__global__ __launch_bounds__(256) void k_morton(const float4* __restrict__ tlo, const float4* __restrict__ thi,
                                                int64_t n, const float* __restrict__ cb,
                                                uint64_t* __restrict__ keys, int32_t* __restrict__ vals) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 lo = tlo[i], hi = thi[i];
    const float c[3] = {(lo.x + hi.x) * 0.5f, (lo.y + hi.y) * 0.5f, (lo.z + hi.z) * 0.5f};
    uint64_t code = 0;
    for (int a = 0; a < 3; a++) {
        const float mn = cb[a], mx = cb[3 + a];
        const float ext = mx - mn;
        float f = ext > 0.f ? (c[a] - mn) / ext : 0.5f;
        f = fminf(fmaxf(f, 0.f), 1.f);
        const uint64_t q = uint64_t(fminf(f * 2097152.0f, 2097151.0f));
        code |= spread21(q) << (2 - a);
    }
    keys[i] = code;
    vals[i] = int32_t(i);
}


// flag = 1 if keys[i] > keys[i + 1] for some i
__global__ __launch_bounds__(256) void k_check_sorted(const uint64_t* __restrict__ keys, int64_t n,
                                                      int32_t* __restrict__ flag) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i + 1 < n && keys[i] > keys[i + 1]) *flag = 1;
}

__device__ __forceinline__ int delta(const uint64_t* __restrict__ k, int64_t n, int64_t i, int64_t j) {
    if (j < 0 || j >= n) return -1;
    const uint64_t a = k[i], b = k[j];
    if (a == b) return 64 + __clzll(uint64_t(i ^ j));
    return __clzll(a ^ b);
}

__global__ __launch_bounds__(256) void k_lbvh(const uint64_t* __restrict__ k, int64_t n, BNode* __restrict__ bn,
                                              int32_t* __restrict__ parent_int, int32_t* __restrict__ parent_leaf) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = (delta(k, n, i, i + 1) - delta(k, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(k, n, i, i - d);
    int64_t lmax = 2;
    while (delta(k, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int64_t l = 0;
    for (int64_t t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(k, n, i, i + (l + t) * d) > dmin) l += t;
    const int64_t j = i + l * d;
    const int dnode = delta(k, n, i, j);
    int64_t s = 0;
    int64_t len = l;
    int64_t t = (len + 1) >> 1;
    while (true) {
        if (delta(k, n, i, i + (s + t) * d) > dnode) s += t;
        if (t == 1) break;
        t = (t + 1) >> 1;
    }
    const int64_t g = i + s * d + (d < 0 ? -1 : 0);
    const int64_t lo = i < j ? i : j, hi = i < j ? j : i;
    BNode node;
    node.first = int32_t(lo);
    node.last = int32_t(hi);
    if (lo == g) {
        node.left = ~int32_t(g);
        parent_leaf[g] = int32_t(i);
    } else {
        node.left = int32_t(g);
        parent_int[g] = int32_t(i);
    }
    if (hi == g + 1) {
        node.right = ~int32_t(g + 1);
        parent_leaf[g + 1] = int32_t(i);
    } else {
        node.right = int32_t(g + 1);
        parent_int[g + 1] = int32_t(i);
    }
    bn[i] = node;
}

__device__ __forceinline__ float half_area(float4 lo, float4 hi) {
    const float dx = hi.x - lo.x, dy = hi.y - lo.y, dz = hi.z - lo.z;
    return dx * dy + dy * dz + dz * dx;
}

// Parent links of a binary tree given by its nodes (parent_int[root] stays
// as initialised).
__global__ __launch_bounds__(256) void k_parents(const BNode* __restrict__ bn, int64_t m,
                                                 int32_t* __restrict__ parent_int, int32_t* __restrict__ parent_leaf) {
    const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= m) return;
    const BNode nd = bn[p];
    if (nd.left < 0) parent_leaf[~nd.left] = int32_t(p); else parent_int[nd.left] = int32_t(p);
    if (nd.right < 0) parent_leaf[~nd.right] = int32_t(p); else parent_int[nd.right] = int32_t(p);
}

// Cost tables of the SAH collapse (Ylitie, Karras and Laine, "Efficient
// Incoherent Ray Traversal on GPUs Through Compressed Wide BVHs", HPG 2017,
// sec. 4): for internal binary node p and i = 1..W, C(p, i) is the least SAH
// cost (half areas; a wide-node visit costs 1, a triangle test `ctri`) of
// covering p's subtree with at most i roots, each a wide node or a leaf.
//   C(p, 1) = min(A(p) * N(p) * ctri  [leaf, N(p) <= pmax],
//                 A(p) + D(p, W)       [wide node]),
//   C(p, i) = min(C(p, i - 1), D(p, i)),   D(p, j) = min_k C(L, k) + C(R, j - k),
// and a single triangle j costs A(j) * ctri for every i. choice[p*W + 0] is
// 0xFF for a leaf, else the k of D(p, W); choice[p*W + i - 1] (i >= 2) is 0
// when C(p, i) = C(p, i - 1), else the k of D(p, i).
struct SahDP {
    float* cost;
    uint8_t* choice;
    int pmax;
    float ctri;
};

template <int W>
__device__ __forceinline__ void sah_tables(const SahDP& dp, int32_t p, int32_t left, int32_t right, int cnt,
                                           float area, const float4& l0, const float4& h0, const float4& l1,
                                           const float4& h1) {
    float cl[W], cr[W];
    const float al = half_area(l0, h0) * dp.ctri, ar = half_area(l1, h1) * dp.ctri;
    // loaded for leaves too (from node 0's place), so that the loads need no branch
    const float* tl = dp.cost + int64_t(max(left, 0)) * W;
    const float* tr = dp.cost + int64_t(max(right, 0)) * W;
    for (int i = 0; i < W; i++) {
        cl[i] = tl[i];
        cr[i] = tr[i];
    }
    for (int i = 0; i < W; i++) {
        cl[i] = left < 0 ? al : cl[i];
        cr[i] = right < 0 ? ar : cr[i];
    }
    float dist[W];
    int arg[W];
#pragma unroll
    for (int j = 2; j <= W; j++) {
        float best = __builtin_inff();
        int bk = 1;
#pragma unroll
        for (int k = 1; k < j; k++) {
            const float c = cl[k - 1] + cr[j - k - 1];
            if (c < best) { best = c; bk = k; }
        }
        dist[j - 1] = best;
        arg[j - 1] = bk;
    }
    const float cint = area + dist[W - 1];
    const float cprim = cnt <= dp.pmax ? area * float(cnt) * dp.ctri : __builtin_inff();
    float c = fminf(cprim, cint);
    float* out = dp.cost + int64_t(p) * W;
    uint8_t* ch = dp.choice + int64_t(p) * W;
    out[0] = c;
    ch[0] = cprim <= cint ? uint8_t(0xFF) : uint8_t(arg[W - 1]);
#pragma unroll
    for (int i = 2; i <= W; i++) {
        if (c <= dist[i - 1]) {
            ch[i - 1] = 0;
        } else {
            c = dist[i - 1];
            ch[i - 1] = uint8_t(arg[i - 1]);
        }
        out[i - 1] = c;
    }
}

// Bottom-up refit. A node is done by the thread that counts its second child
// as done, in the round after: rounds are separated by a barrier of the one
// block whose threads wrote both children, so no device-scope fence (a write
// back of the per-XCD L2s) is needed and no launch per level either.
//
// A round is bound by latency, and a mesh of 1.3M triangles takes 22 rounds
// in the blocks and 28 above them: the list holds what a node's loads need, so
// its children and its parent's links are read side by side. That mesh takes
// 214 us in the blocks (with the 42 us of the triangles' gather) and 96 us
// above them; a launch per level over a global list with an atomic per wave
// took 890 us, and the gather was a pass of its own.
struct Refit {
    const BNode* bn;
    const int32_t* parent_int;
    const int32_t* parent_leaf;
    float4* leaf_lo;
    float4* leaf_hi;
    float4* node_lo;
    float4* node_hi;
    int32_t* flags;      // children done, of the nodes that span blocks
    int32_t root;
    SahDP dp;
    BuildHead* head;
};

// A node whose children are done.
struct RefitItem {
    int32_t node, parent, left, right;
    int32_t first, last;
};

__device__ __forceinline__ RefitItem refit_item(const Refit& r, int32_t q) {
    const BNode nd = r.bn[q];
    return RefitItem{q, r.parent_int[q], nd.left, nd.right, nd.first, nd.last};
}

// Bounds and cost tables of a listed node.
template <int W>
__device__ __forceinline__ void refit_node(const Refit& r, const RefitItem it) {
    const float4 l0 = *(it.left < 0 ? r.leaf_lo + ~it.left : r.node_lo + it.left);
    const float4 h0 = *(it.left < 0 ? r.leaf_hi + ~it.left : r.node_hi + it.left);
    const float4 l1 = *(it.right < 0 ? r.leaf_lo + ~it.right : r.node_lo + it.right);
    const float4 h1 = *(it.right < 0 ? r.leaf_hi + ~it.right : r.node_hi + it.right);
    const float4 lo = make_float4(fminf(l0.x, l1.x), fminf(l0.y, l1.y), fminf(l0.z, l1.z), 0.f);
    const float4 hi = make_float4(fmaxf(h0.x, h1.x), fmaxf(h0.y, h1.y), fmaxf(h0.z, h1.z), 0.f);
    if (r.dp.cost)
        sah_tables<W>(r.dp, it.node, it.left, it.right, it.last - it.first + 1, half_area(lo, hi), l0, h0, l1, h1);
    r.node_lo[it.node] = lo;
    r.node_hi[it.node] = hi;
    if (it.node == r.root) {
        r.head->root_lo = lo;
        r.head->root_hi = hi;
    }
}

// The leaves [SPAN * block, + SPAN): their triangles in traversal
// order and bounds, and every node above whose range of leaves lies within
// them, in rounds over a list of ready nodes in LDS (at most half the leaves,
// and never longer than the one before it: each parent enters by exactly one
// child). Children done are counted in LDS too, by the last leaf of the node's
// left child, which no other node shares. A ready node that spans blocks is
// counted in memory and goes to `frontier`: such nodes have disjoint ranges,
// so there are fewer than blocks.
template <int W, int SPAN>
__global__ __launch_bounds__(SPAN / 4) void k_refit_blocks(int64_t n, const int32_t* __restrict__ order,
                                                         const float* __restrict__ verts, TriV* __restrict__ tris,
                                                         Refit r, RefitItem* __restrict__ frontier) {
    constexpr int kBlock = SPAN / 4;
    constexpr int kHalf = SPAN / 2;
    __shared__ int4 links[2 * kHalf];        // RefitItem: node, parent, left, right
    __shared__ uint32_t range[2 * kHalf];    // its first and last leaf, in 16 bits each from the block's first
    __shared__ uint32_t done[SPAN / 4];
    __shared__ int32_t size[2];
    constexpr int kPer = SPAN / kBlock;
    const int32_t lead = int32_t(blockIdx.x) * SPAN;
    const int32_t tail = int32_t(std::min<int64_t>(n, int64_t(lead) + SPAN) - 1);
    if (threadIdx.x < 2) size[threadIdx.x] = 0;
    static_assert(SPAN / 4 <= kBlock && SPAN <= 65536, "one word of `done` per thread, 16-bit ranges");
    if (threadIdx.x < SPAN / 4) done[threadIdx.x] = 0;
    __syncthreads();
    // the child [first, last] of q's node is done
    auto arrive = [&](const RefitItem q, int32_t first, int32_t last, int to) {
        if (q.first >= lead && q.last <= tail) {
            const uint32_t g = uint32_t((q.first == first ? last : first - 1) - lead);
            const uint32_t sh = 8 * (g & 3);
            if ((atomicAdd(&done[g >> 2], 1u << sh) >> sh & 0xffu) != 1u) return;
            const int k = to * kHalf + atomicAdd(&size[to], 1);
            links[k] = make_int4(q.node, q.parent, q.left, q.right);
            range[k] = uint32_t(q.first - lead) | uint32_t(q.last - lead) << 16;
        } else if (atomicAdd(&r.flags[q.node], 1) == 1) {
            frontier[atomicAdd(&r.head->frontier, 1)] = q;
        }
    };
    int32_t ti[kPer], up[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int32_t j = min(lead + int32_t(threadIdx.x) + kBlock * k, tail);
        ti[k] = order[j];
        up[k] = n > 1 ? r.parent_leaf[j] : 0;
    }
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int32_t j = lead + int32_t(threadIdx.x) + kBlock * k;
        if (j > tail) break;
        float v[9];
#pragma unroll
        for (int c = 0; c < 9; c++) v[c] = verts[9 * int64_t(ti[k]) + c];
        RefitItem q{};
        if (n > 1) q = refit_item(r, up[k]);
        TriV t;
        t.v0 = make_float4(v[0], v[1], v[2], __int_as_float(ti[k]));
        t.v1 = make_float4(v[3], v[4], v[5], 0.f);
        t.v2 = make_float4(v[6], v[7], v[8], 0.f);
        tris[j] = t;
        float4 lo, hi;
        tri_bounds(v, lo, hi);
        r.leaf_lo[j] = lo;
        r.leaf_hi[j] = hi;
        if (n > 1) {
            arrive(q, j, j, 0);
        } else {
            r.head->root_lo = lo;
            r.head->root_hi = hi;
        }
    }
    int cur = 0;
    while (true) {
        __syncthreads();
        const int m = size[cur];
        if (m == 0) break;
        for (int i = threadIdx.x; i < m; i += kBlock) {
            const int4 l = links[cur * kHalf + i];
            const uint32_t f = range[cur * kHalf + i];
            const RefitItem it{l.x, l.y, l.z, l.w, lead + int32_t(f & 0xffffu), lead + int32_t(f >> 16)};
            const RefitItem q = refit_item(r, max(it.parent, 0));
            refit_node<W>(r, it);
            if (it.node != r.root) arrive(q, it.first, it.last, cur ^ 1);
        }
        __syncthreads();
        if (threadIdx.x == 0) size[cur] = 0;
        cur ^= 1;
    }
}

// The nodes above the blocks: one block, rounds as above over lists in global
// memory (list0 holds head->frontier items). They are some 1% of the nodes, so
// one block's rate costs less than a launch per level.
template <int W>
__global__ __launch_bounds__(1024) void k_refit_top(Refit r, RefitItem* __restrict__ list0,
                                                    RefitItem* __restrict__ list1) {
    __shared__ int32_t size[2];
    if (threadIdx.x == 0) {
        size[0] = r.head->frontier;
        size[1] = 0;
    }
    const RefitItem* in = list0;
    RefitItem* out = list1;
    int cur = 0;
    while (true) {
        __syncthreads();
        const int m = size[cur];
        if (m == 0) break;
        for (int i = threadIdx.x; i < m; i += 1024) {
            const RefitItem it = in[i];
            const int32_t up = max(it.parent, 0);
            const int32_t before = it.node != r.root ? atomicAdd(&r.flags[up], 1) : 0;
            const RefitItem q = refit_item(r, up);
            refit_node<W>(r, it);
            if (before == 1) out[atomicAdd(&size[cur ^ 1], 1)] = q;
        }
        __syncthreads();
        if (threadIdx.x == 0) size[cur] = 0;
        cur ^= 1;
        RefitItem* t = const_cast<RefitItem*>(in);
        in = out;
        out = t;
    }
}

// One level of the collapse into W-wide nodes: item i of the level is the
// binary ref of the wide node in slot first[level] + i, and the nodes' inner
// children are the next level's items.
struct CollapseArgs {
    const int32_t* in;
    int32_t* out;
    int level;
    const BNode* bn;
    const float4* node_lo;
    const float4* node_hi;
    const float4* leaf_lo;
    const float4* leaf_hi;
    const uint8_t* choice;   // SAH collapse: sah_tables
    int leaf_size;           // greedy collapse
    void* wnodes;
    BuildHead* head;
};

// Runs a level: `expand(bref, ref, nc)` finds the nc <= W refs a wide node of
// `bref` has as children and returns the mask of those that are not leaves. The
// wide children of one node take consecutive slots, so siblings share cache
// lines. Whole blocks take their nodes' slots with one atomic, and the SAH
// sum and leaf count of all a block's items are added once: same-address
// atomics cost 12 ns each on the card, and with four per wave they were most
// of the collapse's time (1.3M triangles, W = 4, 17 levels: 445 us, now
// 220 us, at 10 to 33 us a level mostly the latency of the unfolding).
template <int W, class Expand>
__device__ __forceinline__ void collapse_level(const CollapseArgs& a, Expand expand) {
    __shared__ int32_t wave_sum[4];
    __shared__ int32_t block_base;
    __shared__ double block_sah[4];
    __shared__ int32_t block_leaves[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int32_t count = a.head->count[a.level], first = a.head->first[a.level];
    const int32_t next = first + count;   // slot of the next level's first node
    if (blockIdx.x == 0 && threadIdx.x == 0) a.head->first[a.level + 1] = next;
    WNode<W>* wnodes = static_cast<WNode<W>*>(a.wnodes);
    double sah = 0.0;
    int nleaf = 0;
    for (int64_t base = int64_t(blockIdx.x) * 256; base < count; base += int64_t(gridDim.x) * 256) {
        const int64_t idx = base + threadIdx.x;
        int32_t ref[W];
        int nc = 0, nint = 0;
        uint32_t inner = 0;
        if (idx < count) {
            inner = expand(a.in[idx], ref, nc);
            nint = __popc(inner);
        }
        int inc = nint;
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(inc, off);
            if (lane >= off) inc += y;
        }
        if (lane == 63) wave_sum[w] = inc;
        __syncthreads();
        int before = 0, total = 0;
        for (int k = 0; k < 4; k++) {
            before += k < w ? wave_sum[k] : 0;
            total += wave_sum[k];
        }
        if (threadIdx.x == 0) block_base = total ? atomicAdd(&a.head->count[a.level + 1], total) : 0;
        __syncthreads();
        int32_t q = block_base + before + inc - nint;
        if (idx < count) {
            WNode<W> node;
            for (int c = 0; c < W; c++) {
                if (c < nc) {
                    const int32_t r = ref[c];
                    const float4 lo = r < 0 ? a.leaf_lo[~r] : a.node_lo[r];
                    const float4 hi = r < 0 ? a.leaf_hi[~r] : a.node_hi[r];
                    node.lox[c] = lo.x; node.loy[c] = lo.y; node.loz[c] = lo.z;
                    node.hix[c] = hi.x; node.hiy[c] = hi.y; node.hiz[c] = hi.z;
                    const double area = double(half_area(lo, hi));
                    if (inner >> c & 1u) {
                        node.child[c] = next + q;
                        node.count[c] = 0;
                        sah += area;
                        a.out[q++] = r;
                    } else {
                        const int cnt = r < 0 ? 1 : a.bn[r].last - a.bn[r].first + 1;
                        node.child[c] = r < 0 ? ~r : a.bn[r].first;
                        node.count[c] = cnt;
                        sah += area * cnt;
                        nleaf++;
                    }
                } else {
                    node.lox[c] = node.loy[c] = node.loz[c] = 1e30f;
                    node.hix[c] = node.hiy[c] = node.hiz[c] = -1e30f;
                    node.child[c] = 0;
                    node.count[c] = -1;
                }
            }
            wnodes[first + idx] = node;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        sah += __shfl_xor(sah, off);
        nleaf += __shfl_xor(nleaf, off);
    }
    if (lane == 0) {
        block_sah[w] = sah;
        block_leaves[w] = nleaf;
    }
    __syncthreads();
    if (threadIdx.x == 0 && int64_t(blockIdx.x) * 256 < count) {
        atomicAdd(&a.head->sah, block_sah[0] + block_sah[1] + block_sah[2] + block_sah[3]);
        atomicAdd(&a.head->leaves, block_leaves[0] + block_leaves[1] + block_leaves[2] + block_leaves[3]);
    }
}

// SAH collapse: a wide node's children are the roots the cost tables chose
// for D(p, W) (sah_tables), found by unfolding the choices with a stack of
// (ref, slots) pairs whose slots sum to at most W.
template <int W>
__global__ __launch_bounds__(256) void k_collapse_sah(CollapseArgs a) {
    // a node's W choices as one word, read together with the node itself: a
    // step of the unfolding waits once for memory (17 levels 245 -> 220 us)
    using Row = std::conditional_t<W == 2, uint16_t, std::conditional_t<W == 4, uint32_t, uint64_t>>;
    auto row_of = [&](int32_t r) { return reinterpret_cast<const Row*>(a.choice)[r]; };
    auto choice = [](Row row, int i) { return int(row >> (8 * i)) & 0xff; };
    auto expand = [&](int32_t bref, int32_t (&ref)[W], int& nc) -> uint32_t {
        const Row first = row_of(max(bref, 0));
        const BNode b = a.bn[max(bref, 0)];
        if (bref < 0 || choice(first, 0) == 0xFF) {
            ref[nc++] = bref;   // the whole tree is one leaf (tiny scenes)
            return 0;
        }
        uint32_t inner = 0;
        int32_t sr[W];
        int sj[W];
        int sp = 0;
        const int k = choice(first, 0);
        sr[sp] = b.right; sj[sp++] = W - k;
        sr[sp] = b.left; sj[sp++] = k;
        while (sp > 0) {
            --sp;
            const int32_t m = sr[sp];
            int j = sj[sp];
            const Row row = row_of(max(m, 0));
            const BNode bm = a.bn[max(m, 0)];
            if (m >= 0)
                while (j > 1 && choice(row, j - 1) == 0) j--;
            if (m < 0 || j == 1) {
                if (m >= 0 && choice(row, 0) != 0xFF) inner |= 1u << nc;
                ref[nc++] = m;
                continue;
            }
            const int c = choice(row, j - 1);
            sr[sp] = bm.right; sj[sp++] = j - c;
            sr[sp] = bm.left; sj[sp++] = c;
        }
        return inner;
    };
    collapse_level<W>(a, expand);
}

// Greedy collapse: open the largest-area child until there are W.
template <int W>
__global__ __launch_bounds__(256) void k_collapse(CollapseArgs a) {
    auto cnt_of = [&](int32_t r) -> int { return r < 0 ? 1 : a.bn[r].last - a.bn[r].first + 1; };
    auto lo_of = [&](int32_t r) { return r < 0 ? a.leaf_lo[~r] : a.node_lo[r]; };
    auto hi_of = [&](int32_t r) { return r < 0 ? a.leaf_hi[~r] : a.node_hi[r]; };
    auto is_leaf = [&](int32_t r) { return r < 0 || cnt_of(r) <= a.leaf_size; };
    auto expand = [&](int32_t bref, int32_t (&ref)[W], int& nc) -> uint32_t {
        if (is_leaf(bref)) {
            ref[nc++] = bref;   // whole range is one leaf (tiny scenes)
            return 0;
        }
        ref[nc++] = a.bn[bref].left;
        ref[nc++] = a.bn[bref].right;
        while (nc < W) {
            int best = -1;
            float best_a = -1.f;
            for (int c = 0; c < nc; c++) {
                if (!is_leaf(ref[c])) {
                    const float area = half_area(lo_of(ref[c]), hi_of(ref[c]));
                    if (area > best_a) { best_a = area; best = c; }
                }
            }
            if (best < 0) break;
            const BNode b = a.bn[ref[best]];
            ref[best] = b.left;
            ref[nc++] = b.right;
        }
        uint32_t inner = 0;
        for (int c = 0; c < nc; c++)
            if (!is_leaf(ref[c])) inner |= 1u << c;
        return inner;
    };
    collapse_level<W>(a, expand);
}

__global__ void k_collapse_init(BuildHead* head, int32_t* items, int32_t root_ref) {
    head->count[0] = 1;
    head->first[0] = 0;
    items[0] = root_ref;
}

// ---------------------------------------------------------------------------
// ray-cast kernels
// ---------------------------------------------------------------------------

constexpr int kTraceBlock = 256;
constexpr int kLdsDepth = 24;
constexpr int kPrivDepth = 72;

// Persistent closest-hit / any-hit kernel over a ray array (bvh.h,
// trace_persistent). `next` is this launch's ray counter, zeroed by
// k_zero_counter on the same stream.
template <int W, bool ANY, bool COUNT, class Node>
__global__ __launch_bounds__(kTraceBlock, 6) void k_trace(const Node* __restrict__ nodes,
                                                        const TriV* __restrict__ tris,
                                                        const lmgpu_ray* __restrict__ rays,
                                                        lmgpu_hit* __restrict__ hits, uint8_t* __restrict__ occl,
                                                        uint32_t n, unsigned long long* __restrict__ next,
                                                        int32_t* __restrict__ status,
                                                        unsigned long long* __restrict__ counters, int refill) {
    __shared__ int lds[kLdsDepth + 1][kTraceBlock];
    auto fetch = [&](uint32_t id, f3& o, f3& d, float& tmin, float& tmax) -> int {
        const float4* rp = reinterpret_cast<const float4*>(rays + id);
        const float4 a = rp[0], c = rp[1];
        o = mk(a.x, a.y, a.z);
        d = mk(c.x, c.y, c.z);
        tmin = a.w;
        tmax = c.w;
        return 0;
    };
    auto emit = [&](uint32_t id, const TraceResult& r) {
        if (ANY) {
            occl[id] = r.prim >= 0 ? 1 : 0;
        } else {
            reinterpret_cast<float4*>(hits)[id] =
                make_float4(__int_as_float(r.prim), r.prim >= 0 ? r.t : 0.f, r.u, r.v);
        }
    };
    trace_persistent<W, ANY, COUNT, kLdsDepth, kPrivDepth, kTraceBlock>(nodes, tris, n, next, lds, fetch, emit,
                                                                         status, counters, refill);
}

// Quantised copy of a built W-wide node array (bvh.h, quantise_node), four
// lanes per node: one for each axis's planes, one for the child entries. A
// wave reads and writes 16 whole nodes side by side; a thread per node kept 64
// lines in flight for each of its loads and refetched them (454K nodes, W = 4:
// 171 us, now 31 us).
template <int W>
__global__ __launch_bounds__(256) void k_quantise(const WNode<W>* __restrict__ in, QNode<W>* __restrict__ out,
                                                  int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * 64 + (threadIdx.x >> 2);
    const int a = threadIdx.x & 3;
    if (i >= n) return;   // whole quads
    const WNode<W>& node = in[i];
    QNode<W>& q = out[i];
    const float* planes = reinterpret_cast<const float*>(&node);
    float lo[W], hi[W];   // lane 3: the words of child and count
    for (int c = 0; c < W; c++) {
        lo[c] = planes[(a < 3 ? a : 6) * W + c];
        hi[c] = planes[(a < 3 ? 3 + a : 7) * W + c];
    }
    uint32_t present = 0;
    for (int c = 0; c < W; c++) present |= __float_as_int(hi[c]) >= 0 ? 1u << c : 0u;
    present = __shfl(present, 3, 4);
    QAxis<W> x{};
    if (a < 3) x = quantise_axis<W>(lo, hi, present);
    uint32_t e = a < 3 ? uint32_t(x.e & 0xff) << (8 * a) : 0u;
    for (int off = 1; off < 4; off <<= 1) e |= __shfl_xor(e, off, 4);
    if (a < 3) {
        (a == 0 ? q.ox : a == 1 ? q.oy : q.oz) = x.org;
        for (int k = 0; k < W / 4; k++) {
            q.qlo[a][k] = x.ql[k];
            q.qhi[a][k] = x.qh[k];
        }
    } else {
        q.e = e;
        for (int c = 0; c < W; c++) q.ent[c] = quantised_entry(__float_as_int(lo[c]), __float_as_int(hi[c]));
    }
}

__global__ void k_zero_counter(unsigned long long* c) {
    if (threadIdx.x < kRayCounters) c[threadIdx.x * kRayCounterStride] = 0ull;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

static inline unsigned nblocks(int64_t n, int b) { return unsigned((n + b - 1) / b); }

// Leaves, triangles in traversal order, and every node's bounds (and tables).
template <int W>
static void launch_refit(int64_t n, const int32_t* order, const float* verts, TriV* tris, const Refit& r,
                         RefitItem* list0, RefitItem* list1, hipStream_t s) {
    auto blocks = [&](auto span) {
        constexpr int SPAN = decltype(span)::value;
        hipLaunchKernelGGL((k_refit_blocks<W, SPAN>), dim3(nblocks(n, SPAN)), dim3(SPAN / 4), 0, s, n, order, verts,
                           tris, r, list0);
        if (n > SPAN) hipLaunchKernelGGL(k_refit_top<W>, dim3(1), dim3(1024), 0, s, r, list0, list1);
    };
    if (n < kRefitLargeFrom) blocks(std::integral_constant<int, kRefitSmall>{});
    else blocks(std::integral_constant<int, kRefitLarge>{});
}

template <int W>
static void launch_collapse(bool by_sah, const CollapseArgs& a, unsigned grid, hipStream_t s) {
    if (by_sah) hipLaunchKernelGGL(k_collapse_sah<W>, dim3(grid), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(k_collapse<W>, dim3(grid), dim3(256), 0, s, a);
}

// A buffer kept from the last build serves one of a similar size (it may be up
// to twice what is needed), so that a mesh rebuilt every frame allocates
// nothing: hipMalloc and hipFree of the arrays of 1.3M triangles took 5.5 of a
// rebuild's 7.5 ms.
template <class T>
static bool fits(const DevBuf<T>& b, size_t count) {
    return b.p && b.n >= count && b.n / 2 <= count;
}

template <class T>
static int reserve(DevBuf<T>& b, size_t count) {
    return fits(b, count) ? LMGPU_OK : b.alloc(count);
}

// With what an object keeps from its last tree a build can find less memory
// than a first one would: it then starts again as a first one.
int Accel::build(const float* verts, int64_t n, bool on_device, const lmgpu_build_opts* opts, hipStream_t s) {
    const bool kept = nodes.p != nullptr;
    int rc = build_once(verts, n, on_device, opts, s);
    if (rc == LMGPU_ERR_OUT_OF_MEMORY && kept) {
        release();
        (void)hipGetLastError();
        clear_error();
        rc = build_once(verts, n, on_device, opts, s);
    }
    if (rc != LMGPU_OK && !built) release();
    return rc;
}

int Accel::build_once(const float* verts_in, int64_t n, bool on_device, const lmgpu_build_opts* opts, hipStream_t s) {
    int W = opts && opts->width ? opts->width : 4;
    int leaf = opts && opts->leaf_size ? opts->leaf_size : kDefaultLeafSize;
    const int rf = opts && opts->refill ? opts->refill : kDefaultRefill;
    if (rf < 1 || rf > 64) return fail(LMGPU_ERR_INVALID_ARGUMENT, "refill must be in [1, 64]");
    const int builder = opts ? opts->builder : LMGPU_BUILDER_LBVH;
    if (builder != LMGPU_BUILDER_PLOC && builder != LMGPU_BUILDER_LBVH)
        return fail(LMGPU_ERR_INVALID_ARGUMENT, "unknown builder");
    const int collapse = opts ? opts->collapse : LMGPU_COLLAPSE_SAH;
    if (collapse != LMGPU_COLLAPSE_SAH && collapse != LMGPU_COLLAPSE_GREEDY)
        return fail(LMGPU_ERR_INVALID_ARGUMENT, "unknown collapse");
    const float ctri = opts && opts->sah_tri_cost > 0.f ? opts->sah_tri_cost : kDefaultSahTriCost;
    if (!(ctri > 0.f && ctri < 1e6f)) return fail(LMGPU_ERR_INVALID_ARGUMENT, "sah_tri_cost out of range");
    const int radius = opts && opts->ploc_radius ? opts->ploc_radius : 16;
    if (W != 2 && W != 4 && W != 8) return fail(LMGPU_ERR_INVALID_ARGUMENT, "BVH width must be 2, 4 or 8");
    if (leaf < 1 || leaf > 15) return fail(LMGPU_ERR_INVALID_ARGUMENT, "leaf_size must be in [1, 15]");
    if (n <= 0) return fail(LMGPU_ERR_INVALID_ARGUMENT, "accel build needs at least one triangle");
    if (n >= (int64_t(1) << 27)) return fail(LMGPU_ERR_INVALID_ARGUMENT, "too many triangles (max 2^27)");
    if (!verts_in) return fail(LMGPU_ERR_INVALID_ARGUMENT, "verts is NULL");
    // A rebuild writes over the tree (and the workspace) of the last one:
    // queries still in flight, on whichever stream, come first.
    const bool rebuild = built_here;
    if (nodes.p) LMGPU_HIP(hipDeviceSynchronize());
    built = built_here = false;
    if (!fits(tris, n)) tris.reset();
    if (!fits(nodes, size_t(n) * 2 * W)) {
        nodes.reset();
        qnodes.reset();
    }
    width = W;
    leaf_size = leaf;
    refill = rf;
    num_tris = n;
    struct GiveBack {
        DevBuf<char>& w;
        bool keep;
        ~GiveBack() {
            if (!keep) w.reset();
        }
    } give_back{work, false};   // also when the build fails
    // temporary arrays: one allocation, laid out by the first pass over take()
    const int64_t m = std::max<int64_t>(n - 1, 1);   // binary internal nodes
    const unsigned nb_prep = nblocks(n, 256);
    const size_t sort_bytes = radix_sort_temp_bytes(n);
    const bool sah = collapse == LMGPU_COLLAPSE_SAH;
    float4 *tlo, *thi, *leaf_lo, *leaf_hi, *node_lo, *node_hi;
    float *cb, *partial, *dverts;
    uint64_t *keys, *keys2;
    int32_t *vals, *vals2, *parent_int, *parent_leaf, *flags, *q0, *q1, *perm;
    BNode* bn;
    BuildHead* head;
    char* sort_temp;
    SahDP dp{nullptr, nullptr, leaf, ctri};
    for (int pass = 0; pass < 2; pass++) {
        size_t used = 0;
        auto take = [&](auto*& ptr, size_t count) {
            ptr = pass ? reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(work.p + used) : nullptr;
            used += (count * sizeof(*ptr) + 255) & ~size_t(255);
        };
        take(tlo, n); take(thi, n);
        take(leaf_lo, n); take(leaf_hi, n);
        take(node_lo, m); take(node_hi, m);
        take(cb, 6);
        take(partial, size_t(nb_prep) * 6);
        take(keys, n); take(keys2, n);
        take(vals, n); take(vals2, n);
        take(parent_int, m);
        take(parent_leaf, n);
        take(flags, m);
        take(head, 1);
        take(bn, m);
        take(q0, n); take(q1, n);
        take(sort_temp, sort_bytes);
        take(perm, builder == LMGPU_BUILDER_PLOC ? n : 0);
        take(dverts, on_device ? 0 : size_t(n) * 9);
        take(dp.cost, sah ? size_t(m) * W : 0);
        take(dp.choice, sah ? size_t(m) * W : 0);
        if (pass == 0) LMGPU_TRY(reserve(work, used));
    }
    if (!sah) {
        dp.cost = nullptr;
        dp.choice = nullptr;
    }
    const float* verts = verts_in;
    if (!on_device) {
        LMGPU_HIP(hipMemcpyAsync(dverts, verts_in, sizeof(float) * 9 * n, hipMemcpyHostToDevice, s));
        verts = dverts;
    }
    struct Events {
        hipEvent_t from = nullptr, to = nullptr;
        ~Events() {
            if (from) (void)hipEventDestroy(from);
            if (to) (void)hipEventDestroy(to);
        }
    } ev;
    LMGPU_HIP(hipEventCreate(&ev.from));
    LMGPU_HIP(hipEventCreate(&ev.to));
    LMGPU_HIP(hipEventRecord(ev.from, s));

    LMGPU_HIP(hipMemsetAsync(head, 0, sizeof(BuildHead), s));
    hipLaunchKernelGGL(k_prep, dim3(nb_prep), dim3(256), 0, s, verts, n, tlo, thi, partial);
    hipLaunchKernelGGL(k_reduce_bounds, dim3(1), dim3(256), 0, s, partial, int(nb_prep), cb);
    hipLaunchKernelGGL(k_morton, dim3(nblocks(n, 256)), dim3(256), 0, s, tlo, thi, n, cb, keys, vals);
    bool in_alt = false;
    LMGPU_TRY(radix_sort_pairs_u64(keys, vals, keys2, vals2, n, 63, &in_alt, sort_temp, s));
    const uint64_t* skeys = in_alt ? keys2 : keys;
    const int32_t* svals = in_alt ? vals2 : vals;
    if (n > 1) {
        // the sort's result must be ordered before the tree is built on it
        hipLaunchKernelGGL(k_check_sorted, dim3(nblocks(n - 1, 256)), dim3(256), 0, s, skeys, n, &head->unsorted);
        int32_t unsorted = 0;
        LMGPU_HIP(hipMemcpyAsync(&unsorted, &head->unsorted, sizeof(int32_t), hipMemcpyDeviceToHost, s));
        LMGPU_HIP(hipStreamSynchronize(s));
        if (unsorted) return fail(LMGPU_ERR_DEVICE, "Morton sort produced an unordered key array");
    }
    // binary tree over the sorted triangles: bn, parent links, and `order`
    // (traversal position -> triangle)
    int32_t root_ref = n > 1 ? 0 : ~0;
    const int32_t* order = svals;
    if (n > 1) LMGPU_HIP(hipMemsetAsync(parent_int, 0xff, sizeof(int32_t) * (n - 1), s));
    if (builder == LMGPU_BUILDER_PLOC) {
        LMGPU_TRY(build_ploc(n, svals, tlo, thi, radius, bn, node_lo, node_hi, leaf_lo, leaf_hi,
                             perm, &root_ref, s));
        order = perm;
        if (n > 1)
            hipLaunchKernelGGL(k_parents, dim3(nblocks(n - 1, 256)), dim3(256), 0, s, bn, n - 1, parent_int,
                               parent_leaf);
    } else if (n > 1) {
        hipLaunchKernelGGL(k_lbvh, dim3(nblocks(n - 1, 256)), dim3(256), 0, s, skeys, n, bn, parent_int,
                           parent_leaf);
    }
    // refit (bounds, and the SAH cost tables when collapsing by SAH); q0 and
    // q1 hold the nodes left to its second kernel
    if (n > 1) LMGPU_HIP(hipMemsetAsync(flags, 0, sizeof(int32_t) * (n - 1), s));
    const Refit refit{bn, parent_int, parent_leaf, leaf_lo, leaf_hi, node_lo, node_hi, flags, root_ref,
                      dp, head};
    LMGPU_TRY(reserve(tris, n));
    auto* list0 = reinterpret_cast<RefitItem*>(q0);
    auto* list1 = reinterpret_cast<RefitItem*>(q1);
    if (W == 2) launch_refit<2>(n, order, verts, tris.p, refit, list0, list1, s);
    else if (W == 4) launch_refit<4>(n, order, verts, tris.p, refit, list0, list1, s);
    else launch_refit<8>(n, order, verts, tris.p, refit, list0, list1, s);

    // collapse, level by level
    const size_t node_bytes = size_t(32) * W;
    const int64_t max_nodes = std::max<int64_t>(n, 1);
    LMGPU_TRY(reserve(nodes, size_t(max_nodes) * node_bytes / sizeof(float4)));
    hipLaunchKernelGGL(k_collapse_init, dim3(1), dim3(1), 0, s, head, q0, root_ref);
    CollapseArgs ca{q0, q1, 0, bn, node_lo, node_hi, leaf_lo, leaf_hi, dp.choice, leaf, nodes.p, head};
    // Levels are launched kCollapseLevelsPerSync at a time, each reading its
    // own size; their grids cover what the last size read can have become.
    int64_t bound = 1;
    int levels = 0;
    num_nodes = 0;
    while (levels == ca.level) {
        if (ca.level >= kCollapseMaxLevels) return fail(LMGPU_ERR_DEVICE, "BVH collapse did not terminate");
        const int at = ca.level;
        for (int l = 0; l < kCollapseLevelsPerSync; l++) {
            const unsigned grid = std::min(nblocks(bound, 256), kCollapseMaxBlocks);
            if (W == 2) launch_collapse<2>(sah, ca, grid, s);
            else if (W == 4) launch_collapse<4>(sah, ca, grid, s);
            else launch_collapse<8>(sah, ca, grid, s);
            bound = std::min<int64_t>(bound * W, n);
            ca.level++;
            ca.out = const_cast<int32_t*>(ca.in);
            ca.in = ca.in == q0 ? q1 : q0;
        }
        int32_t sizes[kCollapseLevelsPerSync + 1];
        LMGPU_HIP(hipMemcpyAsync(sizes, head->count + at, sizeof(sizes), hipMemcpyDeviceToHost, s));
        LMGPU_HIP(hipStreamSynchronize(s));
        for (int l = 0; l < kCollapseLevelsPerSync && sizes[l] > 0; l++) {
            num_nodes += sizes[l];
            levels++;
        }
        bound = sizes[kCollapseLevelsPerSync];
        if (bound == 0) break;
    }
    LMGPU_HIP(hipEventRecord(ev.to, s));
    BuildHead h;   // its counters; the level sizes are known
    LMGPU_HIP(hipMemcpyAsync(&h, head, offsetof(BuildHead, count), hipMemcpyDeviceToHost, s));
    LMGPU_HIP(hipStreamSynchronize(s));
    float ms = 0;
    LMGPU_HIP(hipEventElapsedTime(&ms, ev.from, ev.to));
    // root half-area for the SAH normalisation
    const float4 rlo = h.root_lo, rhi = h.root_hi;
    const double ra = double(rhi.x - rlo.x) * (rhi.y - rlo.y) + double(rhi.y - rlo.y) * (rhi.z - rlo.z) +
                      double(rhi.z - rlo.z) * (rhi.x - rlo.x);
    num_leaves = h.leaves;
    depth = levels;
    sah_cost = ra > 0 ? 1.0 + h.sah / ra : 1.0;
    build_ms = ms;
    root_lo[0] = rlo.x; root_lo[1] = rlo.y; root_lo[2] = rlo.z;
    root_hi[0] = rhi.x; root_hi[1] = rhi.y; root_hi[2] = rhi.z;
    LMGPU_TRY(make_trav_nodes(s));
    LMGPU_HIP(hipGetLastError());
    give_back.keep = rebuild && work.n <= kKeptWorkBytes;
    built = built_here = true;
    return LMGPU_OK;
}

bool quantised_width(int width) {
    return (width == 4 && std::is_same<TravNode<4>::type, QNode<4>>::value) ||
           (width == 8 && std::is_same<TravNode<8>::type, QNode<8>>::value);
}

int quantise_nodes(int width, const float4* wnodes, float4* qnodes, int64_t n, hipStream_t s) {
    if (n <= 0) return LMGPU_OK;
    if (width == 4)
        hipLaunchKernelGGL(k_quantise<4>, dim3(nblocks(n, 64)), dim3(256), 0, s,
                           reinterpret_cast<const WNode<4>*>(wnodes), reinterpret_cast<QNode<4>*>(qnodes), n);
    else if (width == 8)
        hipLaunchKernelGGL(k_quantise<8>, dim3(nblocks(n, 64)), dim3(256), 0, s,
                           reinterpret_cast<const WNode<8>*>(wnodes), reinterpret_cast<QNode<8>*>(qnodes), n);
    else
        return fail(LMGPU_ERR_INVALID_ARGUMENT, "quantised nodes are 4- or 8-wide");
    LMGPU_HIP(hipGetLastError());
    return LMGPU_OK;
}

int Accel::make_trav_nodes(hipStream_t s) {
    if (!quantised_width(width)) {
        qnodes.reset();
        return LMGPU_OK;
    }
    LMGPU_TRY(reserve(qnodes, size_t(num_nodes) * width));
    LMGPU_TRY(quantise_nodes(width, nodes.p, qnodes.p, num_nodes, s));
    LMGPU_HIP(hipStreamSynchronize(s));
    return LMGPU_OK;
}

// Resident grid of the persistent kernel: CUs x active blocks per CU.
template <int W, bool ANY, bool COUNT, class Node>
static int persistent_grid() {
    static int grid = 0;
    if (grid == 0) {
        int dev = 0, cus = 0, per = 0;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_trace<W, ANY, COUNT, Node>, kTraceBlock, 0);
        grid = std::max(1, cus) * std::max(1, per);
    }
    return grid;
}

template <int W, bool ANY, bool COUNT>
static void launch_trace(const Accel& a, const lmgpu_ray* rays, lmgpu_hit* hits, uint8_t* occl, int64_t n,
                         unsigned long long* next, int32_t* status, unsigned long long* counters, hipStream_t s) {
    using Node = typename TravNode<W>::type;
    // one launch for all but batches of over 2^30 rays (ray ids are 32 bits on the device)
    for (int64_t at = 0; at < n; at += kMaxLaunchRays) {
        const int64_t m = std::min(n - at, kMaxLaunchRays);
        // a block per 64 rays: few rays spread over the CUs one wave each
        const int grid = int(std::min<int64_t>(persistent_grid<W, ANY, COUNT, Node>(), (m + 63) / 64));
        // few rays are all in the waves' own shares: no counter is read
        const uint32_t nwaves = uint32_t(grid) * (kTraceBlock / 64);
        if (int64_t(nwaves) * ray_share(uint32_t(m), nwaves) < m)
            hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(64), 0, s, next);
        hipLaunchKernelGGL((k_trace<W, ANY, COUNT, Node>), dim3(grid), dim3(kTraceBlock), 0, s,
                           static_cast<const Node*>(a.trav_nodes()), a.tris.p, rays + at, hits ? hits + at : nullptr,
                           occl ? occl + at : nullptr, uint32_t(m), next, status, counters, a.refill);
    }
}

int Accel::trace(const lmgpu_ray* rays, lmgpu_hit* hits, uint8_t* occl, int64_t n, bool any,
                 unsigned long long* counters, hipStream_t s) const {
    LMGPU_TRY(check_trace_args(rays, hits, occl, n, any));
    if (n == 0) return LMGPU_OK;
    int32_t* st = status_dev();
    if (!st) return fail(LMGPU_ERR_OUT_OF_MEMORY, "status buffer");
    unsigned long long* next = next_counter();
    if (!next) return fail(LMGPU_ERR_OUT_OF_MEMORY, "ray counter");
    return trace_with(rays, hits, occl, n, any, counters, next, st, s);
}

int Accel::check_trace_args(const lmgpu_ray* rays, const lmgpu_hit* hits, const uint8_t* occl, int64_t n,
                            bool any) const {
    if (!built) return fail(LMGPU_ERR_INVALID_ARGUMENT, "accel is not built");
    if (n < 0) return fail(LMGPU_ERR_INVALID_ARGUMENT, "negative ray count");
    if (n == 0) return LMGPU_OK;
    if (!rays || (!any && !hits) || (any && !occl))
        return fail(LMGPU_ERR_INVALID_ARGUMENT, "NULL ray or result buffer");
    if ((reinterpret_cast<uintptr_t>(rays) & 15) || (hits && (reinterpret_cast<uintptr_t>(hits) & 15)))
        return fail(LMGPU_ERR_INVALID_ARGUMENT, "rays and hits must be 16-byte aligned");
    return LMGPU_OK;
}

int Accel::trace_with(const lmgpu_ray* rays, lmgpu_hit* hits, uint8_t* occl, int64_t n, bool any,
                      unsigned long long* counters, unsigned long long* next, int32_t* st, hipStream_t s) const {
    LMGPU_TRY(check_trace_args(rays, hits, occl, n, any));
    if (n == 0) return LMGPU_OK;
#define LMGPU_DISPATCH(WW)                                                                          \
    if (width == WW) {                                                                              \
        if (any) launch_trace<WW, true, false>(*this, rays, hits, occl, n, next, st, counters, s);  \
        else if (counters) launch_trace<WW, false, true>(*this, rays, hits, occl, n, next, st, counters, s); \
        else launch_trace<WW, false, false>(*this, rays, hits, occl, n, next, st, counters, s);     \
    }
    LMGPU_DISPATCH(2)
    LMGPU_DISPATCH(4)
    LMGPU_DISPATCH(8)
#undef LMGPU_DISPATCH
    LMGPU_HIP(hipGetLastError());
    return LMGPU_OK;
}

}  // namespace lmgpu
