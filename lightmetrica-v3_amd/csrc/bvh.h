// Wide BVH layout and closest-hit / any-hit traversal (device functions).
//
// Replaces the traversal of accel::sahbvh (src/accel/accel_sahbvh.cpp:269-299:
// FP64 slab test, unordered int[99] stack, Moller-Trumbore) with:
//   * a W-wide BVH (W = 2, 4, 8) whose node is 32*W bytes laid out SoA
//     (lo.x[W], lo.y[W], lo.z[W], hi.x[W], hi.y[W], hi.z[W], child[W], count[W]);
//     W = 4 is exactly one 128-B line,
//   * nearest-first ordered traversal with a per-lane stack in LDS
//     ([depth][lane], bank-conflict free) spilling to private memory,
//   * the watertight FP32 ray/triangle test of Woop, Benthin and Wald
//     (JCGT 2(1), 2013), with the reference's closed edges, closed
//     [tmin, tmax] range and |det| < 1e-8 rejection (accel_sahbvh.cpp:67-71).
#pragma once

#include <algorithm>
#include <cmath>

#include "common.h"
#include "../../include/lmgpu.h"

// Wave-level step vote of the persistent traversal, in quarters:
// a wave takes a leaf step when at least LMGPU_LEAF_VOTE_X4 / 4 times as
// many of its busy lanes sit at a leaf as at an inner node (see
// trace_persistent). 2 measured best on the 1.32M-triangle mesh (incoherent
// rays +11%, coherent +5%, path tracing +5% over no vote; 1, 3, 4 and 8
// slower).
#ifndef LMGPU_LEAF_VOTE_X4
#define LMGPU_LEAF_VOTE_X4 2
#endif

// Traversal of a 4- or 8-wide BVH reads a quantised copy of its nodes
// (QNode<W>: 64 B instead of 128 B for W = 4, 128 B instead of 256 B for
// W = 8) when 1: +15% incoherent closest-hit rays on the 1.32M-triangle mesh
// at W = 4 with identical hits.
#ifndef LMGPU_QNODE
#define LMGPU_QNODE 1
#endif

// Rays a wave takes from a ray counter with one atomic (at least 64, so one
// chunk always covers the idle lanes of a refill); the wave hands them to its
// idle lanes over several refills. 64, 128, 256: 463, 481, 553 us for 2.07M
// primary rays, 44.0, 44.3, 44.8 ms for a 1080p path-traced frame.
#ifndef LMGPU_RAY_CHUNK
#define LMGPU_RAY_CHUNK 64
#endif
static_assert(LMGPU_RAY_CHUNK >= 64, "a ray chunk must cover a whole wave");

namespace lmgpu {

template <int W>
struct alignas(16) WNode {
    float lox[W], loy[W], loz[W];
    float hix[W], hiy[W], hiz[W];
    int32_t child[W];   // internal: wide node index; leaf: first triangle (sorted order)
    int32_t count[W];   // 0 internal, > 0 leaf triangle count, < 0 empty slot
};
static_assert(sizeof(WNode<4>) == 128, "BVH4 node must be one 128-B line");

// Quantised W-wide node (W = 4: 64 B, half a 128-B line; W = 8: 128 B):
// the child boxes are 8-bit planes on a per-node, per-axis grid,
// plane = fma(q, 2^e, origin), rounded outward when built (quantise_node),
// so the decoded boxes contain the exact ones and traversal visits a
// superset of the nodes of the FP32 tree: hits are unchanged. Child c's
// lower / upper plane on axis a is byte c % 4 of qlo[a][c / 4] / qhi[a][c / 4];
// ent[c] is its stack entry (inner node index >= 0, or
// encode_leaf(first, count) < 0), kQEmpty, a leaf of no triangles, for an
// empty slot.
template <int W>
struct alignas(W * 16) QNode {
    float ox, oy, oz;
    uint32_t e;        // exponents of the x, y, z grid steps: signed bytes 0, 1, 2 (read with the origin)
    uint32_t qlo[3][W / 4];
    uint32_t qhi[3][W / 4];
    int32_t ent[W];
};
using QNode4 = QNode<4>;
static_assert(sizeof(QNode<4>) == 64, "quantised BVH4 node must be 64 B");
static_assert(sizeof(QNode<8>) == 128, "quantised BVH8 node must be 128 B");
constexpr int32_t kQEmpty = -1;   // encode_leaf(0, 0)

// Node type the traversal of a W-wide BVH reads.
template <int W>
struct TravNode {
    using type = WNode<W>;
};
#if LMGPU_QNODE
template <>
struct TravNode<4> {
    using type = QNode<4>;
};
template <>
struct TravNode<8> {
    using type = QNode<8>;
};
#endif

// Triangle in traversal order: 3 x float4 = 48 B; v0.w holds the original
// (flattened) triangle index as raw bits.
struct alignas(16) TriV {
    float4 v0, v1, v2;
};

// Stack entries: internal node index (>= 0) or an encoded leaf (< 0).
LMGPU_HD int encode_leaf(int first, int count) { return -((first << 4) | count) - 1; }
LMGPU_HD int leaf_first(int e) { return (-(e + 1)) >> 4; }
LMGPU_HD int leaf_count(int e) { return (-(e + 1)) & 15; }

struct RayPre {
    f3 o, d, inv;
    float Sx, Sy, Sz;
    int kx, ky, kz;
    float dkz_abs;   // |d[kz]|, relates the watertight det to the MT det
};

LMGPU_HD RayPre ray_prepare(f3 o, f3 d) {
    RayPre r;
    r.o = o;
    r.d = d;
    // Reciprocal direction; a zero component becomes a tiny signed value so
    // the slab distances are +-huge rather than NaN.
    const float tiny = 1e-30f;
    const float dx = fabsf(d.x) < tiny ? copysignf(tiny, d.x) : d.x;
    const float dy = fabsf(d.y) < tiny ? copysignf(tiny, d.y) : d.y;
    const float dz = fabsf(d.z) < tiny ? copysignf(tiny, d.z) : d.z;
    r.inv = mk(1.0f / dx, 1.0f / dy, 1.0f / dz);
    const float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    int kz = (ax > ay) ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int kx = kz + 1 == 3 ? 0 : kz + 1;
    int ky = kx + 1 == 3 ? 0 : kx + 1;
    const float dkz = comp(d, kz);
    if (dkz < 0.f) {   // keep the winding of the projected triangle
        const int t = kx; kx = ky; ky = t;
    }
    r.kx = kx; r.ky = ky; r.kz = kz;
    r.Sx = comp(d, kx) / dkz;
    r.Sy = comp(d, ky) / dkz;
    r.Sz = 1.0f / dkz;
    r.dkz_abs = fabsf(dkz);
    return r;
}

// Watertight ray/triangle test of a triangle given relative to the ray origin
// and permuted to (kx, ky, kz): (ax, ay, az), (bx, by, bz), (cx, cy, cz). On
// acceptance (t in [tmin, tmax], closed edges, |det_MT| >= 1e-8 as the
// reference), writes t and the barycentric weights (u, v) of v1 and v2.
// Watertightness needs each edge function to be the exact negative of the
// same edge's function in the neighbouring triangle (a*b - c*d against
// c*d - a*b). Both products must therefore be rounded before the
// subtraction: fusing one of them into an FMA would break the antisymmetry
// and let a ray through a shared edge miss both triangles, so contraction is
// switched off for the three edge functions.
LMGPU_HD bool tri_test(const RayPre& r, float ax, float ay, float Akz, float bx, float by, float Bkz, float cx,
                       float cy, float Ckz, float tmin, float tmax, float& t, float& u, float& v) {
    const float Ax = fmaf(-r.Sx, Akz, ax);
    const float Ay = fmaf(-r.Sy, Akz, ay);
    const float Bx = fmaf(-r.Sx, Bkz, bx);
    const float By = fmaf(-r.Sy, Bkz, by);
    const float Cx = fmaf(-r.Sx, Ckz, cx);
    const float Cy = fmaf(-r.Sy, Ckz, cy);
    float U, V, Wt;
    {
#pragma clang fp contract(off)
        U = Cx * By - Cy * Bx;
        V = Ax * Cy - Ay * Cx;
        Wt = Bx * Ay - By * Ax;
    }
    if (U == 0.0f || V == 0.0f || Wt == 0.0f) {
        // Exact edge: recompute the edge functions in FP64 (Woop et al., sec. 3).
        U = float(double(Cx) * double(By) - double(Cy) * double(Bx));
        V = float(double(Ax) * double(Cy) - double(Ay) * double(Cx));
        Wt = float(double(Bx) * double(Ay) - double(By) * double(Ax));
    }
    if ((U < 0.f || V < 0.f || Wt < 0.f) && (U > 0.f || V > 0.f || Wt > 0.f)) return false;
    const float det = U + V + Wt;
    if (det == 0.f) return false;
    // |det_MT| = |d . (e1 x e2)| = |det| |d[kz]| for a unit-length direction
    if (fabsf(det) * r.dkz_abs < 1e-8f) return false;
    const float Az = r.Sz * Akz, Bz = r.Sz * Bkz, Cz = r.Sz * Ckz;
    const float T = U * Az + V * Bz + Wt * Cz;
    const float sdet = fabsf(det);
    const float sT = det < 0.f ? -T : T;
    if (sT < tmin * sdet || sT > tmax * sdet) return false;
    const float rcp = 1.0f / det;
    t = T * rcp;
    u = V * rcp;
    v = Wt * rcp;
    return true;
}

// The same test on the triangle's world-space vertices.
LMGPU_HD bool tri_intersect(const RayPre& r, float4 p0, float4 p1, float4 p2, float tmin, float tmax, float& t,
                            float& u, float& v) {
    const f3 A = mk(p0.x - r.o.x, p0.y - r.o.y, p0.z - r.o.z);
    const f3 B = mk(p1.x - r.o.x, p1.y - r.o.y, p1.z - r.o.z);
    const f3 C = mk(p2.x - r.o.x, p2.y - r.o.y, p2.z - r.o.z);
    return tri_test(r, comp(A, r.kx), comp(A, r.ky), comp(A, r.kz), comp(B, r.kx), comp(B, r.ky), comp(B, r.kz),
                    comp(C, r.kx), comp(C, r.ky), comp(C, r.kz), tmin, tmax, t, u, v);
}

// Slab test of one child box; conservative against FP32 rounding by scaling
// the far distance with 1 + 2*gamma(3) (Ize, "Robust BVH Ray Traversal",
// JCGT 2(2), 2013).
__device__ __forceinline__ float box_near(const RayPre& r, float lx, float ly, float lz, float hx, float hy,
                                          float hz, float tmin, float tmax, bool& hit) {
    const float t1x = (lx - r.o.x) * r.inv.x, t2x = (hx - r.o.x) * r.inv.x;
    const float t1y = (ly - r.o.y) * r.inv.y, t2y = (hy - r.o.y) * r.inv.y;
    const float t1z = (lz - r.o.z) * r.inv.z, t2z = (hz - r.o.z) * r.inv.z;
    const float tn = fmaxf(fmaxf(fminf(t1x, t2x), fminf(t1y, t2y)), fmaxf(fminf(t1z, t2z), tmin));
    const float tf = fminf(fminf(fmaxf(t1x, t2x), fmaxf(t1y, t2y)), fminf(fmaxf(t1z, t2z), tmax));
    hit = tn <= tf * 1.00000036f;
    return tn;
}

// Slab keys of the W children of one node: key[c] is the entry distance of
// a hit child (+inf otherwise), ent[c] its stack entry.
template <int W>
__device__ __forceinline__ void child_keys(const WNode<W>& nd, const RayPre& r, float tmin, float tmax,
                                           float (&key)[W], int (&ent)[W]) {
#pragma unroll
    for (int c = 0; c < W; c++) {
        bool hit;
        const float tn = box_near(r, nd.lox[c], nd.loy[c], nd.loz[c], nd.hix[c], nd.hiy[c], nd.hiz[c], tmin, tmax, hit);
        const int cnt = nd.count[c];
        const int ch = nd.child[c];
        hit = hit && cnt >= 0;
        key[c] = hit ? tn : __builtin_inff();
        ent[c] = cnt == 0 ? ch : encode_leaf(ch, cnt);
    }
}

LMGPU_HD float qplane(uint32_t q, int c, float step, float origin) {
    return std::fma(float((q >> (8 * c)) & 0xffu), step, origin);
}

// Slab keys of the W children of a quantised node. The slab distance of
// grid plane q on axis x is computed as one fma, t = q * ax + bx, with
//   ax = step_x * inv_x   (exact: the step is a power of two),
//   bx = (ox - o_x) * inv_x,
// and no decoded plane: the planes are the exact reals ox + q * step. Each
// axis picks its near and far plane by the sign of inv_x, so one fma gives
// the entry and one the exit distance (no per-axis min / max). Bounds, with
// u = 2^-24: bx is within 2u |bx| of (ox - o_x) * inv_x; the exact plane
// ox + q step lies within u (|ox| + 255 step) of the FP32 plane the builder
// rounded outward (quantise_node); the fma and inv_x round relatively, which
// the 1 + 2 gamma(3) factor on the exit distance covers (box_near). The entry
// offset is lowered and the exit offset raised by
//   Ex = 16u (|bx| + |inv_x| |ox| + 255 |ax|),
// which exceeds the absolute terms with their own rounding, so every child
// box the FP32 test of the decoded planes would hit is hit here too.
// The keys order the traversal, and where coplanar triangles tie in t (a box
// standing on a floor) the one visited last is the hit: the keys' rounding
// is part of the result, and a cheaper bound for Ex is not a free choice.
template <int W>
LMGPU_HD void child_keys(const QNode<W>& nd, const RayPre& r, float tmin, float tmax, float (&key)[W],
                         int (&ent)[W]) {
    const float org[3] = {nd.ox, nd.oy, nd.oz};
    const float inv[3] = {r.inv.x, r.inv.y, r.inv.z};
    const float o[3] = {r.o.x, r.o.y, r.o.z};
    float a[3], bn[3], bf[3];
    uint32_t wn[3][W / 4], wf[3][W / 4];
    // both plane words of every axis as loaded (whole 16-B loads of the node);
    // the empty asm keeps the compiler from turning the sign choice below into
    // per-lane dword loads from chosen addresses
    uint32_t ql[3][W / 4], qh[3][W / 4];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int w = 0; w < W / 4; w++) {
            ql[k][w] = nd.qlo[k][w];
            qh[k][w] = nd.qhi[k][w];
#if defined(__HIP_DEVICE_COMPILE__)
            asm("" : "+v"(ql[k][w]), "+v"(qh[k][w]));
#endif
        }
#pragma unroll
    for (int k = 0; k < 3; k++) {
        a[k] = ldexpf(inv[k], int32_t(nd.e << (24 - 8 * k)) >> 24);
        const float b = (org[k] - o[k]) * inv[k];
        const float x = fabsf(b) + fmaf(fabsf(org[k]), fabsf(inv[k]), 255.f * fabsf(a[k]));
        bn[k] = fmaf(x, -0x1p-20f, b);   // Ex = 2^-20 x
        bf[k] = fmaf(x, 0x1p-20f, b);
        const bool pos = inv[k] >= 0.f;
#pragma unroll
        for (int w = 0; w < W / 4; w++) {
            wn[k][w] = pos ? ql[k][w] : qh[k][w];
            wf[k][w] = pos ? qh[k][w] : ql[k][w];
        }
    }
#pragma unroll
    for (int c = 0; c < W; c++) {
        const int w = c >> 2, sh = 8 * (c & 3);
        float tn[3], tf[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            tn[k] = fmaf(float((wn[k][w] >> sh) & 0xffu), a[k], bn[k]);
            tf[k] = fmaf(float((wf[k][w] >> sh) & 0xffu), a[k], bf[k]);
        }
        const float n = fmaxf(fmaxf(tn[0], tn[1]), fmaxf(tn[2], tmin));
        const float f = fminf(fminf(tf[0], tf[1]), fminf(tf[2], tmax));
        const int e = nd.ent[c];
        const bool hit = n <= f * 1.00000036f && (c < 2 || e != kQEmpty);
        key[c] = hit ? n : __builtin_inff();
        ent[c] = e;
    }
}

// One axis of a quantised node: grid origin, exponent of the step, and the
// children's lower and upper planes (bytes).
template <int W>
struct QAxis {
    float org;
    int e;
    uint32_t ql[W / 4], qh[W / 4];
};

// Quantises the children's bounds on one axis (bit c of `present`: slot c holds
// a child): the grid starts at the smallest child plane, with the smallest
// power-of-two step that spans the node in 255 steps; each plane is rounded
// outward in the exact FP32 expression the traversal decodes (qplane), so every
// decoded box contains the original.
template <int W>
LMGPU_HD QAxis<W> quantise_axis(const float (&lo)[W], const float (&hi)[W], uint32_t present) {
    QAxis<W> q{};
    float mn = __builtin_inff(), mx = -__builtin_inff();
    for (int c = 0; c < W; c++)
        if (present >> c & 1u) {
            mn = std::min(mn, lo[c]);
            mx = std::max(mx, hi[c]);
        }
    if (!(mn <= mx)) mn = mx = 0.f;   // no child (not produced by the builder)
    q.org = mn;
    // smallest e with fma(255, 2^e, mn) >= mx; steps of at least 2^-126.
    // Start from ceil(log2(span / 255)), read off the binary exponent:
    // x = m 2^k with m in [0.5, 1) gives ceil(log2 x) = k, or k - 1 when
    // m = 0.5 exactly.
    int e = -126;
    const double span = double(mx) - double(mn);
    if (span > 0.0) {
        int k = 0;
        const double m = std::frexp(span / 255.0, &k);
        e = std::max(-126, m == 0.5 ? k - 1 : k);
    }
    while (e < 127 && std::fma(255.f, std::ldexp(1.f, e), mn) < mx) e++;
    q.e = e;
    const float step = std::ldexp(1.f, e);
    for (int c = 0; c < W; c++) {
        if (!(present >> c & 1u)) continue;
        // division by the power-of-two step is an exact scaling
        int l = int(std::floor(std::ldexp(double(lo[c]) - double(mn), -e)));
        l = std::min(std::max(l, 0), 255);
        while (l > 0 && std::fma(float(l), step, mn) > lo[c]) l--;
        int h = int(std::ceil(std::ldexp(double(hi[c]) - double(mn), -e)));
        h = std::min(std::max(h, 0), 255);
        while (h < 255 && std::fma(float(h), step, mn) < hi[c]) h++;
        q.ql[c >> 2] |= uint32_t(l) << (8 * (c & 3));
        q.qh[c >> 2] |= uint32_t(h) << (8 * (c & 3));
    }
    return q;
}

// Stack entry of a wide node's child (WNode::child, WNode::count).
LMGPU_HD int32_t quantised_entry(int32_t child, int32_t count) {
    return count < 0 ? kQEmpty : (count == 0 ? child : encode_leaf(child, count));
}

// A whole quantised node.
template <int W>
LMGPU_HD QNode<W> quantise_node(const WNode<W>& n) {
    QNode<W> q;
    uint32_t present = 0;
    for (int c = 0; c < W; c++) present |= n.count[c] >= 0 ? 1u << c : 0u;
    const QAxis<W> x[3] = {quantise_axis<W>(n.lox, n.hix, present), quantise_axis<W>(n.loy, n.hiy, present),
                           quantise_axis<W>(n.loz, n.hiz, present)};
    q.ox = x[0].org;
    q.oy = x[1].org;
    q.oz = x[2].org;
    q.e = 0;
    for (int a = 0; a < 3; a++) {
        q.e |= uint32_t(x[a].e & 0xff) << (8 * a);
        for (int k = 0; k < W / 4; k++) {
            q.qlo[a][k] = x[a].ql[k];
            q.qhi[a][k] = x[a].qh[k];
        }
    }
    for (int c = 0; c < W; c++) q.ent[c] = quantised_entry(n.child[c], n.count[c]);
    return q;
}

struct TraceResult {
    int prim;        // original triangle index, -1 for a miss
    float t, u, v;   // of the hit; t of a miss is the ray's tmax
    bool overflow;
};

// Hit record of the accepted triangle re-evaluated once in FP64 with the
// reference's Moller-Trumbore formula (accel_sahbvh.cpp:58-75), whose Hit
// carries FP64 t and uv. The hit decision itself stays the FP32 watertight
// test; this only removes the FP32 conditioning error of t at grazing
// incidence (error ~ eps * edge / (t * cos)). A triangle whose FP64
// determinant vanishes keeps the FP32 values.
__device__ __forceinline__ void refine_hit(const TriV& tv, const RayPre& r, float tmin, float& t, float& u, float& v) {
    const f3 o = r.o, d = r.d;
    const double p1x = tv.v0.x, p1y = tv.v0.y, p1z = tv.v0.z;
    const double e1x = double(tv.v1.x) - p1x, e1y = double(tv.v1.y) - p1y, e1z = double(tv.v1.z) - p1z;
    const double e2x = double(tv.v2.x) - p1x, e2y = double(tv.v2.y) - p1y, e2z = double(tv.v2.z) - p1z;
    const double dx = d.x, dy = d.y, dz = d.z;
    const double px = dy * e2z - dz * e2y, py = dz * e2x - dx * e2z, pz = dx * e2y - dy * e2x;
    const double tx = double(o.x) - p1x, ty = double(o.y) - p1y, tz = double(o.z) - p1z;
    const double qx = ty * e1z - tz * e1y, qy = tz * e1x - tx * e1z, qz = tx * e1y - ty * e1x;
    const double det = e1x * px + e1y * py + e1z * pz;
    if (det == 0.0) {
        (void)tri_intersect(r, tv.v0, tv.v1, tv.v2, tmin, __builtin_inff(), t, u, v);
        return;
    }
    const double inv = 1.0 / det;
    t = float((e2x * qx + e2y * qy + e2z * qz) * inv);
    u = float((tx * px + ty * py + tz * pz) * inv);
    v = float((dx * qx + dy * qy + dz * qz) * inv);
}

// Orders the (key, entry) pairs of a node's children by key. Equal keys (a ray
// starting inside several boxes, boxes that share a plane) stay in place at
// each compare: their order decides which of coplanar triangles is hit, so
// the network's own order on ties is part of the result.
__device__ __forceinline__ void cswap(float& ka, int& ea, float& kb, int& eb) {
    const bool s = kb < ka;
    const float tk = s ? kb : ka;
    const int te = s ? eb : ea;
    kb = s ? ka : kb;
    eb = s ? ea : eb;
    ka = tk;
    ea = te;
}

template <int W>
__device__ __forceinline__ void sort_children(float (&k)[W], int (&e)[W]) {
    auto cs = [&](int a, int b) { cswap(k[a], e[a], k[b], e[b]); };
    if constexpr (W == 2) {
        cs(0, 1);
    } else if constexpr (W == 4) {
        cs(0, 1); cs(2, 3); cs(0, 2); cs(1, 3); cs(1, 2);
    } else {
        // Batcher odd-even merge sort network for 8 inputs (19 comparators).
        cs(0, 1); cs(2, 3); cs(4, 5); cs(6, 7);
        cs(0, 2); cs(1, 3); cs(4, 6); cs(5, 7);
        cs(1, 2); cs(5, 6);
        cs(0, 4); cs(1, 5); cs(2, 6); cs(3, 7);
        cs(2, 4); cs(3, 5);
        cs(1, 2); cs(3, 4); cs(5, 6);
    }
}

// Stack entry of a lane with nothing left to visit: the bottom of every
// stack, so that popping an empty stack needs no test.
constexpr int32_t kDone = INT32_MAX;
// Ray id of a lane without a ray; ray ids stay below 2^31 (n of a launch).
constexpr uint32_t kNoRay = UINT32_MAX;
// Most rays of one launch of the persistent traversal.
constexpr int64_t kMaxLaunchRays = int64_t(1) << 30;
// Ray counters of one launch, in cache lines of their own; zeroed before it.
constexpr uint32_t kRayCounters = 8;
constexpr uint32_t kRayCounterStride = 16;   // in 64-bit words
constexpr uint32_t kRayCounterWords = kRayCounters * kRayCounterStride;
// Rays a wave starts with: its whole part of an even split in whole waves of
// rays when that is at most 256 rays (room at 256x256, 85 rays a wave: 2.03 ms
// with half of it, 1.48 with all; 2M rays of uneven cost, 325 a wave: 889 us
// with half, 1030 with all), else half of it, at most 256 rays (2730 a wave at
// 1080p: half 45.9 ms a frame, 256 rays 44.0); the ray counters hand out the rest.
__device__ __host__ inline uint32_t ray_share(uint32_t n, uint32_t nwaves) {
    const uint32_t per = (n + nwaves - 1) / nwaves;
    return per <= 256u ? (per + 63u) & ~63u : (per < 512u ? per / 2u : 256u) & ~63u;
}

// Persistent traversal: every lane owns one ray at a time; when at least
// `refill` lanes of a wave have finished (or the whole wave has), the
// finished lanes hand over their results together and take new rays from the
// wave's pool: a share of its own, then chunks of LMGPU_RAY_CHUNK from the ray
// counters with one atomic (Aila & Laine, HPG 2009, "persistent threads"), so
// lanes do not sit idle behind a wave's slowest ray and the counters see few
// atomics. refill = 64 keeps whole
// waves of consecutive rays together (best for coherent rays), smaller
// values keep lanes busy.
// Each loop iteration advances the lanes of one kind of step: a wide node or
// a leaf, chosen per wave by vote. Closest hit (ANY = false) keeps shrinking
// tmax; an accepted triangle is replaced by a later one at t == tmax, as the
// reference's closed [tmin, tmax] test does. `fetch(id, o, d, tmin, tmax)` loads ray
// `id` and returns the node its traversal starts from (0, or a root inside a
// multi-BVH arena);
// `emit(id, res)` consumes its result.
//
// The loop is bound by the instructions it issues (29 of 64 lanes active; vector
// issue busy 78% on incoherent rays) and by the return of its divergent 16-B
// node loads (data return busy 77%, address unit 68%), so a node step has no branch in the common case: lds[0][lane] holds kDone
// and entry i of the lane's stack lds[1 + i][lane]; each child is written at
// the top of the stack and the stack grows by one only if the child was hit,
// so what lies above the top is garbage that the next push overwrites; and
// the entry to pop is read before the test, with the node's own load. The
// first LDS_DEPTH entries live there, at [entry][lane] (bank-conflict free),
// the rest in private memory: a wave with a lane that could pass LDS_DEPTH in
// this step takes a separate, branchy path. Results are emitted
// only when lanes are refilled: done as each ray ends, the FP64
// re-evaluation ran in most iterations for a lane or two.
// Measured on the 1.32M-triangle mesh together with the waves' own shares
// (below), timed in turn: 2.07M primary rays 719 -> 459 us, 2M incoherent rays
// 1018 -> 904, 500K any-hit rays on the 8-wide tree 516 -> 353.
template <int W, bool ANY, bool COUNT, int LDS_DEPTH, int PRIV_DEPTH, int BLOCK, class Node, class Fetch, class Emit>
__device__ __forceinline__ void trace_persistent(const Node* __restrict__ nodes, const TriV* __restrict__ tris,
                                                 uint32_t n, unsigned long long* next, int (*lds)[BLOCK],
                                                 Fetch fetch, Emit emit, int32_t* status,
                                                 unsigned long long* counters, int refill) {
    constexpr uint32_t chunk_rays = LMGPU_RAY_CHUNK;
    static_assert(LDS_DEPTH >= W, "one node's children must fit the LDS part of an empty stack");
    const int lane = threadIdx.x & 63;
    const int tid = threadIdx.x;
    int priv[PRIV_DEPTH];
    RayPre r{};
    f3 ok = mk(0.f, 0.f, 0.f);   // ray origin permuted to (kx, ky, kz)
    uint32_t kk = 0;             // 1 << kx, 1 << ky, 1 << kz in bits 0-2, 3-5, 6-8
    uint32_t rid = kNoRay;       // ray of this lane whose result is still to be emitted
    float tmin = 0.f, tfar = 0.f;
    int best = -1;               // hit triangle in traversal order
    bool overflow = false;
    int cur = kDone;             // node (>= 0), leaf (< 0) or kDone
    int sp = 0;                  // stack entries
    lds[0][tid] = kDone;
    // Wave-uniform: ray ids of the wave not yet handed to a lane, and whether
    // ids are left beyond them. Every wave starts with a share of its own
    // (ray_share) and takes chunks of what lies past all shares from the ray
    // counters. Atomics on one address from all XCDs take 12 ns each, so one per
    // wave before any ray started took 74 us of every launch, and a last,
    // empty-handed one per wave as much of its end. Group g of the blocks takes
    // chunks g, g + 8, ... from a counter of its own: an eighth of the
    // updates wait for each other, and all groups work on all parts of the
    // rays. Shares go to the waves of a block in a row, whose rays then meet in
    // its L1; with fewer shares than waves they go to the blocks in turn, over
    // all CUs.
    const uint32_t nblk = gridDim.x, nwaves = nblk * (BLOCK / 64);
    const uint32_t share = ray_share(n, nwaves);
    const uint32_t in_blk = threadIdx.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(n < nwaves * 64u ? in_blk * nblk + blockIdx.x
                                                                         : blockIdx.x * (BLOCK / 64) + in_blk);
    const uint32_t shared_from = nwaves * share;   // < n + 64 nwaves
    const uint32_t groups = min(kRayCounters, nblk), group = blockIdx.x % groups;
    uint32_t pool_next = min(n, wave * share), pool_end = min(n, wave * share + share);
    bool more = shared_from < n;                   // ids of the group beyond the pool may be left
    bool exhausted = pool_next == pool_end && !more;
    unsigned long long nv = 0, nt = 0;
    // component kx (shift 0), ky (3) or kz (6) of v: tests of single bits
    // stay two selects, where a test of the number itself becomes branches
    auto pick = [&](int shift, float x, float y, float z) {
        return kk & (1u << shift) ? x : (kk & (2u << shift) ? y : z);
    };
    // the ray with what the loop does not hold in registers of its own
    auto with_axes = [&]() {
        RayPre q = r;
        q.dkz_abs = fabsf(pick(6, r.d.x, r.d.y, r.d.z));
        return q;
    };
    // pop for a wave with stacks past LDS_DEPTH
    auto pop_deep = [&]() -> int {
        int v = lds[min(sp, LDS_DEPTH)][tid];
        asm volatile("" : "+v"(v));   // keep the ds_read apart from the private read
        if (sp > LDS_DEPTH) v = priv[sp - 1 - LDS_DEPTH];
        if (sp > 0) sp--;
        return v;
    };
    while (true) {
        const unsigned long long busy = __ballot(cur != kDone);
        if (busy == 0 || (!exhausted && 64 - __popcll(busy) >= refill)) {
            // hand over the results of the lanes that finished
            if (rid != kNoRay && cur == kDone) {
                TraceResult res;
                res.prim = -1;
                res.t = tfar;
                res.u = res.v = 0.f;
                res.overflow = overflow;
                if (overflow) atomicOr(status, 1);
                if (best >= 0) {
                    const TriV tv = tris[best];
                    res.prim = __float_as_int(tv.v0.w);
                    if (!ANY) {
                        RayPre q = with_axes();
                        q.kx = kk & 1u ? 0 : (kk & 2u ? 1 : 2);
                        q.ky = kk & 8u ? 0 : (kk & 16u ? 1 : 2);
                        q.kz = kk & 64u ? 0 : (kk & 128u ? 1 : 2);
                        refine_hit(tv, q, tmin, res.t, res.u, res.v);
                    }
                }
                emit(rid, res);
                rid = kNoRay;
            }
            if (!exhausted) {
                // idle lanes take, in lane order, the rest of the wave's pool
                // and then the start of a new chunk (chunk_end - chunk rays)
                const bool idle = cur == kDone;
                const unsigned long long idle_mask = ~busy;
                const uint32_t nidle = __popcll(idle_mask);
                const uint32_t avail = pool_end - pool_next;
                uint32_t chunk = n, chunk_end = n;
                if (avail < nidle && more) {
                    uint32_t b = 0;
                    if (lane == 0) b = uint32_t(atomicAdd(next + group * kRayCounterStride, 1ull));
                    // wave-uniform from here on: scalar registers for the pool
                    const uint32_t at = (__builtin_amdgcn_readfirstlane(b) * groups + group) * chunk_rays;
                    chunk = min(n, shared_from + at);
                    chunk_end = min(n, chunk + chunk_rays);
                    more = chunk + groups * chunk_rays < n;
                }
                if (idle) {
                    const uint32_t rank = __popcll(idle_mask & ((1ull << lane) - 1ull));
                    const uint32_t id = rank < avail ? pool_next + rank : chunk + (rank - avail);
                    if (rank < avail || id < chunk_end) {
                        rid = id;
                        f3 o, d;
                        cur = fetch(id, o, d, tmin, tfar);
                        r = ray_prepare(o, d);
                        ok = mk(comp(o, r.kx), comp(o, r.ky), comp(o, r.kz));
                        kk = (1u << r.kx) | (8u << r.ky) | (64u << r.kz);
                        best = -1;
                        overflow = false;
                        sp = 0;
                    }
                }
                if (avail < nidle) {
                    pool_next = min(chunk + (nidle - avail), chunk_end);
                    pool_end = chunk_end;
                } else {
                    pool_next += nidle;
                }
                exhausted = pool_next == pool_end && !more;
            }
            if (__ballot(cur != kDone) == 0) break;
        }
        // One kind of step per iteration for the whole wave, so inner-node
        // and leaf code do not both run, each for a part of the lanes: leaves
        // when enough lanes sit at a leaf, else inner nodes; the other lanes
        // wait one iteration.
        const unsigned long long leaf_mask = __ballot(cur < 0);
        const int nleaf = __popcll(leaf_mask);
        const int nnode = __popcll(__ballot(cur != kDone)) - nleaf;
        if (4 * nleaf >= LMGPU_LEAF_VOTE_X4 * nnode) {
            if (cur < 0) {
                const int first = leaf_first(cur), cnt = leaf_count(cur);
                const RayPre q = with_axes();
                bool hit = false;
                for (int k = 0; k < cnt; k++) {
                    if (COUNT) nt++;
                    const TriV tv = tris[first + k];
                    float t, u, v;
                    const float4 a = tv.v0, b = tv.v1, c = tv.v2;
                    if (tri_test(q, pick(0, a.x, a.y, a.z) - ok.x, pick(3, a.x, a.y, a.z) - ok.y,
                                 pick(6, a.x, a.y, a.z) - ok.z, pick(0, b.x, b.y, b.z) - ok.x,
                                 pick(3, b.x, b.y, b.z) - ok.y, pick(6, b.x, b.y, b.z) - ok.z,
                                 pick(0, c.x, c.y, c.z) - ok.x, pick(3, c.x, c.y, c.z) - ok.y,
                                 pick(6, c.x, c.y, c.z) - ok.z, tmin, tfar, t, u, v)) {
                        tfar = t;
                        best = first + k;
                        hit = true;
                        if (ANY) break;
                    }
                }
                if (ANY && hit) cur = kDone;
                else if (__ballot(sp > LDS_DEPTH) != 0) cur = pop_deep();
                else {
                    cur = lds[sp][tid];
                    sp = max(sp - 1, 0);
                }
            }
        } else if (uint32_t(cur) < uint32_t(kDone)) {
            if (COUNT) nv++;
            const Node& nd = nodes[cur];
            const int top = lds[min(sp, LDS_DEPTH)][tid];
            float key[W];
            int ent[W];
            child_keys<W>(nd, r, tmin, tfar, key, ent);
            sort_children<W>(key, ent);
            const float kInfF = __builtin_inff();
            if (__ballot(sp + W - 1 > LDS_DEPTH) == 0) {
#pragma unroll
                for (int c = W - 1; c >= 1; c--) {
                    lds[sp + 1][tid] = ent[c];
                    sp += key[c] != kInfF ? 1 : 0;
                }
                const bool any_child = key[0] != kInfF;
                cur = any_child ? ent[0] : top;
                sp = any_child ? sp : max(sp - 1, 0);
            } else {
                bool full = false;
#pragma unroll
                for (int c = W - 1; c >= 1; c--)
                    if (key[c] != kInfF) {
                        if (sp < LDS_DEPTH) lds[sp + 1][tid] = ent[c];
                        else if (sp < LDS_DEPTH + PRIV_DEPTH) priv[sp - LDS_DEPTH] = ent[c];
                        else full = true;
                        if (!full) sp++;
                    }
                if (full) {
                    overflow = true;
                    cur = kDone;
                } else if (key[0] != kInfF) {
                    cur = ent[0];
                } else {
                    cur = pop_deep();
                }
            }
        }
    }
    if (COUNT) {
        for (int off = 32; off > 0; off >>= 1) {
            nv += __shfl_xor(nv, off);
            nt += __shfl_xor(nt, off);
        }
        if (lane == 0) {
            atomicAdd(&counters[0], nv);
            atomicAdd(&counters[1], nt);
        }
    }
}

}  // namespace lmgpu
