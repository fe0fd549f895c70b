// Device BVH construction for sgpu_scene_commit (the replacement of Embree's rtcCommitScene,
// Source/Core/SceneLib/ModelResource.cpp:447-472).
//
// Pipeline (all on the device, one stream):
//   1. k_prep     triangle records (v0, e1, e2, ids), per-triangle boxes and centroids, and a
//                 block-reduced scene box and centroid box.
//   2. k_morton   63-bit Morton codes (21 bits per axis) of centroids in the centroid box.
//   3. rocPRIM    device radix sort of (code, triangle) pairs.
//   4. k_box_*    a pyramid of boxes over the leaves in sorted order: level k holds the union of
//                 every aligned run of 2^k leaves.
//   5. k_karras   binary radix tree over the sorted codes (Karras 2012, "Maximizing Parallelism
//                 in the Construction of BVHs, Octrees, and k-d Trees", Alg. 1 + 2); equal codes
//                 are split by position, so every key is distinct. A node covers a run of leaves,
//                 and so does each child: the node's record (both child boxes + child links) is
//                 written at once from the pyramid's aligned runs.
//   6. k_depth    the deepest leaf (traversal stack size); then the 8-wide tree (build_wide) with the
//                 triangle records in its slots.
//
// Boxes are inflated by 2^-18 of the scene's largest absolute coordinate. The boxes only cull;
// the inflation keeps culling conservative with respect to the triangle test's rounding, so
// closest hits do not depend on the tree's shape.
#include "sgpu_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>  // rocprim/iterator/texture_cache_iterator.hpp uses memset without including it
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ uint32_t f2ord(float f)
{
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u)
{
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// bounds layout (12 ordered-uint slots): [0..2] scene lo, [3..5] scene hi (stored as ~ord so that
// atomicMin works for both), [6..8] centroid lo, [9..11] centroid hi (also as ~ord).
__global__ __launch_bounds__(kBlock) void k_prep(const float* __restrict pos, uint32_t n,
                                                 const uint32_t* __restrict tri_geom,
                                                 const uint32_t* __restrict geom_first,
                                                 TriRecord* __restrict rec, float4* __restrict blo,
                                                 float4* __restrict bhi, float4* __restrict cent,
                                                 uint32_t* __restrict bounds)
{
    __shared__ uint32_t red[12][kBlock / 64];
    uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    uint32_t v[12];
    for (int k = 0; k < 12; ++k) v[k] = 0xFFFFFFFFu;
    if (i < n) {
        const float* p = pos + (size_t)i * 9;
        f3 v0 = mk3(p[0], p[1], p[2]);
        f3 v1 = mk3(p[3], p[4], p[5]);
        f3 v2 = mk3(p[6], p[7], p[8]);
        f3 e1 = v1 - v0;
        f3 e2 = v2 - v0;
        uint32_t g = tri_geom[i];
        // quad geometries (bit 31 of their first index) keep prim = 2 * quad + half, flagged in bit 31
        const uint32_t fg = geom_first[g];
        uint32_t prim = (i - (fg & 0x7FFFFFFFu)) | (fg & 0x80000000u);
        TriRecord r;
        r.a = make_float4(v0.x, v0.y, v0.z, __uint_as_float(i));
        r.b = make_float4(e1.x, e1.y, e1.z, __uint_as_float(g));
        r.c = make_float4(e2.x, e2.y, e2.z, __uint_as_float(prim));
        r.pad = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        rec[i] = r;
        f3 lo = mk3(fminf(v0.x, fminf(v1.x, v2.x)), fminf(v0.y, fminf(v1.y, v2.y)), fminf(v0.z, fminf(v1.z, v2.z)));
        f3 hi = mk3(fmaxf(v0.x, fmaxf(v1.x, v2.x)), fmaxf(v0.y, fmaxf(v1.y, v2.y)), fmaxf(v0.z, fmaxf(v1.z, v2.z)));
        f3 c = mk3(0.5f * (lo.x + hi.x), 0.5f * (lo.y + hi.y), 0.5f * (lo.z + hi.z));
        blo[i] = make_float4(lo.x, lo.y, lo.z, 0.0f);
        bhi[i] = make_float4(hi.x, hi.y, hi.z, 0.0f);
        cent[i] = make_float4(c.x, c.y, c.z, 0.0f);
        v[0] = f2ord(lo.x); v[1] = f2ord(lo.y); v[2] = f2ord(lo.z);
        v[3] = ~f2ord(hi.x); v[4] = ~f2ord(hi.y); v[5] = ~f2ord(hi.z);
        v[6] = f2ord(c.x); v[7] = f2ord(c.y); v[8] = f2ord(c.z);
        v[9] = ~f2ord(c.x); v[10] = ~f2ord(c.y); v[11] = ~f2ord(c.z);
    }
    // wave64 min-reduction, then across the block's waves, then one atomic per slot per block
    for (int k = 0; k < 12; ++k) {
        uint32_t x = v[k];
        for (int off = 32; off > 0; off >>= 1) x = min(x, (uint32_t)__shfl_xor((int)x, off, 64));
        v[k] = x;
    }
    int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 12; ++k) red[k][wave] = v[k];
    __syncthreads();
    if (threadIdx.x < 12) {
        uint32_t x = red[threadIdx.x][0];
        for (int w = 1; w < kBlock / 64; ++w) x = min(x, red[threadIdx.x][w]);
        atomicMin(&bounds[threadIdx.x], x);
    }
}

__device__ __forceinline__ uint64_t spread21(uint64_t x)
{
    x &= 0x1fffffULL;
    x = (x | (x << 32)) & 0x1f00000000ffffULL;
    x = (x | (x << 16)) & 0x1f0000ff0000ffULL;
    x = (x | (x << 8)) & 0x100f00f00f00f00fULL;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ULL;
    x = (x | (x << 2)) & 0x1249249249249249ULL;
    return x;
}

__global__ __launch_bounds__(kBlock) void k_morton(const float4* __restrict cent, uint32_t n,
                                                   const uint32_t* __restrict bounds,
                                                   uint64_t* __restrict keys, uint32_t* __restrict vals)
{
    uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    float lo[3], ext[3];
    for (int k = 0; k < 3; ++k) {
        lo[k] = ord2f(bounds[6 + k]);
        float hi = ord2f(~bounds[9 + k]);
        ext[k] = hi - lo[k];
    }
    float4 c = cent[i];
    float cc[3] = {c.x, c.y, c.z};
    uint64_t q[3];
    for (int k = 0; k < 3; ++k) {
        float f = ext[k] > 0.0f ? (cc[k] - lo[k]) / ext[k] : 0.0f;
        f = fminf(fmaxf(f, 0.0f), 1.0f);
        q[k] = (uint64_t)fminf(f * 2097152.0f, 2097151.0f);
    }
    keys[i] = (spread21(q[0]) << 2) | (spread21(q[1]) << 1) | spread21(q[2]);
    vals[i] = i;
}

__device__ __forceinline__ int delta(const uint64_t* __restrict k, int n, int i, int j)
{
    if (j < 0 || j >= n) return -1;
    uint64_t a = k[i], b = k[j];
    if (a == b) return 64 + __clz((int)((uint32_t)i ^ (uint32_t)j));
    return __clzll((long long)(a ^ b));
}

__device__ __forceinline__ float inflate_eps(const uint32_t* __restrict bounds)
{
    float m = 0.0f;
    for (int k = 0; k < 3; ++k) {
        m = fmaxf(m, fabsf(ord2f(bounds[k])));
        m = fmaxf(m, fabsf(ord2f(~bounds[3 + k])));
    }
    return m * (1.0f / 262144.0f);
}

__device__ __forceinline__ void leaf_box(const float4* __restrict blo, const float4* __restrict bhi,
                                         const uint32_t* __restrict order, int j, float eps,
                                         float4& lo, float4& hi)
{
    uint32_t t = order[j];
    lo = blo[t];
    hi = bhi[t];
    lo.x -= eps; lo.y -= eps; lo.z -= eps;
    hi.x += eps; hi.y += eps; hi.z += eps;
}

// The box pyramid: level 0 the inflated leaf boxes in sorted order, level k the union of each
// aligned run of 2^k of them (the last run of a level may be short). Boxes of a radix tree's nodes
// are read from it as O(log n) aligned runs, most of them one or two (half of a tree's nodes cover
// two or three leaves). It takes the place of a bottom-up pass with an arrival counter per node,
// whose two device-scope fences per step write back and invalidate an XCD's L2: 500K triangles
// 3.96 ms with that pass, 0.06 ms with the pyramid; the boxes are the same unions.
struct LeafBox {
    float4 lo, hi;
};
constexpr int kMaxBoxLevels = 31;
struct BoxLevels {
    const LeafBox* level[kMaxBoxLevels];
};

__device__ __forceinline__ void grow_box(float4& lo, float4& hi, const LeafBox& b)
{
    lo.x = fminf(lo.x, b.lo.x);
    lo.y = fminf(lo.y, b.lo.y);
    lo.z = fminf(lo.z, b.lo.z);
    hi.x = fmaxf(hi.x, b.hi.x);
    hi.y = fmaxf(hi.y, b.hi.y);
    hi.z = fmaxf(hi.z, b.hi.z);
}

// Union of the leaves first..last (inclusive).
__device__ __forceinline__ void range_box(const BoxLevels& levels, uint32_t first, uint32_t last, float4& lo, float4& hi)
{
    const float inf = __int_as_float(0x7f800000);
    lo = make_float4(inf, inf, inf, 0.0f);
    hi = make_float4(-inf, -inf, -inf, 0.0f);
    uint32_t l = first, r = last + 1;
    for (int k = 0; l < r; ++k, l >>= 1, r >>= 1) {
        if (l & 1u) grow_box(lo, hi, levels.level[k][l++]);
        if (r & 1u) grow_box(lo, hi, levels.level[k][--r]);
    }
}

// Level 0: the leaf boxes, inflated, in sorted order.
__global__ __launch_bounds__(kBlock) void k_box_leaves(uint32_t n, const float4* __restrict blo,
                                                       const float4* __restrict bhi, const uint32_t* __restrict order,
                                                       const uint32_t* __restrict bounds, LeafBox* __restrict out)
{
    const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= n) return;
    LeafBox b;
    leaf_box(blo, bhi, order, (int)j, inflate_eps(bounds), b.lo, b.hi);
    out[j] = b;
}

// The kBoxStep levels over one given level of m boxes: each block reduces kBlock of them through
// LDS, writing every level's runs (level k has ceil(m / 2^k) boxes at out[k]).
constexpr int kBoxStep = 8;  // log2 kBlock
struct BoxOut {
    LeafBox* level[kBoxStep];
};
__global__ __launch_bounds__(kBlock) void k_box_levels(uint32_t m, const LeafBox* __restrict in, BoxOut out)
{
    __shared__ LeafBox s[kBlock];
    const uint32_t t = threadIdx.x, base = blockIdx.x * kBlock;
    const uint32_t count = min((uint32_t)kBlock, m - base);
    if (t < count) s[t] = in[base + t];
    __syncthreads();
    uint32_t c = count;
    for (int k = 0; k < kBoxStep; ++k) {
        const uint32_t h = (c + 1) / 2;
        LeafBox b;
        if (t < h) {
            b = s[2 * t];
            if (2 * t + 1 < c) grow_box(b.lo, b.hi, s[2 * t + 1]);
        }
        __syncthreads();
        if (t < h) {
            s[t] = b;
            out.level[k][(base >> (k + 1)) + t] = b;
        }
        __syncthreads();
        c = h;
    }
}

// Internal node i of n-1: its children (internal index, or ~leaf for leaves), their boxes and the
// children's parent links.
__global__ __launch_bounds__(kBlock) void k_karras(const uint64_t* __restrict keys, int n, BoxLevels levels,
                                                   BvhNode* __restrict nodes, int* __restrict parent_int,
                                                   int* __restrict parent_leaf)
{
    int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n - 1) return;
    int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = delta(keys, n, i, j);
    int s = 0;
    int div = 2;
    while (true) {
        int t = (l + div - 1) / div;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
        if (t <= 1) break;
        div <<= 1;
    }
    int gamma = i + s * d + min(d, 0);
    int left, right;
    const int first = min(i, j), last = max(i, j);
    if (first == gamma) {
        left = ~gamma;
        parent_leaf[gamma] = i;
    } else {
        left = gamma;
        parent_int[gamma] = i;
    }
    if (last == gamma + 1) {
        right = ~(gamma + 1);
        parent_leaf[gamma + 1] = i;
    } else {
        right = gamma + 1;
        parent_int[gamma + 1] = i;
    }
    float4 lo0, hi0, lo1, hi1;
    range_box(levels, (uint32_t)first, (uint32_t)gamma, lo0, hi0);
    range_box(levels, (uint32_t)gamma + 1u, (uint32_t)last, lo1, hi1);
    BvhNode nd;
    nd.x = make_float4(lo0.x, hi0.x, lo1.x, hi1.x);
    nd.y = make_float4(lo0.y, hi0.y, lo1.y, hi1.y);
    nd.z = make_float4(lo0.z, hi0.z, lo1.z, hi1.z);
    nd.child = make_int4(left, right, 0, 0);
    nodes[i] = nd;
    if (i == 0) parent_int[0] = -1;
}

// Single-triangle scene: one root whose two children are the same leaf.
__global__ void k_single(const float4* __restrict blo, const float4* __restrict bhi,
                         const uint32_t* __restrict bounds, BvhNode* __restrict nodes)
{
    float eps = inflate_eps(bounds);
    float4 lo = blo[0], hi = bhi[0];
    lo.x -= eps; lo.y -= eps; lo.z -= eps;
    hi.x += eps; hi.y += eps; hi.z += eps;
    BvhNode nd;
    nd.x = make_float4(lo.x, hi.x, lo.x, hi.x);
    nd.y = make_float4(lo.y, hi.y, lo.y, hi.y);
    nd.z = make_float4(lo.z, hi.z, lo.z, hi.z);
    nd.child = make_int4(~0, ~0, 0, 0);
    nodes[0] = nd;
}

// ---- PLOC: the binary tree by parallel locally-ordered clustering ----------------------------------
//
// Meister and Bittner, "Parallel Locally-Ordered Clustering for Bounding Volume Hierarchy
// Construction" (IEEE TVCG 2018). The clusters start as the leaves in Morton order; every round,
// each cluster finds the neighbour within kPlocRadius positions whose union box has the smallest
// surface area, mutual nearest neighbours merge into a new internal node (at the lower position),
// and the surviving clusters are compacted in order. Edges are ordered by (area, lower position,
// higher position), so the nearest-neighbour relation has no cycles and every round merges at
// least one pair. Node indices are handed out from n - 2 downwards in position order, so the last
// merge is the root, node 0, and the tree is deterministic.

constexpr int kPlocRadius = 16;

__device__ __forceinline__ float union_area(float4 alo, float4 ahi, float4 blo, float4 bhi)
{
    const float dx = fmaxf(ahi.x, bhi.x) - fminf(alo.x, blo.x);
    const float dy = fmaxf(ahi.y, bhi.y) - fminf(alo.y, blo.y);
    const float dz = fmaxf(ahi.z, bhi.z) - fminf(alo.z, blo.z);
    return dx * dy + dy * dz + dz * dx;
}

// The leaves as the first clusters: leaf j (Morton order) with its inflated box, height 0.
__global__ __launch_bounds__(kBlock) void k_ploc_init(uint32_t n, const float4* __restrict blo,
                                                      const float4* __restrict bhi, const uint32_t* __restrict order,
                                                      const uint32_t* __restrict bounds, int* __restrict cid,
                                                      float4* __restrict clo, float4* __restrict chi,
                                                      uint32_t* __restrict height)
{
    const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= n) return;
    const float eps = inflate_eps(bounds);
    float4 lo, hi;
    leaf_box(blo, bhi, order, (int)j, eps, lo, hi);
    cid[j] = ~(int)j;
    clo[j] = lo;
    chi[j] = hi;
    height[j] = 0;
}

// nn[i] = the neighbour of cluster i (within kPlocRadius positions) of least union area, edges
// ordered by (area, lower position, higher position). The block's clusters and the radius on both
// sides are staged in LDS.
__global__ __launch_bounds__(kBlock) void k_ploc_nn(uint32_t m, const float4* __restrict clo,
                                                    const float4* __restrict chi, uint32_t* __restrict nn)
{
    __shared__ float4 slo[kBlock + 2 * kPlocRadius], shi[kBlock + 2 * kPlocRadius];
    const int first = (int)(blockIdx.x * kBlock) - kPlocRadius;
    for (int k = threadIdx.x; k < kBlock + 2 * kPlocRadius; k += kBlock) {
        const int g = first + k;
        if (g >= 0 && g < (int)m) {
            slo[k] = clo[g];
            shi[k] = chi[g];
        }
    }
    __syncthreads();
    const int i = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (i >= (int)m) return;
    const int li = i - first;
    const float4 lo = slo[li], hi = shi[li];
    float best = 0.0f;
    int bj = -1;
    const int j0 = i - kPlocRadius < 0 ? 0 : i - kPlocRadius;
    const int j1 = i + kPlocRadius >= (int)m ? (int)m - 1 : i + kPlocRadius;
    for (int j = j0; j <= j1; ++j) {
        if (j == i) continue;
        const float a = union_area(lo, hi, slo[j - first], shi[j - first]);
        // (a, min, max) against the best edge so far; with i fixed, a smaller other end wins ties
        if (bj < 0 || a < best || (a == best && j < bj)) {
            best = a;
            bj = j;
        }
    }
    nn[i] = (uint32_t)bj;
}

// Per position: bit 0 of keep = the cluster survives this round (it is not the higher end of a
// merging pair), bit 32 = it is the lower end of a merging pair (a new node).
__global__ __launch_bounds__(kBlock) void k_ploc_flags(uint32_t m, const uint32_t* __restrict nn,
                                                       uint64_t* __restrict flags)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= m) return;
    const uint32_t j = nn[i];
    const bool mutual = nn[j] == i;
    const uint64_t keep = (mutual && j < i) ? 0ull : 1ull;
    const uint64_t lead = (mutual && i < j) ? 1ull : 0ull;
    flags[i] = keep | (lead << 32);
}

// The round's merges (node base + rank among this round's merges, written as BvhNodes) and the
// surviving clusters, compacted in position order into the other buffers.
__global__ __launch_bounds__(kBlock) void k_ploc_merge(uint32_t m, uint32_t node_base, const uint32_t* __restrict nn,
                                                       const uint64_t* __restrict flags,
                                                       const uint64_t* __restrict prefix, const int* __restrict cid,
                                                       const float4* __restrict clo, const float4* __restrict chi,
                                                       const uint32_t* __restrict height, int* __restrict ncid,
                                                       float4* __restrict nlo, float4* __restrict nhi,
                                                       uint32_t* __restrict nheight, BvhNode* __restrict nodes)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= m) return;
    const uint64_t f = flags[i];
    if (!(f & 1ull)) return;
    const uint32_t pos = (uint32_t)(prefix[i] & 0xFFFFFFFFull);
    if (f >> 32) {
        const uint32_t j = nn[i];
        const uint32_t id = node_base + (uint32_t)(prefix[i] >> 32);
        const float4 lo0 = clo[i], hi0 = chi[i], lo1 = clo[j], hi1 = chi[j];
        BvhNode nd;
        nd.x = make_float4(lo0.x, hi0.x, lo1.x, hi1.x);
        nd.y = make_float4(lo0.y, hi0.y, lo1.y, hi1.y);
        nd.z = make_float4(lo0.z, hi0.z, lo1.z, hi1.z);
        nd.child = make_int4(cid[i], cid[j], 0, 0);
        nodes[id] = nd;
        ncid[pos] = (int)id;
        nlo[pos] = make_float4(fminf(lo0.x, lo1.x), fminf(lo0.y, lo1.y), fminf(lo0.z, lo1.z), 0.0f);
        nhi[pos] = make_float4(fmaxf(hi0.x, hi1.x), fmaxf(hi0.y, hi1.y), fmaxf(hi0.z, hi1.z), 0.0f);
        nheight[pos] = 1 + max(height[i], height[j]);
    } else {
        ncid[pos] = cid[i];
        nlo[pos] = clo[i];
        nhi[pos] = chi[i];
        nheight[pos] = height[i];
    }
}

__global__ __launch_bounds__(kBlock) void k_depth(int n, const int* __restrict parent_int,
                                                  const int* __restrict parent_leaf, uint32_t* maxdepth)
{
    int j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= n) return;
    uint32_t d = 1;
    int p = parent_leaf[j];
    while (p > 0 && p < n - 1 && d <= (uint32_t)n) {
        p = parent_int[p];
        ++d;
    }
    atomicMax(maxdepth, d);
}

// ---- 8-wide collapse (breadth-first, one level per pair of launches) ----
//
// A wide node starts from its binary node's two children and repeatedly opens the internal child
// of largest surface area (the first such child on ties) until it has 8 children or only leaves.
// A task is a binary node and the slot its wide node goes to. k_wide_expand writes each task's
// children (binary refs and boxes) and the counts of its internal children and of the slots its
// children take; a scan of those counts numbers the next level's tasks and slots in task order, so the
// numbering (and the tree) is deterministic and a node's children are contiguous;
// k_wide_emit quantizes the boxes and writes the node's first slot (internal children first), the
// next level's tasks and the leaves' slots. In the top tree of an instanced scene leaves are nodes
// too: a task ~k stands for leaf k, whose node is its instance's (InstNode). A node has 8 children
// or only leaves, so there are at most 4 n / 7 nodes over n leaves.

struct WideTask {
    int ref;        // binary node, or ~leaf in a top tree
    uint32_t slot;
};

__device__ __forceinline__ float half_area(const float* b)
{
    float dx = fmaxf(b[3] - b[0], 0.0f), dy = fmaxf(b[4] - b[1], 0.0f), dz = fmaxf(b[5] - b[2], 0.0f);
    return dx * dy + dy * dz + dz * dx;
}

__device__ __forceinline__ void child_box(const BvhNode& nd, int c, float* b)
{
    b[0] = c ? nd.x.z : nd.x.x;
    b[1] = c ? nd.y.z : nd.y.x;
    b[2] = c ? nd.z.z : nd.z.x;
    b[3] = c ? nd.x.w : nd.x.y;
    b[4] = c ? nd.y.w : nd.y.y;
    b[5] = c ? nd.z.w : nd.z.y;
}

template <bool TOP>
__global__ __launch_bounds__(kBlock) void k_wide_expand(const WideTask* __restrict tasks, uint32_t n_tasks,
                                                        const BvhNode* __restrict bn, int* __restrict cref,
                                                        float* __restrict cbox, uint32_t* __restrict nchild,
                                                        uint64_t* __restrict counts)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= n_tasks) return;
    const int task = tasks[t].ref;
    if (TOP && task < 0) {  // an instance's node
        cref[8 * (size_t)t] = task;
        nchild[t] = 0;
        counts[t] = 0;
        return;
    }
    int ref[8];
    float box[8][6];
    const BvhNode root = bn[task];
    ref[0] = root.child.x;
    ref[1] = root.child.y;
    child_box(root, 0, box[0]);
    child_box(root, 1, box[1]);
    uint32_t m = 2;
    while (m < 8) {
        int best = -1;
        float best_a = -1.0f;
        for (uint32_t k = 0; k < m; ++k)
            if (ref[k] >= 0) {
                float a = half_area(box[k]);
                if (a > best_a) {
                    best_a = a;
                    best = (int)k;
                }
            }
        if (best < 0) break;
        const BvhNode nd = bn[ref[best]];
        ref[best] = nd.child.x;
        child_box(nd, 0, box[best]);
        ref[m] = nd.child.y;
        child_box(nd, 1, box[m]);
        ++m;
    }
    uint32_t internal = 0, out = 0;
    for (uint32_t k = 0; k < m; ++k) internal += (TOP || ref[k] >= 0) ? 1u : 0u;
    // internal children first, both kinds in the order found
    for (int pass = 0; pass < 2; ++pass)
        for (uint32_t k = 0; k < m; ++k) {
            if ((TOP || ref[k] >= 0) != (pass == 0)) continue;
            cref[8 * (size_t)t + out] = ref[k];
            for (int a = 0; a < 6; ++a) cbox[48 * (size_t)t + 6 * out + a] = box[k][a];
            ++out;
        }
    nchild[t] = internal | (m << 8);
    // slots: two per node, one per leaf after the first, an even number (nodes stay 128-byte aligned)
    const uint32_t slots = (2 * internal + (m > internal ? m - internal - 1 : 0) + 1) & ~1u;
    counts[t] = (uint64_t)internal | ((uint64_t)slots << 32);
}

// Smallest e in [-126, 127] with ext <= 254 * 2^e (ext >= 0).
__device__ __forceinline__ int plane_exponent(double ext)
{
    if (!(ext > 0.0)) return -126;
    int k;
    double f = frexp(ext / 254.0, &k);  // ext / 254 = f * 2^k, f in [0.5, 1)
    int e = f == 0.5 ? k - 1 : k;
    return e < -126 ? -126 : (e > 127 ? 127 : e);
}

// The largest float not above x whose low 11 bits are zero.
__device__ __forceinline__ float origin_floor(float x)
{
    uint32_t u = __float_as_uint(x);
    if (x < 0.0f && (u & ~kOriginMask)) u += ~kOriginMask + 1u;
    return __uint_as_float(u & kOriginMask);
}

// The first slot of a node (or an instance's node), as the traversal reads it.
struct NodeSlot {
    uint32_t w[16];
};

template <bool TOP>
__global__ __launch_bounds__(kBlock) void k_wide_emit(uint32_t n_tasks, uint32_t level_base, uint32_t slot_base,
                                                      const WideTask* __restrict tasks,
                                                      const uint64_t* __restrict ends, const uint64_t* __restrict counts,
                                                      const int* __restrict cref,
                                                      const float* __restrict cbox, const uint32_t* __restrict nchild,
                                                      NodeSlot* __restrict out, uint32_t* __restrict out_slot,
                                                      WideTask* __restrict next_tasks,
                                                      uint32_t* __restrict leaf_slot,
                                                      const InstRecord* __restrict insts,
                                                      const uint32_t* __restrict order, uint32_t* __restrict bad)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= n_tasks) return;
    const uint32_t ni = nchild[t] & 0xFFu, m = nchild[t] >> 8, slot = tasks[t].slot;
    out_slot[level_base + t] = slot;
    NodeSlot w;
    if (TOP && m == 0) {
        InstNode in;
        in.index = order[~cref[8 * (size_t)t]];
        in.unused[0] = in.unused[1] = 0;
        in.meta = 0;
        for (int r = 0; r < 3; ++r) in.w2l[r] = insts[in.index].w2l[r];
        *reinterpret_cast<InstNode*>(&out[level_base + t]) = in;
        return;
    }
    const float* B = cbox + 48 * (size_t)t;
    float lo[3] = {B[0], B[1], B[2]}, hi[3] = {B[3], B[4], B[5]};
    for (uint32_t k = 1; k < m; ++k)
        for (int a = 0; a < 3; ++a) {
            lo[a] = fminf(lo[a], B[6 * k + a]);
            hi[a] = fmaxf(hi[a], B[6 * k + 3 + a]);
        }
    const uint64_t offset = ends[t] - counts[t];
    const uint32_t base = slot_base + (uint32_t)(offset >> 32);
    uint32_t meta = ni << 24 | m << 28;
    for (int a = 0; a < 3; ++a) {
        const float og = origin_floor(lo[a]);
        w.w[a] = __float_as_uint(og) | ((a == 0 ? base : a == 1 ? base >> 11 : base >> 22) & ~kOriginMask);
        const int e = plane_exponent((double)hi[a] - (double)og);
        const float sc = __uint_as_float((uint32_t)(e + 127) << 23);
        const double sd = (double)sc;
        meta |= ((uint32_t)e & 0xFFu) << (8 * a);
        uint32_t qw[2][2] = {{0, 0}, {0, 0}};
        for (uint32_t k = 0; k < 8; ++k) {
            int qlo = 255, qhi = 0;  // an empty box
            if (k < m) {
                const float clo = B[6 * k + a], chi = B[6 * k + 3 + a];
                double ql = floor(((double)clo - (double)og) / sd);
                double qh = ceil(((double)chi - (double)og) / sd);
                qlo = ql < 0.0 ? 0 : (ql > 255.0 ? 255 : (int)ql);
                qhi = qh < 0.0 ? 0 : (qh > 255.0 ? 255 : (int)qh);
                // the decoded planes (one FP32 rounding) must contain the box
                while (qlo > 0 && fmaf((float)qlo, sc, og) > clo) --qlo;
                while (qhi < 255 && fmaf((float)qhi, sc, og) < chi) ++qhi;
                if (fmaf((float)qlo, sc, og) > clo || fmaf((float)qhi, sc, og) < chi) atomicOr(bad, 1u);
            }
            qw[0][k >> 2] |= (uint32_t)qlo << (8 * (k & 3));
            qw[1][k >> 2] |= (uint32_t)qhi << (8 * (k & 3));
        }
        for (int h = 0; h < 2; ++h) {
            w.w[4 + 2 * a + h] = qw[0][h];
            w.w[10 + 2 * a + h] = qw[1][h];
        }
    }
    w.w[3] = meta;
    const uint32_t task_off = (uint32_t)(offset & 0xFFFFFFFFull);
    for (uint32_t k = 0; k < m; ++k) {
        const int r = cref[8 * (size_t)t + k];
        if (k < ni)
            next_tasks[task_off + k] = WideTask{r, base + 2 * k};
        else
            leaf_slot[~r] = k == ni ? slot + 1 : base + ni + k - 1;  // leaf k - ni: the node's second slot, or base + 2 ni + (k - ni) - 1
    }
    out[level_base + t] = w;
}

// The nodes' first slots and the leaves' records in their slots.
__global__ __launch_bounds__(kBlock) void k_place_nodes(const NodeSlot* __restrict in, const uint32_t* __restrict slot,
                                                        uint32_t n, NodeSlot* __restrict out)
{
    // four lanes a slot
    const size_t k = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (k / 4 >= n) return;
    reinterpret_cast<uint4*>(out + slot[k / 4])[k % 4] = reinterpret_cast<const uint4*>(in + k / 4)[k % 4];
}

// (`stride` bytes from a record to the next, of which a slot's worth is placed)
__global__ __launch_bounds__(kBlock) void k_place_records(const char* __restrict in, uint32_t stride,
                                                          const uint32_t* __restrict order,
                                                          const uint32_t* __restrict leaf_slot, uint32_t n,
                                                          NodeSlot* __restrict out)
{
    const size_t k = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const size_t j = k / 4;
    if (j >= n) return;
    reinterpret_cast<uint4*>(out + leaf_slot[j])[k % 4] = reinterpret_cast<const uint4*>(in + (size_t)order[j] * stride)[k % 4];
}

// The binary tree's leaves named by their records' slots.
__global__ __launch_bounds__(kBlock) void k_relabel(BvhNode* __restrict nodes, uint32_t n_int,
                                                    const uint32_t* __restrict leaf_slot)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n_int) return;
    int4 c = nodes[i].child;
    if (c.x < 0) c.x = ~(int)leaf_slot[~c.x];
    if (c.y < 0) c.y = ~(int)leaf_slot[~c.y];
    nodes[i].child = c;
}

// An array in the build's scratch.
template <typename T>
struct DevBuf {
    T* p = nullptr;
    hipError_t alloc(sgpu_scratch& s, size_t count)
    {
        p = s.get<T>(count);
        return s.err;
    }
};

// Scratch bytes a build over n primitives takes at its widest, in the binary tree: per primitive the
// record (64 for triangles, 80 for curves), order and places (12), positions (40, triangles), boxes and
// centroid (48), sorted codes (8), parents (8) and the box pyramid (64); the sort before it and the 8-wide
// tree after it take the same memory and need less. In a top tree or with PLOC more, taken as needed.
size_t build_scratch(size_t n) { return 240 * n + ((size_t)1 << 20); }

struct WideTree {
    WideNode* wide = nullptr;
    uint32_t n_slots = 0, n_wide = 0, depth = 0;
};

// Collapses the binary tree (nodes, root 0, over n leaves) into an 8-wide tree, with the records rec[order[j]]
// (rec_bytes apart, the first 64 a leaf's slot) of its leaves j; d_leaf_slot: their slots. The top tree of
// an instanced scene passes its instance records instead (order[j]: the instance of leaf j): its leaves
// become nodes.
int build_wide(sgpu_scratch& S, const BvhNode* nodes, uint32_t n, hipStream_t stream, const uint32_t* order,
               const void* rec, uint32_t rec_bytes, const InstRecord* insts, WideTree& tree,
               DevBuf<uint32_t>& d_leaf_slot)
{
    const bool top = insts != nullptr;
    const uint32_t n_leaves = std::max(n, 2u);  // a tree of one leaf has a root with two children, the leaf twice
    const size_t max_nodes = (size_t)n_leaves * 4 / 7 + 2 + (top ? n_leaves : 0);
    SGPU_HIP_TRY(d_leaf_slot.alloc(S, n_leaves));
    sgpu_scratch::Frame frame(S);
    DevBuf<WideTask> d_tasks, d_next;
    DevBuf<uint32_t> d_bad, d_slot;
    DevBuf<NodeSlot> d_all;
    SGPU_HIP_TRY(d_tasks.alloc(S, max_nodes));
    SGPU_HIP_TRY(d_next.alloc(S, max_nodes));
    SGPU_HIP_TRY(d_bad.alloc(S, 1));
    SGPU_HIP_TRY(d_all.alloc(S, max_nodes));
    SGPU_HIP_TRY(d_slot.alloc(S, max_nodes));
    const WideTask root{0, 0};
    SGPU_HIP_TRY(hipMemcpyAsync(d_tasks.p, &root, sizeof(root), hipMemcpyHostToDevice, stream));
    SGPU_HIP_TRY(hipMemsetAsync(d_bad.p, 0, sizeof(uint32_t), stream));
    uint32_t level_base = 0, n_tasks = 1, depth = 0;
    uint64_t slot_base = 2;
    // a level's tasks at most this many at a time: their children take 250 bytes a task, which for the last
    // level of a top tree (its instances) would be the most of a build's scratch
    const uint32_t chunk = std::max(1u << 17, n_leaves / 8);
    while (n_tasks > 0) {
        uint32_t n_next = 0;
        for (uint32_t c0 = 0; c0 < n_tasks; c0 += chunk) {
            const uint32_t nc = std::min(chunk, n_tasks - c0);
            const WideTask* const tasks = d_tasks.p + c0;
            sgpu_scratch::Frame children(S);
            DevBuf<int> d_cref;
            DevBuf<float> d_cbox;
            DevBuf<uint32_t> d_nch;
            DevBuf<uint64_t> d_cnt, d_off;
            DevBuf<uint8_t> d_tmp;
            SGPU_HIP_TRY(d_cref.alloc(S, 8 * (size_t)nc));
            SGPU_HIP_TRY(d_cbox.alloc(S, 48 * (size_t)nc));
            SGPU_HIP_TRY(d_nch.alloc(S, nc));
            SGPU_HIP_TRY(d_cnt.alloc(S, nc));
            SGPU_HIP_TRY(d_off.alloc(S, nc));
            size_t tmp_bytes = 0;
            SGPU_HIP_TRY(rocprim::inclusive_scan(nullptr, tmp_bytes, d_cnt.p, d_off.p, (size_t)nc,
                                                 rocprim::plus<uint64_t>(), stream));
            SGPU_HIP_TRY(d_tmp.alloc(S, tmp_bytes));
            const uint32_t grid = (nc + kBlock - 1) / kBlock;
            if (top)
                hipLaunchKernelGGL(k_wide_expand<true>, dim3(grid), dim3(kBlock), 0, stream, tasks, nc, nodes, d_cref.p,
                                   d_cbox.p, d_nch.p, d_cnt.p);
            else
                hipLaunchKernelGGL(k_wide_expand<false>, dim3(grid), dim3(kBlock), 0, stream, tasks, nc, nodes, d_cref.p,
                                   d_cbox.p, d_nch.p, d_cnt.p);
            SGPU_HIP_TRY(hipGetLastError());
            SGPU_HIP_TRY(rocprim::inclusive_scan(d_tmp.p, tmp_bytes, d_cnt.p, d_off.p, (size_t)nc,
                                                 rocprim::plus<uint64_t>(), stream));
            SGPU_HIP_TRY(hipMemcpyAsync(S.pinned(), d_off.p + nc - 1, sizeof(uint64_t), hipMemcpyDeviceToHost, stream));
            SGPU_HIP_TRY(hipStreamSynchronize(stream));
            const uint64_t total = S.pinned()[0];
            const uint32_t n_child = (uint32_t)(total & 0xFFFFFFFFull), n_new = (uint32_t)(total >> 32);
            if ((uint64_t)level_base + n_tasks + n_next + n_child > max_nodes)
                return sgpu_fail(SGPU_E_STATE, "wide tree larger than its bound");
            if (slot_base + n_new > 0x7FFFFFFFull)
                return sgpu_fail(SGPU_E_RANGE, "wide tree takes more than 2^31 slots");
            if (top)
                hipLaunchKernelGGL(k_wide_emit<true>, dim3(grid), dim3(kBlock), 0, stream, nc, level_base + c0,
                                   (uint32_t)slot_base, tasks, d_off.p, d_cnt.p, d_cref.p, d_cbox.p, d_nch.p, d_all.p,
                                   d_slot.p, d_next.p + n_next, d_leaf_slot.p, insts, order, d_bad.p);
            else
                hipLaunchKernelGGL(k_wide_emit<false>, dim3(grid), dim3(kBlock), 0, stream, nc, level_base + c0,
                                   (uint32_t)slot_base, tasks, d_off.p, d_cnt.p, d_cref.p, d_cbox.p, d_nch.p, d_all.p,
                                   d_slot.p, d_next.p + n_next, d_leaf_slot.p, insts, order, d_bad.p);
            SGPU_HIP_TRY(hipGetLastError());
            n_next += n_child;
            slot_base += n_new;
        }
        std::swap(d_tasks.p, d_next.p);
        level_base += n_tasks;
        n_tasks = n_next;
        ++depth;
    }
    SGPU_HIP_TRY(hipMemcpyAsync(S.pinned(), d_bad.p, sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    SGPU_HIP_TRY(hipStreamSynchronize(stream));
    if (*(const uint32_t*)S.pinned()) return sgpu_fail(SGPU_E_RANGE, "wide node quantization could not contain a child box");
    if (sgpu_device_malloc((void**)&tree.wide, slot_base * kSlotBytes) != hipSuccess)
        return sgpu_fail(SGPU_E_NOMEM, "hipMalloc of triangle records and 8-wide nodes failed");
    tree.n_slots = (uint32_t)slot_base;
    tree.n_wide = level_base;
    tree.depth = depth;
    NodeSlot* const slots = reinterpret_cast<NodeSlot*>(tree.wide);
    auto grid4 = [](size_t k) { return dim3((uint32_t)((4 * k + kBlock - 1) / kBlock)); };
    hipLaunchKernelGGL(k_place_nodes, grid4(level_base), dim3(kBlock), 0, stream, d_all.p, d_slot.p, level_base, slots);
    SGPU_HIP_TRY(hipGetLastError());
    if (!top) {
        hipLaunchKernelGGL(k_place_records, grid4(n), dim3(kBlock), 0, stream, (const char*)rec, rec_bytes, order,
                           d_leaf_slot.p, n, slots);
        SGPU_HIP_TRY(hipGetLastError());
        if (n == 1)  // a single leaf is both children of the root: slots 1 and 2
            for (int k = 1; k <= 2; ++k)
                SGPU_HIP_TRY(hipMemcpyAsync(slots + k, rec, kSlotBytes, hipMemcpyDeviceToDevice, stream));
    }
    SGPU_HIP_TRY(hipStreamSynchronize(stream));
    return SGPU_OK;
}

// build_wide as the scene's own tree (of triangles, or of instances).
int build_scene_wide(sgpu_scene scene, sgpu_scratch& S, BvhNode* nodes, uint32_t n, hipStream_t stream,
                     const uint32_t* order, const TriRecord* rec, const InstRecord* insts)
{
    WideTree t;
    DevBuf<uint32_t> leaf_slot;
    const int rc = build_wide(S, nodes, n, stream, order, rec, sizeof(TriRecord), insts, t, leaf_slot);
    scene->d_wide = t.wide;
    scene->n_slots = t.n_slots;
    scene->n_wide = t.n_wide;
    scene->wide_depth = t.depth;
    if (rc != SGPU_OK || insts) return rc;
    const uint32_t n_int = n > 1 ? n - 1 : 1;
    hipLaunchKernelGGL(k_relabel, dim3((n_int + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, nodes, n_int, leaf_slot.p);
    SGPU_HIP_TRY(hipGetLastError());
    SGPU_HIP_TRY(hipStreamSynchronize(stream));
    return SGPU_OK;
}

// Words of traversal stack an 8-wide tree of `levels` levels can need: an entry of two words for every
// node above the walked one's parent (whose group is in registers) but the root's level and the last,
// whose nodes have no nodes below.
uint32_t wide_stack_words(uint32_t levels) { return levels > 2 ? 2 * (levels - 2) : 0; }

}  // namespace

namespace {

float host_ord2f(uint32_t u)
{
    const uint32_t b = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
    float f;
    std::memcpy(&f, &b, sizeof(f));
    return f;
}

uint32_t host_f2ord(float f)
{
    uint32_t u;
    std::memcpy(&u, &f, sizeof(u));
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The binary tree over n primitive boxes (d_blo, d_bhi, centroids d_cent, bounds as k_prep
// leaves them): Morton codes, radix sort, box pyramid, Karras hierarchy. On success *nodes_out holds
// max(n - 1, 1) nodes (the caller's array, or where it is NULL a new one), d_order (the caller's) the
// primitive of each leaf in leaf order and *depth the deepest leaf.
int build_binary(sgpu_scratch& S, uint32_t n, const float4* d_blo, const float4* d_bhi, const float4* d_cent, const uint32_t* d_bounds,
                 hipStream_t stream, BvhNode** nodes_out, const DevBuf<uint32_t>& d_order, uint32_t* depth_out,
                 uint32_t builder)
{
    sgpu_scratch::Frame frame(S);
    const uint32_t n_int = n > 1 ? n - 1 : 1;
    BvhNode* nodes = *nodes_out;
    if (!nodes) SGPU_HIP_TRY(sgpu_device_malloc((void**)&nodes, (size_t)n_int * sizeof(BvhNode)));
    auto fail_free = [&](int code, const std::string& msg) {
        if (!*nodes_out) (void)hipFree(nodes);
        return sgpu_fail(code, msg);
    };
#define SGPU_BUILD_TRY(expr)                                                                  \
    do {                                                                                      \
        hipError_t _e = (expr);                                                               \
        if (_e != hipSuccess) return fail_free(SGPU_E_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
    } while (0)
    if (n == 1) {
        hipLaunchKernelGGL(k_single, dim3(1), dim3(1), 0, stream, d_blo, d_bhi, d_bounds, nodes);
        SGPU_BUILD_TRY(hipGetLastError());
        SGPU_BUILD_TRY(hipMemsetAsync(d_order.p, 0, sizeof(uint32_t), stream));
        SGPU_BUILD_TRY(hipStreamSynchronize(stream));
        *nodes_out = nodes;
        *depth_out = 1;
        return SGPU_OK;
    }
    const uint32_t grid = (n + kBlock - 1) / kBlock;
    DevBuf<uint64_t> d_keys2;
    SGPU_BUILD_TRY(d_keys2.alloc(S, n));
    {
        sgpu_scratch::Frame sort(S);
        DevBuf<uint64_t> d_keys;
        DevBuf<uint32_t> d_vals;
        DevBuf<uint8_t> d_tmp;
        SGPU_BUILD_TRY(d_keys.alloc(S, n));
        SGPU_BUILD_TRY(d_vals.alloc(S, n));
        hipLaunchKernelGGL(k_morton, dim3(grid), dim3(kBlock), 0, stream, d_cent, n, d_bounds, d_keys.p, d_vals.p);
        SGPU_BUILD_TRY(hipGetLastError());
        size_t tmp_bytes = 0;
        SGPU_BUILD_TRY(rocprim::radix_sort_pairs(nullptr, tmp_bytes, d_keys.p, d_keys2.p, d_vals.p, d_order.p,
                                                 (size_t)n, 0, 63, stream));
        SGPU_BUILD_TRY(d_tmp.alloc(S, tmp_bytes));
        SGPU_BUILD_TRY(rocprim::radix_sort_pairs(d_tmp.p, tmp_bytes, d_keys.p, d_keys2.p, d_vals.p, d_order.p,
                                                 (size_t)n, 0, 63, stream));
    }
    if (builder == 1) {
        // PLOC over the Morton-ordered leaves
        DevBuf<int> cid[2];
        DevBuf<float4> clo[2], chi[2];
        DevBuf<uint32_t> hgt[2], nn;
        DevBuf<uint64_t> flags, prefix;
        for (int b = 0; b < 2; ++b) {
            SGPU_BUILD_TRY(cid[b].alloc(S, n));
            SGPU_BUILD_TRY(clo[b].alloc(S, n));
            SGPU_BUILD_TRY(chi[b].alloc(S, n));
            SGPU_BUILD_TRY(hgt[b].alloc(S, n));
        }
        SGPU_BUILD_TRY(nn.alloc(S, n));
        SGPU_BUILD_TRY(flags.alloc(S, n));
        SGPU_BUILD_TRY(prefix.alloc(S, n));
        size_t scan_bytes = 0;
        SGPU_BUILD_TRY(rocprim::exclusive_scan(nullptr, scan_bytes, flags.p, prefix.p, (uint64_t)0, (size_t)n,
                                               rocprim::plus<uint64_t>(), stream));
        DevBuf<uint8_t> d_scan;
        SGPU_BUILD_TRY(d_scan.alloc(S, scan_bytes));
        hipLaunchKernelGGL(k_ploc_init, dim3(grid), dim3(kBlock), 0, stream, n, d_blo, d_bhi, d_order.p, d_bounds,
                           cid[0].p, clo[0].p, chi[0].p, hgt[0].p);
        SGPU_BUILD_TRY(hipGetLastError());
        uint32_t m = n, next_id = n - 1, cur = 0;
        uint64_t tail[2] = {0, 0};
        while (m > 1) {
            const uint32_t g = (m + kBlock - 1) / kBlock;
            hipLaunchKernelGGL(k_ploc_nn, dim3(g), dim3(kBlock), 0, stream, m, clo[cur].p, chi[cur].p, nn.p);
            hipLaunchKernelGGL(k_ploc_flags, dim3(g), dim3(kBlock), 0, stream, m, nn.p, flags.p);
            SGPU_BUILD_TRY(hipGetLastError());
            SGPU_BUILD_TRY(rocprim::exclusive_scan(d_scan.p, scan_bytes, flags.p, prefix.p, (uint64_t)0, (size_t)m,
                                                   rocprim::plus<uint64_t>(), stream));
            SGPU_BUILD_TRY(hipMemcpyAsync(&tail[0], prefix.p + m - 1, sizeof(uint64_t), hipMemcpyDeviceToHost, stream));
            SGPU_BUILD_TRY(hipMemcpyAsync(&tail[1], flags.p + m - 1, sizeof(uint64_t), hipMemcpyDeviceToHost, stream));
            SGPU_BUILD_TRY(hipStreamSynchronize(stream));
            const uint64_t tot = tail[0] + tail[1];
            const uint32_t kept = (uint32_t)(tot & 0xFFFFFFFFull), merges = (uint32_t)(tot >> 32);
            if (merges == 0 || merges > next_id || kept != m - merges)
                return fail_free(SGPU_E_STATE, "PLOC: a clustering round made no progress");
            next_id -= merges;
            hipLaunchKernelGGL(k_ploc_merge, dim3(g), dim3(kBlock), 0, stream, m, next_id, nn.p, flags.p, prefix.p,
                               cid[cur].p, clo[cur].p, chi[cur].p, hgt[cur].p, cid[1 - cur].p, clo[1 - cur].p,
                               chi[1 - cur].p, hgt[1 - cur].p, nodes);
            SGPU_BUILD_TRY(hipGetLastError());
            cur = 1 - cur;
            m = kept;
        }
        uint32_t h = 0;
        SGPU_BUILD_TRY(hipMemcpyAsync(&h, hgt[cur].p, sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
        SGPU_BUILD_TRY(hipStreamSynchronize(stream));
        if (next_id != 0) return fail_free(SGPU_E_STATE, "PLOC: the tree does not end at node 0");
        *nodes_out = nodes;
        *depth_out = h;
        return SGPU_OK;
    }
    DevBuf<int> d_pint, d_pleaf;
    DevBuf<uint32_t> d_depth;
    SGPU_BUILD_TRY(d_pint.alloc(S, n_int));
    SGPU_BUILD_TRY(d_pleaf.alloc(S, n));
    SGPU_BUILD_TRY(d_depth.alloc(S, 1));
    SGPU_BUILD_TRY(hipMemsetAsync(d_pint.p, 0xFF, (size_t)n_int * sizeof(int), stream));
    SGPU_BUILD_TRY(hipMemsetAsync(d_pleaf.p, 0xFF, (size_t)n * sizeof(int), stream));
    SGPU_BUILD_TRY(hipMemsetAsync(d_depth.p, 0, sizeof(uint32_t), stream));
    // the pyramid's levels one after another: level k has ceil(n / 2^k) boxes
    DevBuf<LeafBox> d_boxes;
    SGPU_BUILD_TRY(d_boxes.alloc(S, 2 * (size_t)n + 2 * kMaxBoxLevels));
    LeafBox* level[kMaxBoxLevels + kBoxStep];
    uint32_t size[kMaxBoxLevels + kBoxStep];
    size_t used = 0;
    for (int k = 0; k < kMaxBoxLevels + kBoxStep; ++k) {
        const uint32_t m = k < kMaxBoxLevels ? (uint32_t)(((uint64_t)n + (1ull << k) - 1) >> k) : 1u;
        size[k] = m;
        level[k] = k < kMaxBoxLevels ? d_boxes.p + used : level[kMaxBoxLevels - 1];
        if (k < kMaxBoxLevels) used += m;
    }
    hipLaunchKernelGGL(k_box_leaves, dim3(grid), dim3(kBlock), 0, stream, n, d_blo, d_bhi, d_order.p, d_bounds, level[0]);
    SGPU_BUILD_TRY(hipGetLastError());
    for (int k = 0; k < kMaxBoxLevels && size[k] > 1; k += kBoxStep) {
        BoxOut out;
        for (int j = 0; j < kBoxStep; ++j) out.level[j] = level[k + 1 + j];
        hipLaunchKernelGGL(k_box_levels, dim3((size[k] + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, size[k],
                           level[k], out);
        SGPU_BUILD_TRY(hipGetLastError());
    }
    BoxLevels levels;
    for (int k = 0; k < kMaxBoxLevels; ++k) levels.level[k] = level[k];
    const uint32_t grid_int = (n - 1 + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(k_karras, dim3(grid_int), dim3(kBlock), 0, stream, d_keys2.p, (int)n, levels, nodes, d_pint.p,
                       d_pleaf.p);
    SGPU_BUILD_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_depth, dim3(grid), dim3(kBlock), 0, stream, (int)n, d_pint.p, d_pleaf.p, d_depth.p);
    SGPU_BUILD_TRY(hipGetLastError());
    uint32_t depth = 0;
    SGPU_BUILD_TRY(hipMemcpyAsync(&depth, d_depth.p, sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    SGPU_BUILD_TRY(hipStreamSynchronize(stream));
#undef SGPU_BUILD_TRY
    *nodes_out = nodes;
    *depth_out = depth;
    return SGPU_OK;
}

}  // namespace

namespace {

// Box of each curve segment (its control points' box grown by the largest radius: the B-spline
// basis weights are non-negative and sum to one, so the swept balls stay inside), centroid, and the
// ordered-uint bounds k_prep computes. TIGHT: the box and centroid of the same cubic's Bezier points,
// which span the segment alone and not its neighbours' two thirds of the control polygon (a third of
// the length along a blade of grass); the bounds' scene box stays that of the control points.
template <bool TIGHT>
__global__ __launch_bounds__(kBlock) void k_curve_prep(const CurveRecord* __restrict rec, uint32_t n,
                                                       float4* __restrict blo, float4* __restrict bhi,
                                                       float4* __restrict cent, uint32_t* __restrict bounds)
{
    __shared__ uint32_t red[12][kBlock / 64];
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    uint32_t v[12];
    for (int k = 0; k < 12; ++k) v[k] = 0xFFFFFFFFu;
    if (i < n) {
        const CurveRecord r = rec[i];
        f3 lo = mk3(r.p[0].x, r.p[0].y, r.p[0].z), hi = lo;
        float rmax = r.p[0].w;
        for (int j = 1; j < 4; ++j) {
            lo = mk3(fminf(lo.x, r.p[j].x), fminf(lo.y, r.p[j].y), fminf(lo.z, r.p[j].z));
            hi = mk3(fmaxf(hi.x, r.p[j].x), fmaxf(hi.y, r.p[j].y), fmaxf(hi.z, r.p[j].z));
            rmax = fmaxf(rmax, r.p[j].w);
        }
        lo = mk3(lo.x - rmax, lo.y - rmax, lo.z - rmax);
        hi = mk3(hi.x + rmax, hi.y + rmax, hi.z + rmax);
        v[0] = f2ord(lo.x); v[1] = f2ord(lo.y); v[2] = f2ord(lo.z);
        v[3] = ~f2ord(hi.x); v[4] = ~f2ord(hi.y); v[5] = ~f2ord(hi.z);
        if (TIGHT) {
            const float4 p0 = r.p[0], p1 = r.p[1], p2 = r.p[2], p3 = r.p[3];
            auto bezier = [&](float a, float b, float c, float e, float& l, float& h) {
                const float q0 = (a + 4.0f * b + c) * (1.0f / 6.0f), q1 = (2.0f * b + c) * (1.0f / 3.0f);
                const float q2 = (b + 2.0f * c) * (1.0f / 3.0f), q3 = (b + 4.0f * c + e) * (1.0f / 6.0f);
                l = fminf(fminf(q0, q1), fminf(q2, q3)) - rmax;
                h = fmaxf(fmaxf(q0, q1), fmaxf(q2, q3)) + rmax;
            };
            bezier(p0.x, p1.x, p2.x, p3.x, lo.x, hi.x);
            bezier(p0.y, p1.y, p2.y, p3.y, lo.y, hi.y);
            bezier(p0.z, p1.z, p2.z, p3.z, lo.z, hi.z);
        }
        const f3 c = mk3(0.5f * (lo.x + hi.x), 0.5f * (lo.y + hi.y), 0.5f * (lo.z + hi.z));
        blo[i] = make_float4(lo.x, lo.y, lo.z, 0.0f);
        bhi[i] = make_float4(hi.x, hi.y, hi.z, 0.0f);
        cent[i] = make_float4(c.x, c.y, c.z, 0.0f);
        v[6] = f2ord(c.x); v[7] = f2ord(c.y); v[8] = f2ord(c.z);
        v[9] = ~f2ord(c.x); v[10] = ~f2ord(c.y); v[11] = ~f2ord(c.z);
    }
    for (int k = 0; k < 12; ++k) {
        uint32_t x = v[k];
        for (int off = 32; off > 0; off >>= 1) x = min(x, (uint32_t)__shfl_xor((int)x, off, 64));
        v[k] = x;
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 12; ++k) red[k][wave] = v[k];
    __syncthreads();
    if (threadIdx.x < 12) {
        uint32_t x = red[threadIdx.x][0];
        for (int w = 1; w < kBlock / 64; ++w) x = min(x, red[threadIdx.x][w]);
        atomicMin(&bounds[threadIdx.x], x);
    }
}

// Each segment's place in the leaf order `order`.
__global__ __launch_bounds__(kBlock) void k_curve_places(const uint32_t* __restrict order, uint32_t n,
                                                         uint32_t* __restrict place)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) place[order[i]] = i;
}

// The ids of the segment in each leaf's slot (a single segment is in slots 1 and 2).
__global__ __launch_bounds__(kBlock) void k_curve_ids(const CurveRecord* __restrict rec, const uint32_t* __restrict order,
                                                      const uint32_t* __restrict leaf_slot,
                                                      const uint32_t* __restrict place, uint32_t n,
                                                      uint4* __restrict ids)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t k = order[i];
    const uint4 v = make_uint4(rec[k].geom, rec[k].prim, rec[k].inst, place[k]);
    ids[leaf_slot[i]] = v;
    if (n == 1) ids[1] = ids[2] = v;
}

}  // namespace

int sgpu_curve_build(sgpu_scene scene, const std::vector<float>& cp, const std::vector<uint32_t>& geom,
                     const std::vector<uint32_t>& prim, const std::vector<uint32_t>& inst, hipStream_t stream)
{
    const uint32_t n = (uint32_t)geom.size();
    scene->n_curves = 0;
    if (n == 0) return SGPU_OK;
    if (n > (1u << 28)) return sgpu_fail(SGPU_E_RANGE, "scene has more than 2^28 curve segments");
    std::vector<CurveRecord> rec(n);
    for (uint32_t s = 0; s < n; ++s) {
        const float* c = cp.data() + 16 * (size_t)s;
        for (int j = 0; j < 4; ++j) rec[s].p[j] = make_float4(c[4 * j], c[4 * j + 1], c[4 * j + 2], c[4 * j + 3]);
        rec[s].geom = geom[s];
        rec[s].prim = prim[s];
        rec[s].inst = inst[s];
        rec[s].pad = 0;
    }
    sgpu_scratch S(scene->ctx, stream, build_scratch(n) + n * sizeof(BvhNode));
    DevBuf<CurveRecord> d_rec;
    DevBuf<uint32_t> d_bounds, d_order, d_place, d_leaf_slot;
    SGPU_HIP_TRY(d_rec.alloc(S, n));
    SGPU_HIP_TRY(d_bounds.alloc(S, 12));
    SGPU_HIP_TRY(d_order.alloc(S, n));
    SGPU_HIP_TRY(d_place.alloc(S, n));
    SGPU_HIP_TRY(hipMemcpyAsync(d_rec.p, rec.data(), n * sizeof(CurveRecord), hipMemcpyHostToDevice, stream));
    const uint32_t grid = (n + kBlock - 1) / kBlock;
    uint32_t hb[12], depth = 0;
    DevBuf<BvhNode> walked;
    SGPU_HIP_TRY(walked.alloc(S, n));
    // the tree that orders hits at equal distance, then the one that is walked, over the tight boxes
    for (int tight = 0; tight < 2; ++tight) {
        sgpu_scratch::Frame boxes(S);
        DevBuf<float4> d_blo, d_bhi, d_cent;
        SGPU_HIP_TRY(d_blo.alloc(S, n));
        SGPU_HIP_TRY(d_bhi.alloc(S, n));
        SGPU_HIP_TRY(d_cent.alloc(S, n));
        SGPU_HIP_TRY(hipMemsetAsync(d_bounds.p, 0xFF, 12 * sizeof(uint32_t), stream));
        if (tight)
            hipLaunchKernelGGL(k_curve_prep<true>, dim3(grid), dim3(kBlock), 0, stream, d_rec.p, n, d_blo.p, d_bhi.p,
                               d_cent.p, d_bounds.p);
        else
            hipLaunchKernelGGL(k_curve_prep<false>, dim3(grid), dim3(kBlock), 0, stream, d_rec.p, n, d_blo.p, d_bhi.p,
                               d_cent.p, d_bounds.p);
        SGPU_HIP_TRY(hipGetLastError());
        if (!tight) SGPU_HIP_TRY(hipMemcpyAsync(hb, d_bounds.p, sizeof(hb), hipMemcpyDeviceToHost, stream));
        const int rc = build_binary(S, n, d_blo.p, d_bhi.p, d_cent.p, d_bounds.p, stream,
                                    tight ? &walked.p : &scene->d_cnodes, d_order, &depth, 0);
        if (rc != SGPU_OK) return rc;
        if (tight) continue;
        if (depth + 1 > kCurveStack)
            return sgpu_fail(SGPU_E_RANGE, "curve tree deeper than the curve traversal's stack");
        hipLaunchKernelGGL(k_curve_places, dim3(grid), dim3(kBlock), 0, stream, d_order.p, n, d_place.p);
        SGPU_HIP_TRY(hipGetLastError());
    }
    WideTree tree;
    const int rc = build_wide(S, walked.p, n, stream, d_order.p, d_rec.p, sizeof(CurveRecord), nullptr, tree, d_leaf_slot);
    scene->d_cwide = tree.wide;
    scene->n_cslots = tree.n_slots;
    if (rc != SGPU_OK) return rc;
    SGPU_HIP_TRY(sgpu_device_malloc((void**)&scene->d_cids, (size_t)tree.n_slots * sizeof(uint4)));
    hipLaunchKernelGGL(k_curve_ids, dim3(grid), dim3(kBlock), 0, stream, d_rec.p, d_order.p, d_leaf_slot.p, d_place.p, n,
                       scene->d_cids);
    SGPU_HIP_TRY(hipGetLastError());
    SGPU_HIP_TRY(hipStreamSynchronize(stream));
    scene->n_curves = n;
    scene->wide_stack = std::max(scene->wide_stack, wide_stack_words(tree.depth));
    scene->stack_cap = std::max(scene->stack_cap, scene->wide_stack);
    // the scene's box takes in the curves
    for (int k = 0; k < 3; ++k) {
        const float lo = host_ord2f(hb[k]), hi = host_ord2f(~hb[3 + k]);
        if (scene->box[k] > scene->box[3 + k]) {
            scene->box[k] = lo;
            scene->box[3 + k] = hi;
        } else {
            scene->box[k] = std::min(scene->box[k], lo);
            scene->box[3 + k] = std::max(scene->box[3 + k], hi);
        }
    }
    return SGPU_OK;
}

int sgpu_bvh_build(sgpu_scene scene, hipStream_t stream)
{
    const uint32_t n = (uint32_t)scene->tri_geom.size();
    scene->n_tris = n;
    scene->n_nodes = 0;
    scene->max_depth = 0;
    if (n == 0) return SGPU_OK;
    if (n > (1u << 30)) return sgpu_fail(SGPU_E_RANGE, "scene has more than 2^30 triangles");

    sgpu_scratch S(scene->ctx, stream, build_scratch(n));
    DevBuf<uint32_t> d_bounds, d_order;
    DevBuf<TriRecord> d_rec;
    SGPU_HIP_TRY(d_bounds.alloc(S, 12));
    SGPU_HIP_TRY(d_order.alloc(S, n));
    SGPU_HIP_TRY(d_rec.alloc(S, n));
    BvhNode* nodes = nullptr;
    uint32_t depth = 0, hb[12];
    {
        sgpu_scratch::Frame input(S);
        DevBuf<float> d_pos;
        DevBuf<uint32_t> d_geom, d_first;
        DevBuf<float4> d_blo, d_bhi, d_cent;
        SGPU_HIP_TRY(d_pos.alloc(S, (size_t)n * 9));
        SGPU_HIP_TRY(d_geom.alloc(S, n));
        SGPU_HIP_TRY(d_first.alloc(S, scene->geom_first.size()));
        SGPU_HIP_TRY(d_blo.alloc(S, n));
        SGPU_HIP_TRY(d_bhi.alloc(S, n));
        SGPU_HIP_TRY(d_cent.alloc(S, n));
        SGPU_HIP_TRY(hipMemcpyAsync(d_pos.p, scene->tri_pos.data(), (size_t)n * 9 * sizeof(float), hipMemcpyHostToDevice,
                                    stream));
        SGPU_HIP_TRY(hipMemcpyAsync(d_geom.p, scene->tri_geom.data(), (size_t)n * sizeof(uint32_t), hipMemcpyHostToDevice,
                                    stream));
        // device copy of the geometries' first indices with bit 31 set for quad geometries
        std::vector<uint32_t> first_flagged(scene->geom_first.size());
        for (size_t g = 0; g < first_flagged.size(); ++g)
            first_flagged[g] = scene->geom_first[g] | (scene->geom_quad[g] == 1 ? 0x80000000u : 0u);
        SGPU_HIP_TRY(hipMemcpy(d_first.p, first_flagged.data(), first_flagged.size() * sizeof(uint32_t),
                               hipMemcpyHostToDevice));
        SGPU_HIP_TRY(hipMemsetAsync(d_bounds.p, 0xFF, 12 * sizeof(uint32_t), stream));
        const uint32_t grid = (n + kBlock - 1) / kBlock;
        hipLaunchKernelGGL(k_prep, dim3(grid), dim3(kBlock), 0, stream, d_pos.p, n, d_geom.p, d_first.p, d_rec.p, d_blo.p,
                           d_bhi.p, d_cent.p, d_bounds.p);
        SGPU_HIP_TRY(hipGetLastError());
        SGPU_HIP_TRY(hipMemcpyAsync(hb, d_bounds.p, sizeof(hb), hipMemcpyDeviceToHost, stream));
        const int rc = build_binary(S, n, d_blo.p, d_bhi.p, d_cent.p, d_bounds.p, stream, &nodes, d_order, &depth,
                                    scene->ctx->bvh_builder);
        if (rc != SGPU_OK) return rc;
    }
    for (int k = 0; k < 3; ++k) {
        scene->box[k] = host_ord2f(hb[k]);
        scene->box[3 + k] = host_ord2f(~hb[3 + k]);
    }
    scene->d_nodes = nodes;
    scene->n_nodes = n > 1 ? n - 1 : 1;
    scene->max_depth = depth;
    const int rc = build_scene_wide(scene, S, nodes, n, stream, d_order.p, d_rec.p, nullptr);
    scene->wide_stack = wide_stack_words(scene->wide_depth);
    // the binary tree's stack: a word per level
    scene->stack_cap = std::max(scene->max_depth + 1, scene->wide_stack);
    return rc;
}

namespace {

// r = a * b for row-major 3x4 affine transforms (the implicit last row 0 0 0 1)
void affine_mul(const double* a, const double* b, double* r)
{
    for (int i = 0; i < 3; ++i) {
        for (int j = 0; j < 4; ++j) {
            double v = a[4 * i + 0] * b[0 + j] + a[4 * i + 1] * b[4 + j] + a[4 * i + 2] * b[8 + j];
            if (j == 3) v += a[4 * i + 3];
            r[4 * i + j] = v;
        }
    }
}

// inverse of a row-major 3x4 affine transform; false when singular
bool affine_inverse(const double* m, double* r)
{
    const double a = m[0], b = m[1], c = m[2], d = m[4], e = m[5], f = m[6], g = m[8], h = m[9], k = m[10];
    const double A = e * k - f * h, B = -(d * k - f * g), C = d * h - e * g;
    const double det = a * A + b * B + c * C;
    if (!(std::fabs(det) > 0.0) || !std::isfinite(det)) return false;
    const double id = 1.0 / det;
    const double inv[9] = {A * id, -(b * k - c * h) * id, (b * f - c * e) * id,
                           B * id, (a * k - c * g) * id,  -(a * f - c * d) * id,
                           C * id, -(a * h - b * g) * id, (a * e - b * d) * id};
    for (int i = 0; i < 3; ++i) {
        r[4 * i + 0] = inv[3 * i + 0];
        r[4 * i + 1] = inv[3 * i + 1];
        r[4 * i + 2] = inv[3 * i + 2];
        r[4 * i + 3] = -(inv[3 * i + 0] * m[3] + inv[3 * i + 1] * m[7] + inv[3 * i + 2] * m[11]);
    }
    return true;
}

}  // namespace

namespace {

// The curves of the composed instances (placed scene, local-to-world row-major 3 x 4 in double) in
// world space, each segment tagged with its composed instance, and the instanced scene's curve
// tree over them. A placement that scales unevenly or shears would turn the swept spheres into
// ellipsoids, which the world-space curve test does not represent: such a placement is refused.
int bake_instance_curves(sgpu_scene scene, const std::vector<std::pair<sgpu_scene, const double*>>& comp,
                         hipStream_t stream)
{
    std::vector<float> cp;
    std::vector<uint32_t> geom, prim, inst;
    for (uint32_t k = 0; k < comp.size(); ++k) {
        const sgpu_scene b = comp[k].first;
        const double* m = comp[k].second;
        if (b->curve_geom.empty()) continue;
        double n2[3], s2 = 0.0;
        for (int c = 0; c < 3; ++c) {
            n2[c] = m[c] * m[c] + m[4 + c] * m[4 + c] + m[8 + c] * m[8 + c];
            s2 += n2[c] / 3.0;
        }
        bool similar = s2 > 0.0;
        for (int c = 0; c < 3 && similar; ++c) {
            similar &= std::fabs(n2[c] - s2) <= 1e-5 * s2;
            for (int e = c + 1; e < 3; ++e)
                similar &= std::fabs(m[c] * m[e] + m[4 + c] * m[4 + e] + m[8 + c] * m[8 + e]) <= 1e-5 * s2;
        }
        if (!similar)
            return sgpu_fail(SGPU_E_INVALID, "an instance placing curves is not a similarity (rotation, uniform scale, "
                                             "translation)");
        const double sc = std::sqrt(s2);
        const size_t nseg = b->curve_geom.size(), base = cp.size();
        cp.resize(base + 16 * nseg);
        for (size_t i = 0; i < nseg; ++i) {
            const float* src = b->curve_cp.data() + 16 * i;
            float* dst = cp.data() + base + 16 * i;
            for (int j = 0; j < 4; ++j) {
                const double p[3] = {src[4 * j], src[4 * j + 1], src[4 * j + 2]};
                for (int r = 0; r < 3; ++r)
                    dst[4 * j + r] = (float)(m[4 * r] * p[0] + m[4 * r + 1] * p[1] + m[4 * r + 2] * p[2] + m[4 * r + 3]);
                dst[4 * j + 3] = (float)(src[4 * j + 3] * sc);
            }
            geom.push_back(b->curve_geom[i]);
            prim.push_back(b->curve_prim[i]);
            inst.push_back(k);
        }
    }
    return sgpu_curve_build(scene, cp, geom, prim, inst, stream);
}

}  // namespace

int sgpu_bvh_build_instances(sgpu_scene scene, hipStream_t stream)
{
    // compose the levels: (instance i of a scene of geometries) or (instance i of an instanced
    // scene, its instance j), in that order
    struct Flat {
        sgpu_scene blas;
        double l2w[12];
        uint32_t id0, id1;
    };
    std::vector<Flat> flat;
    uint32_t levels = 1;
    for (size_t i = 0; i < scene->instances.size(); ++i) {
        const auto& in = scene->instances[i];
        if (in.child->instances.empty()) {
            Flat f{in.child, {}, (uint32_t)i, SGPU_INVALID_ID};
            std::memcpy(f.l2w, in.l2w, sizeof(f.l2w));
            flat.push_back(f);
        } else {
            levels = 2;
            for (size_t j = 0; j < in.child->instances.size(); ++j) {
                const auto& in2 = in.child->instances[j];
                Flat f{in2.child, {}, (uint32_t)i, (uint32_t)j};
                affine_mul(in.l2w, in2.l2w, f.l2w);
                flat.push_back(f);
            }
        }
    }
    // scenes without triangles are not in the top tree; those with curves are composed after the
    // tree's instances (the curve pass reaches them through their curves), the others place nothing
    std::vector<Flat> extra;
    for (const Flat& f : flat)
        if (f.blas->n_tris == 0 && !f.blas->curve_geom.empty()) extra.push_back(f);
    flat.erase(std::remove_if(flat.begin(), flat.end(), [](const Flat& f) { return f.blas->n_tris == 0; }), flat.end());
    if (flat.size() + extra.size() > (1u << 30)) return sgpu_fail(SGPU_E_RANGE, "scene has more than 2^30 composed instances");
    const uint32_t n = (uint32_t)flat.size();
    scene->n_tris = 0;
    scene->n_nodes = 0;
    scene->max_depth = 0;
    scene->inst_levels = levels;
    scene->comp_blas.clear();
    scene->comp_l2w.clear();
    // composed instances past the tree's: records (world-to-local), ids, placed scene and transform
    std::vector<InstRecord> xrec(extra.size());
    std::vector<uint32_t> xids(2 * extra.size());
    for (size_t e = 0; e < extra.size(); ++e) {
        double w2l[12];
        if (!affine_inverse(extra[e].l2w, w2l)) return sgpu_fail(SGPU_E_INVALID, "instance transform is singular");
        for (int r = 0; r < 3; ++r)
            xrec[e].w2l[r] = make_float4((float)w2l[4 * r], (float)w2l[4 * r + 1], (float)w2l[4 * r + 2], (float)w2l[4 * r + 3]);
        xrec[e].wide = nullptr;
        xrec[e].pad = 0;
        xids[2 * e] = extra[e].id0;
        xids[2 * e + 1] = extra[e].id1;
    }
    auto composed = [&]() {
        std::vector<std::pair<sgpu_scene, const double*>> c;
        for (const Flat& f : flat) c.emplace_back(f.blas, f.l2w);
        for (const Flat& f : extra) c.emplace_back(f.blas, f.l2w);
        return c;
    };
    auto push_extra_shading = [&]() {
        for (const Flat& f : extra) {
            scene->comp_blas.push_back(f.blas);
            for (int r = 0; r < 3; ++r)
                for (int c = 0; c < 3; ++c) scene->comp_l2w.push_back((float)f.l2w[4 * r + c]);
        }
    };
    if (n == 0) {
        if (extra.empty()) return SGPU_OK;
        // only curves: no top tree; the composed instances' records for the curve pass and shading
        push_extra_shading();
        hipError_t e = sgpu_device_malloc((void**)&scene->d_inst, xrec.size() * sizeof(InstRecord));
        if (e == hipSuccess) e = sgpu_device_malloc((void**)&scene->d_inst_ids, xids.size() * sizeof(uint32_t));
        if (e == hipSuccess) e = hipMemcpy(scene->d_inst, xrec.data(), xrec.size() * sizeof(InstRecord), hipMemcpyHostToDevice);
        if (e == hipSuccess)
            e = hipMemcpy(scene->d_inst_ids, xids.data(), xids.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
        if (e != hipSuccess) return sgpu_fail(SGPU_E_HIP, std::string("instance records: ") + hipGetErrorString(e));
        scene->n_inst = 0;
        scene->wide_stack = 0;
        scene->stack_cap = 1;
        return bake_instance_curves(scene, composed(), stream);
    }

    // The top tree's box of an instance: the boxes of the placed scene's root children (decoded
    // from its 8-wide root as the traversal decodes them) through the transform, their 8 corners in
    // double, united and rounded outward: much tighter than the transformed box of the whole scene
    // when the transform rotates. The scene's own box (the IBL's emission sphere) takes the 8
    // corners of each placed scene's box.
    std::vector<std::pair<sgpu_scene, std::vector<float>>> root_boxes;
    auto child_boxes = [&](sgpu_scene b, std::vector<float>& out) -> int {
        for (const auto& rb : root_boxes)
            if (rb.first == b) {
                out = rb.second;
                return SGPU_OK;
            }
        WideNode w;
        SGPU_HIP_TRY(hipMemcpy(&w, b->d_wide, sizeof(WideNode), hipMemcpyDeviceToHost));
        const uint32_t nch = w.meta >> 28;
        float o[3], sc[3];
        for (int a = 0; a < 3; ++a) {
            const uint32_t bits = w.origin_base[a] & kOriginMask;
            std::memcpy(&o[a], &bits, sizeof(float));
        }
        for (int a = 0; a < 3; ++a) sc[a] = std::ldexp(1.0f, (int)(int8_t)((w.meta >> (8 * a)) & 0xFFu));
        out.clear();
        for (uint32_t c = 0; c < nch && c < 8; ++c)
            for (int side = 0; side < 2; ++side)
                for (int a = 0; a < 3; ++a) {
                    const uint32_t word = side ? w.qhi[a][c >> 2] : w.qlo[a][c >> 2];
                    out.push_back(std::fma((float)((word >> (8 * (c & 3))) & 0xFFu), sc[a], o[a]));
                }
        root_boxes.emplace_back(b, out);
        return SGPU_OK;
    };
    std::vector<float4> blo(n), bhi(n), cent(n);
    std::vector<InstRecord> rec(n);
    std::vector<uint32_t> ids(2 * (size_t)n);
    float slo[3] = {INFINITY, INFINITY, INFINITY}, shi[3] = {-INFINITY, -INFINITY, -INFINITY};
    float clo[3] = {INFINITY, INFINITY, INFINITY}, chi[3] = {-INFINITY, -INFINITY, -INFINITY};
    uint32_t blas_cap = 0;
    for (uint32_t k = 0; k < n; ++k) {
        const Flat& f = flat[k];
        double w2l[12];
        if (!affine_inverse(f.l2w, w2l)) return sgpu_fail(SGPU_E_INVALID, "instance transform is singular");
        // the 8 corners of a local box through the transform, in double
        auto world_box = [&](const float* b6, double* lo, double* hi) {
            for (int c = 0; c < 8; ++c) {
                const double p[3] = {b6[(c & 1) ? 3 : 0], b6[(c & 2) ? 4 : 1], b6[(c & 4) ? 5 : 2]};
                for (int r = 0; r < 3; ++r) {
                    const double w =
                        f.l2w[4 * r] * p[0] + f.l2w[4 * r + 1] * p[1] + f.l2w[4 * r + 2] * p[2] + f.l2w[4 * r + 3];
                    lo[r] = std::min(lo[r], w);
                    hi[r] = std::max(hi[r], w);
                }
            }
        };
        double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        world_box(f.blas->box, lo, hi);
        std::vector<float> cb;
        int rcb = child_boxes(f.blas, cb);
        if (rcb != SGPU_OK) return rcb;
        double tlo[3] = {INFINITY, INFINITY, INFINITY}, thi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (size_t c = 0; c + 6 <= cb.size(); c += 6) world_box(cb.data() + c, tlo, thi);
        if (cb.empty())
            for (int r = 0; r < 3; ++r) {
                tlo[r] = lo[r];
                thi[r] = hi[r];
            }
        float l[3], h[3];
        for (int r = 0; r < 3; ++r) {
            const float sl = std::nextafter((float)lo[r], -INFINITY), sh = std::nextafter((float)hi[r], INFINITY);
            l[r] = std::nextafter((float)std::max(tlo[r], lo[r]), -INFINITY);
            h[r] = std::nextafter((float)std::min(thi[r], hi[r]), INFINITY);
            if (!std::isfinite(sl) || !std::isfinite(sh))
                return sgpu_fail(SGPU_E_RANGE, "instance box is not finite in single precision");
            slo[r] = std::min(slo[r], sl);
            shi[r] = std::max(shi[r], sh);
            const float cc = 0.5f * (l[r] + h[r]);
            clo[r] = std::min(clo[r], cc);
            chi[r] = std::max(chi[r], cc);
        }
        blo[k] = make_float4(l[0], l[1], l[2], 0.0f);
        bhi[k] = make_float4(h[0], h[1], h[2], 0.0f);
        cent[k] = make_float4(0.5f * (l[0] + h[0]), 0.5f * (l[1] + h[1]), 0.5f * (l[2] + h[2]), 0.0f);
        for (int r = 0; r < 3; ++r)
            rec[k].w2l[r] = make_float4((float)w2l[4 * r], (float)w2l[4 * r + 1], (float)w2l[4 * r + 2], (float)w2l[4 * r + 3]);
        rec[k].wide = f.blas->d_wide;
        rec[k].pad = 0;
        scene->comp_blas.push_back(f.blas);
        for (int r = 0; r < 3; ++r)
            for (int c = 0; c < 3; ++c) scene->comp_l2w.push_back((float)f.l2w[4 * r + c]);
        ids[2 * k] = f.id0;
        ids[2 * k + 1] = f.id1;
        blas_cap = std::max(blas_cap, f.blas->wide_stack);
    }
    push_extra_shading();
    rec.insert(rec.end(), xrec.begin(), xrec.end());
    ids.insert(ids.end(), xids.begin(), xids.end());
    uint32_t hb[12];
    for (int r = 0; r < 3; ++r) {
        hb[r] = host_f2ord(slo[r]);
        hb[3 + r] = ~host_f2ord(shi[r]);
        hb[6 + r] = host_f2ord(clo[r]);
        hb[9 + r] = ~host_f2ord(chi[r]);
        scene->box[r] = slo[r];
        scene->box[3 + r] = shi[r];
    }
    sgpu_scratch S(scene->ctx, stream, build_scratch(n));
    DevBuf<uint32_t> d_order;
    SGPU_HIP_TRY(d_order.alloc(S, n));
    BvhNode* nodes = nullptr;
    uint32_t depth = 0;
    int rc = SGPU_OK;
    {
        sgpu_scratch::Frame boxes(S);
        DevBuf<float4> d_blo, d_bhi, d_cent;
        DevBuf<uint32_t> d_bounds;
        SGPU_HIP_TRY(d_blo.alloc(S, n));
        SGPU_HIP_TRY(d_bhi.alloc(S, n));
        SGPU_HIP_TRY(d_cent.alloc(S, n));
        SGPU_HIP_TRY(d_bounds.alloc(S, 12));
        SGPU_HIP_TRY(hipMemcpyAsync(d_blo.p, blo.data(), n * sizeof(float4), hipMemcpyHostToDevice, stream));
        SGPU_HIP_TRY(hipMemcpyAsync(d_bhi.p, bhi.data(), n * sizeof(float4), hipMemcpyHostToDevice, stream));
        SGPU_HIP_TRY(hipMemcpyAsync(d_cent.p, cent.data(), n * sizeof(float4), hipMemcpyHostToDevice, stream));
        SGPU_HIP_TRY(hipMemcpyAsync(d_bounds.p, hb, sizeof(hb), hipMemcpyHostToDevice, stream));
        rc = build_binary(S, n, d_blo.p, d_bhi.p, d_cent.p, d_bounds.p, stream, &nodes, d_order, &depth,
                          scene->ctx->bvh_builder);
        if (rc != SGPU_OK) return rc;
    }
    InstRecord* d_inst = nullptr;
    uint32_t* d_ids = nullptr;
    hipError_t e = sgpu_device_malloc((void**)&d_inst, rec.size() * sizeof(InstRecord));
    if (e == hipSuccess) e = sgpu_device_malloc((void**)&d_ids, ids.size() * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMemcpy(d_inst, rec.data(), rec.size() * sizeof(InstRecord), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d_ids, ids.data(), ids.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(nodes);
        if (d_inst) (void)hipFree(d_inst);
        if (d_ids) (void)hipFree(d_ids);
        return sgpu_fail(SGPU_E_HIP, std::string("instance records: ") + hipGetErrorString(e));
    }
    scene->d_nodes = nodes;
    scene->d_inst = d_inst;
    scene->d_inst_ids = d_ids;
    scene->n_inst = n;
    scene->n_nodes = n > 1 ? n - 1 : 1;
    scene->max_depth = depth;
    // instance nodes name composed instances by their composition index (instance i, then its instance
    // j), so the closest-hit tie rule follows (inst_id0, inst_id1)
    rc = build_scene_wide(scene, S, nodes, n, stream, d_order.p, nullptr, d_inst);
    // the top tree's groups above an instance's node (its last level), the exit entry and the deepest
    // placed tree's stack; the binary top tree is not walked
    scene->wide_stack = 2 * scene->wide_depth + blas_cap;
    scene->stack_cap = scene->wide_stack;
    if (rc != SGPU_OK) return rc;
    return bake_instance_curves(scene, composed(), stream);
}
