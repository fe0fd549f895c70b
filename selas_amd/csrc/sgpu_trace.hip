// Closest-hit and any-hit BVH traversal: the replacement of Embree's rtcIntersect1/8 and
// rtcOccluded1/8 (called from RayPick / OcclusionRay, Source/Applications/Selas/Source/PathTracer.cpp:71-139,
// and the packet tracers, Source/Applications/Selas/Source/DeferredPathTracer.cpp:151-280).
//
// One ray per lane, 64-lane waves, rays read from SoA arrays with coalesced loads. The traversal
// stack is per lane: its top SGPU_STACK_LDS entries live in LDS laid out [slot][lane] (one bank
// per lane), deeper entries spill to a global buffer laid out [depth][thread] (coalesced).
//
// Triangle test (the arithmetic restated in oracle/sgpu_oracle.c, orc_tri_test):
//   pvec = cross_fma(d, e2); det = dot_fma(e1, pvec); tvec = o - v0;
//   U = dot_fma(tvec, pvec); qvec = cross_fma(tvec, e1); V = dot_fma(d, qvec); T = dot_fma(e2, qvec)
//   det == 0 -> miss; if det < 0 negate U, V, T; a = |det|
//   barycentric accept: U >= 0 && V >= 0 && U + V <= a
//   t = T / a, u = U / a, v = V / a (IEEE division); accept tnear < t <= tfar.
// Closest hit: smallest t, ties to the smaller global triangle index (= smaller (geomID, primID)).
#include "sgpu_wide.h"

#include <algorithm>

namespace {

using sgpu::safe_rcp;

// The test but for the barycentrics' divisions: u = U / a, v = V / a of the hit kept in the end.
__device__ __forceinline__ bool tri_hit(const TriRecord& r, const f3& o, const f3& d, float tnear, float& t, float& U,
                                        float& V, float& a)
{
    f3 v0 = mk3(r.a.x, r.a.y, r.a.z);
    f3 e1 = mk3(r.b.x, r.b.y, r.b.z);
    f3 e2 = mk3(r.c.x, r.c.y, r.c.z);
    f3 pvec = cross_fma(d, e2);
    float det = dot_fma(e1, pvec);
    f3 tvec = o - v0;
    U = dot_fma(tvec, pvec);
    f3 qvec = cross_fma(tvec, e1);
    V = dot_fma(d, qvec);
    float T = dot_fma(e2, qvec);
    if (det == 0.0f) return false;
    if (det < 0.0f) {
        U = -U;
        V = -V;
        T = -T;
    }
    a = fabsf(det);
    if (!(U >= 0.0f && V >= 0.0f && U + V <= a)) return false;
    t = T / a;
    return t > tnear;
}

__device__ __forceinline__ bool tri_test(const TriRecord& r, const f3& o, const f3& d, float tnear, float& t,
                                         float& u, float& v)
{
    float U, V, a;
    if (!tri_hit(r, o, d, tnear, t, U, V, a)) return false;
    u = U / a;
    v = V / a;
    return true;
}

// The query's result: occlusion flag, or Embree's hit fields (quad hits reported as the quad and its
// own (u, v): triangle 2q + h of quad q, second triangle (1 - u, 1 - v)).
template <bool ANY>
__device__ __forceinline__ void write_result(uint32_t i, bool hit_any, uint32_t best_tri, float best_t, float best_u,
                                             float best_v, const TriRecord* __restrict rt, sgpu_hits_soa& hits,
                                             uint32_t* __restrict occluded, uint32_t id0 = SGPU_INVALID_ID,
                                             uint32_t id1 = SGPU_INVALID_ID)
{
    if (ANY) {
        occluded[i] = hit_any ? 1u : 0u;
        return;
    }
    bool found = best_tri != 0xFFFFFFFFu;
    uint32_t prim = SGPU_INVALID_ID, geom = SGPU_INVALID_ID;
    f3 ng = mk3(0.0f, 0.0f, 0.0f);
    if (found) {
        const TriRecord r = rt[best_tri];
        geom = __float_as_uint(r.b.w);
        prim = __float_as_uint(r.c.w);
        if (hits.ng_x) ng = cross3(mk3(r.b.x, r.b.y, r.b.z), mk3(r.c.x, r.c.y, r.c.z));
        if (prim & 0x80000000u) {
            if (prim & 1u) {
                best_u = 1.0f - best_u;
                best_v = 1.0f - best_v;
            }
            prim = (prim & 0x7FFFFFFFu) >> 1;
        }
    }
    if (hits.t) hits.t[i] = best_t;
    if (hits.u) hits.u[i] = found ? best_u : 0.0f;
    if (hits.v) hits.v[i] = found ? best_v : 0.0f;
    if (hits.prim_id) hits.prim_id[i] = prim;
    if (hits.geom_id) hits.geom_id[i] = geom;
    if (hits.ng_x) {
        hits.ng_x[i] = ng.x;
        hits.ng_y[i] = ng.y;
        hits.ng_z[i] = ng.z;
    }
    if (hits.inst_id0) hits.inst_id0[i] = found ? id0 : SGPU_INVALID_ID;
    if (hits.inst_id1) hits.inst_id1[i] = found ? id1 : SGPU_INVALID_ID;
}

template <bool ANY, bool STATS, bool MULTI>
__global__ __launch_bounds__(SGPU_TRACE_BLOCK) void k_trace(const BvhNode* __restrict nodes,
                                                            const TriRecord* __restrict tris, uint32_t n_tris,
                                                            const TraceScene* __restrict table,
                                                            const uint32_t* __restrict ray_scene,
                                                            sgpu_rays_soa rays, sgpu_hits_soa hits,
                                                            uint32_t* __restrict occluded, uint32_t n,
                                                            const uint32_t* __restrict n_ptr,
                                                            uint32_t* __restrict spill, uint32_t stack_cap,
                                                            unsigned long long* __restrict stats,
                                                            uint32_t* __restrict overflow)
{
    __shared__ uint32_t lds_stack[SGPU_STACK_LDS][SGPU_TRACE_BLOCK];
    const uint32_t lane = threadIdx.x;
    const uint32_t gtid = blockIdx.x * SGPU_TRACE_BLOCK + threadIdx.x;
    const uint32_t stride = gridDim.x * SGPU_TRACE_BLOCK;
    unsigned long long cnt_nodes = 0, cnt_tris = 0;
    if (n_ptr) n = *n_ptr;  // the count written on the device by the kernel that queued the rays

    for (uint32_t i = gtid; i < n; i += stride) {
        f3 o = mk3(rays.org_x[i], rays.org_y[i], rays.org_z[i]);
        f3 d = mk3(rays.dir_x[i], rays.dir_y[i], rays.dir_z[i]);
        float tnear = rays.tnear[i];
        float tfar = rays.tfar[i];
        f3 inv = mk3(safe_rcp(d.x), safe_rcp(d.y), safe_rcp(d.z));
        f3 oinv = mk3(o.x * inv.x, o.y * inv.y, o.z * inv.z);
        // the ray's scene: the launch's one, or its own entry of the table in a multi-scene launch
        const BvhNode* __restrict rn = nodes;
        const TriRecord* __restrict rt = tris;
        uint32_t rnt = n_tris;
        if (MULTI) {
            const TraceScene ts = table[ray_scene[i]];
            rn = ts.nodes;
            rt = reinterpret_cast<const TriRecord*>(ts.wide);
            rnt = ts.n_tris;
        }

        float best_t = tfar;
        uint32_t best_key = 0xFFFFFFFFu;
        uint32_t best_tri = 0xFFFFFFFFu;
        float best_u = 0.0f, best_v = 0.0f;
        bool hit_any = false;

        uint32_t sp = 0;
        int node = rnt > 0 ? 0 : 0x7FFFFFFF;
        bool done = rnt == 0;
        while (!done) {
            if (node >= 0) {
                const BvhNode nd = rn[node];
                if (STATS) ++cnt_nodes;
                float l0x = fmaf(nd.x.x, inv.x, -oinv.x), h0x = fmaf(nd.x.y, inv.x, -oinv.x);
                float l1x = fmaf(nd.x.z, inv.x, -oinv.x), h1x = fmaf(nd.x.w, inv.x, -oinv.x);
                float l0y = fmaf(nd.y.x, inv.y, -oinv.y), h0y = fmaf(nd.y.y, inv.y, -oinv.y);
                float l1y = fmaf(nd.y.z, inv.y, -oinv.y), h1y = fmaf(nd.y.w, inv.y, -oinv.y);
                float l0z = fmaf(nd.z.x, inv.z, -oinv.z), h0z = fmaf(nd.z.y, inv.z, -oinv.z);
                float l1z = fmaf(nd.z.z, inv.z, -oinv.z), h1z = fmaf(nd.z.w, inv.z, -oinv.z);
                float tmin0 = fmaxf(fmaxf(fminf(l0x, h0x), fminf(l0y, h0y)), fmaxf(fminf(l0z, h0z), tnear));
                float tmax0 = fminf(fminf(fmaxf(l0x, h0x), fmaxf(l0y, h0y)), fminf(fmaxf(l0z, h0z), best_t));
                float tmin1 = fmaxf(fmaxf(fminf(l1x, h1x), fminf(l1y, h1y)), fmaxf(fminf(l1z, h1z), tnear));
                float tmax1 = fminf(fminf(fmaxf(l1x, h1x), fmaxf(l1y, h1y)), fminf(fmaxf(l1z, h1z), best_t));
                bool hit0 = tmin0 <= tmax0;
                bool hit1 = tmin1 <= tmax1;
                if (hit0 && hit1) {
                    int near_c = tmin0 <= tmin1 ? nd.child.x : nd.child.y;
                    int far_c = tmin0 <= tmin1 ? nd.child.y : nd.child.x;
                    if (sp >= stack_cap) {
                        atomicOr(overflow, 1u);
                        done = true;
                        break;
                    }
                    if (sp < SGPU_STACK_LDS) {
                        lds_stack[sp][lane] = (uint32_t)far_c;
                    } else {
                        // ring over the LDS slots: evict position sp-K to global before reuse
                        uint32_t slot = sp % SGPU_STACK_LDS;
                        spill[(size_t)(sp - SGPU_STACK_LDS) * stride + gtid] = lds_stack[slot][lane];
                        lds_stack[slot][lane] = (uint32_t)far_c;
                    }
                    ++sp;
                    node = near_c;
                    continue;
                } else if (hit0) {
                    node = nd.child.x;
                    continue;
                } else if (hit1) {
                    node = nd.child.y;
                    continue;
                }
            } else {
                const uint32_t j = (uint32_t)(~node);
                const TriRecord r = rt[j];
                if (STATS) ++cnt_tris;
                float t, u, v;
                if (tri_test(r, o, d, tnear, t, u, v)) {
                    if (ANY) {
                        if (t <= tfar) {
                            hit_any = true;
                            break;
                        }
                    } else {
                        uint32_t key = __float_as_uint(r.a.w);
                        if (t < best_t || (t == best_t && key < best_key)) {
                            best_t = t;
                            best_key = key;
                            best_tri = j;
                            best_u = u;
                            best_v = v;
                        }
                    }
                }
            }
            // pop
            if (sp == 0) break;
            --sp;
            uint32_t slot = sp % SGPU_STACK_LDS;
            node = (int)lds_stack[slot][lane];
            if (sp >= SGPU_STACK_LDS) lds_stack[slot][lane] = spill[(size_t)(sp - SGPU_STACK_LDS) * stride + gtid];
        }

        write_result<ANY>(i, hit_any, best_tri, best_t, best_u, best_v, rt, hits, occluded);
    }
    if (STATS) {
        atomicAdd(&stats[0], cnt_nodes);
        atomicAdd(&stats[1], cnt_tris);
    }
}

// A ray into an instance's space: x' = w.x x + w.y y + w.z z (+ w.w for points), summed by fused
// multiply-adds from the last term (the arithmetic the oracle restates).
__device__ __forceinline__ f3 inst_point(const float4* w, f3 p)
{
    return mk3(fmaf(w[0].x, p.x, fmaf(w[0].y, p.y, fmaf(w[0].z, p.z, w[0].w))),
               fmaf(w[1].x, p.x, fmaf(w[1].y, p.y, fmaf(w[1].z, p.z, w[1].w))),
               fmaf(w[2].x, p.x, fmaf(w[2].y, p.y, fmaf(w[2].z, p.z, w[2].w))));
}
__device__ __forceinline__ f3 inst_vector(const float4* w, f3 v)
{
    return mk3(fmaf(w[0].x, v.x, fmaf(w[0].y, v.y, w[0].z * v.z)), fmaf(w[1].x, v.x, fmaf(w[1].y, v.y, w[1].z * v.z)),
               fmaf(w[2].x, v.x, fmaf(w[2].y, v.y, w[2].z * v.z)));
}


// Wide nodes of a single-scene launch that may be kept in LDS (sgpu_tuning.trace_lds_nodes): the root
// and the next breadth-first nodes (the root's children when it has 8 internal ones), visited by
// nearly every ray. Measured on MI355X they hit in L1/L2 anyway, and the LDS branch costs 1-3 %.
constexpr uint32_t kTopNodes = 9;
constexpr uint32_t kTraceChunk = 64;  // rays a wave takes from the launch's counter at a time
// Finished lanes for which a wave stops to write results and take rays (16M closest-hit rays in 2M
// triangles: 12.1 ms at 1, 10.9 at 4, 10.6 at 8, 10.3 at 16 and 24; 4M any-hit rays 1.83, 1.72, 1.69,
// 1.71, 1.78 ms).
template <bool ANY>
constexpr int kRefill = ANY ? 8 : 16;
constexpr int kNext = -2;             // a lane that takes its next node once its triangles are tested

// Launches of few rays: eight lanes a ray, lane c testing child c of the node and, where that is a leaf,
// its triangle, so that a visit is one box test long and the node's triangles are tested at once. A wave
// of one ray per lane is a chain of some 40 trips of 400 instructions whatever it holds; up to kGroupRays
// rays the chip has waves to spare and that chain is what a launch takes (61 rays: 107 -> 36 us; a 64 x 64
// image of one vertex-merging iteration, 42 such launches: 2.57 -> 1.57 ms). What is left is a chain of
// node and triangle fetches. The ray's stack holds (slot, entry distance) pairs in LDS, pushed by the
// lanes that hit, far to near, and entries beyond the closest hit so far are dropped when popped. Hits
// are the same bits (the ties of k_trace8).
// The line: closest hits of random rays through 65 536 triangles take 271 us this way and 335 lane by lane
// at 131 072 rays, 401 and 376 at 200 000; any hits through a million 220 and 273 at 98 304, 284 and 277
// at 131 072; 1024 rays 80 and 253, 58 and 176.
template <bool ANY>
constexpr uint32_t kGroupRays = ANY ? 98304u : 131072u;
constexpr int kTailRays = 64 / 8;  // a ray of a wave's last to each group
constexpr uint32_t kGroupStack = 128;  // entries a ray's stack holds
// The entries a tree can need whose 8-wide stack takes `words` words (two a level but two): a visit takes
// one entry and leaves eight, on every level but the last, and an instanced ray has an exit entry.
constexpr uint32_t group_stack(uint32_t words) { return 7 * (words / 2) + 9; }
constexpr uint32_t kGroupExit = 0xFFFFFFFFu;  // the entry that returns to the top tree

template <int CTRL>
__device__ __forceinline__ int dpp(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}

// How many of the group's eight keys are smaller than this lane's (keys differ).
__device__ __forceinline__ uint32_t group_rank(int k)
{
    const int m = dpp<0x141>(k);  // lane ^ 7
    return (uint32_t)(dpp<0xB1>(k) < k) + (uint32_t)(dpp<0x4E>(k) < k) + (uint32_t)(dpp<0x1B>(k) < k) + (uint32_t)(m < k) +
           (uint32_t)(dpp<0xB1>(m) < k) + (uint32_t)(dpp<0x4E>(m) < k) + (uint32_t)(dpp<0x1B>(m) < k);
}

// A node as a lane of a group reads it: its header and the lane's child's box.
struct GroupNode
{
    uint4 w;
    uint32_t lx, ly, lz, hx, hy, hz;
    __device__ __forceinline__ GroupNode() {}
    __device__ __forceinline__ GroupNode(const WideNode* __restrict rw, int node, uint32_t gl)
    {
        const uint8_t* __restrict np = reinterpret_cast<const uint8_t*>(rw) + (size_t)(uint32_t)node * kSlotBytes;
        w = *reinterpret_cast<const uint4*>(np);
        lx = np[16 + gl], ly = np[24 + gl], lz = np[32 + gl];
        hx = np[40 + gl], hy = np[48 + gl], hz = np[56 + gl];
    }
    __device__ __forceinline__ uint32_t base() const
    {
        return (w.x & ~kOriginMask) | (w.y & ~kOriginMask) << 11 | w.z << 22;
    }
    // whether the ray enters the lane's child, and where (wide_boxes' arithmetic)
    __device__ __forceinline__ bool enters(uint32_t gl, f3 inv, f3 oinv, float tnear, float best, float& tmin) const
    {
        const float ax = __builtin_amdgcn_ldexpf(inv.x, (int)(w.w << 24) >> 24);
        const float ay = __builtin_amdgcn_ldexpf(inv.y, (int)(w.w << 16) >> 24);
        const float az = __builtin_amdgcn_ldexpf(inv.z, (int)(w.w << 8) >> 24);
        const float bx = fmaf(__uint_as_float(w.x & kOriginMask), inv.x, -oinv.x);
        const float by = fmaf(__uint_as_float(w.y & kOriginMask), inv.y, -oinv.y);
        const float bz = fmaf(__uint_as_float(w.z & kOriginMask), inv.z, -oinv.z);
        const bool sx = __float_as_int(inv.x) < 0, sy = __float_as_int(inv.y) < 0, sz = __float_as_int(inv.z) < 0;
        const float t0x = fmaf((float)(sx ? hx : lx), ax, bx), t1x = fmaf((float)(sx ? lx : hx), ax, bx);
        const float t0y = fmaf((float)(sy ? hy : ly), ay, by), t1y = fmaf((float)(sy ? ly : hy), ay, by);
        const float t0z = fmaf((float)(sz ? hz : lz), az, bz), t1z = fmaf((float)(sz ? lz : hz), az, bz);
        tmin = fmaxf(fmaxf(t0x, t0y), fmaxf(t0z, tnear));
        return gl < w.w >> 28 && tmin <= fminf(fminf(t1x, t1y), fminf(t1z, best));
    }
};

// The lane of the group with the smallest (t, key) among those that found a closer hit.
__device__ __forceinline__ uint32_t group_closest(bool closer, float t, uint32_t key)
{
    float ct = closer ? t : __int_as_float(0x7f800000);
    uint32_t ck = closer ? key : 0xFFFFFFFFu, from = threadIdx.x & 7u;
#pragma unroll
    for (uint32_t x = 1; x < 8; x <<= 1) {
        const float ot = __shfl_xor(ct, x, 8);
        const uint32_t ok = (uint32_t)__shfl_xor((int)ck, x, 8), of = (uint32_t)__shfl_xor((int)from, x, 8);
        if (ot < ct || (ot == ct && ok < ck)) {
            ct = ot;
            ck = ok;
            from = of;
        }
    }
    return from;
}

template <bool ANY, bool STATS, bool MULTI, bool INST>
__device__ void trace_groups(const TraceScene& scene, const uint32_t* __restrict inst_ids,
                             const TraceScene* __restrict table, const uint32_t* __restrict ray_scene,
                             const sgpu_rays_soa& rays, sgpu_hits_soa& hits, uint32_t* __restrict occluded, uint32_t n,
                             unsigned long long* __restrict stats, uint32_t* __restrict comp_out, uint2* lds)
{
    const uint32_t gl = threadIdx.x & 7u, shift = threadIdx.x & 56u;
    const uint32_t group = (blockIdx.x * SGPU_TRACE_BLOCK + threadIdx.x) >> 3, groups = gridDim.x * SGPU_TRACE_BLOCK >> 3;
    uint2* const stack = lds + kGroupStack * (threadIdx.x >> 3);
    unsigned long long cnt_nodes = 0, cnt_tris = 0;
    for (uint32_t i = group; i < n; i += groups) {
        f3 o, d, inv, oinv;
        auto load_ray = [&]() {
            o = mk3(rays.org_x[i], rays.org_y[i], rays.org_z[i]);
            d = mk3(rays.dir_x[i], rays.dir_y[i], rays.dir_z[i]);
        };
        auto set_slopes = [&]() {
            inv = mk3(safe_rcp(d.x), safe_rcp(d.y), safe_rcp(d.z));
            oinv = mk3(o.x * inv.x, o.y * inv.y, o.z * inv.z);
        };
        load_ray();
        set_slopes();
        const float tnear = rays.tnear[i];
        float best_t = rays.tfar[i];
        const TraceScene ts = MULTI ? table[ray_scene[i]] : scene;
        const WideNode* rw = ts.wide;
        uint32_t best_key = 0xFFFFFFFFu, best_tri = 0xFFFFFFFFu, best_inst = SGPU_INVALID_ID, cur = SGPU_INVALID_ID;
        float best_u = 0.0f, best_v = 0.0f, best_a = 1.0f;
        bool hit_any = false;
        uint32_t sp = 0;
        int node = ts.n_tris > 0 || (INST && ts.n_inst > 0) ? 0 : -1;
        GroupNode gn;
        auto fetch = [&]() { gn = GroupNode(rw, node, gl); };
        if (node >= 0) fetch();
        while (node >= 0) {
            if (INST && (gn.w.w >> 28) == 0) {
                // an instance: into its space, at its root
                const InstNode* __restrict in = reinterpret_cast<const InstNode*>(rw) + node;
                const float4 rows[3] = {in->w2l[0], in->w2l[1], in->w2l[2]};
                const f3 wo = o, wd = d;
                o = inst_point(rows, wo);
                d = inst_vector(rows, wd);
                set_slopes();
                cur = gn.w.x;
                rw = ts.insts[cur].wide;
                stack[sp++] = make_uint2(kGroupExit, 0);
                node = 0;
                fetch();
                continue;
            }
            if (STATS && gl == 0) ++cnt_nodes;
            const uint32_t ni = (gn.w.w >> 24) & 15u, base = gn.base();
            float tmin;
            const bool in = gn.enters(gl, inv, oinv, tnear, best_t, tmin);
            // internal children, far to near (any hit: last to first) onto the stack
            const bool inner = in && gl < ni, leaf = in && gl >= ni;
            const uint32_t inners = (uint32_t)(__ballot(inner) >> shift) & 0xFFu;
            const int k = inner ? (__float_as_int(tmin) & ~7) | (int)gl : 0x7FFFFFF8 | (int)gl;
            const uint32_t rank = ANY ? (uint32_t)__popc(inners & ((1u << gl) - 1u)) : group_rank(k);
            const uint32_t cnt = (uint32_t)__popc(inners);
            if (inner) stack[sp + cnt - 1u - rank] = make_uint2(base + 2u * gl, __float_as_uint(tmin));
            sp += cnt;
            asm volatile("" ::: "memory");
            // leaf children's triangles and, with them in flight, the node on top of the stack (65 536 rays:
            // 194 -> 167 us). Not over instances: the top entry may leave the one whose triangles these
            // are, and telling that apart costs more than the wait (494 -> 522 us).
            const uint32_t slot = gl == ni ? (uint32_t)node + 1u : base + ni + gl - 1u;
            const TriRecord* __restrict rt = reinterpret_cast<const TriRecord*>(rw);
            TriRecord r;
            if (leaf) r = rt[slot];
            uint2 e = make_uint2(kGroupExit, 0);
            const bool ahead = !INST && sp > 0;
            if (ahead) {
                e = stack[--sp];
                node = (int)e.x;
                fetch();
            }
            float t = 0.0f, U = 0.0f, V = 0.0f, a = 1.0f;
            uint32_t key = 0xFFFFFFFFu;
            bool closer = false;
            if (leaf) {
                if (STATS) ++cnt_tris;
                if (tri_hit(r, o, d, tnear, t, U, V, a)) {
                    key = __float_as_uint(r.a.w);
                    const bool first = INST ? (cur < best_inst || (cur == best_inst && key < best_key)) : key < best_key;
                    closer = ANY ? t <= best_t : t < best_t || (t == best_t && first);
                }
            }
            if ((uint32_t)(__ballot(closer) >> shift) & 0xFFu) {
                if (ANY) {
                    hit_any = true;
                    break;
                }
                const uint32_t from = group_closest(closer, t, key);
                best_t = __shfl(t, (int)from, 8);
                best_key = (uint32_t)__shfl((int)key, (int)from, 8);
                best_tri = (uint32_t)__shfl((int)slot, (int)from, 8);
                best_inst = cur;
                best_u = __shfl(U, (int)from, 8);
                best_v = __shfl(V, (int)from, 8);
                best_a = __shfl(a, (int)from, 8);
            }
            if (ahead && (ANY || __uint_as_float(e.y) <= best_t)) continue;
            node = -1;
            while (sp > 0) {
                e = stack[--sp];
                if (INST && e.x == kGroupExit) {
                    load_ray();
                    set_slopes();
                    rw = ts.wide;
                    cur = SGPU_INVALID_ID;
                    continue;
                }
                if (ANY || __uint_as_float(e.y) <= best_t) {
                    node = (int)e.x;
                    fetch();
                    break;
                }
            }
            asm volatile("" ::: "memory");
        }
        if (gl == 0) {
            uint32_t id0 = SGPU_INVALID_ID, id1 = SGPU_INVALID_ID;
            const WideNode* bw = ts.wide;
            if (INST && !ANY && best_tri != 0xFFFFFFFFu && best_inst != SGPU_INVALID_ID) {
                bw = ts.insts[best_inst].wide;
                if (inst_ids) {
                    id0 = inst_ids[2 * best_inst];
                    id1 = inst_ids[2 * best_inst + 1];
                }
            }
            write_result<ANY>(i, hit_any, best_tri, best_t, best_u / best_a, best_v / best_a,
                              reinterpret_cast<const TriRecord*>(bw), hits, occluded, id0, id1);
            if (INST && !ANY && comp_out) comp_out[i] = best_tri != 0xFFFFFFFFu ? best_inst : SGPU_INVALID_ID;
        }
    }
    if (STATS) {
        atomicAdd(&stats[0], cnt_nodes);
        atomicAdd(&stats[1], cnt_tris);
    }
}

// 8-wide traversal of the collapsed tree (WideNode), one ray per lane. In a trip of the wave's loop
// every lane has at most one 64-byte slot to read: a triangle to test, or else a node to visit.
// (Letting the lanes with triangles wait until 4, 8 or 16 of a wave have one cost 1-25 %.)
//
// Slots are fetched by the wave together (WaveFetch). A node visit (wide_boxes) turns leaf children hit
// into the lane's triangles to test (a slot base and a mask) and internal children hit into a group:
// the base of the node's children and a list of their numbers, 4 bits each (closest hit: by entry
// distance, a min/max network over keys that carry the number in their low bits; any hit: the mask, in
// order). The group being walked is in registers, the groups above it on the stack, so a visit pushes
// or pops one 8-byte entry at most and the stack is as deep as the tree. Hits are the triangle test's,
// independent of the tree and of the visiting order.
//
// INST: scenes of instances. Leaves of the top tree are nodes (InstNode); visiting one saves the
// group, pushes an exit entry (an empty group), moves the ray into the instance's space (t keeps its
// meaning: the direction is not renormalized) and goes on at the instance's root; popping the exit
// entry restores the world ray. Composed instances are numbered in composition order (instance i of
// the scene, then its instance j), so the closest hit is the smallest t with ties to the smaller
// (composed instance, triangle) = (inst_id0, inst_id1, geomID, primID).
//
// Waves take rays in chunks of 64 and a lane whose ray is done takes the next one of its wave's
// chunk at once, so lanes do not wait for the wave's longest ray; a wave whose chunk is used up
// takes the next from a counter, so waves do not wait for the launch's longest chunk.
//
// Bound by vector instructions (81 % of the issue cycles on the traversal workload with kRefill = 1,
// address unit 69 %); 32 KB of LDS a block allow 5 waves per SIMD. Against the version that read nodes
// and triangles lane by lane, sorted (distance, child) pairs and kept a stack of children: 16M rays in
// 2M triangles 15.2 -> 10.2 ms, 4M shadow rays in 1M triangles 2.66 -> 1.57 ms, 250K rays 0.62 -> 0.32
// ms (back to back; a call alone 0.35), 4M rays through 256 instances (which had no refill) 9.8 -> 3.0
// ms; hits the same bits.
template <bool ANY, bool STATS, bool MULTI, bool INST, bool TOP>
__global__ __launch_bounds__(SGPU_TRACE_BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_trace8(
    TraceScene scene, const uint32_t* __restrict inst_ids, const TraceScene* __restrict table,
    const uint32_t* __restrict ray_scene, sgpu_rays_soa rays, sgpu_hits_soa hits, uint32_t* __restrict occluded,
    uint32_t n, const uint32_t* __restrict n_ptr, uint2* __restrict spill, uint32_t stack_cap,
    unsigned long long* __restrict stats, uint32_t* __restrict overflow, uint32_t* __restrict work,
    uint32_t* __restrict comp_out, uint32_t n_top, uint32_t group_max)
{
    // each lane's fetched slot (4 KB a wave) and the stacks; or the stacks of 32 groups
    __shared__ uint4 lds_all[4 * SGPU_TRACE_BLOCK + kWideStackLds * SGPU_TRACE_BLOCK / 2];
    static_assert(sizeof(uint2) * kGroupStack * (SGPU_TRACE_BLOCK / 8) <= sizeof(lds_all), "the groups' stacks");
    uint4* const lds_slots = lds_all;
    uint2(*const lds_stack)[SGPU_TRACE_BLOCK] = reinterpret_cast<uint2(*)[SGPU_TRACE_BLOCK]>(lds_all + 4 * SGPU_TRACE_BLOCK);
    __shared__ uint4 lds_top[TOP ? 4 * kTopNodes : 1];
    uint32_t lane = threadIdx.x;  // the stack's column, and its spilled part's
    uint32_t gtid = blockIdx.x * SGPU_TRACE_BLOCK + threadIdx.x;
    const uint32_t stride = gridDim.x * SGPU_TRACE_BLOCK;
    unsigned long long cnt_nodes = 0, cnt_tris = 0;
    if (n_ptr) n = *n_ptr;  // the count written on the device by the kernel that queued the rays
    if (!TOP && n <= group_max) {
        trace_groups<ANY, STATS, MULTI, INST>(scene, inst_ids, table, ray_scene, rays, hits, occluded, n, stats, comp_out,
                                              reinterpret_cast<uint2*>(lds_all));
        return;
    }
    if (TOP) {
        for (uint32_t k = threadIdx.x; k < 4 * n_top; k += SGPU_TRACE_BLOCK)
            lds_top[k] = reinterpret_cast<const uint4*>(scene.wide + k / 4)[k % 4];
        __syncthreads();
    }

    // Rays come in chunks of 64: wave w's first chunk is chunk w, the next ones come from the
    // launch's counter (work[0], zeroed before the launch) past the grid's first chunks. A launch of
    // at most one chunk per wave takes no atomic. Positions in a chunk come from a ballot, so `next`
    // and `end` stay wave-uniform.
    const uint32_t grid_rays = (gridDim.x * SGPU_TRACE_BLOCK / 64) * kTraceChunk;
    uint32_t next = min(n, (uint32_t)__builtin_amdgcn_readfirstlane(gtid >> 6) * kTraceChunk);
    uint32_t end = min(n, next + kTraceChunk);
    bool drained = false;
    const unsigned long long below = (1ull << (threadIdx.x & 63u)) - 1ull;

    bool active = false;
    uint32_t i = 0;
    f3 o = mk3(0, 0, 0), d = mk3(0, 0, 0), inv = mk3(0, 0, 0), oinv = mk3(0, 0, 0);
    float tnear = 0.0f;
    float best_t = 0.0f;  // the any-hit query's tfar
    uint32_t best_key = 0xFFFFFFFFu, best_tri = 0xFFFFFFFFu, best_inst = SGPU_INVALID_ID;
    float best_u = 0.0f, best_v = 0.0f, best_a = 1.0f;  // u and v times the hit's |det|, and that
    bool hit_any = false;
    const WideNode* rw = scene.wide;
    uint32_t cur = SGPU_INVALID_ID;  // INST: the instance being walked (none: the top tree)
    int node = -1;                   // the slot of the node to visit, kNext: to be taken, -1: none left
    uint32_t gbase = 0, glist = 0;   // the group being walked: children's base, children still to visit
    uint32_t pfirst = 0, pbase = 0, pmask = 0;  // triangles to test: slot of leaf 0, base of the others, mask
    uint32_t sp = 0;

    const sgpu::WaveFetch wf(lds_slots);

    auto load_ray = [&](bool with_range) {
        o = mk3(rays.org_x[i], rays.org_y[i], rays.org_z[i]);
        d = mk3(rays.dir_x[i], rays.dir_y[i], rays.dir_z[i]);
        if (with_range) {
            tnear = rays.tnear[i];
            best_t = rays.tfar[i];
        }
    };
    auto set_slopes = [&]() {
        inv = mk3(safe_rcp(d.x), safe_rcp(d.y), safe_rcp(d.z));
        oinv = mk3(o.x * inv.x, o.y * inv.y, o.z * inv.z);
    };
    // the stack: entries below kWideStackLds deep in LDS (a ring), deeper ones spilled
    auto push = [&](uint32_t base, uint32_t list) {
        if (sp >= stack_cap) {
            atomicOr(overflow, 1u);
            return;
        }
        const uint32_t slot = sp % kWideStackLds;
        if (sp >= kWideStackLds) spill[(size_t)(sp - kWideStackLds) * stride + gtid] = lds_stack[slot][lane];
        lds_stack[slot][lane] = make_uint2(base, list);
        ++sp;
    };
    auto pop = [&]() {
        --sp;
        const uint32_t slot = sp % kWideStackLds;
        const uint2 e = lds_stack[slot][lane];
        if (sp >= kWideStackLds) lds_stack[slot][lane] = spill[(size_t)(sp - kWideStackLds) * stride + gtid];
        gbase = e.x;
        glist = e.y;
    };
    // the next node: the walked group's next child, or the top entry's
    auto advance = [&]() {
        while (glist == 0 && sp > 0) {
            pop();
            if (INST && glist == 0) {  // an exit entry: back in the top tree
                load_ray(false);
                set_slopes();
                rw = MULTI ? table[ray_scene[i]].wide : scene.wide;
                cur = SGPU_INVALID_ID;
            }
        }
        node = glist ? sgpu::wide_take<ANY>(gbase, glist) : -1;
    };

    auto finish = [&]() {
        uint32_t id0 = SGPU_INVALID_ID, id1 = SGPU_INVALID_ID;
        const WideNode* bw = rw;
        if (INST && !ANY && best_tri != 0xFFFFFFFFu) {
            if (best_inst != SGPU_INVALID_ID) {
                bw = (MULTI ? table[ray_scene[i]].insts : scene.insts)[best_inst].wide;
                if (inst_ids) {
                    id0 = inst_ids[2 * best_inst];
                    id1 = inst_ids[2 * best_inst + 1];
                }
            } else {
                bw = MULTI ? table[ray_scene[i]].wide : scene.wide;
            }
        }
        write_result<ANY>(i, hit_any, best_tri, best_t, best_u / best_a, best_v / best_a,
                          reinterpret_cast<const TriRecord*>(bw), hits, occluded, id0, id1);
        if (INST && !ANY && comp_out) comp_out[i] = best_tri != 0xFFFFFFFFu ? best_inst : SGPU_INVALID_ID;
    };
    bool tail = false;

    for (;;) {
        // Finished rays are written and their lanes take the next rays of the chunk (a new chunk when it
        // is used up) kRefill at a time: the work of that is a hundred instructions of the wave, and
        // nearly every trip has a lane or two that are done.
        const bool done = pmask == 0 && node == -1;
        const unsigned long long finished = __ballot(active && done), free_lanes = __ballot(done);
        // the launch's last rays: handed over below, once the finished ones are written
        const bool few = !TOP && drained && 64 - __popcll(free_lanes) <= kTailRays;
        if (free_lanes == ~0ull || few || __popcll(drained ? finished : free_lanes) >= kRefill<ANY>) {
            if (active && done) {
                finish();
                active = false;
            }
            const unsigned long long idle = free_lanes;
            if (next >= end && !drained) {
                if (grid_rays >= n) {
                    drained = true;  // the first chunks held every ray
                } else {
                    uint32_t base = 0;
                    if ((threadIdx.x & 63u) == 0) base = grid_rays + atomicAdd(&work[0], kTraceChunk);
                    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                    if (base >= n) {
                        drained = true;
                    } else {
                        next = base;
                        end = min(n, base + kTraceChunk);
                    }
                }
            }
            if (next < end) {
                const uint32_t r = next + (uint32_t)__popcll(idle & below);
                if (!active && r < end) {
                    i = r;
                    active = true;
                    load_ray(true);
                    set_slopes();
                    bool walk;
                    if (MULTI) {
                        const TraceScene ts = table[ray_scene[i]];
                        rw = ts.wide;
                        walk = ts.n_tris > 0 || (INST && ts.n_inst > 0);
                    } else {
                        rw = scene.wide;
                        walk = scene.n_tris > 0 || (INST && scene.n_inst > 0);
                    }
                    best_key = 0xFFFFFFFFu;
                    best_tri = 0xFFFFFFFFu;
                    best_inst = SGPU_INVALID_ID;
                    best_u = 0.0f;
                    best_v = 0.0f;
                    best_a = 1.0f;
                    hit_any = false;
                    sp = 0;
                    glist = 0;
                    pmask = 0;
                    cur = SGPU_INVALID_ID;
                    node = walk ? 0 : -1;
                }
                next = min(end, next + (uint32_t)__popcll(idle));
            }
            if (__ballot(active) == 0) break;
            if (few) {
                tail = true;
                break;
            }
        }

        const bool test = pmask != 0;
        const bool visit = pmask == 0 && node >= 0;
        int slot = visit ? node : -1;
        if (test) {
            const uint32_t k = (uint32_t)__builtin_ctz(pmask);
            slot = (int)(k == 0 ? pfirst : pbase + k);
            pmask &= pmask - 1;
        }
        const bool in_top = TOP && visit && (uint32_t)slot < 2 * n_top;
        wf.fetch<MULTI || INST>(in_top ? -1 : slot, rw);
        uint4 w0, w1, w2, w3;
        if (in_top) {
            const uint4* t = lds_top + 2 * slot;
            w0 = t[0], w1 = t[1], w2 = t[2], w3 = t[3];
        } else {
            w0 = wf.read(0), w1 = wf.read(1), w2 = wf.read(2), w3 = wf.read(3);
        }
        if (test) {
            // ---- one triangle test ----
            TriRecord r;
            r.a = make_float4(__uint_as_float(w0.x), __uint_as_float(w0.y), __uint_as_float(w0.z), __uint_as_float(w0.w));
            r.b = make_float4(__uint_as_float(w1.x), __uint_as_float(w1.y), __uint_as_float(w1.z), __uint_as_float(w1.w));
            r.c = make_float4(__uint_as_float(w2.x), __uint_as_float(w2.y), __uint_as_float(w2.z), __uint_as_float(w2.w));
            if (STATS) ++cnt_tris;
            float t, U, V, a;
            if (tri_hit(r, o, d, tnear, t, U, V, a)) {
                if (ANY) {
                    if (t <= best_t) {
                        hit_any = true;
                        pmask = 0;
                        node = -1;
                    }
                } else {
                    const uint32_t key = __float_as_uint(r.a.w);
                    const bool first = INST ? (cur < best_inst || (cur == best_inst && key < best_key)) : key < best_key;
                    if (t < best_t || (t == best_t && first)) {
                        best_t = t;
                        best_key = key;
                        best_tri = (uint32_t)slot;
                        if (INST) best_inst = cur;
                        best_u = U;
                        best_v = V;
                        best_a = a;
                    }
                }
            }
        }
        if (visit) {
            // ---- one node visit ----
            if (INST && (w0.w >> 28) == 0) {
                // an instance: into its space, at its root
                if (glist) push(gbase, glist);
                push(0, 0);
                const f3 wo = o, wd = d;
                const float4 rows[3] = {make_float4(__uint_as_float(w1.x), __uint_as_float(w1.y), __uint_as_float(w1.z), __uint_as_float(w1.w)),
                                        make_float4(__uint_as_float(w2.x), __uint_as_float(w2.y), __uint_as_float(w2.z), __uint_as_float(w2.w)),
                                        make_float4(__uint_as_float(w3.x), __uint_as_float(w3.y), __uint_as_float(w3.z), __uint_as_float(w3.w))};
                o = inst_point(rows, wo);
                d = inst_vector(rows, wd);
                set_slopes();
                cur = w0.x;
                rw = (MULTI ? table[ray_scene[i]].insts : scene.insts)[cur].wide;
                node = 0;
                glist = 0;
            } else {
                if (STATS) ++cnt_nodes;
                const sgpu::WideHits h = sgpu::wide_boxes<ANY>(w0, w1, w2, w3, inv, oinv, tnear, best_t);
                pmask = h.leaves;
                pfirst = (uint32_t)node + 1;
                pbase = h.leaf_base;
                if (h.list) {
                    if (glist) push(gbase, glist);
                    gbase = h.base;
                    glist = h.list;
                }
                node = kNext;
            }
        }
        // the triangles found in a node come before the next node: leaving an instance changes the ray
        if (pmask == 0 && node == kNext) advance();
    }
    if (tail) {
        // The wave's last eight rays, with none to come, end a launch with a chain of trips for one lane in
        // eight or fewer: eight lanes each take over a ray where its lane stands, as in trace_groups but on
        // the lane's stack (250K rays 394 -> 315 us, 4M any-hit rays 1.68 -> 1.57 ms, 4M rays through 256
        // instances 3.30 -> 3.01 ms, a 256 x 256 image of 16 paths a pixel 5.9 -> 5.3 ms).
        unsigned long long left = __ballot(active);
        const uint32_t gl = threadIdx.x & 7u, shift = threadIdx.x & 56u;
#pragma unroll
        for (uint32_t k = 0; k < kTailRays - 1; ++k)  // group g: the g-th of them
            if (k < shift >> 3) left &= left - 1;
        const bool mine = left != 0;
        const int own = mine ? __builtin_ctzll(left) : 0;
        auto take = [&](uint32_t v) { return (uint32_t)__shfl((int)v, own); };
        auto takef = [&](float v) { return __shfl(v, own); };
        i = take(i);
        o = mk3(takef(o.x), takef(o.y), takef(o.z));
        d = mk3(takef(d.x), takef(d.y), takef(d.z));
        set_slopes();
        tnear = takef(tnear);
        best_t = takef(best_t);
        best_key = take(best_key);
        best_tri = take(best_tri);
        best_inst = take(best_inst);
        best_u = takef(best_u);
        best_v = takef(best_v);
        best_a = takef(best_a);
        if (MULTI || INST) {
            const uint64_t a = (uint64_t)rw;
            rw = (const WideNode*)((uint64_t)take((uint32_t)(a >> 32)) << 32 | take((uint32_t)a));
            cur = take(cur);
        }
        node = (int)take((uint32_t)node);
        gbase = take(gbase);
        glist = take(glist);
        pfirst = take(pfirst);
        pbase = take(pbase);
        pmask = take(pmask);
        sp = take(sp);
        hit_any = false;
        __threadfence_block();  // the spilled entries are the owners' stores
        lane = (lane & ~63u) | (uint32_t)own;
        gtid = (gtid & ~63u) | (uint32_t)own;
        while (mine) {
            if (pmask) {
                const uint32_t slot = gl == 0 ? pfirst : pbase + gl;
                float t = 0.0f, U = 0.0f, V = 0.0f, a = 1.0f;
                uint32_t key = 0xFFFFFFFFu;
                bool closer = false;
                if ((pmask >> gl) & 1u) {
                    const TriRecord r = reinterpret_cast<const TriRecord*>(rw)[slot];
                    if (STATS) ++cnt_tris;
                    if (tri_hit(r, o, d, tnear, t, U, V, a)) {
                        key = __float_as_uint(r.a.w);
                        const bool first = INST ? (cur < best_inst || (cur == best_inst && key < best_key)) : key < best_key;
                        closer = ANY ? t <= best_t : t < best_t || (t == best_t && first);
                    }
                }
                pmask = 0;
                if ((uint32_t)(__ballot(closer) >> shift) & 0xFFu) {
                    if (ANY) {
                        hit_any = true;
                        break;
                    }
                    const uint32_t from = group_closest(closer, t, key);
                    best_t = __shfl(t, (int)from, 8);
                    best_key = (uint32_t)__shfl((int)key, (int)from, 8);
                    best_tri = (uint32_t)__shfl((int)slot, (int)from, 8);
                    if (INST) best_inst = cur;
                    best_u = __shfl(U, (int)from, 8);
                    best_v = __shfl(V, (int)from, 8);
                    best_a = __shfl(a, (int)from, 8);
                }
            }
            if (node == kNext) advance();
            if (node < 0) break;
            const GroupNode gn(rw, node, gl);
            if (INST && (gn.w.w >> 28) == 0) {
                const InstNode* __restrict in = reinterpret_cast<const InstNode*>(rw) + node;
                const float4 rows[3] = {in->w2l[0], in->w2l[1], in->w2l[2]};
                if (glist) push(gbase, glist);
                push(0, 0);
                const f3 wo = o, wd = d;
                o = inst_point(rows, wo);
                d = inst_vector(rows, wd);
                set_slopes();
                cur = gn.w.x;
                rw = (MULTI ? table[ray_scene[i]].insts : scene.insts)[cur].wide;
                node = 0;
                glist = 0;
                continue;
            }
            if (STATS && gl == 0) ++cnt_nodes;
            const uint32_t ni = (gn.w.w >> 24) & 15u, base = gn.base();
            float tmin;
            const bool in = gn.enters(gl, inv, oinv, tnear, best_t, tmin);
            const uint32_t found = (uint32_t)(__ballot(in) >> shift) & 0xFFu;
            pmask = found >> ni;
            pfirst = (uint32_t)node + 1u;
            pbase = base + 2u * ni - 1u;
            uint32_t list = found & ((1u << ni) - 1u);
            if (!ANY) {
                const bool inner = in && gl < ni;
                const uint32_t rank = group_rank(inner ? (__float_as_int(tmin) & ~7) | (int)gl : 0x7FFFFFF8 | (int)gl);
                list = inner ? (8u | gl) << (4u * rank) : 0u;
#pragma unroll
                for (uint32_t x = 1; x < 8; x <<= 1) list |= (uint32_t)__shfl_xor((int)list, x, 8);
            }
            if (list) {
                if (glist) push(gbase, glist);
                gbase = base;
                glist = list;
            }
            node = kNext;
        }
        if (mine && gl == 0) finish();
    }
    if (STATS) {
        atomicAdd(&stats[0], cnt_nodes);
        atomicAdd(&stats[1], cnt_tris);
    }
}

}  // namespace

namespace {

__global__ void k_zero_work(uint32_t* __restrict w)
{
    if (threadIdx.x < kTraceWorkWords) w[threadIdx.x] = 0u;
}

}  // namespace

// The ray counters, then each lane's stack words past those in LDS.
size_t sgpu_trace_spill_words(uint32_t stack_words, size_t threads)
{
    const uint32_t deep = stack_words > SGPU_STACK_LDS ? stack_words - SGPU_STACK_LDS : 1;
    return kTraceWorkWords + deep * threads;
}

void sgpu_trace_work_zero(uint32_t* spill, hipStream_t stream)
{
    hipLaunchKernelGGL(k_zero_work, dim3(1), dim3(kTraceWorkWords), 0, stream, spill);
}

namespace {

// One traversal launch over n rays: of one scene (`scene`, its instances' ids `inst_ids`), or (table
// != nullptr) of the scenes of a batch, ray i in table[ray_scene[i]]; stack_words bounds every
// scene's stack. The context's trace_tree picks the tree kind; scenes of instances are walked on the
// 8-wide one.
int trace_launch(sgpu_context ctx, const TraceScene& scene, uint32_t n_wide, const uint32_t* inst_ids,
                 uint32_t stack_words, uint32_t* overflow, const TraceScene* table, const uint32_t* ray_scene,
                 const sgpu_rays_soa* rays, const sgpu_hits_soa* hits, uint32_t* occluded, uint32_t n, bool any_hit,
                 uint64_t* d_stats, hipStream_t stream, uint32_t* spill_buf, const uint32_t* n_ptr, bool instanced,
                 uint32_t* comp_out, uint32_t cap_blocks = 0)
{
    if (n == 0) return SGPU_OK;
    const uint32_t cus = (uint32_t)ctx->props.multiProcessorCount;
    const bool binary = ctx->trace_tree == 0 && !instanced;
    const bool multi = table != nullptr;
    // top nodes in LDS: single-scene launches over geometries
    const uint32_t n_top = binary || multi || instanced ? 0u : std::min(n_wide, std::min(ctx->trace_lds_nodes, kTopNodes));
    // launches of few rays go eight lanes a ray, where the trees' depth lets their stacks be in LDS
    const uint32_t group_max = binary || n_top || group_stack(stack_words) > kGroupStack ? 0u : any_hit ? kGroupRays<true> : kGroupRays<false>;
    const uint32_t lanes = n <= group_max ? 8u : 1u;
    uint32_t blocks = (uint32_t)(((uint64_t)n * lanes + SGPU_TRACE_BLOCK - 1) / SGPU_TRACE_BLOCK);
    uint32_t max_blocks = cus * std::min(ctx->trace_blocks_per_cu, kMaxTraceBlocksPerCu);
    if (cap_blocks && max_blocks > cap_blocks) max_blocks = cap_blocks;
    if (blocks > max_blocks) blocks = max_blocks;

    // stream-ordered scratch for the spilled part of the stacks, private to this call, unless the
    // caller lends a buffer of sgpu_trace_spill_words (sized for the largest grid); its first
    // kTraceWorkWords words are the launch's ray counters. A launch whose rays the grid holds at once
    // and whose stacks fit LDS touches neither (a stream-ordered free makes the host wait for the
    // kernel: 150 us of a small query).
    const bool counts = !binary && blocks < (n + SGPU_TRACE_BLOCK - 1) / SGPU_TRACE_BLOCK;
    uint32_t* buf = spill_buf;
    if (!buf && (counts || (n > group_max && stack_words > SGPU_STACK_LDS)))
        SGPU_HIP_TRY(sgpu_device_malloc_async((void**)&buf,
                                    sgpu_trace_spill_words(stack_words, (size_t)blocks * SGPU_TRACE_BLOCK) *
                                        sizeof(uint32_t),
                                    stream));
    uint32_t* const work = buf;
    uint32_t* const spill = buf ? buf + kTraceWorkWords : nullptr;
    sgpu_hits_soa h = {};
    if (hits) h = *hits;
    unsigned long long* st = (unsigned long long*)d_stats;
    const dim3 g(blocks), b(SGPU_TRACE_BLOCK);
    if (binary) {
#define SGPU_LAUNCH_2(A, S, M)                                                                                      \
    hipLaunchKernelGGL((k_trace<A, S, M>), g, b, 0, stream, scene.nodes,                      \
                       reinterpret_cast<const TriRecord*>(scene.wide), scene.n_tris, table, ray_scene,            \
                       *rays, h, occluded, n, n_ptr, spill, stack_words, st, overflow)
        if (any_hit) {
            if (st) { if (multi) SGPU_LAUNCH_2(true, true, true); else SGPU_LAUNCH_2(true, true, false); }
            else { if (multi) SGPU_LAUNCH_2(true, false, true); else SGPU_LAUNCH_2(true, false, false); }
        } else {
            if (st) { if (multi) SGPU_LAUNCH_2(false, true, true); else SGPU_LAUNCH_2(false, true, false); }
            else { if (multi) SGPU_LAUNCH_2(false, false, true); else SGPU_LAUNCH_2(false, false, false); }
        }
#undef SGPU_LAUNCH_2
    } else {
        if (counts) sgpu_trace_work_zero(work, stream);
#define SGPU_LAUNCH_8(A, S, M, I, T)                                                                               \
    hipLaunchKernelGGL((k_trace8<A, S, M, I, T>), g, b, 0, stream, scene, inst_ids, table, ray_scene, *rays, h,    \
                       occluded, n, n_ptr, (uint2*)spill, std::max(stack_words / 2, kWideStackLds), st, overflow, work, comp_out, n_top, group_max)
#define SGPU_LAUNCH_8S(A, S)                                                                                      \
    do {                                                                                                          \
        if (multi && instanced) SGPU_LAUNCH_8(A, S, true, true, false);                                           \
        else if (multi) SGPU_LAUNCH_8(A, S, true, false, false);                                                  \
        else if (instanced) SGPU_LAUNCH_8(A, S, false, true, false);                                              \
        else if (n_top) SGPU_LAUNCH_8(A, S, false, false, true);                                                  \
        else SGPU_LAUNCH_8(A, S, false, false, false);                                                            \
    } while (0)
        if (any_hit) {
            if (st) SGPU_LAUNCH_8S(true, true);
            else SGPU_LAUNCH_8S(true, false);
        } else {
            if (st) SGPU_LAUNCH_8S(false, true);
            else SGPU_LAUNCH_8S(false, false);
        }
#undef SGPU_LAUNCH_8S
#undef SGPU_LAUNCH_8
    }
    SGPU_HIP_TRY(hipGetLastError());
    if (buf && !spill_buf) SGPU_HIP_TRY(hipFreeAsync(buf, stream));
    return SGPU_OK;
}

}  // namespace

size_t sgpu_trace_spill_words(sgpu_context ctx, uint32_t stack_words)
{
    const uint32_t cus = (uint32_t)ctx->props.multiProcessorCount;
    return sgpu_trace_spill_words(stack_words, (size_t)cus * kMaxTraceBlocksPerCu * SGPU_TRACE_BLOCK);
}

uint32_t sgpu_trace_stack_words(sgpu_scene scene) { return scene->wide_stack; }

size_t sgpu_trace_spill_words(sgpu_scene scene) { return sgpu_trace_spill_words(scene->ctx, scene->stack_cap); }

int sgpu_trace_launch(sgpu_scene scene, const sgpu_rays_soa* rays, const sgpu_hits_soa* hits, uint32_t* occluded,
                      uint32_t n, bool any_hit, uint64_t* d_stats, hipStream_t stream, uint32_t* spill_buf,
                      const uint32_t* n_ptr, uint32_t* overflow, uint32_t* comp_out, uint32_t max_blocks,
                      uint64_t* curve_stats)
{
    const TraceScene ts = sgpu_trace_scene(scene);
    const int rc = trace_launch(scene->ctx, ts, scene->n_wide, scene->d_inst_ids,
                                scene->ctx->trace_tree == 1 ? scene->wide_stack : scene->stack_cap,
                                overflow ? overflow : scene->d_overflow, nullptr, nullptr, rays, hits, occluded, n,
                                any_hit, d_stats, stream, spill_buf, n_ptr, !scene->instances.empty(), comp_out,
                                max_blocks);
    if (rc != SGPU_OK || scene->n_curves == 0) return rc;
    return sgpu_curve_launch(scene->ctx, ts, scene->d_inst_ids, scene->wide_stack, nullptr, nullptr, rays, hits, occluded, n, any_hit, n_ptr, comp_out,
                             overflow ? overflow : scene->d_overflow, stream, spill_buf, max_blocks, curve_stats);
}

int sgpu_trace_launch_multi(sgpu_context ctx, const TraceScene* table, const uint32_t* ray_scene, uint32_t stack_cap,
                            uint32_t* overflow, const sgpu_rays_soa* rays, const sgpu_hits_soa* hits,
                            uint32_t* occluded, uint32_t n, bool any_hit, uint64_t* d_stats, hipStream_t stream,
                            uint32_t* spill_buf, const uint32_t* n_ptr, bool instanced, uint32_t* comp_out,
                            bool curves)
{
    const int rc = trace_launch(ctx, TraceScene{}, 0, nullptr, stack_cap, overflow, table, ray_scene, rays, hits, occluded,
                                n, any_hit, d_stats, stream, spill_buf, n_ptr, instanced, comp_out);
    if (rc != SGPU_OK || !curves) return rc;
    return sgpu_curve_launch(ctx, TraceScene{}, nullptr, stack_cap, table, ray_scene, rays, hits, occluded, n, any_hit,
                             n_ptr, comp_out, overflow, stream, spill_buf);
}
