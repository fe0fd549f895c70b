// The curve pass: rays against a scene's round B-spline curves (rtcIntersect1 / rtcOccluded1 on
// RTC_GEOMETRY_TYPE_ROUND_BSPLINE_CURVE geometry, ModelResource.cpp:300-330), after the triangle
// traversal over the same rays. Curves sit in a tree of their own (built by sgpu_curve_build), so that
// the triangle kernels keep their registers; this pass runs only for scenes that hold curves.
//
// One ray per lane, refilled as rays finish. A ray's work is a mix of very unequal steps: node visits
// (200 instructions), segments rejected or not by one capsule (150), some segments' sixteen piece
// capsules (1,700 one after another) and piece searches (4,000). Run by each lane where it met them, a
// wave had 1.7 of its 64 lanes active; so each lane carries the step it is at and a trip of the wave's
// loop does one kind of step for the lanes that are at it: searches once kSearchLanes lanes wait for
// one, the piece capsules of four segments at a time on 16 lanes each, else visits and segment tests
// (or what the lanes that are left wait for).
//
// The tree is 8-wide, over the segments' tight boxes, and walked like the triangles' (sgpu_wide.h);
// control points are slots like nodes, and a segment's points stay in the lane's slot in LDS for its
// piece tests and searches. The closest entry of a ray that starts outside every tube does not depend on
// the order of the walk but where two segments meet: the ball between them can be both segments' first
// entry at the same t. Such a tie goes
// to the segment that the binary tree over the control points' boxes, walked nearer child first,
// comes to first.
//
// 1M rays (camera and ground) in a field of 65,536 blades, 458,752 segments: 27.8 ms by a lane-by-lane
// walk of that binary tree (185 visits, 30 segment tests a ray), 12.7 in steps, 3.92 on the 8-wide tree
// of tight boxes (24 visits, 4.4 segment tests), the same bits. Bound by the searches' vector
// instructions.
#include "sgpu_curve.h"
#include "sgpu_wide.h"

#include <algorithm>

namespace {

constexpr int kCurveBlock = 256;
// Lanes waiting for a search for which a trip searches: 1M rays over 459K segments take 6.0 ms at 12,
// 4.7 at 20, 4.2 at 28, 4.0 at 36 and 40, 4.2 at 48. (Searching in two steps, the crossing pieces' entries
// apart, came to 4.2 ms at best; segment tests gain nothing by waiting for each other.)
constexpr int kSearchLanes = 38;
constexpr unsigned kCurveWaves = 4;  // waves per SIMD: 4.0 ms; 3: 4.2, 5 (registers spilled): 4.6
static_assert(sgpu::kCurvePieces == 16, "a segment's pieces are 16 lanes");
constexpr int kCurveRefill = 8;
constexpr uint32_t kCurveChunk = 64;

__device__ __forceinline__ bool child_box(float lx, float hx, float ly, float hy, float lz, float hz, f3 o, f3 inv,
                                          float tmin, float tmax, float& tent)
{
    const float ax = (lx - o.x) * inv.x, bx = (hx - o.x) * inv.x;
    const float ay = (ly - o.y) * inv.y, by = (hy - o.y) * inv.y;
    const float az = (lz - o.z) * inv.z, bz = (hz - o.z) * inv.z;
    const float tn = fmaxf(fmaxf(tmin, fminf(ax, bx)), fmaxf(fminf(ay, by), fminf(az, bz)));
    const float tf = fminf(fminf(tmax, fmaxf(ax, bx)), fminf(fmaxf(ay, by), fmaxf(az, bz)));
    tent = tn;
    return tn <= tf;
}

__device__ __forceinline__ float safe_inv(float x)
{
    return 1.0f / (fabsf(x) > 1e-30f ? x : copysignf(1e-30f, x));
}

__device__ __forceinline__ float4 as_f4(uint4 v)
{
    return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
}

// Whether the binary tree's walk (of a ray that hits both) comes to leaf a before leaf b: at the node
// where they part, leaf children come before nodes, the first before the second, and of two nodes the
// nearer one. A radix tree's node parts leaves 0..g from g + 1 on, g the index of its first child.
__device__ bool walked_before(const BvhNode* __restrict nodes, int a, int b, f3 o, f3 inv, float tnear, float best)
{
    int node = 0;
    for (uint32_t k = 0; k < kCurveStack; ++k) {
        const BvhNode nd = nodes[node];
        const int c0 = nd.child.x, c1 = nd.child.y;
        const int g = c0 < 0 ? ~c0 : c0;
        if (a <= g && b <= g && c0 >= 0) {
            node = c0;
        } else if (a > g && b > g && c1 >= 0) {
            node = c1;
        } else {
            bool first = true;  // child 0 comes first
            if (c0 >= 0 && c1 < 0) first = false;
            if (c0 >= 0 && c1 >= 0) {
                float t0, t1;
                child_box(nd.x.x, nd.x.y, nd.y.x, nd.y.y, nd.z.x, nd.z.y, o, inv, tnear, best, t0);
                child_box(nd.x.z, nd.x.w, nd.y.z, nd.y.w, nd.z.z, nd.z.w, o, inv, tnear, best, t1);
                first = t0 <= t1;
            }
            return (a <= g) == first;
        }
    }
    return false;
}

// The step a lane is at.
enum Step : int { kIdle, kVisit, kSegment, kPieces, kSearch, kDone };

template <bool ANY, bool MULTI, bool STATS>
__global__ __launch_bounds__(kCurveBlock) __attribute__((amdgpu_waves_per_eu(kCurveWaves))) void k_curves(
    TraceScene scene, const uint32_t* __restrict inst_ids, const TraceScene* __restrict table,
    const uint32_t* __restrict ray_scene, sgpu_rays_soa rays, sgpu_hits_soa hits, uint32_t* __restrict occluded,
    uint32_t n, const uint32_t* __restrict n_ptr, uint32_t* __restrict work, uint2* __restrict spill,
    uint32_t stack_cap, uint32_t* __restrict comp_out, uint32_t* __restrict overflow,
    unsigned long long* __restrict stats)
{
    __shared__ uint2 lds_stack[kWideStackLds][kCurveBlock];
    __shared__ uint4 lds_slots[4 * kCurveBlock];  // each lane's fetched slot, 4 KB a wave
    const uint32_t lane = threadIdx.x;
    const uint32_t gtid = blockIdx.x * kCurveBlock + threadIdx.x;
    const uint32_t stride = gridDim.x * kCurveBlock;
    const uint32_t count = n_ptr ? min(*n_ptr, n) : n;
    unsigned long long cnt_nodes = 0, cnt_segs = 0;
    const sgpu::WaveFetch wf(lds_slots);
    const uint32_t wl = wf.lane;

    // chunks of 64 rays: wave w's first is chunk w, the next ones come from the counter work[0]
    const uint32_t grid_rays = gridDim.x * kCurveBlock / 64 * kCurveChunk;
    uint32_t next = min(count, (uint32_t)__builtin_amdgcn_readfirstlane((blockIdx.x * kCurveBlock + threadIdx.x) >> 6) * kCurveChunk);
    uint32_t end = min(count, next + kCurveChunk);
    bool drained = false;
    const unsigned long long below = (1ull << wl) - 1ull;

    int step = kIdle;
    uint32_t i = 0;
    f3 o = mk3(0, 0, 0), d = mk3(0, 0, 0), inv = mk3(0, 0, 0), oinv = mk3(0, 0, 0);
    float tnear = 0.0f, best = 0.0f;
    int best_rec = -1;    // the slot of the closest entry's segment
    float best_u = 0.0f;  // the ball of the closest entry (its contact parameter is found at the end)
    const WideNode* rw = scene.cwide;
    int node = -1;                              // the node to visit after the segments below; -1: none
    uint32_t gbase = 0, glist = 0;              // the group being walked
    uint32_t pfirst = 0, pbase = 0, pmask = 0;  // segments to test: slot of leaf 0, base of the others, mask
    uint32_t sp = 0;
    // the segment being searched: its slot, entry and ball of its closest entry so far, pieces left
    int seg = -1;
    float seg_t = 0.0f, seg_u = 0.0f;
    bool seg_found = false;
    uint32_t pieces = 0;

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
    // what follows a segment or a visit: the next segment of the node, the next node, or the end
    auto proceed = [&]() {
        if (pmask) {
            const uint32_t k = (uint32_t)__builtin_ctz(pmask);
            seg = (int)(k == 0 ? pfirst : pbase + k);
            pmask &= pmask - 1;
            step = kSegment;
            return;
        }
        if (glist == 0 && sp > 0) {
            --sp;
            const uint32_t slot = sp % kWideStackLds;
            const uint2 e = lds_stack[slot][lane];
            if (sp >= kWideStackLds) lds_stack[slot][lane] = spill[(size_t)(sp - kWideStackLds) * stride + gtid];
            gbase = e.x;
            glist = e.y;
        }
        step = glist ? kVisit : kDone;
        if (glist) node = sgpu::wide_take<ANY>(gbase, glist);
    };
    // the segment's last piece is done
    auto segment_done = [&]() {
        bool better = seg_found && (ANY || seg_t < best);
        if (!ANY && seg_found && seg_t == best && best_rec >= 0) {
            // two segments' entries at one t
            const TraceScene ts = MULTI ? table[ray_scene[i]] : scene;
            const f3 inv_d = mk3(safe_inv(d.x), safe_inv(d.y), safe_inv(d.z));
            better = walked_before(ts.cnodes, (int)ts.cids[seg].w, (int)ts.cids[best_rec].w, o, inv_d, tnear, best);
        }
        if (better) {
            best = seg_t;
            best_u = seg_u;
            best_rec = seg;
        }
        if (ANY && best_rec >= 0) step = kDone;
        else proceed();
    };
    auto points = [&](sgpu::CurveSeg& s) {
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) s.p[c] = as_f4(wf.read(c));
    };

    for (;;) {
        const unsigned long long free_lanes = __ballot(step == kIdle || step == kDone);
        const unsigned long long done = __ballot(step == kDone);
        if (free_lanes == ~0ull || __popcll(drained ? done : free_lanes) >= kCurveRefill) {
            if (step == kDone) {
                if (ANY) {
                    if (best_rec >= 0) occluded[i] = 1u;
                } else if (best_rec >= 0) {
                    sgpu::CurveSeg s;
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        s.p[c] = reinterpret_cast<const CurvePoints*>(reinterpret_cast<const char*>(rw) + (size_t)best_rec * kSlotBytes)->p[c];
                    float u;
                    f3 ng;
                    sgpu::curve_finish(s, o, d, best, best_u, u, ng);
                    const InstRecord* ins = MULTI ? table[ray_scene[i]].insts : scene.insts;
                    const uint4 ids = (MULTI ? table[ray_scene[i]].cids : scene.cids)[best_rec];  // geom, prim, inst
                    uint32_t id0 = SGPU_INVALID_ID, id1 = SGPU_INVALID_ID;
                    if (ids.z != SGPU_INVALID_ID && ins) {
                        // Embree reports an instanced geometry's normal in its own space: through the linear
                        // part of the world-to-local transform (a similarity, so the normal's direction is kept)
                        const InstRecord ir = ins[ids.z];
                        ng = mk3(ir.w2l[0].x * ng.x + ir.w2l[0].y * ng.y + ir.w2l[0].z * ng.z,
                                 ir.w2l[1].x * ng.x + ir.w2l[1].y * ng.y + ir.w2l[1].z * ng.z,
                                 ir.w2l[2].x * ng.x + ir.w2l[2].y * ng.y + ir.w2l[2].z * ng.z);
                        if (inst_ids) {
                            id0 = inst_ids[2 * ids.z];
                            id1 = inst_ids[2 * ids.z + 1];
                        }
                    }
                    if (hits.t) hits.t[i] = best;
                    if (hits.u) hits.u[i] = u;
                    if (hits.v) hits.v[i] = 0.0f;
                    if (hits.prim_id) hits.prim_id[i] = ids.y;
                    if (hits.geom_id) hits.geom_id[i] = ids.x;
                    if (hits.ng_x) {
                        hits.ng_x[i] = ng.x;
                        hits.ng_y[i] = ng.y;
                        hits.ng_z[i] = ng.z;
                    }
                    if (hits.inst_id0) hits.inst_id0[i] = id0;
                    if (hits.inst_id1) hits.inst_id1[i] = id1;
                    if (comp_out) comp_out[i] = ids.z;
                }
                step = kIdle;
            }
            if (next >= end && !drained) {
                if (grid_rays >= count) {
                    drained = true;  // the first chunks held every ray
                } else {
                    uint32_t base = 0;
                    if (wl == 0) base = grid_rays + atomicAdd(&work[0], kCurveChunk);
                    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                    if (base >= count) {
                        drained = true;
                    } else {
                        next = base;
                        end = min(count, base + kCurveChunk);
                    }
                }
            }
            if (next < end) {
                const uint32_t r = next + (uint32_t)__popcll(free_lanes & below);
                if (step == kIdle && r < end) {
                    i = r;
                    uint32_t nc = scene.n_curves;
                    if (MULTI) {
                        const TraceScene ts = table[ray_scene[i]];
                        rw = ts.cwide;
                        nc = ts.n_curves;
                    }
                    if (nc > 0 && !(ANY && occluded[i])) {
                        o = mk3(rays.org_x[i], rays.org_y[i], rays.org_z[i]);
                        d = mk3(rays.dir_x[i], rays.dir_y[i], rays.dir_z[i]);
                        inv = mk3(sgpu::safe_rcp(d.x), sgpu::safe_rcp(d.y), sgpu::safe_rcp(d.z));
                        oinv = mk3(o.x * inv.x, o.y * inv.y, o.z * inv.z);
                        tnear = rays.tnear[i];
                        // the triangle pass left its hit distance (or tfar on a miss) in hits.t
                        best = (!ANY && hits.t) ? hits.t[i] : rays.tfar[i];
                        best_rec = -1;
                        sp = 0;
                        glist = 0;
                        pmask = 0;
                        node = 0;
                        step = kVisit;
                    }
                }
                next = min(end, next + (uint32_t)__popcll(free_lanes));
            }
            if (__ballot(step != kIdle) == 0) {
                if (next >= end && drained) break;
                continue;
            }
        }

        const int n_search = __popcll(__ballot(step == kSearch)), n_pieces = __popcll(__ballot(step == kPieces));
        const bool light = __ballot(step == kVisit || step == kSegment) != 0;
        if (n_search >= kSearchLanes || (!light && n_search > 0 && n_search >= n_pieces)) {
            // ---- one piece searched ----
            if (step == kSearch) {
                sgpu::CurveSeg s;
                points(s);
                float a, m2, m2r;
                const sgpu::CurveRay ray = sgpu::curve_ray(o, d, a);
                sgpu::curve_bounds(s, m2, m2r);
                const int k = __builtin_ctz(pieces);
                pieces &= pieces - 1;
                const float h = 1.0f / sgpu::kCurvePieces;
                f3 A, B;
                float ra, rb;
                sgpu::curve_eval(s, (float)k * h, A, ra);
                sgpu::curve_eval(s, (float)(k + 1) * h, B, rb);
                float near, t, u;
                // (the entry found in an earlier piece may have ruled this one out)
                if (sgpu::curve_piece_candidate(ray, a, A, ra, B, rb, sgpu::curve_deviation(m2, m2r), tnear, seg_t) &&
                    sgpu::curve_piece_search(s, ray, k, near) &&
                    sgpu::curve_piece_entry(s, ray, k, near, tnear, seg_t, t, u)) {
                    seg_t = t;
                    seg_u = u;
                    seg_found = true;
                    if (ANY) pieces = 0;
                }
                if (pieces == 0) segment_done();
            }
        } else if (n_pieces >= 4 || (!light && n_pieces > 0)) {
            // ---- the piece capsules of four segments, 16 lanes each ----
            const unsigned long long waiting = __ballot(step == kPieces);
            // the lane whose segment this lane's group takes: the (wl / 16)-th that waits
            unsigned long long m = waiting;
            int who = -1;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int first = m ? __builtin_ctzll(m) : -1;
                if ((int)(wl >> 4) == g) who = first;
                m &= m - 1;
            }
            const int src = 4 * (who < 0 ? 0 : who);
            auto from = [&](float x) { return __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(x))); };
            const f3 ro = mk3(from(o.x), from(o.y), from(o.z)), rd = mk3(from(d.x), from(d.y), from(d.z));
            const float rnear = from(tnear), rbest = from(best);
            bool candidate = false;
            if (who >= 0) {
                sgpu::CurveSeg s;
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c) s.p[c] = as_f4(wf.read(c, (uint32_t)who));
                float a, m2, m2r;
                const sgpu::CurveRay ray = sgpu::curve_ray(ro, rd, a);
                sgpu::curve_bounds(s, m2, m2r);
                const float h = 1.0f / sgpu::kCurvePieces;
                const int k = (int)(wl & 15u);
                f3 A, B;
                float ra, rb;
                sgpu::curve_eval(s, (float)k * h, A, ra);
                sgpu::curve_eval(s, (float)(k + 1) * h, B, rb);
                candidate = sgpu::curve_piece_candidate(ray, a, A, ra, B, rb, sgpu::curve_deviation(m2, m2r), rnear, rbest);
            }
            const unsigned long long cand = __ballot(candidate);
            const uint32_t rank = (uint32_t)__popcll(waiting & below);
            if (step == kPieces && rank < 4) {
                pieces = (uint32_t)(cand >> (16 * rank)) & 0xFFFFu;
                seg_t = best;
                seg_found = false;
                if (pieces) step = kSearch;
                else proceed();
            }
        } else {
            // ---- node visits and segments' capsules ----
            const bool visit = step == kVisit, segment = step == kSegment;
            wf.fetch<MULTI>(visit ? node : segment ? seg : -1, rw);
            if (segment) {
                if (STATS) ++cnt_segs;
                sgpu::CurveSeg s;
                points(s);
                float a, m2, m2r;
                const sgpu::CurveRay ray = sgpu::curve_ray(o, d, a);
                sgpu::curve_bounds(s, m2, m2r);
                if (sgpu::curve_start(s, ray, a, m2, m2r, tnear, best)) step = kPieces;
                else proceed();
            }
            if (visit) {
                if (STATS) ++cnt_nodes;
                const sgpu::WideHits h =
                    sgpu::wide_boxes<ANY>(wf.read(0), wf.read(1), wf.read(2), wf.read(3), inv, oinv, tnear, best);
                pmask = h.leaves;
                pfirst = (uint32_t)node + 1;
                pbase = h.leaf_base;
                if (h.list) {
                    if (glist) push(gbase, glist);
                    gbase = h.base;
                    glist = h.list;
                }
                proceed();
            }
        }
    }
    if (STATS) {
        atomicAdd(&stats[0], cnt_nodes);
        atomicAdd(&stats[1], cnt_segs);
    }
}

}  // namespace

int sgpu_curve_launch(sgpu_context ctx, const TraceScene& scene, const uint32_t* inst_ids, uint32_t stack_words,
                      const TraceScene* table, const uint32_t* ray_scene, const sgpu_rays_soa* rays,
                      const sgpu_hits_soa* hits, uint32_t* occluded, uint32_t n, bool any_hit, const uint32_t* n_ptr,
                      uint32_t* comp_out, uint32_t* overflow, hipStream_t stream, uint32_t* spill,
                      uint32_t max_blocks, uint64_t* stats)
{
    if (n == 0) return SGPU_OK;
    sgpu_hits_soa h = {};
    if (hits) h = *hits;
    // as many blocks as are resident at once (4 waves per SIMD); what is past them comes from the counter
    const uint32_t needed = (n + kCurveBlock - 1) / kCurveBlock;
    uint32_t blocks = std::min(needed, kCurveWaves * (uint32_t)ctx->props.multiProcessorCount);
    if (max_blocks) blocks = std::min(blocks, max_blocks);  // a lent buffer's
    uint32_t* buf = spill;
    if (!buf && (blocks < needed || stack_words > SGPU_STACK_LDS))
        SGPU_HIP_TRY(sgpu_device_malloc_async((void**)&buf,
                                    sgpu_trace_spill_words(stack_words, (size_t)blocks * kCurveBlock) * sizeof(uint32_t),
                                    stream));
    if (blocks < needed) sgpu_trace_work_zero(buf, stream);
    const dim3 g(blocks), b(kCurveBlock);
    const bool multi = table != nullptr;
    unsigned long long* st = (unsigned long long*)stats;
#define SGPU_LAUNCH_C(A, M, S)                                                                                      \
    hipLaunchKernelGGL((k_curves<A, M, S>), g, b, 0, stream, scene, inst_ids, table, ray_scene, *rays, h, occluded, \
                       n, n_ptr, buf, buf ? (uint2*)(buf + kTraceWorkWords) : nullptr,                              \
                       std::max(stack_words / 2, kWideStackLds), comp_out, overflow, st)
    if (st) {  // counting: single-scene queries (sgpu_intersect_stats)
        if (any_hit) SGPU_LAUNCH_C(true, false, true);
        else SGPU_LAUNCH_C(false, false, true);
    } else if (any_hit) {
        if (multi) SGPU_LAUNCH_C(true, true, false);
        else SGPU_LAUNCH_C(true, false, false);
    } else {
        if (multi) SGPU_LAUNCH_C(false, true, false);
        else SGPU_LAUNCH_C(false, false, false);
    }
#undef SGPU_LAUNCH_C
    SGPU_HIP_TRY(hipGetLastError());
    if (buf && !spill) SGPU_HIP_TRY(hipFreeAsync(buf, stream));
    return SGPU_OK;
}
