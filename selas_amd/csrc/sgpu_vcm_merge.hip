// Vertex merging (the camera side of VCM's photon range search), in a translation unit of its own.
// Built with correctly rounded division and square root like the rest of the path (a build with fast
// ones held more registers and ran no faster).
#include "sgpu_vcm_common.h"

namespace sgpu_vcm {

namespace {

// What the photons of a query are found and evaluated with, in LDS: its BSDF for the view direction, the
// camera vertex's MIS terms, the slice's constants, position and squared radius. 68 words, so that the
// queries of a wave, read at once, lie in different banks.
struct alignas(16) QueryView {
    DisneyView q;
    float dvcm, dvm, ccp, vc_weight;
    uint32_t plen, max_len, transparent;
    const float* materials;
    const uint32_t* geom_material;
    float pos[3], radius_sq;
};
static_assert(sizeof(QueryView) == 68 * 4, "a query's view takes 68 words");

// The photon ranges of a query's 2x2x2 cells as one list: entry i lies in the first cell k with i <
// end[k] and is photon i + base[k] (mod 2^32).
struct QueryCells {
    uint32_t end[8], base[8];
};

// Vertex merging (SearchHashGrid + MergeVertices, VCMHashGrid.cpp:107-157, VCM.cpp:362-409). A wave takes
// the queries of a bounce up to kBatch at a time, grid-stride: a lane each prepares its BSDF and constants in
// LDS, eight lanes each look up its cells. Then the wave's groups of GW lanes take a query each, round by
// round: the lanes of a group scan the photons of its cells as one list (the cells' ranges in the
// reference's visiting order, strided over the lanes) and append those within the radius to the group's
// LDS queue (ballot and prefix count, queue order = scan order). Once the wave's groups have 64 photons
// queued between them (or nothing more to scan) the wave evaluates the camera BSDF for up to 64, one per
// lane, whichever of the round's queries they belong to, and each group adds its photons' contributions
// in queue order, strided over its lanes; a fixed butterfly over the group's lanes gives the query's sum.
//
// A query has about 14 photons within the radius and 92 in its cells on the 1M-triangle workload. With
// the query's values in every lane's registers and each group evaluating its own photons (168 VGPRs, 3
// waves per SIMD, passes half empty, a query's preparation run by 4 queries at a time) the 512 x 512 x 32
// job's merging took 15.3 ms; the values in LDS (5 waves) 11.0, photons of all groups in one pass 10.6,
// preparation in batches 8.8 (16 lanes a group; 9.0 with 8, 10.7 with 32). Bound by vector instructions.
// A batch is as many rounds as it takes for the waves that are resident to hold every query: full batches
// on a part of the chip took longer than the smaller preparation gains (the merges of a 64 x 64 image of
// one iteration, ten launches: 90 us, 140 with full batches, 83 before the pooling; 128 x 128 x 4 161, 241
// and 175; 256 x 256 x 8 494, 580 and 762; with 32 lanes a group 87, 170, 79; 181, 325, 221; 652, 845,
// 1215). With `order` (the
// queries of the bounce in spatial order) blocks are numbered xcd-major, so that the queries running at
// once on one XCD are neighbours in space and read the same photon cells through that XCD's L2.
template <uint32_t GW>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kMergeWavesPerSimd))) void k_cam_merge(Wave w, const uint32_t* __restrict count_ptr,
                                                      const uint32_t* __restrict order,
                                                      const CamVertex* __restrict cam_vm,
                                                      const uint32_t* __restrict path_slice, GridView G, CamSlots S,
                                                      uint32_t resident, unsigned long long* __restrict mstat)
{
    static_assert(GW == 8 || GW == 16 || GW == 32, "a group divides the wave");
    constexpr uint32_t kQ = 64 / GW;                   // groups of a wave
    constexpr uint32_t kBatch = GW == 8 ? 8 : 16;      // (8 and 16: LDS for 5 waves per SIMD)
    constexpr uint32_t kQueue = 64 + GW;               // fewer than 64 queued before a scan step adds at most GW
    const uint32_t count = *count_ptr;
    __shared__ QueryView view_lds[kMergeWaves][kBatch];
    __shared__ QueryCells cell_lds[kMergeWaves][kBatch];
    __shared__ uint32_t list_lds[kMergeWaves][kQ][kQueue];
    __shared__ float sum_lds[kMergeWaves][3][64];
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    const uint32_t grp = lane / GW, gl = lane % GW;  // group and lane within it
    uint32_t* list = list_lds[wid][grp];
    const unsigned long long below = (1ull << lane) - 1ull;
    const unsigned long long group_bits = ((1ull << GW) - 1ull) << (grp * GW);
    if (*G.nv_ptr == 0) return;
    const uint32_t waves = min(gridDim.x * kMergeWaves, resident);
    const uint32_t batch = min(kBatch, kQ * max(1u, (count + kQ * waves - 1) / (kQ * waves)));
    const uint32_t stride = batch * gridDim.x * kMergeWaves;
    const uint32_t block = order ? xcd_major_block(blockIdx.x, gridDim.x) : blockIdx.x;
    // work counters of this wave, flushed at the end
    __shared__ uint32_t cnt_lds[kMergeWaves][4];
    if (mstat && lane < 4) cnt_lds[wid][lane] = 0;
    __builtin_amdgcn_wave_barrier();

    // The contribution of photon q to query qv (zero where it has none).
    auto merge = [&](const QueryView& qv, uint32_t q) -> f3 {
        // the query's values are read from LDS for each evaluation, not held in registers over the loop
        asm volatile("" ::: "memory");
        const LightVertex& lv = G.sverts[q];
        const uint32_t lgp = lv.geom_plen;
        if (qv.plen + (lgp & 31u) > qv.max_len) return mk3(0, 0, 0);
        const float* lmat = qv.materials + 22 * (size_t)qv.geom_material[lgp >> 5];
        // the reference's transparency rule (VCM.cpp:381-383)
        if (qv.transparent != ((uint32_t)lmat[21] & kMatTransparent)) return mk3(0, 0, 0);
        f3 lw = mk3(lv.wfix[0], lv.wfix[1], lv.wfix[2]);
        // a photon arriving in the surface's plane is not evaluated (measure zero; 0/0 below)
        const float nl = dot3(qv.q.n, lw);
        if (nl == 0.0f) return mk3(0, 0, 0);
        float fwd, rev;
        f3 f = bsdf_eval_view(qv.q, lw, fwd, rev);
        if (is_zero3(f)) return mk3(0, 0, 0);
        float cos_l = absf_(nl);
        fwd *= qv.ccp;
        rev *= lv.cp;
        float w_light = lv.dvcm * qv.vc_weight + lv.dvm * fwd;
        float w_cam = qv.dvcm * qv.vc_weight + qv.dvm * rev;
        float mis = 1.0f / (w_light + 1.0f + w_cam);
        return (f * mk3(lv.thr[0], lv.thr[1], lv.thr[2])) * (mis / cos_l);
    };

    for (uint32_t j0 = batch * (block * kMergeWaves + wid); j0 < count; j0 += stride) {
        // ---- the batch's queries, a lane each (none past the end, or without a query, or outside the box) ----
        const uint32_t jj = j0 + lane;
        const bool in_batch = lane < batch && jj < count;
        const uint32_t j = order && in_batch ? order[jj] : jj;
        bool active = false;
        uint32_t si = 0, cell_base = 0, cell_count = 1;
        int32_t mn[3] = {0, 0, 0};
        if (in_batch) {
            const CamVertex v = cam_vm[j];
            active = v.geom_plen != kNoQuery;
            if (active) {
                si = path_slice[v.path];
                const Slice& sl = w.slices[si];
                const uint32_t* box = G.box + 8 * si;
                for (int k = 0; k < 3; ++k) {
                    const float dmin = v.pos[k] - ord2f(box[k]);
                    const float dmax = ord2f(~box[3 + k]) - v.pos[k];
                    if (dmin < 0.0f || dmax < 0.0f) active = false;
                    const float cp = sl.inv_cell * dmin;
                    const float cf = floorf(cp);
                    mn[k] = (int32_t)cf;
                    if (cp - cf < 0.5f) --mn[k];
                }
            }
            if (active) {
                const Slice& sl = w.slices[si];
                cell_base = sl.path_base;
                cell_count = sl.N;
                const uint32_t geom = v.geom_plen >> 5;
                const f3 view = mk3(v.view[0], v.view[1], v.view[2]);
                Surface s;
                s.position = mk3(v.pos[0], v.pos[1], v.pos[2]);
                s.error = 0.0f;
                surface_material(sl.materials + 22 * (size_t)sl.geom_material[geom], mk3(v.n[0], v.n[1], v.n[2]), view, s);
                if (geom_has_tangents(sl, geom)) tangent_frame(s.n, w.cam_tan[j], s);
                s.base_color = mk3(v.base[0], v.base[1], v.base[2]);
                QueryView& qv = view_lds[wid][lane];
                qv.dvcm = v.dvcm;
                qv.dvm = v.dvm;
                qv.ccp = cont_prob(s);
                qv.vc_weight = sl.vc_weight;
                qv.plen = v.geom_plen & 31u;
                qv.max_len = sl.L;
                qv.transparent = s.flags & kMatTransparent;
                qv.materials = sl.materials;
                qv.geom_material = sl.geom_material;
                for (int k = 0; k < 3; ++k) qv.pos[k] = v.pos[k];
                qv.radius_sq = sl.radius_sq;
                bsdf_view(s, view, qv.q);
            }
        }
        const unsigned long long actives = __ballot(active);
        if (mstat && lane == 0) {
            atomicAdd(&cnt_lds[wid][0], min(batch, count - j0));
            atomicAdd(&cnt_lds[wid][1], (uint32_t)__popcll(actives));
        }
        if (actives == 0) continue;
        // ---- their cells, eight lanes a query: cell k = (x, y, z) bits of k, its photon range ----
#pragma unroll
        for (uint32_t part = 0; part < kBatch / 8; ++part) {
            const uint32_t b = 8 * part + (lane >> 3), k = lane & 7u;
            const int32_t cx = __shfl(mn[0], (int)b, 64) + (int32_t)(k & 1u);
            const int32_t cy = __shfl(mn[1], (int)b, 64) + (int32_t)((k >> 1) & 1u);
            const int32_t cz = __shfl(mn[2], (int)b, 64) + (int32_t)(k >> 2);
            const uint32_t cells = (uint32_t)__shfl((int)cell_count, (int)b, 64);
            const uint32_t cell0 = (uint32_t)__shfl((int)cell_base, (int)b, 64);
            uint32_t cb = 0, cn = 0;
            if ((actives >> b) & 1ull) {
                const uint32_t cell = cell0 + cell_hash(cx, cy, cz, cells);
                cb = cell == 0 ? 0 : G.cell_ends[cell - 1];
                cn = G.cell_ends[cell] - cb;
            }
            uint32_t incl = cn;
            for (uint32_t d = 1; d < 8; d <<= 1) {
                const uint32_t y = (uint32_t)__shfl_up((int)incl, d, 8);
                if (k >= d) incl += y;
            }
            cell_lds[wid][b].end[k] = incl;
            cell_lds[wid][b].base[k] = cb - (incl - cn);
        }
        __builtin_amdgcn_wave_barrier();

        for (uint32_t round = 0; round < batch / kQ; ++round) {
            const uint32_t b = round * kQ + grp;  // this group's query
            const QueryCells& cells = cell_lds[wid][b];
            const QueryView& mine = view_lds[wid][b];
            uint32_t ends[8];
            for (int k = 0; k < 8; ++k) ends[k] = cells.end[k];
            const uint32_t total = ends[7];  // 0 for a group without a query
            const f3 x = mk3(mine.pos[0], mine.pos[1], mine.pos[2]);
            const float radius_sq = mine.radius_sq;
            f3 acc = mk3(0, 0, 0);
            uint32_t head = 0, listed = 0;  // the group's queue; same in every lane of the group
            uint32_t n_near = 0;            // photons within the radius (counted only for mstat)
            for (uint32_t c0 = 0;; c0 += GW) {
                const bool more = __ballot(c0 < total) != 0;
                if (more) {
                    const uint32_t i = c0 + gl;
                    bool near = false;
                    uint32_t q = 0;
                    if (i < total) {
                        uint32_t k = 0;
                        for (int m = 0; m < 7; ++m) k += i >= ends[m] ? 1u : 0u;
                        q = i + cells.base[k];
                        const float4 lp = G.spos[q];
                        const f3 dv = x - mk3(lp.x, lp.y, lp.z);
                        near = dot3(dv, dv) <= radius_sq;
                    }
                    const unsigned long long m = __ballot(near) & group_bits;
                    uint32_t at = head + listed + (uint32_t)__popcll(m & below);
                    at = at >= kQueue ? at - kQueue : at;
                    if (near) list[at] = q;
                    listed += (uint32_t)__popcll(m);
                    n_near += (uint32_t)__popcll(m);
                    __builtin_amdgcn_wave_barrier();
                }
                // the queues end to end: where this group's begins, and this lane's photon: its group and place
                uint32_t all = 0, first = 0, of = 0, at = lane;
#pragma unroll
                for (uint32_t g = 0; g < kQ; ++g) {
                    const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)listed, (int)(g * GW));
                    if (g < grp) first += n;
                    if (lane >= all) {
                        of = g;
                        at = lane - all;
                    }
                    all += n;
                }
                if (all >= 64 || (!more && all > 0)) {
                    at += (uint32_t)__shfl((int)head, (int)(of * GW), 64);
                    at = at >= kQueue ? at - kQueue : at;
                    f3 c = mk3(0, 0, 0);
                    if (lane < all) c = merge(view_lds[wid][round * kQ + of], list_lds[wid][of][at]);
                    sum_lds[wid][0][lane] = c.x;
                    sum_lds[wid][1][lane] = c.y;
                    sum_lds[wid][2][lane] = c.z;
                    __builtin_amdgcn_wave_barrier();
                    const uint32_t taken = first < 64 ? min(listed, 64 - first) : 0;
                    for (uint32_t e = gl; e < taken; e += GW)
                        acc += mk3(sum_lds[wid][0][first + e], sum_lds[wid][1][first + e], sum_lds[wid][2][first + e]);
                    __builtin_amdgcn_wave_barrier();
                    head += taken;
                    head = head >= kQueue ? head - kQueue : head;
                    listed -= taken;
                }
                if (!more) break;
            }
            for (uint32_t off = 1; off < GW; off <<= 1) {
                acc.x += __shfl_xor(acc.x, off, GW);
                acc.y += __shfl_xor(acc.y, off, GW);
                acc.z += __shfl_xor(acc.z, off, GW);
            }
            const uint32_t qj = (uint32_t)__shfl((int)j, (int)b, 64), qsi = (uint32_t)__shfl((int)si, (int)b, 64);
            if (gl == 0 && ((actives >> b) & 1ull)) {
                if (mstat) {
                    atomicAdd(&cnt_lds[wid][2], total);
                    atomicAdd(&cnt_lds[wid][3], n_near);
                }
                const CamVertex& cv = cam_vm[qj];
                const size_t slot = (size_t)cv.path * w.nslots + w.nslots - 1;
                s3(S.c, slot, (mk3(cv.thr[0], cv.thr[1], cv.thr[2]) * acc) * w.slices[qsi].vm_norm);
                S.valid[slot] = 1;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (mstat) {
        __builtin_amdgcn_wave_barrier();
        if (lane < 4 && cnt_lds[wid][lane]) atomicAdd(mstat + lane, (unsigned long long)cnt_lds[wid][lane]);
    }
}

}  // namespace

void launch_cam_merge(uint32_t lanes, uint32_t blocks, hipStream_t stream, const Wave& w, const uint32_t* count_ptr,
                      const uint32_t* order, const CamVertex* cam_vm, const uint32_t* path_slice, const GridView& G,
                      const CamSlots& S, uint32_t resident, unsigned long long* mstat)
{
    if (lanes == 32)
        hipLaunchKernelGGL(k_cam_merge<32>, dim3(blocks), dim3(kBlock), 0, stream, w, count_ptr, order, cam_vm,
                           path_slice, G, S, resident, mstat);
    else if (lanes == 8)
        hipLaunchKernelGGL(k_cam_merge<8>, dim3(blocks), dim3(kBlock), 0, stream, w, count_ptr, order, cam_vm,
                           path_slice, G, S, resident, mstat);
    else
        hipLaunchKernelGGL(k_cam_merge<16>, dim3(blocks), dim3(kBlock), 0, stream, w, count_ptr, order, cam_vm,
                           path_slice, G, S, resident, mstat);
}

}  // namespace sgpu_vcm
