// What the traversals of 8-wide trees share (the triangle and instance traversal, the curve pass): the
// wave's cooperative fetch of 64-byte slots and the box tests of a node.
#pragma once

#include "sgpu_internal.h"

namespace sgpu {

__device__ __forceinline__ float safe_rcp(float x)
{
    float ax = fabsf(x);
    float y = ax < 1e-20f ? copysignf(1e-20f, x) : x;
    return __builtin_amdgcn_rcpf(y);
}

// Compare-exchange of sort keys, ascending.
__device__ __forceinline__ void cswap(int& a, int& b)
{
    const int lo = min(a, b);
    b = max(a, b);
    a = lo;
}

// A wave's fetch of at most one 64-byte slot per lane: lane l asks for 16 bytes of the slot of lane
// 16 k + l / 4 in the k-th of four loads, straight into LDS, and each lane reads its own slot from
// there. A divergent 16-byte load costs the address unit two cycles a lane whatever it hits; read lane
// by lane (5 loads a node, 3 a triangle) the traversal workload kept that unit busy 84 % of the time.
// The 16-byte pieces of a slot are permuted by bits 2-3 of its lane, so that the reads' banks differ.
struct WaveFetch {
    uint4* slots;          // the wave's 4 KB of LDS
    uint32_t lane, piece;  // this lane of the wave and the piece of a slot it asks for

    __device__ __forceinline__ WaveFetch(uint4* block_slots)
    {
        lane = threadIdx.x & 63u;
        slots = block_slots + 4 * 64 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        piece = (lane & 3u) ^ ((lane >> 4) & 3u);
    }

    // Every lane of the wave calls it: lane's slot `ask` (none: -1) of the array at `base` (per lane, or
    // one for the wave).
    template <bool PER_LANE>
    __device__ __forceinline__ void fetch(int ask, const void* base) const
    {
        const unsigned long long at = (unsigned long long)base;
        unsigned long long from[4];
        int s[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int src = 4 * (16 * k + (int)(lane >> 2));
            s[k] = __builtin_amdgcn_ds_bpermute(src, ask);
            from[k] = at;
            if (PER_LANE)
                from[k] = (unsigned long long)(uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)(uint32_t)at) |
                          (unsigned long long)(uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)(uint32_t)(at >> 32)) << 32;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (s[k] >= 0)
                __builtin_amdgcn_global_load_lds(
                    (const __attribute__((address_space(1))) uint32_t*)(from[k] + (unsigned long long)(uint32_t)s[k] * kSlotBytes + 16 * piece),
                    (__attribute__((address_space(3))) uint32_t*)(slots + 64 * k), 16, 0, 0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }

    // Piece c of the slot last fetched for lane `of`.
    __device__ __forceinline__ uint4 read(uint32_t c, uint32_t of) const { return slots[4 * of + (c ^ ((of >> 2) & 3u))]; }
    __device__ __forceinline__ uint4 read(uint32_t c) const { return read(c, lane); }
};

// The children of a node that a ray enters: `list` the internal ones (their slots are base + 2 c;
// closest hit: 4 bits each, c | 8, by entry distance from the lowest up; any hit: a mask), `leaves` a
// mask of the leaf children (leaf 0 in the slot after the node's, leaf k >= 1 at leaf_base + k).
struct WideHits {
    uint32_t base, list, leaf_base, leaves;
};

// The 8 quantized child boxes (WideNode's first slot in w0..w3) against a ray (inv = 1 / d, oinv =
// o / d) over [tnear, best], near and far planes picked by the direction's signs, each plane one fused
// multiply-add t = q (2^e / d) + (origin - o) / d.
template <bool ANY>
__device__ __forceinline__ WideHits wide_boxes(uint4 w0, uint4 w1, uint4 w2, uint4 w3, f3 inv, f3 oinv, float tnear,
                                               float best)
{
    const uint32_t meta = w0.w;
    const uint32_t ni = (meta >> 24) & 15u, nch = meta >> 28;
    // per axis: slope a (per quantization step) and intercept b of the planes' distances
    const float ax = __builtin_amdgcn_ldexpf(inv.x, (int)(meta << 24) >> 24);
    const float ay = __builtin_amdgcn_ldexpf(inv.y, (int)(meta << 16) >> 24);
    const float az = __builtin_amdgcn_ldexpf(inv.z, (int)(meta << 8) >> 24);
    const float bx = fmaf(__uint_as_float(w0.x & kOriginMask), inv.x, -oinv.x);
    const float by = fmaf(__uint_as_float(w0.y & kOriginMask), inv.y, -oinv.y);
    const float bz = fmaf(__uint_as_float(w0.z & kOriginMask), inv.z, -oinv.z);
    const bool sx = __float_as_int(inv.x) < 0, sy = __float_as_int(inv.y) < 0, sz = __float_as_int(inv.z) < 0;
    const uint32_t nx[2] = {sx ? w2.z : w1.x, sx ? w2.w : w1.y}, fx[2] = {sx ? w1.x : w2.z, sx ? w1.y : w2.w};
    const uint32_t ny[2] = {sy ? w3.x : w1.z, sy ? w3.y : w1.w}, fy[2] = {sy ? w1.z : w3.x, sy ? w1.w : w3.y};
    const uint32_t nz[2] = {sz ? w3.z : w2.x, sz ? w3.w : w2.y}, fz[2] = {sz ? w2.x : w3.z, sz ? w2.y : w3.w};
    int key[8];
    uint32_t hit = 0;
#pragma unroll
    for (int c = 7; c >= 0; --c) {
        const int sh = 8 * (c & 3), wi = c >> 2;
        const float t0x = fmaf((float)((nx[wi] >> sh) & 0xFFu), ax, bx);
        const float t0y = fmaf((float)((ny[wi] >> sh) & 0xFFu), ay, by);
        const float t0z = fmaf((float)((nz[wi] >> sh) & 0xFFu), az, bz);
        const float t1x = fmaf((float)((fx[wi] >> sh) & 0xFFu), ax, bx);
        const float t1y = fmaf((float)((fy[wi] >> sh) & 0xFFu), ay, by);
        const float t1z = fmaf((float)((fz[wi] >> sh) & 0xFFu), az, bz);
        const float tmin = fmaxf(fmaxf(t0x, t0y), fmaxf(t0z, tnear));
        const float tmax = fminf(fminf(t1x, t1y), fminf(t1z, best));
        const bool in = tmin <= tmax;
        hit = hit + hit + (in ? 1u : 0u);
        // internal children: entry distance as the sort key, the child's number (and 8) in its low bits
        if (!ANY) key[c] = in && (uint32_t)c < ni ? (__float_as_int(tmin) & ~15) | (8 | c) : 0x7FFFFFF0;
    }
    WideHits r;
    r.base = (w0.x & ~kOriginMask) | (w0.y & ~kOriginMask) << 11 | w0.z << 22;
    r.leaf_base = r.base + 2 * ni - 1;
    r.leaves = __builtin_amdgcn_ubfe(hit, ni, nch - ni);
    if (ANY) {
        r.list = __builtin_amdgcn_ubfe(hit, 0, ni);
    } else {
        // Batcher's odd-even merge sort network for 8 keys
        cswap(key[0], key[1]); cswap(key[2], key[3]); cswap(key[4], key[5]); cswap(key[6], key[7]);
        cswap(key[0], key[2]); cswap(key[1], key[3]); cswap(key[4], key[6]); cswap(key[5], key[7]);
        cswap(key[1], key[2]); cswap(key[5], key[6]);
        cswap(key[0], key[4]); cswap(key[1], key[5]); cswap(key[2], key[6]); cswap(key[3], key[7]);
        cswap(key[2], key[4]); cswap(key[3], key[5]);
        cswap(key[1], key[2]); cswap(key[3], key[4]); cswap(key[5], key[6]);
        // the low 4 bits of each key, the nearest lowest
        r.list = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) r.list = __builtin_amdgcn_alignbit((uint32_t)key[c], r.list, 4);
    }
    return r;
}

// The next internal child of a group (its list not empty): its slot, taken off the list.
template <bool ANY>
__device__ __forceinline__ int wide_take(uint32_t base, uint32_t& list)
{
    int slot;
    if (ANY) {
        slot = (int)(base + 2u * (uint32_t)__builtin_ctz(list));
        list &= list - 1;
    } else {
        slot = (int)(base + 2u * (list & 7u));
        list >>= 4;
    }
    return slot;
}

}  // namespace sgpu
