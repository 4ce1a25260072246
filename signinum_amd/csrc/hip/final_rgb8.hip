// Final stage of 8-bit RGB tiles under 5/3 and RCT (lossless slides), in
// 16-bit packed integers.
//
// A work-group synthesises one 64x64 block of the last level of all three
// components.  Horizontal lifting runs in registers on row pairs (an even and
// an odd row share a dword, so one packed operation lifts both); the lifted
// rows of the three components go through LDS once; vertical lifting, the
// inverse colour transform, level shift, clamp and packing then run in
// registers on 4x4 pixels per thread (two columns share a dword), which leave
// as 12-byte stores.  Values equal the reference's (idwt.rs:741-764, rows then
// columns; mct.rs:71-156) because no sum leaves 16 bits: from inputs of
// magnitude at most M = 2048 a direction of lifting gives at most 2.5 M + 1,
// two give 12,804, and the largest sum of the colour transform is 32,139.
// Code-block samples are bounded by their bit-planes (the host admits K <= 11);
// low-pass samples from lower levels are checked as they are loaded, and a
// block with a larger one is listed for the 32-bit kernel instead.
//
// What bounds it: HBM (int16 bands, int32 low-pass, packed pixels).  About 11
// VALU operations per sample against 38 in the 32-bit kernel, and one barrier a
// block against fifteen: 4096 x 256x256 RGB take 682 us (2.8 GB, 4.1 TB/s)
// against 1377 there.
#include <hip/hip_runtime.h>

#include "../host/plan_types.h"

namespace sgn {

using i16x2 = int16_t __attribute__((ext_vector_type(2)));

constexpr int kRgbRows = kBlk + 4;       // rows a block's vertical lifting reads
constexpr int kRgbPitch = kBlk / 2 + 4;  // dwords of a row in LDS (16-byte aligned)
constexpr uint32_t kRgbMax = 2048;       // inputs in [-kRgbMax, kRgbMax) keep to 16 bits

__device__ __forceinline__ i16x2 as_pk(uint32_t v) { return __builtin_bit_cast(i16x2, v); }
__device__ __forceinline__ uint32_t as_u32(i16x2 v) { return __builtin_bit_cast(uint32_t, v); }
// Low and high halves of a and b: (a.lo, b.lo) and (a.hi, b.hi).
__device__ __forceinline__ uint32_t pk_lo(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_perm(b, a, 0x05040100u);
}
__device__ __forceinline__ uint32_t pk_hi(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_perm(b, a, 0x07060302u);
}
// 5/3 steps on packed samples (idwt.rs:741-764).
__device__ __forceinline__ i16x2 lift_even(i16x2 s, i16x2 a, i16x2 b) {
    return s - ((a + b + (int16_t)2) >> 2);
}
__device__ __forceinline__ i16x2 lift_odd(i16x2 s, i16x2 a, i16x2 b) { return s + ((a + b) >> 1); }

// One component's bands as a block reads them (uniform over the work-group).
struct RgbBands {
    const uint8_t *ll, *hl, *lh, *hh;
    uint32_t pll, phl, plh, phh;  // row pitches in bytes
    int w, h;
    bool ll16;
};

__device__ __forceinline__ RgbBands rgb_bands(const LevelJob *lj, const uint32_t *coef) {
    RgbBands b;
    const uint8_t *base = reinterpret_cast<const uint8_t *>(coef);
    b.ll16 = (lj->narrow & 1u) != 0;
    b.ll = base + ((size_t)lj->band[0] << (b.ll16 ? 1 : 2));
    b.hl = base + ((size_t)lj->band[1] << 1);
    b.lh = base + ((size_t)lj->band[2] << 1);
    b.hh = base + ((size_t)lj->band[3] << 1);
    b.pll = lj->bw[0] << (b.ll16 ? 1 : 2);
    b.phl = lj->bw[1] << 1;
    b.plh = lj->bw[2] << 1;
    b.phh = lj->bw[3] << 1;
    b.w = (int)(lj->x1 - lj->x0);
    b.h = (int)(lj->y1 - lj->y0);
    return b;
}

// What one lane loads of a row pair: eight columns (four low-pass, four
// high-pass samples) of an even and an odd row, and, in the lanes at the
// block's sides, the columns beside it.
struct RgbChunk {
    uint32_t ll[4], lh[2], hl[2], hh[2];
    int32_t xll, xlh, xhl, xhh;
};

// Row pair j of the block (rows oy - 2 + 2 j and the next), columns 8 seg ..
// 8 seg + 7.  x0 and y0 are even: even positions are low-pass.
__device__ __forceinline__ void rgb_load(const RgbBands &b, int ox, int oy, int j, int seg,
                                         RgbChunk &k) {
    const int ye = oy - 2 + 2 * j, yo = ye + 1;
    // whole-sample symmetric extension; rows further out are not read by any
    // output row
    const int re = ye < 0 ? -ye : ye >= b.h ? 2 * (b.h - 1) - ye : ye;
    const int ro = yo < 0 ? -yo : yo >= b.h ? 2 * (b.h - 1) - yo : yo;
    const uint32_t e = (uint32_t)max(re, 0) >> 1, o = (uint32_t)max(ro, 0) >> 1;
    const int wl = (b.w + 1) >> 1, wh = b.w >> 1;
    const int c = (ox >> 1) + 4 * seg;
#pragma unroll
    for (int t = 0; t < 4; ++t) k.ll[t] = 0;
#pragma unroll
    for (int t = 0; t < 2; ++t) k.lh[t] = k.hl[t] = k.hh[t] = 0;
    k.xll = k.xlh = k.xhl = k.xhh = 0;
    const uint8_t *ll = b.ll + (size_t)e * b.pll, *hl = b.hl + (size_t)e * b.phl;
    const uint8_t *lh = b.lh + (size_t)o * b.plh, *hh = b.hh + (size_t)o * b.phh;
    if (c < wl) {
        if (b.ll16) {
            const uint2 v = *reinterpret_cast<const uint2 *>(ll + 2 * c);
            k.ll[0] = (uint32_t)((int32_t)(v.x << 16) >> 16);
            k.ll[1] = (uint32_t)((int32_t)v.x >> 16);
            k.ll[2] = (uint32_t)((int32_t)(v.y << 16) >> 16);
            k.ll[3] = (uint32_t)((int32_t)v.y >> 16);
        } else {
            const uint4 v = *reinterpret_cast<const uint4 *>(ll + 4 * c);
            k.ll[0] = v.x, k.ll[1] = v.y, k.ll[2] = v.z, k.ll[3] = v.w;
        }
        const uint2 v = *reinterpret_cast<const uint2 *>(lh + 2 * c);
        k.lh[0] = v.x, k.lh[1] = v.y;
    }
    if (c < wh) {
        const uint2 u = *reinterpret_cast<const uint2 *>(hl + 2 * c);
        const uint2 v = *reinterpret_cast<const uint2 *>(hh + 2 * c);
        k.hl[0] = u.x, k.hl[1] = u.y;
        k.hh[0] = v.x, k.hh[1] = v.y;
    }
    if (seg == 0 || seg == 7) {
        const int x = seg ? c + 4 : c - 1;  // column beside the block
        if (x >= 0 && x < wh) {
            k.xhl = *reinterpret_cast<const int16_t *>(hl + 2 * x);
            k.xhh = *reinterpret_cast<const int16_t *>(hh + 2 * x);
        }
        if (seg && x < wl) {
            k.xll = b.ll16 ? (int32_t)*reinterpret_cast<const int16_t *>(ll + 2 * x)
                           : *reinterpret_cast<const int32_t *>(ll + 4 * x);
            k.xlh = *reinterpret_cast<const int16_t *>(lh + 2 * x);
        }
    }
}

// Horizontal lifting of the chunk's row pair into rows 2 j and 2 j + 1 of the
// LDS tile.  Called by whole groups of eight lanes (a row pair's segments).
// Sets bits above kRgbMax's in `over` for a low-pass sample out of range.
__device__ __forceinline__ void rgb_rows(const RgbBands &b, int ox, int j, int seg, RgbChunk &k,
                                         uint32_t *tile, uint32_t &over) {
    const int wl = (b.w + 1) >> 1, wh = b.w >> 1;
    const int c = (ox >> 1) + 4 * seg;
    const bool edge = ox + kBlk >= b.w;  // the level's last column is in or beside the block
    if (edge) {
        // columns past the level's end: whatever the row's padding holds
#pragma unroll
        for (int t = 0; t < 4; ++t) k.ll[t] = c + t < wl ? k.ll[t] : 0u;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) over |= k.ll[t] + kRgbMax;
    over |= (uint32_t)k.xll + kRgbMax;
    // (even row, odd row) of each column
    i16x2 s[4], h[4];
    s[0] = as_pk(pk_lo(k.ll[0], k.lh[0]));
    s[1] = as_pk(__builtin_amdgcn_perm(k.lh[0], k.ll[1], 0x07060100u));
    s[2] = as_pk(pk_lo(k.ll[2], k.lh[1]));
    s[3] = as_pk(__builtin_amdgcn_perm(k.lh[1], k.ll[3], 0x07060100u));
    h[0] = as_pk(pk_lo(k.hl[0], k.hh[0]));
    h[1] = as_pk(pk_hi(k.hl[0], k.hh[0]));
    h[2] = as_pk(pk_lo(k.hl[1], k.hh[1]));
    h[3] = as_pk(pk_hi(k.hl[1], k.hh[1]));
    const uint32_t xh = pk_lo((uint32_t)k.xhl, (uint32_t)k.xhh);
    // the high-pass column to the left: the lane before, or the block before,
    // or (mirrored) the first one
    const uint32_t from_left =
        (uint32_t)__builtin_amdgcn_update_dpp(0, (int)as_u32(h[3]), 0x111, 0xF, 0xF, true);
    i16x2 hm = as_pk(seg ? from_left : c ? xh : as_u32(h[0]));
    if (edge) {
        // odd width: the column past the last high-pass one mirrors it
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (c + t == wh) h[t] = t ? h[t - 1] : hm;
    }
    i16x2 e[5];
    e[0] = lift_even(s[0], hm, h[0]);
#pragma unroll
    for (int t = 1; t < 4; ++t) e[t] = lift_even(s[t], h[t - 1], h[t]);
    if (edge) {
        // even width: the even column past the end mirrors the last one
        const uint32_t em =
            (uint32_t)__builtin_amdgcn_update_dpp(0, (int)as_u32(e[3]), 0x111, 0xF, 0xF, true);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (c + t == wl) e[t] = t ? e[t - 1] : as_pk(em);
    }
    // the even column to the right: the lane after, or computed from the block
    // after (whose first high-pass column may lie past the end), or the last
    const uint32_t from_right =
        (uint32_t)__builtin_amdgcn_update_dpp(0, (int)as_u32(e[0]), 0x101, 0xF, 0xF, true);
    const i16x2 hx = c + 4 < wh ? as_pk(xh) : h[3];
    const i16x2 ex = c + 4 < wl
                         ? lift_even(as_pk(pk_lo((uint32_t)k.xll, (uint32_t)k.xlh)), h[3], hx)
                         : e[3];
    e[4] = seg == 7 ? ex : as_pk(from_right);
    i16x2 o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] = lift_odd(h[t], e[t], e[t + 1]);
    // columns 2 t, 2 t + 1 of each row
    uint4 r0, r1;
    r0.x = pk_lo(as_u32(e[0]), as_u32(o[0]));
    r0.y = pk_lo(as_u32(e[1]), as_u32(o[1]));
    r0.z = pk_lo(as_u32(e[2]), as_u32(o[2]));
    r0.w = pk_lo(as_u32(e[3]), as_u32(o[3]));
    r1.x = pk_hi(as_u32(e[0]), as_u32(o[0]));
    r1.y = pk_hi(as_u32(e[1]), as_u32(o[1]));
    r1.z = pk_hi(as_u32(e[2]), as_u32(o[2]));
    r1.w = pk_hi(as_u32(e[3]), as_u32(o[3]));
    uint4 *d = reinterpret_cast<uint4 *>(tile + 2 * j * kRgbPitch + 4 * seg);
    d[0] = r0;
    d[kRgbPitch / 4] = r1;
}

// One 64x64 block per work-group: block list[i] of the plan's final blocks.
// Blocks with a low-pass sample out of range write nothing and append
// themselves to `redo` (count in *redo_n).
extern "C" __global__ void __launch_bounds__(kIdwtThreads)
sgn_final_rgb8(const FinalJob *jobs, const uint32_t *list, const uint32_t *block_job,
               const LevelJob *lv, const uint32_t *coef, uint32_t *redo, uint32_t *redo_n) {
    __shared__ __attribute__((aligned(16))) uint32_t s_rows[3][kRgbRows * kRgbPitch];
    const uint32_t blk = list[xcd_remap(blockIdx.x, gridDim.x)];
    const FinalJob *fj = jobs + block_job[blk];
    const uint32_t local = blk - fj->block_base, nbx = fj->nbx;
    const int ox = (int)(fj->bx0 + local % nbx) * kBlk, oy = (int)(fj->by0 + local / nbx) * kBlk;
    const int tid = threadIdx.x, seg = tid & 7;
    const RgbBands B[3] = {rgb_bands(lv + fj->level[0], coef), rgb_bands(lv + fj->level[1], coef),
                           rgb_bands(lv + fj->level[2], coef)};
    const int w = B[0].w, h = B[0].h;
    uint32_t over = 0;
    {
        // row pairs 0..31 of the three components, loads first
        RgbChunk k[3];
        const int j = tid >> 3;
        const bool need = oy - 2 + 2 * j <= h + 1;
        if (need) {
#pragma unroll
            for (int c = 0; c < 3; ++c) rgb_load(B[c], ox, oy, j, seg, k[c]);
#pragma unroll
            for (int c = 0; c < 3; ++c) rgb_rows(B[c], ox, j, seg, k[c], s_rows[c], over);
        }
    }
    if (tid < 64 && oy + 62 <= h + 1) {
        // row pairs 32 and 33 (the first wave; lanes 48.. idle)
        const int c = min(tid >> 4, 2), j = 32 + ((tid >> 3) & 1);
        const RgbBands b = c == 0 ? B[0] : c == 1 ? B[1] : B[2];
        if (tid < 48) {
            RgbChunk k;
            rgb_load(b, ox, oy, j, seg, k);
            rgb_rows(b, ox, j, seg, k, s_rows[c], over);
        }
    }
    // a sample out of range sets bit 12 or above after the bias
    if (__syncthreads_or((int)(over >> 12))) {
        if (tid == 0) redo[atomicAdd(redo_n, 1u)] = blk;
        return;
    }
    // columns 4 g .. 4 g + 3, rows 4 r .. 4 r + 3 of the block
    const int g = tid & 15, r = tid >> 4;
    const int x = ox + 4 * g, y = oy + 4 * r;
    if (x >= w || y >= h) return;
    i16x2 v[3][4][2];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const uint32_t *t = s_rows[c] + (4 * r + 1) * kRgbPitch + 2 * g;
        i16x2 a[7][2];
#pragma unroll
        for (int q = 0; q < 7; ++q) {
            const uint2 u = *reinterpret_cast<const uint2 *>(t + q * kRgbPitch);
            a[q][0] = as_pk(u.x);
            a[q][1] = as_pk(u.y);
        }
        // tile rows 4 r + 1 .. 4 r + 7; outputs are rows 4 r + 2 .. 4 r + 5
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const i16x2 e0 = lift_even(a[1][d], a[0][d], a[2][d]);
            const i16x2 e1 = lift_even(a[3][d], a[2][d], a[4][d]);
            const i16x2 e2 = lift_even(a[5][d], a[4][d], a[6][d]);
            v[c][0][d] = e0;
            v[c][1][d] = lift_odd(a[2][d], e0, e1);
            v[c][2][d] = e1;
            v[c][3][d] = lift_odd(a[4][d], e1, e2);
        }
    }
    uint8_t *const dst = reinterpret_cast<uint8_t *>(fj->dst) + (size_t)y * fj->pitch + (size_t)x * 3;
    const bool words = ((fj->dst | fj->pitch) & 3u) == 0 && x + 4 <= w;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (y + q >= h) break;
        // G = Y - ((Cb + Cr) >> 2), R = Cr + G, B = Cb + G, each plus 128
        uint32_t p[2][3];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const i16x2 gg = v[0][q][d] - ((v[1][q][d] + v[2][q][d]) >> 2) + (int16_t)128;
            const i16x2 rr = v[2][q][d] + gg, bb = v[1][q][d] + gg;
            auto clamp = [](i16x2 s) -> uint32_t {
                const i16x2 z = {0, 0}, m = {255, 255};
                return as_u32(__builtin_elementwise_min(__builtin_elementwise_max(s, z), m));
            };
            p[d][0] = clamp(rr);
            p[d][1] = clamp(gg);
            p[d][2] = clamp(bb);
        }
        // bytes r0 g0 b0 r1 | g1 b1 r2 g2 | b2 r3 g3 b3
        const uint32_t rg0 = p[0][0] | (p[0][1] << 8), rg1 = p[1][0] | (p[1][1] << 8);
        const uint32_t w0 = __builtin_amdgcn_perm(rg0, p[0][2], 0x06000504u);
        const uint32_t t0 = __builtin_amdgcn_perm(rg0, p[0][2], 0x0C0C0207u);  // g1 b1
        const uint32_t w1 = (t0 & 0xFFFFu) | (rg1 << 16);
        const uint32_t w2 = __builtin_amdgcn_perm(rg1, p[1][2], 0x02070600u);
        uint8_t *o = dst + (size_t)q * fj->pitch;
        if (words) {
            uint32_t *ow = reinterpret_cast<uint32_t *>(o);
            ow[0] = w0;
            ow[1] = w1;
            ow[2] = w2;
        } else {
            const int n = min(4, w - x) * 3;
#pragma unroll
            for (int t = 0; t < 12; ++t)
                if (t < n) o[t] = (uint8_t)((t < 4 ? w0 : t < 8 ? w1 : w2) >> (8 * (t & 3)));
        }
    }
}

}  // namespace sgn
