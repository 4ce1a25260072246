// Synthesis of 64x64 blocks whose level has an even origin, sides of at least
// 8 and 16-byte aligned rows: the case of every tile that starts at an even
// position of its image (x0, y0 multiples of 2).
//
// Horizontal lifting runs in registers: a lane holds eight columns (four
// low-pass, four high-pass samples) of an even and an odd row, and takes what
// lies beside them from the neighbouring lane step by step, so nothing is
// computed twice but a few columns at the block's sides.  The lifted rows go
// through LDS once; vertical lifting runs in registers on 4x4 samples per
// thread.  Where the signal ends, the missing neighbour of a step is the
// present one, which is what whole-sample symmetric extension gives at every
// step (idwt.rs:741-835; the same operations in the same order, so the values
// are those of the general kernels in idwt.hip).
#include <hip/hip_runtime.h>

#include "../host/plan_types.h"

namespace sgn {

// REV: 5/3 in integers, else 9/7 in f32.  HI16 / LL16: int16 samples in the
// high-pass bands / the low-pass band (else 32-bit words; the low-pass of a 9/7
// level then holds f32 samples if LLF).
template <bool REV>
struct RowTile {
    static constexpr int H = REV ? 2 : 4;          // rows above and below the block
    static constexpr int kRows = kBlk + 2 * H;
    static constexpr int kPairs = kRows / 2;
    static constexpr int kPitch = kBlk + 4;        // words
    static constexpr int kIn = REV ? 7 : 11;       // inputs of four vertical outputs
    using T = typename Sample<REV>::T;
};

// One level's bands (uniform over the work-group).
struct RowBands {
    const uint8_t *p[4];
    uint32_t pitch[4];  // bytes
    float delta[4];
    int w, h;
};

template <bool HI16, bool LL16>
__device__ __forceinline__ RowBands row_bands(const LevelJob *lj, const uint32_t *coef) {
    RowBands b;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int sh = (k ? HI16 : LL16) ? 1 : 2;
        b.p[k] = reinterpret_cast<const uint8_t *>(coef) + ((size_t)lj->band[k] << sh);
        b.pitch[k] = lj->bw[k] << sh;
        b.delta[k] = lj->delta[k];
    }
    b.w = (int)(lj->x1 - lj->x0);
    b.h = (int)(lj->y1 - lj->y0);
    return b;
}

// What one lane loads of a row pair, as stored (int16: two samples a word):
// four samples of each band, and in the lanes at the block's sides the two
// samples beside them.
struct RowChunk {
    uint32_t v[4][4], x[4][2];
};

// Row pair j of the block (rows oy - H + 2 j and the next), columns 8 seg ..
// 8 seg + 7.
template <bool REV, bool HI16, bool LL16>
__device__ __forceinline__ void row_load(const RowBands &b, int ox, int oy, int j, int seg,
                                         RowChunk &k) {
    const int ye = oy - RowTile<REV>::H + 2 * j, yo = ye + 1;
    // rows further out than one reflection are not read by any output row
    const int re = ye < 0 ? -ye : ye >= b.h ? 2 * (b.h - 1) - ye : ye;
    const int ro = yo < 0 ? -yo : yo >= b.h ? 2 * (b.h - 1) - yo : yo;
    const uint32_t e = (uint32_t)max(re, 0) >> 1, o = (uint32_t)max(ro, 0) >> 1;
    const int wl = (b.w + 1) >> 1, wh = b.w >> 1;
    const int c = (ox >> 1) + 4 * seg, x = seg ? c + 4 : c - 2;
    // columns past the level's end: its first ones instead (their values reach
    // no output inside the level)
    const uint32_t cl = c < wl ? c : 0, ch = c < wh ? c : 0;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const uint8_t *r = b.p[n] + (size_t)(n & 2 ? o : e) * b.pitch[n];
        const uint32_t cc = n & 1 ? ch : cl;
        if (n ? HI16 : LL16) {
            const uint2 t = *reinterpret_cast<const uint2 *>(r + 2 * cc);
            k.v[n][0] = t.x, k.v[n][1] = t.y;
        } else {
            const uint4 t = *reinterpret_cast<const uint4 *>(r + 4 * cc);
            k.v[n][0] = t.x, k.v[n][1] = t.y, k.v[n][2] = t.z, k.v[n][3] = t.w;
        }
    }
    if (seg == 0 || seg == 7) {
        const uint32_t xl = x >= 0 && x < wl ? x : 0, xh = x >= 0 && x < wh ? x : 0;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const uint8_t *r = b.p[n] + (size_t)(n & 2 ? o : e) * b.pitch[n];
            const uint32_t xx = n & 1 ? xh : xl;
            if (n ? HI16 : LL16) {
                k.x[n][0] = *reinterpret_cast<const uint32_t *>(r + 2 * xx);
            } else {
                const uint2 t = *reinterpret_cast<const uint2 *>(r + 4 * xx);
                k.x[n][0] = t.x, k.x[n][1] = t.y;
            }
        }
    }
}

// Samples of a band's words: sign-extended, dequantised and scaled for the
// 9/7 (F.3.8.2: low-pass by kappa, high-pass by its inverse).
template <bool REV, bool NAR, bool ISF, int N>
__device__ __forceinline__ void row_samples(const uint32_t *raw, float delta, float scale,
                                            typename Sample<REV>::T *out) {
#pragma clang fp contract(off)
#pragma unroll
    for (int t = 0; t < N; ++t) {
        int32_t s;
        if constexpr (NAR)
            s = t & 1 ? (int32_t)raw[t >> 1] >> 16 : (int32_t)(raw[t >> 1] << 16) >> 16;
        else
            s = (int32_t)raw[t];
        if constexpr (REV)
            out[t] = s;
        else if constexpr (ISF)
            out[t] = __int_as_float(s) * scale;
        else
            out[t] = ((float)s * delta) * scale;
    }
}

template <int CTRL, typename T>
__device__ __forceinline__ T lane_dpp(T v) {
    const int r = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(T, r);
}

// Horizontal lifting of one row: e and o are the lane's low- and high-pass
// samples (columns c + t of their bands), lo and hi the two columns beside the
// block in its first and last segment.  Called by whole groups of eight lanes.
template <bool REV>
__device__ __forceinline__ void lift_row(typename Sample<REV>::T (&e)[4],
                                         typename Sample<REV>::T (&o)[4],
                                         typename Sample<REV>::T (&lo)[2],
                                         typename Sample<REV>::T (&hi)[2], int seg, int c, int wl,
                                         int wh, bool edge) {
#pragma clang fp contract(off)
    using T = typename Sample<REV>::T;
    const bool first = seg == 0, last = seg == 7;
    // neighbours of e[0] and o[3] (whose value beside the block is `side`)
    auto left = [&](T side) -> T {
        const T v = lane_dpp<0x111>(o[3]);
        if (c == 0) side = o[0];
        return first ? side : v;
    };
    auto right = [&](T side) -> T {
        const T v = lane_dpp<0x101>(e[0]);
        const T n = last ? side : v;
        return edge && c + 4 >= wl ? e[3] : n;
    };
    // the high-pass column past the level's end mirrors the last one, and so
    // does the low-pass column past it
    auto mirror_o = [&](T om) {
        if (!edge) return;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (c + t == wh) o[t] = t ? o[t - 1] : om;
    };
    auto mirror_e = [&]() {
        if (!edge) return;
#pragma unroll
        for (int t = 1; t < 4; ++t)
            if (c + t == wl) e[t] = e[t - 1];
    };
    if constexpr (REV) {
        const T om = left(hi[1]);
        mirror_o(om);
        const T x0 = lo[0] - ((o[3] + (edge && c + 4 >= wh ? o[3] : hi[0]) + 2) >> 2);
        e[0] -= (om + o[0] + 2) >> 2;
#pragma unroll
        for (int t = 1; t < 4; ++t) e[t] -= (o[t - 1] + o[t] + 2) >> 2;
        mirror_e();
        const T e4 = right(x0);
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] += (e[t] + (t < 3 ? e[t + 1] : e4)) >> 1;
    } else {
        T om = left(hi[1]);
        mirror_o(om);
        // beside the block: columns c - 2, c - 1 or c + 4, c + 5
        if (edge && last) {
            if (c + 4 >= wh) hi[0] = o[3];
            if (c + 5 >= wh) hi[1] = hi[0];
        }
        const T x0 = fmaf(o[3] + hi[0], kNegDelta, lo[0]);
        T x1 = fmaf(hi[0] + hi[1], kNegDelta, lo[1]);
        if (edge && last && c + 5 >= wl) x1 = x0;
        e[0] = fmaf(om + o[0], kNegDelta, e[0]);
#pragma unroll
        for (int t = 1; t < 4; ++t) e[t] = fmaf(o[t - 1] + o[t], kNegDelta, e[t]);
        mirror_e();
        T e4 = right(x0);
        // the high-pass column c - 1 or c + 4
        T y = fmaf((first ? e[0] : x0) + x1, kNegGamma, first ? hi[1] : hi[0]);
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] = fmaf(e[t] + (t < 3 ? e[t + 1] : e4), kNegGamma, o[t]);
        om = left(y);
        mirror_o(om);
        if (edge && last && c + 4 >= wh) y = o[3];
        const T z = fmaf(o[3] + y, kNegBeta, x0);
        e[0] = fmaf(om + o[0], kNegBeta, e[0]);
#pragma unroll
        for (int t = 1; t < 4; ++t) e[t] = fmaf(o[t - 1] + o[t], kNegBeta, e[t]);
        mirror_e();
        e4 = right(z);
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] = fmaf(e[t] + (t < 3 ? e[t + 1] : e4), kNegAlpha, o[t]);
    }
}

// Horizontal lifting of the chunk's row pair into rows 2 j and 2 j + 1 of the
// LDS tile.
template <bool REV, bool HI16, bool LL16, bool LLF>
__device__ __forceinline__ void row_lift(const RowBands &b, int ox, int j, int seg,
                                         const RowChunk &k, typename Sample<REV>::T *tile) {
    using T = typename Sample<REV>::T;
    const int wl = (b.w + 1) >> 1, wh = b.w >> 1;
    const int c = (ox >> 1) + 4 * seg;
    const bool edge = ox + kBlk + 4 > b.w;  // the level ends in the block or right beside it
    constexpr float kl = kKappa, kh = 1.0f / kKappa;
    auto one = [&](T (&e)[4], T (&o)[4], T (&lo)[2], T (&hi)[2], int r) {
        lift_row<REV>(e, o, lo, hi, seg, c, wl, wh, edge);
        uint4 *d = reinterpret_cast<uint4 *>(tile + (2 * j + r) * RowTile<REV>::kPitch + 8 * seg);
        d[0] = make_uint4(__builtin_bit_cast(uint32_t, e[0]), __builtin_bit_cast(uint32_t, o[0]),
                          __builtin_bit_cast(uint32_t, e[1]), __builtin_bit_cast(uint32_t, o[1]));
        d[1] = make_uint4(__builtin_bit_cast(uint32_t, e[2]), __builtin_bit_cast(uint32_t, o[2]),
                          __builtin_bit_cast(uint32_t, e[3]), __builtin_bit_cast(uint32_t, o[3]));
    };
    T e[4], o[4], lo[2], hi[2];
    row_samples<REV, LL16, LLF, 4>(k.v[0], b.delta[0], kl, e);
    row_samples<REV, HI16, false, 4>(k.v[1], b.delta[1], kh, o);
    row_samples<REV, LL16, LLF, 2>(k.x[0], b.delta[0], kl, lo);
    row_samples<REV, HI16, false, 2>(k.x[1], b.delta[1], kh, hi);
    one(e, o, lo, hi, 0);
    row_samples<REV, HI16, false, 4>(k.v[2], b.delta[2], kl, e);
    row_samples<REV, HI16, false, 4>(k.v[3], b.delta[3], kh, o);
    row_samples<REV, HI16, false, 2>(k.x[2], b.delta[2], kl, lo);
    row_samples<REV, HI16, false, 2>(k.x[3], b.delta[3], kh, hi);
    one(e, o, lo, hi, 1);
}

// Vertical lifting of columns 4 g .. 4 g + 3, rows 4 r .. 4 r + 3 of the block.
template <bool REV>
__device__ __forceinline__ void col_lift(const typename Sample<REV>::T *tile, int g, int r,
                                         typename Sample<REV>::T (&out)[4][4]) {
#pragma clang fp contract(off)
    using T = typename Sample<REV>::T;
    using R = RowTile<REV>;
    T a[R::kIn][4];
#pragma unroll
    for (int q = 0; q < R::kIn; ++q) {
        const uint4 u =
            *reinterpret_cast<const uint4 *>(tile + (4 * r + 1 + q) * R::kPitch + 4 * g);
        a[q][0] = __builtin_bit_cast(T, u.x);
        a[q][1] = __builtin_bit_cast(T, u.y);
        a[q][2] = __builtin_bit_cast(T, u.z);
        a[q][3] = __builtin_bit_cast(T, u.w);
    }
    // a[0] is an odd row
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        if constexpr (REV) {
#pragma unroll
            for (int q = 1; q < 6; q += 2) a[q][d] -= (a[q - 1][d] + a[q + 1][d] + 2) >> 2;
            a[2][d] += (a[1][d] + a[3][d]) >> 1;
            a[4][d] += (a[3][d] + a[5][d]) >> 1;
#pragma unroll
            for (int q = 0; q < 4; ++q) out[q][d] = a[q + 1][d];
        } else {
            const float kl = kKappa, kh = 1.0f / kKappa;
#pragma unroll
            for (int q = 0; q < 11; ++q) a[q][d] = a[q][d] * (q & 1 ? kl : kh);
#pragma unroll
            for (int q = 1; q < 10; q += 2)
                a[q][d] = fmaf(a[q - 1][d] + a[q + 1][d], kNegDelta, a[q][d]);
#pragma unroll
            for (int q = 2; q < 9; q += 2)
                a[q][d] = fmaf(a[q - 1][d] + a[q + 1][d], kNegGamma, a[q][d]);
#pragma unroll
            for (int q = 3; q < 8; q += 2)
                a[q][d] = fmaf(a[q - 1][d] + a[q + 1][d], kNegBeta, a[q][d]);
#pragma unroll
            for (int q = 4; q < 7; q += 2)
                a[q][d] = fmaf(a[q - 1][d] + a[q + 1][d], kNegAlpha, a[q][d]);
#pragma unroll
            for (int q = 0; q < 4; ++q) out[q][d] = a[q + 3][d];
        }
    }
}

// One 64x64 block of a level below the last into the coefficient arena: 256
// threads, the rows past the 32nd pair by the first wave.
template <bool REV, bool HI16, bool LL16, bool LLF>
__device__ __forceinline__ void level_rows(const LevelJob *lj, uint32_t local, uint32_t *coef,
                                           typename Sample<REV>::T *tile) {
    using R = RowTile<REV>;
    const RowBands b = row_bands<HI16, LL16>(lj, coef);
    const uint32_t nbx = lj->nbx;
    const int ox = (int)(lj->bx0 + local % nbx) * kBlk, oy = (int)(lj->by0 + local / nbx) * kBlk;
    const int tid = threadIdx.x, seg = tid & 7, j = tid >> 3;
    const int rows = b.h + R::H - oy + R::H;  // rows of the tile that outputs read
    RowChunk k{};
    if (2 * j < rows) {
        row_load<REV, HI16, LL16>(b, ox, oy, j, seg, k);
        row_lift<REV, HI16, LL16, LLF>(b, ox, j, seg, k, tile);
    }
    if (tid < 8 * (R::kPairs - 32) && 2 * (32 + j) < rows) {
        row_load<REV, HI16, LL16>(b, ox, oy, 32 + j, seg, k);
        row_lift<REV, HI16, LL16, LLF>(b, ox, 32 + j, seg, k, tile);
    }
    __syncthreads();
    const int g = tid & 15, r = tid >> 4;
    const int x = ox + 4 * g, y = oy + 4 * r;
    if (x >= b.w || y >= b.h) return;
    typename Sample<REV>::T v[4][4];
    col_lift<REV>(tile, g, r, v);
    // rows are padded to 16 elements: whole groups of four can be written
    const uint32_t pitch = coef_pitch((uint32_t)b.w);
    uint32_t *out = coef + lj->out + (uint32_t)y * pitch + (uint32_t)x;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (y + q < b.h)
            *reinterpret_cast<uint4 *>(out + (uint32_t)q * pitch) = make_uint4(
                __builtin_bit_cast(uint32_t, v[q][0]), __builtin_bit_cast(uint32_t, v[q][1]),
                __builtin_bit_cast(uint32_t, v[q][2]), __builtin_bit_cast(uint32_t, v[q][3]));
}

// The levels of a launch whose jobs all fit (rows_level on the host).  What
// bounds it: HBM.  The 256x256 levels of 192 tiles of 512x512 under 9/7 take 67 us
// (80 in the general kernel), the 128x128 levels of 4096 tiles of 256x256 under
// 5/3 287 (330; 1.3 GB, 4.5 TB/s).
template <bool REV>
__device__ __forceinline__ void level_rows_any(const LevelJob *lj, uint32_t local, uint32_t *coef) {
    __shared__ __attribute__((aligned(16)))
        typename Sample<REV>::T tile[RowTile<REV>::kRows * RowTile<REV>::kPitch];
    const bool hi16 = (lj->narrow & 2u) != 0, ll16 = (lj->narrow & 1u) != 0;
    const bool llf = !REV && (lj->float_in & 1u);
    if (hi16) {
        if (ll16)
            level_rows<REV, true, true, false>(lj, local, coef, tile);
        else if (REV || !llf)
            level_rows<REV, true, false, false>(lj, local, coef, tile);
        else
            level_rows<REV, true, false, true>(lj, local, coef, tile);
    } else if (ll16) {
        level_rows<REV, false, true, false>(lj, local, coef, tile);
    } else if (REV || !llf) {
        level_rows<REV, false, false, false>(lj, local, coef, tile);
    } else {
        level_rows<REV, false, false, true>(lj, local, coef, tile);
    }
}
template <bool REV>
__device__ __forceinline__ void level_rows_body(const LevelJob *jobs, uint32_t njobs,
                                                uint32_t block_offset, const uint32_t *block_job,
                                                uint32_t *coef) {
    const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x) + block_offset;
    const LevelJob *lj = job_of(jobs, njobs, block_job, blk);
    level_rows_any<REV>(lj, blk - lj->block_base, coef);
}
extern "C" __global__ void __launch_bounds__(kIdwtThreads)
sgn_idwt_rows_rev(const LevelJob *jobs, uint32_t njobs, uint32_t block_offset,
                  const uint32_t *block_job, uint32_t *coef) {
    level_rows_body<true>(jobs, njobs, block_offset, block_job, coef);
}
extern "C" __global__ void __launch_bounds__(kIdwtThreads)
sgn_idwt_rows_irr(const LevelJob *jobs, uint32_t njobs, uint32_t block_offset,
                  const uint32_t *block_job, uint32_t *coef) {
    level_rows_body<false>(jobs, njobs, block_offset, block_job, coef);
}

// The lowest levels of tile-components, one block each, one after the other in
// one work-group per component: job first[d] + blockIdx.x is its d-th, whose
// low-pass band the one before wrote; bit d of `general`: some job of that depth
// needs the general kernel.  A launch of its own takes a level of few components
// about 5 us, most of it the launch and the loads' latency.
struct LevelChain {
    uint32_t first[8];
    uint32_t levels, general;
};
template <bool REV>
__device__ __forceinline__ void chain_body(const LevelJob *jobs, const LevelChain &c, uint32_t *coef) {
    const uint32_t j = xcd_remap(blockIdx.x, gridDim.x);
    for (uint32_t d = 0; d < c.levels; ++d) {
        if ((c.general >> d) & 1u)
            level_block<REV, Big>(jobs + c.first[d] + j, 0, coef);
        else
            level_rows_any<REV>(jobs + c.first[d] + j, 0, coef);
        __syncthreads();  // the level's samples are the next one's low-pass band
    }
}
extern "C" __global__ void __launch_bounds__(kIdwtThreads)
sgn_idwt_chain_rev(const LevelJob *jobs, LevelChain c, uint32_t *coef) {
    chain_body<true>(jobs, c, coef);
}
extern "C" __global__ void __launch_bounds__(kIdwtThreads)
sgn_idwt_chain_irr(const LevelJob *jobs, LevelChain c, uint32_t *coef) {
    chain_body<false>(jobs, c, coef);
}

// Rounds half away from zero and saturates to 8 bits, as `as u8` of a rounded
// f32 does (NaN: 0).  From 0 up the largest f32 below a half, added before
// truncation, rounds every f32 below 2^23 right.
__device__ __forceinline__ uint32_t round_u8(float v) {
    return (uint32_t)fminf(fmaxf(v + 0.49999997f, 0.0f), 255.0f);
}

// Final stage of 8-bit RGB tiles under 9/7 and ICT: block list[i] of the plan's
// 9/7 final blocks per work-group.  One component at a time through the LDS
// tile; the next one's loads are in flight during the vertical lifting.
//
// What bounds it: VALU issue, about 25 operations a sample.  192 tiles of 512x512
// take 221 us (0.53 GB, 2.4 TB/s) against 665 in the general kernel, which
// computes every lifting segment's neighbours again and passes each component
// through LDS four times.  Band types are compile-time (selecting them per
// block took 304 us), and 96 registers keep five waves a SIMD.
constexpr int kIctThreads = 320;  // 36 row pairs of 8 lanes; 256 threads for the columns
extern "C" __global__ void __launch_bounds__(kIctThreads, 5)
sgn_final_ict8(const FinalJob *jobs, const uint32_t *list, const uint32_t *block_job,
               const LevelJob *lv, const uint32_t *coef) {
#pragma clang fp contract(off)
    using R = RowTile<false>;
    static_assert(kIctThreads >= 8 * R::kPairs, "a row pair per group of eight lanes");
    __shared__ __attribute__((aligned(16))) float tile[R::kRows * R::kPitch];
    const uint32_t blk = list[xcd_remap(blockIdx.x, gridDim.x)];
    const FinalJob *fj = jobs + block_job[blk];
    const uint32_t local = blk - fj->block_base, nbx = fj->nbx;
    const int ox = (int)(fj->bx0 + local % nbx) * kBlk, oy = (int)(fj->by0 + local / nbx) * kBlk;
    const int tid = threadIdx.x, seg = tid & 7, j = tid >> 3;
    const LevelJob *l0 = lv + fj->level[0];
    const int w = (int)(l0->x1 - l0->x0), h = (int)(l0->y1 - l0->y0);
    const bool rows = j < R::kPairs && oy - R::H + 2 * j <= h + 3;
    const int g = tid & 15, r = tid >> 4;
    const int x = ox + 4 * g, y = oy + 4 * r;
    const bool cols = tid < 256 && x < w && y < h;
    float v[3][4][4];
    RowChunk k{};
    if (rows) row_load<false, true, false>(row_bands<true, false>(l0, coef), ox, oy, j, seg, k);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (rows)
            row_lift<false, true, false, true>(row_bands<true, false>(lv + fj->level[c], coef), ox, j,
                                               seg, k, tile);
        __syncthreads();
        if (c < 2 && rows)
            row_load<false, true, false>(row_bands<true, false>(lv + fj->level[c + 1], coef), ox,
                                         oy, j, seg, k);
        if (cols) col_lift<false>(tile, g, r, v[c]);
        if (c < 2) __syncthreads();
    }
    if (!cols) return;
    uint8_t *const dst = reinterpret_cast<uint8_t *>(fj->dst) + (size_t)y * fj->pitch + (size_t)x * 3;
    const bool words = ((fj->dst | fj->pitch) & 3u) == 0 && x + 4 <= w;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (y + q >= h) break;
        uint32_t o[4][3];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            // mct.rs:71-156, then the level shift
            const float y0 = v[0][q][d], y1 = v[1][q][d], y2 = v[2][q][d];
            o[d][0] = round_u8(fmaf(y2, 1.402f, y0) + 128.0f);
            o[d][1] = round_u8(fmaf(y2, -0.71414f, fmaf(y1, -0.34413f, y0)) + 128.0f);
            o[d][2] = round_u8(fmaf(y1, 1.772f, y0) + 128.0f);
        }
        const uint32_t w0 = o[0][0] | (o[0][1] << 8) | (o[0][2] << 16) | (o[1][0] << 24);
        const uint32_t w1 = o[1][1] | (o[1][2] << 8) | (o[2][0] << 16) | (o[2][1] << 24);
        const uint32_t w2 = o[2][2] | (o[3][0] << 8) | (o[3][1] << 16) | (o[3][2] << 24);
        uint8_t *p = dst + (size_t)q * fj->pitch;
        if (words) {
            uint32_t *pw = reinterpret_cast<uint32_t *>(p);
            pw[0] = w0;
            pw[1] = w1;
            pw[2] = w2;
        } else {
            const int n = min(4, w - x) * 3;
#pragma unroll
            for (int t = 0; t < 12; ++t)
                if (t < n) p[t] = (uint8_t)((t < 4 ? w0 : t < 8 ? w1 : w2) >> (8 * (t & 3)));
        }
    }
}

}  // namespace sgn
