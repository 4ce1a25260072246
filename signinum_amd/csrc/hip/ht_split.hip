// HT cleanup decode in three kernels, each with the shape of its own work:
//
//   sgn_ht_clean    sixteen (or four) lanes per code-block: removes the bit stuffing of
//                   the VLC stream, eight bytes a lane, into a plain bit string
//                   in the block's workspace;
//   sgn_ht_symbols  one block per lane (L of a wave's 64 lanes in use): the
//                   serial MEL / VLC / UVLC chain, reading plain bits, writing
//                   16 bits per quad into the workspace;
//   sgn_ht_magsgn   as many lanes per block, a quad pair each: magnitudes and
//                   signs of a quad row at once, each quad's place in the
//                   MagSgn stream a prefix sum of the quads' bit counts.
//
// The steps are those of crates/signinum-j2k-native/src/j2c/ht_block_decode.rs
// (decode_cleanup_symbols :1056-1204, decode_magnitude_sign_phase :1435-1560);
// only the order in which independent work happens differs: the chain never
// needs a magnitude (its contexts are significance bits alone), so all symbols
// of a block come first.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../host/plan_types.h"
#include "ht_common.hpp"
#include "ht_readers4.hpp"
#include "ht_refine.hpp"

namespace sgn {

constexpr int kSplitWaves = 4;  // waves per work-group of the three kernels

// A block's part of its group's workspace.
struct HtWork {
    uint4 *head, *vlc, *mel, *sym;
};
__device__ __forceinline__ HtWork ht_work(uint4 *work, const HtGroup *groups, uint32_t i) {
    const HtGroup g = groups[i / kHtGroup];
    HtWork w;
    w.head = work + g.base + i % kHtGroup;
    w.vlc = w.head + kHtGroup;
    w.mel = w.vlc + size_t(kHtGroup) * g.vlc_units;
    w.sym = w.mel + kHtGroup * kHtMelUnits + i % kHtGroup;  // two units a block
    return w;
}

// Header of a block's workspace.
struct HtHead {
    uint32_t vlc_last;  // last 16-byte unit of the VLC string (all zeros)
    uint32_t scup;      // length of the MEL + VLC segment; 0: nothing to decode
    uint32_t bad;       // malformed
    uint32_t pad;
};

// Decode tables of the symbol kernel, fields where the chain uses them.
// Context entries (index: 7 stream bits, then the context): bits 0-2 codeword
// length, 8 u-offset, 9-11 the context that the quad gives its right neighbour
// (first row: sigma_0 | sigma_1, sigma_2, sigma_3; other rows: bit 9 sigma_2 |
// sigma_3, bits 10-11 come from the row above), 16-23 two bits per sample (0
// insignificant, 1 significant, 2 exponent known to be 0, 3 to be 1), 30
// sigma_3, 31 sigma_1.  u-offset entries (index: 6 stream bits, the quads'
// u-offset flags): bits 0-4 prefix length plus 2, 5-9 suffix length, 10-14 the
// first quad's part of it, 16-20 both lengths; then the same number of words
// with the prefixes' values in bytes 1 and 3.
struct HtSplitTables {
    uint32_t first[1024], other[1024];
    uint32_t ufirst[2 * 320], uother[2 * 256];
};

// From the tables of T.814 (length, u_off, rho, e_1, e_k; prefix and suffix).
inline void ht_split_tables(const uint16_t *vlc0, const uint16_t *vlc1, const uint16_t *u0,
                            const uint16_t *u1, HtSplitTables &T) {
    auto entry = [](uint32_t t, bool first) {
        uint32_t code = 0;
        for (uint32_t s = 0; s < 4; ++s) {
            const uint32_t sig = (t >> (4 + s)) & 1u, e1 = (t >> (8 + s)) & 1u,
                           ek = (t >> (12 + s)) & 1u;
            code |= (sig ? 1u + ek + (ek & e1) : 0u) << (2 * s);
        }
        const uint32_t r0 = (t >> 4) & 1u, r1 = (t >> 5) & 1u, r2 = (t >> 6) & 1u, r3 = (t >> 7) & 1u;
        const uint32_t right = first ? (r0 | r1) | r2 << 1 | r3 << 2 : r2 | r3;
        return (t & 7u) | ((t >> 3) & 1u) << 8 | right << 9 | code << 16 | r3 << 30 | r1 << 31;
    };
    for (uint32_t k = 0; k < 1024; ++k) {
        T.first[k] = entry(vlc0[k], true);
        // context bits: left, (sigma_3 of the quad above or sigma_1 of the one
        // after it), (sigma_1 of the quad above or sigma_3 of the one before)
        const uint32_t left = (k >> 7) & 1u, after = (k >> 8) & 1u, before = (k >> 9) & 1u;
        T.other[k] = entry(vlc1[(k & 0x7Fu) | before << 7 | left << 8 | after << 9], false);
    }
    auto uentry = [](uint32_t e, uint32_t add, uint32_t &word, uint32_t &base) {
        const uint32_t lp = e & 7u, ls = (e >> 3) & 0xFu, n0 = (e >> 7) & 7u;
        word = (lp + 2) | ls << 5 | n0 << 10 | (lp + ls) << 16;
        base = (((e >> 10) & 7u) + add) << 8 | ((e >> 13) + add) << 24;
    };
    for (uint32_t k = 0; k < 320; ++k) uentry(u0[k], 1, T.ufirst[k], T.ufirst[320 + k]);
    for (uint32_t k = 0; k < 256; ++k) uentry(u1[k], 0, T.uother[k], T.uother[256 + k]);
}

// The clean, magnitude and refinement kernels give a block one DPP row (16 lanes),
// so that neighbours, prefix sums and broadcasts inside a block are single VALU
// operations that never cross into the next block; or one quad (4 lanes) where all
// blocks of the list are at most 16 wide and would leave the rest of a row idle.
// Cleanup in us with rows, with quads, and in one kernel of a lane a block that
// these replaced: 2.4 million 4x4 blocks 994, 431, 492; 614,400 8x8 blocks 354, 166,
// 202; 310,800 16x16 blocks 320, 200, 244 (1.2 million 1190, 869, 725).
constexpr uint32_t kSplitLanes = 16, kQuadLanes = 4, kQuadWidth = 16;
constexpr uint32_t split_blocks(uint32_t lanes) { return kSplitWaves * 64 / lanes; }  // per work-group

// Value of another lane of the row (CTRL), 0 past the row's ends.
template <int CTRL>
__device__ __forceinline__ uint32_t row_dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}

// The L lanes of a block, this one being lane q.  Called by all lanes.
template <uint32_t L>
struct BlockLanes {
    static_assert(L == 16 || L == 4, "a DPP row or quad");
    uint32_t q;
    // Value of the lane before (0 for the first) and after (0 for the last).
    __device__ __forceinline__ uint32_t before(uint32_t v) const {
        if constexpr (L == 16) return row_dpp<0x111>(v);  // row_shr:1
        const uint32_t x = row_dpp<0x90>(v);              // quad_perm:[0,0,1,2]
        return q ? x : 0u;
    }
    __device__ __forceinline__ uint32_t after(uint32_t v) const {
        if constexpr (L == 16) return row_dpp<0x101>(v);  // row_shl:1
        const uint32_t x = row_dpp<0xF9>(v);              // quad_perm:[1,2,3,3]
        return q < 3 ? x : 0u;
    }
    // Inclusive prefix sum.
    __device__ __forceinline__ uint32_t scan(uint32_t v) const {
        v += before(v);
        if constexpr (L == 16) {
            v += row_dpp<0x112>(v);  // row_shr:2
            v += row_dpp<0x114>(v);  // row_shr:4
            v += row_dpp<0x118>(v);  // row_shr:8
        } else {
            const uint32_t x = row_dpp<0x40>(v);  // quad_perm:[0,0,0,1]
            v += q >= 2 ? x : 0u;
        }
        return v;
    }
    // The last lane's value (row_newbcast:15, quad_perm:[3,3,3,3]).
    __device__ __forceinline__ uint32_t last(uint32_t v) const {
        return L == 16 ? row_dpp<0x15F>(v) : row_dpp<0xFF>(v);
    }
};

// Orders the LDS accesses of one wave for the compiler; the LDS unit executes
// a wave's instructions in order, so nothing is waited for.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ---- stuffing removal ------------------------------------------------------

// Dwords of a block's ring: a partly filled unit and a round's 2 L + 1.
template <uint32_t L>
constexpr uint32_t kCleanRing = 4 * L;

// A plain bit string that a block's L lanes write to its interleaved
// units, 8 L bytes of stream a round, through a ring of words in LDS that whole
// units leave.  Every byte is ORed in at its place.
template <uint32_t L>
struct PlainString {
    static constexpr uint32_t kMask = kCleanRing<L> - 1;
    uint32_t *buf;  // the ring, 16-byte aligned
    BlockLanes<L> lanes;
    uint32_t q;  // lane of the block
    uint4 *d;    // unit 0
    uint32_t units, fill, done;

    __device__ __forceinline__ PlainString(uint32_t *b, uint32_t lane, uint4 *out, uint32_t n,
                                           uint32_t head, uint32_t bits)
        : buf(b), lanes{lane}, q(lane), d(out), units(n), fill(bits), done(0) {
        if (q < 4) buf[q] = q == 0 ? head : 0u;
    }
    // This lane's n0 and n1 next bits (25 to 32 each; a value may reach one bit
    // past its count).  Called by all lanes; blocks that are not `act` sit out.
    __device__ __forceinline__ void round(bool act, uint32_t v0, uint32_t n0, uint32_t v1,
                                          uint32_t n1) {
        const uint32_t incl = lanes.scan(n0 + n1), tot = lanes.last(incl);
        if (act) {
            const uint32_t z = (fill >> 5) + 1 + q;
            buf[z & kMask] = 0;
            buf[(z + L) & kMask] = 0;
        }
        wave_lds_fence();
        if (act) {
            // the lane's 50 to 64 bits: three words at most
            const uint64_t v = (uint64_t)v0 | ((uint64_t)v1 << n0);
            const uint32_t pos = fill + incl - (n0 + n1), wi = pos >> 5, sh = pos & 31u;
            const uint64_t a = v << sh;
            const uint32_t x2 = sh ? (uint32_t)(v >> 32) >> (32u - sh) : 0u;
            if ((uint32_t)a) atomicOr(&buf[wi & kMask], (uint32_t)a);
            if ((uint32_t)(a >> 32))
                atomicOr(&buf[(wi + 1) & kMask], (uint32_t)(a >> 32));
            if (x2) atomicOr(&buf[(wi + 2) & kMask], x2);
            fill += tot;
        }
        wave_lds_fence();
        // whole units (at most 9 a round, 2 of a quad; the padding of the last round's
        // bytes may reach past the string's last unit)
        const uint32_t full = min(fill >> 7, units), u = done + q;
        if (act && u < full)
            d[kHtGroup * u] = *reinterpret_cast<uint4 *>(&buf[4 * u & kMask]);
        done = act ? full : done;
    }
    // The partly filled unit, then zeros up to and with unit `units`
    // (seven-bit bytes leave the string short of it).
    __device__ __forceinline__ void finish() {
        const uint32_t last = fill >> 5;
        for (uint32_t u = done + q; u <= units; u += L) {
            uint4 v = make_uint4(0, 0, 0, 0);
            if (u < units) {
                const uint32_t *x = &buf[4 * u & kMask];
                v.x = 4 * u <= last ? x[0] : 0u;
                v.y = 4 * u + 1 <= last ? x[1] : 0u;
                v.z = 4 * u + 2 <= last ? x[2] : 0u;
                v.w = 4 * u + 3 <= last ? x[3] : 0u;
            }
            d[kHtGroup * u] = v;
        }
    }
};

// Stream bytes that carry 7 bits (bit 0 of each byte of s) close up: the
// dword's bits from bit 0, and their count.
__device__ __forceinline__ uint32_t close_up(uint32_t d, uint32_t s, uint32_t &bits) {
    // running counts, a byte each
    uint32_t c = s + (s << 8);
    c += c << 16;
    bits = 32u - (c >> 24);
    return (d & 0xFFu) | ((d & 0xFF00u) >> (c & 31u)) | ((d & 0xFF0000u) >> ((c >> 8) & 31u)) |
           ((d & 0xFF000000u) >> ((c >> 16) & 31u));
}
// Bit 7 of every byte of d that is 0xFF.
__device__ __forceinline__ uint32_t bytes_ff(uint32_t d) {
    return ((d & 0x7F7F7F7Fu) + 0x01010101u) & d & 0x80808080u;
}
// Bit 7 of every byte above 0x8F, and of every byte whose low 7 bits are ones.
__device__ __forceinline__ uint32_t bytes_above(uint32_t d) {
    return ((d & 0x7F7F7F7Fu) + 0x70707070u) & d & 0x80808080u;
}
__device__ __forceinline__ uint32_t bytes_7f(uint32_t d) {
    return ((d & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u;
}

// The VLC string of one block per L lanes: two zero bits, the 3 or 4 bits of the
// segment's second last byte, and from there it runs backward from the byte before; a byte
// whose low 7 bits are ones after a byte > 0x8F carries 7 bits, and is ORed in
// whole, as the byte-wise reader does (ht_block_decode.rs:931-999); zeros
// follow it.  Two dependent trips to memory per block bound it (the first
// bytes are asked for beside the length field); a round takes eight bytes a
// lane, through a ring of words in LDS that whole 16-byte units leave.  *clear
// (null: none) is a counter of a later launch, set to 0.
template <uint32_t L>
__global__ void __launch_bounds__(kSplitWaves * 64)
sgn_ht_clean(const CbJob *__restrict__ jobs, uint32_t n, const uint8_t *__restrict__ arena,
             const HtGroup *__restrict__ groups, uint4 *__restrict__ work, uint32_t *clear) {
    if (clear && blockIdx.x == 0 && threadIdx.x == 0) *clear = 0;
    __shared__ __attribute__((aligned(16))) uint32_t s_buf[split_blocks(L)][kCleanRing<L>];
    const uint32_t row = threadIdx.x / L, q = threadIdx.x % L;
    const BlockLanes<L> lanes{q};
    uint32_t *buf = s_buf[row];
    const uint32_t i = blockIdx.x * split_blocks(L) + row;
    const bool valid = i < n;
    CbJob j{};
    if (valid) j = jobs[i];
    const bool coded = valid && !(j.flags & kCbZero) && j.lcup >= 2;
    const uint32_t lcup = coded ? j.lcup : 0, seg1 = j.src + lcup;
    // the four bytes e - 3 .. e (e: arena address), the last in the top byte
    auto load4 = [&](uint32_t e) -> uint32_t {
        uint32_t x;
        if (e >= 3) {
            __builtin_memcpy(&x, arena + e - 3, 4);
            return x;
        }
        __builtin_memcpy(&x, arena, 4);
        return x << (8 * (3 - e));
    };
    // this lane's eight bytes of a round, k0 bytes into the stream
    uint32_t hi = 0, lo = 0;
    auto fetch = [&](uint32_t k0, uint32_t len) {
        hi = lo = 0;
        if (k0 < len) hi = load4(seg1 - 3 - k0);
        if (k0 + 4 < len) lo = load4(seg1 - 3 - k0 - 4);
    };
    uint32_t b0 = 0, top = 0;
    if (coded) {
        b0 = arena[seg1 - 2];
        top = arena[seg1 - 1];
    }
    // (bytes past a shorter segment are dropped below)
    fetch(8 * q, lcup > 2 ? lcup - 2 : 0);
    uint32_t scup = (top << 4) + (b0 & 0x0F);
    uint32_t bad = 0;
    if (valid && !(j.flags & kCbZero))
        bad = lcup < 2 || j.zblk >= 30 || scup < 2 || scup > lcup || scup > 4079;
    if (!coded || bad) scup = 0;
    const HtWork w = ht_work(work, groups, valid ? i : 0);
    // the first MEL bytes, as they are
    for (uint32_t u = q; u < kHtMelUnits && scup > 16 * u; u += L) {
        uint4 v;
        __builtin_memcpy(&v, arena + (seg1 - scup) + 16 * u, 16);
        w.mel[kHtGroup * u] = v;
    }
    const uint32_t len = scup ? scup - 2 : 0;
    const uint32_t units = (6 + 8 * len + 127) >> 7;  // 16-byte units that hold stream bits
    const uint32_t first = b0 >> 4;
    // two bits in front
    PlainString<L> str(buf, q, w.vlc, units, first << 2, 6u - ((first & 7u) == 7u ? 1u : 0u));
    uint32_t carry = b0 | 0x0Fu;  // the byte before this round's

    for (uint32_t at = 0; __any(at < len); at += 8 * L) {
        const uint32_t k0 = at + 8 * q;
        uint32_t d0 = __builtin_bswap32(hi), d1 = __builtin_bswap32(lo);
        if (k0 + 4 > len) d0 &= k0 < len ? 0xFFFFFFFFu >> (8 * (4 - (len - k0))) : 0u;
        if (k0 + 8 > len) d1 &= k0 + 4 < len ? 0xFFFFFFFFu >> (8 * (8 - (len - k0))) : 0u;
        fetch(k0 + 8 * L, len);
        const uint32_t g0 = bytes_above(d0), g1 = bytes_above(d1);
        uint32_t pg = lanes.before(g1);
        if (q == 0) pg = carry > 0x8Fu ? 0x80000000u : 0u;
        carry = lanes.last(d1 >> 24);
        uint32_t n0, n1;
        const uint32_t v0 =
            close_up(d0, (bytes_7f(d0) & __builtin_amdgcn_alignbit(g0, pg, 24)) >> 7, n0);
        const uint32_t v1 =
            close_up(d1, (bytes_7f(d1) & __builtin_amdgcn_alignbit(g1, g0, 24)) >> 7, n1);
        str.round(at < len, v0, n0, v1, n1);
    }
    if (scup) str.finish();
    if (valid && q == 0) *reinterpret_cast<HtHead *>(w.head) = HtHead{units, scup, bad, 0};
}

// ---- MEL / VLC / UVLC chain --------------------------------------------------

// MEL events as a bit queue: bit n is the outcome of the n-th quad (or, in the
// first row, u-offset pair) from here that asks the MEL decoder.  A run symbol
// (ht_block_decode.rs:860-929) adds its zeros and, if the run ended early, a
// one; so the chain takes one bit per question instead of counting runs down.
struct MelQueue {
    uint64_t buf;   // undecoded MEL bits, next in bit 63
    uint64_t ev;    // events, next in bit 0
    uint32_t bits;  // valid bits of buf
    uint32_t n;     // valid events
    uint32_t k;     // run-length state, 0..12
    uint32_t next;  // four stream bytes, loaded ahead
    int32_t left;   // stream bytes from `next` on
    uint32_t at;    // their arena address
    uint32_t idx;   // their dword index in the string
    uint32_t ff;    // the byte before them was 0xFF
    const uint4 *copy;  // the string's first units in the workspace
};

// The four bytes at `at` (from the workspace as far as its copy goes).
__device__ __forceinline__ void mel_queue_load(MelQueue &m, const uint8_t *arena) {
    const uint8_t *p = m.idx < 4 * kHtMelUnits
                           ? reinterpret_cast<const uint8_t *>(m.copy + kHtGroup * (m.idx >> 2)) +
                                 4 * (m.idx & 3u)
                           : arena + m.at;
    __builtin_memcpy(&m.next, p, 4);
}

// Appends the four bytes loaded ahead (MSB-first, 7 bits after 0xFF, the
// segment's last byte ORed with 0x0F, 0xFF past it) and asks for the next
// (past the segment for bytes inside it, which are not used).
__device__ __forceinline__ void mel_queue_bytes(MelQueue &m, const uint8_t *arena) {
    uint32_t w = m.next;
    if (m.left <= 4) {
        if (m.left > 0) w |= 0x0Fu << (8 * (m.left - 1));
        if (m.left < 4) w |= 0xFFFFFFFFu << (8 * max(m.left, 0));
    }
    m.left -= 4;
    m.at += m.left > 0 ? 4u : 0u;
    m.idx += m.left > 0 ? 1u : 0u;
    mel_queue_load(m, arena);
    uint32_t v = 0, n = 0;
#pragma unroll
    for (uint32_t t = 0; t < 4; ++t) {
        const uint32_t b = (w >> (8 * t)) & 0xFFu;
        const uint32_t nb = 8u - m.ff;
        v = (v << nb) | (b & (0xFFu >> m.ff));
        n += nb;
        m.ff = b == 0xFFu ? 1u : 0u;
    }
    m.buf |= (uint64_t)v << (64u - m.bits - n);
    m.bits += n;
}

// Decodes run symbols until every lane of the wave that is `on` holds `need`
// (at most 32) events; lanes with room and bits join in.  Sixteen events take
// 41 bits at most when they start from the longest runs, so the buffer (over 32
// bits at a segment's start) hardly ever has to wait for its next bytes here.
__device__ __forceinline__ void mel_queue_fill(MelQueue &m, uint32_t need, bool on,
                                               const uint8_t *arena) {
    // E for k = 0..12, four bits each
    constexpr uint64_t kExp = 0x5433222111000ull;
    while (__any(on && m.n < need)) {
        if (on && (m.n < need || (m.n < 32u && m.bits >= 6u))) {
            if (m.bits < 6u) mel_queue_bytes(m, arena);
            const uint32_t e = (uint32_t)(kExp >> (4u * m.k)) & 0xFu;
            const uint32_t hi = (uint32_t)(m.buf >> 32), one = hi >> 31;
            // run length bits of an early end (none for E = 0)
            const uint32_t v = __builtin_amdgcn_ubfe(hi, 31u - e, e);
            const uint32_t used = one ? 1u : 1u + e;
            m.buf <<= used;
            m.bits -= used;
            m.k = one ? min(m.k + 1u, 12u) : max(m.k, 1u) - 1u;
            m.n += one ? 1u << e : v + 1u;
            m.ev |= (uint64_t)(one ^ 1u) << (m.n - 1u);
        }
    }
}

// Symbols of the blocks jobs[0 .. n): lane l < L of wave k takes block k * L +
// l.  Fewer lanes a wave spread few blocks over more waves (every SIMD gets
// some).  The VLC string is staged through a ring of four 16-byte units per
// lane in LDS, two units loaded ahead in registers, so that no read of the
// chain waits for memory.  Everything else of a lane's state is in
// registers: the significance that contexts need is two bits per quad of the
// row above, as one bit string with the left neighbours' bits beside it.
//
// The chain is bound by latency when waves are few (three dependent LDS reads a
// pair: two context tables and the u-offset table; the stream window is kept in
// registers, its next dword read a pair ahead) and by VALU issue when they are
// many, so a pair is straight-line code of about 60 operations: the tables
// (HtSplitTables) hold every field where it is used, a quad past the block's edge
// is a quad whose table entry is masked to zero (whole segments go without), and
// the MEL question is arithmetic on 0/1 words.  One 512x512 RGB tile takes 165
// us, half of it VALU issue and a third LDS waits; with the window read in the
// chain 171.
//
// TIMED (the decode-cost model's samples, with L = 1): each wave records the
// shader-clock cycles of its block's chain.
template <int L, bool TIMED = false>
__global__ void __launch_bounds__(kSplitWaves * 64)
sgn_ht_symbols(const CbJob *__restrict__ jobs, uint32_t n, const uint8_t *__restrict__ arena,
               const HtGroup *__restrict__ groups, uint4 *__restrict__ work,
               const HtSplitTables *__restrict__ tables, uint64_t *__restrict__ cycles) {
    __shared__ __attribute__((aligned(16))) HtSplitTables s_t;
    __shared__ uint32_t s_ring[kSplitWaves][16][L];
    for (uint32_t t = threadIdx.x; t < sizeof(HtSplitTables) / 16; t += kSplitWaves * 64)
        reinterpret_cast<uint4 *>(&s_t)[t] = reinterpret_cast<const uint4 *>(tables)[t];
    __syncthreads();
    const uint64_t began = TIMED ? clock64() : 0;
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t i = (blockIdx.x * kSplitWaves + wv) * L + lane;
    const bool valid = lane < (uint32_t)L && i < n;
    uint32_t(*ring)[L] = s_ring[wv];
    const uint32_t rl = lane < (uint32_t)L ? lane : 0u;  // idle lanes read, never write

    uint32_t width = 0, height = 0;
    const HtWork w = ht_work(work, groups, valid ? i : 0);
    HtHead hd{0, 0, 0, 0};
    uint32_t seg1 = 0;
    if (valid) {
        const CbJob j = jobs[i];
        width = j.w;
        height = j.h;
        seg1 = j.src + j.lcup;
        if (!(j.flags & kCbZero)) hd = *reinterpret_cast<const HtHead *>(w.head);
    }
    const bool on = hd.scup != 0;
    uint32_t d0 = 0, d1 = 0;  // the string's dwords at pos
    const uint32_t nq = (width + 1) >> 1, npairs = (width + 3) >> 2;
    const uint32_t nrows = on ? (height + 1) >> 1 : 0, nseg = (npairs + 7) >> 3;
    auto vlc = [&](uint32_t u) -> uint4 { return w.vlc[kHtGroup * min(u, hd.vlc_last)]; };
    uint4 *sym = w.sym;

    MelQueue mel{0, 0, 0, 0, 0, 0, (int32_t)hd.scup - 1, seg1 - hd.scup, 0, 0, w.mel};
    uint4 pend0 = make_uint4(0, 0, 0, 0), pend1 = pend0;
    uint32_t res = 4;  // unit that pend0 holds (pend1 the next): those below are or were in the ring
    auto put = [&](uint32_t unit, const uint4 &v) {
        const uint32_t s = (unit & 3u) * 4u;
        ring[s + 0][rl] = v.x;
        ring[s + 1][rl] = v.y;
        ring[s + 2][rl] = v.z;
        ring[s + 3][rl] = v.w;
    };
    if (on) {
        mel_queue_load(mel, arena);
        uint4 u[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) u[k] = vlc(k);
        pend0 = vlc(4);
        pend1 = vlc(5);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) put(k, u[k]);
        d0 = u[0].x;
        d1 = u[0].y;
        mel_queue_bytes(mel, arena);
    }
    // next bit of the VLC string less two (the string starts at bit 2): the
    // window's next bit is bit 2, a table's byte offset
    uint32_t pos = 0;
    uint32_t x0 = 0, x1 = 0;    // contexts from the row above, two bits per quad, first quad on top
    uint32_t sig0 = 0;          // this row's sigma_1, sigma_3 bits of its first 16 quads
    uint32_t t1 = 0;            // table entry of the quad to the left
    uint32_t row = 0, seg = 0;

    const uint8_t *ctx0 = reinterpret_cast<const uint8_t *>(s_t.first);
    const uint8_t *ctx1 = reinterpret_cast<const uint8_t *>(s_t.other);

    while (__any(row < nrows)) {
        const bool run = row < nrows;
        const bool first = row == 0;
        // events of up to 16 quads and, in the first row, 8 u-offset pairs
        mel_queue_fill(mel, first ? 24u : 16u, run, arena);
        // events leave at bit 0; a one above the 24 that a segment may take
        // says at the end how many did
        uint32_t ev = ((uint32_t)mel.ev & 0xFFFFFFu) | 0x80000000u;
        uint32_t acc = 0;
        uint32_t out[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        const uint32_t pa = 8 * seg;
        const uint32_t pairs = run ? npairs - pa : 0;           // from here to the row's end
        const uint32_t quads = run ? min(nq - 2 * pa, 16u) : 0;
        const uint32_t exist = (1u << quads) - 1u;              // bit per quad
        // one pair: FIRST rows take contexts from the left alone and may ask
        // MEL for the u-offsets; later rows add the row above
        uint32_t x = (seg ? x1 : x0) | (quads < 16u ? 0xFFFFFFFFu >> (2u * quads) : 0u);
        auto pair = [&](auto is_first, auto is_full, uint32_t p) {
            constexpr bool kFirst = decltype(is_first)::value, kFull = decltype(is_full)::value;
            // a pair takes at most 30 bits, so the next one starts in the first
            // or the second dword: the third is read here, off the chain
            const uint32_t d2 = ring[((pos >> 5) + 2u) & 15u][rl];
            uint32_t win = __builtin_amdgcn_alignbit(d1, d0, pos);
            uint32_t t0;
#pragma unroll
            for (uint32_t q = 2 * p; q < 2 * p + 2; ++q) {
                // context: table offset bits 9-11
                uint32_t c;
                if constexpr (kFirst) {
                    c = t1 & 0xE00u;
                } else {
                    const uint32_t above = q < 10 ? x >> (20 - 2 * q) : x << (2 * q - 20);
                    c = (above & 0xC00u) | (t1 & 0x200u);
                }
                uint32_t t = *reinterpret_cast<const uint32_t *>((kFirst ? ctx0 : ctx1) +
                                                                 ((win & 0x1FCu) | c));
                // a quad without context asks MEL; its 0 makes the entry 0
                uint32_t ask = (c - 1u) >> 31;
                if constexpr (kFirst) ask &= exist >> q;
                const uint32_t drop = ask & ~ev;
                ev >>= ask;
                t &= drop - 1u;
                if constexpr (!kFull) t &= (uint32_t)__builtin_amdgcn_sbfe((int)exist, q, 1);
                win >>= t & 31u;  // bits 3 to 7 are 0
                acc = __builtin_amdgcn_alignbit(acc, t, 30);
                if (q & 1)
                    t1 = t;
                else
                    t0 = t1 = t;
            }
            uint32_t mode = (t0 & 0x100u) | ((t1 & 0x100u) << 1);
            if constexpr (kFirst) {
                const uint32_t both = (mode >> 8) & (mode >> 9);
                mode += (ev & both) << 8;
                ev >>= both;
            }
            const uint32_t *ut = (kFirst ? s_t.ufirst : s_t.uother) + (((win & 0xFCu) | mode) >> 2);
            const uint32_t e = ut[0], base = ut[kFirst ? 320 : 256];
            // (field operands count modulo 32)
            const uint32_t sfx = __builtin_amdgcn_ubfe(win, e, e >> 5);
            const uint32_t n0 = e >> 10;
            const uint32_t low = __builtin_amdgcn_ubfe(sfx, 0, n0), high = sfx >> (n0 & 31u);
            out[p] = __builtin_amdgcn_perm(t1, t0, 0x0C060C02u) + (base + (low << 8) + (high << 24));
            const uint32_t was = pos;
            pos += ((t0 + t1) & 0xFFu) + (e >> 16);
            const bool next = ((was ^ pos) & 32u) != 0;
            d0 = next ? d1 : d0;
            d1 = next ? d2 : d1;
        };
        if (__any(run && first)) {
            // the wave's other lanes (blocks of other heights start their rows
            // together, so there are none but idle ones) sit this out
            if (first) {
#pragma unroll
                for (uint32_t p = 0; p < 8; ++p) {
                    if (p < pairs) pair(std::true_type{}, std::false_type{}, p);
                    else acc <<= 4;
                }
            }
        }
        if (!__any(run && (first || quads < 16u))) {
            // whole segments: no quad to mask
            if (run) {
#pragma unroll
                for (uint32_t p = 0; p < 8; ++p) pair(std::false_type{}, std::true_type{}, p);
            }
        } else if (run && !first) {
#pragma unroll
            for (uint32_t p = 0; p < 8; ++p) {
                if (p && p % 2 == 0 && !__any(p < pairs)) {
                    acc <<= 4 * (8 - p);
                    break;
                }
                pair(std::false_type{}, std::false_type{}, p);
            }
        }
        const uint32_t used = (uint32_t)__builtin_clz(ev);
        mel.ev >>= used;
        mel.n -= used;
        // What was loaded a segment ago goes into the ring (eight pairs take at
        // most 240 bits: two units fill it again) and the MEL buffer, and the
        // next loads go out; all before this segment's stores, whose
        // completion the next wait for a load would include.
        if (run && res < (pos >> 7) + 4u) {
            put(res, pend0);
            ++res;
            if (res < (pos >> 7) + 4u) {
                put(res, pend1);
                ++res;
            }
            pend0 = vlc(res);
            pend1 = vlc(res + 1);
        }
        if (run && mel.bits <= 32u) mel_queue_bytes(mel, arena);
        if (run) {
            sym[0] = make_uint4(out[0], out[1], out[2], out[3]);
            sym[1] = make_uint4(out[4], out[5], out[6], out[7]);
            sym += 2 * kHtGroup;
        }
        if (seg + 1 < nseg) {
            sig0 = acc;
            ++seg;
        } else {
            // contexts of the next row: sigma_1 of the quad or sigma_3 of the
            // one before, sigma_3 of the quad or sigma_1 of the one after; in
            // the bit string s1 s3 s1 s3 ... each bit joins its neighbour on
            // the other quad's side
            const uint32_t lo = seg ? sig0 : acc, hi = seg ? acc : 0u;
            x0 = lo | ((lo >> 1) & 0xAAAAAAAAu) |
                 (__builtin_amdgcn_alignbit(lo, hi, 31) & 0x55555555u);
            x1 = hi | (__builtin_amdgcn_alignbit(lo, hi, 1) & 0xAAAAAAAAu) |
                 ((hi << 1) & 0x55555555u);
            t1 = 0;
            seg = 0;
            ++row;
        }
    }
    if constexpr (TIMED) {
        if (valid && lane == 0) cycles[i] = clock64() - began;
    }
}

// ---- magnitudes and signs ------------------------------------------------------

// Dwords of a block's unstuffed MagSgn ring (a power of two).
template <uint32_t L>
constexpr uint32_t kMagRingOf = 16 * L;

using s16x2 = int16_t __attribute__((ext_vector_type(2)));

// One block per L lanes, a quad pair (eight samples) per lane.  A quad row
// takes at most 2 L quads * 4 samples * 31 bits = 31 L bytes of the ring's 64 L,
// which is topped up eight bytes a lane at a time, from words loaded a round
// ahead.  Sample rows leave as whole 128-byte (int16) lines.
// Bound by VALU issue.
template <typename C, uint32_t L>
__global__ void __launch_bounds__(kSplitWaves * 64)
sgn_ht_magsgn(const CbJob *__restrict__ jobs, uint32_t n, const uint8_t *__restrict__ arena,
              C *__restrict__ coef, const HtGroup *__restrict__ groups, uint4 *__restrict__ work,
              uint8_t *__restrict__ status) {
    // one dword more than the ring: a copy of the first, so that two adjacent
    // dwords can be read at any place
    constexpr uint32_t kMagRing = kMagRingOf<L>;
    __shared__ uint32_t s_ring[split_blocks(L)][kMagRing + 1];
    // per symbol code: byte s of .x is 0xFF where sample s is significant, of
    // .y 1 where its exponent is known, of .z that exponent bit
    __shared__ uint4 s_code[256];
    {
        const uint32_t t = threadIdx.x;
        uint32_t sig = 0, known = 0, bit = 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t c = (t >> (2 * k)) & 3u;
            sig |= (c ? 0xFFu : 0u) << (8 * k);
            known |= (c >> 1) << (8 * k);
            bit |= (c == 3 ? 1u : 0u) << (8 * k);
        }
        s_code[t] = make_uint4(sig, known, bit, 0);
    }
    __syncthreads();
    const uint32_t row = threadIdx.x / L, q = threadIdx.x % L;
    const BlockLanes<L> lanes{q};
    uint32_t *ring = s_ring[row];
    const uint32_t i = blockIdx.x * split_blocks(L) + row;
    const bool valid = i < n;
    CbJob j{};
    if (valid) j = jobs[i];
    const uint32_t w = j.w, h = j.h, stride = j.stride;
    HtHead hd{0, 0, 0, 0};
    const HtWork ws = ht_work(work, groups, valid ? i : 0);
    if (valid && !(j.flags & kCbZero)) hd = *reinterpret_cast<const HtHead *>(ws.head);
    // (the planner makes a block with zblk >= K a zero block; the 16-bit samples'
    // windows rest on it)
    const bool on = hd.scup != 0 && (sizeof(C) == 4 || j.zblk < 15u);
    const uint32_t nrows = (h + 1) >> 1;
    // pair q of a row: dword q % 8 of the row's chunk q / 8
    const uint32_t *sym = reinterpret_cast<const uint32_t *>(ws.sym) +
                          (q >> 3) * (8 * kHtGroup) + (q & 7u);
    const uint32_t spitch = ((w + 31) >> 5) * (8 * kHtGroup);  // dwords per symbol row
    // columns of this lane (4 q .. 4 q + 3) inside the block
    const uint32_t cols = 4 * q < w ? min(w - 4 * q, 4u) : 0u;
    // the samples of its two quads, two bits each
    const uint32_t mask = !on || !cols ? 0u
                          : cols >= 4  ? 0xFFFFu
                          : cols == 3  ? 0x0FFFu
                          : cols == 2  ? 0x00FFu
                                       : 0x000Fu;
    const uint32_t p = 30 - j.zblk, mmsbp2 = j.zblk + 2u;
    const uint32_t shift = j.kmax >= 31 ? 0u : 31u - j.kmax;
    const bool vec = ((j.dst | stride) & 3u) == 0 && cols == 4;
    C *out = coef + j.dst + 4 * q;

    // MagSgn bytes [next, end): forward, a byte after 0xFF carries 7 bits and
    // is ORed in whole, 0xFF past the end (ht_block_decode.rs:881-929).  `raw`
    // holds the eight bytes at `next`, whatever lies there.
    const uint32_t end = on ? j.src + j.lcup - hd.scup : 0;
    uint32_t next = (on ? j.src : 0) + 8 * q;
    uint2 raw = make_uint2(0, 0);
    if (next < end) __builtin_memcpy(&raw, arena + next, 8);
    uint32_t fill = 0, prev = 0, pos = 0;
    if (q == 0) ring[0] = ring[kMagRing] = 0;
    uint32_t bad = hd.bad;
    uint32_t e1 = 0, e3 = 0, e5 = 0, e7 = 0;  // exponents of the bottom samples of the row above
    uint32_t s_next = mask && nrows ? *sym : 0u;
    uint32_t rows_max = (uint32_t)__builtin_amdgcn_readlane((int)nrows, 0);
#pragma unroll
    for (int k = L; k < 64; k += L)
        rows_max = max(rows_max, (uint32_t)__builtin_amdgcn_readlane((int)nrows, k));
    for (uint32_t r = 0; r < rows_max; ++r) {
        const bool live = r < nrows;
        const uint32_t s = s_next;
        if (mask && r + 1 < nrows) s_next = *(sym += spitch);
        uint32_t uq0 = (s >> 8) & 0xFFu, uq1 = s >> 24;
        if (r) {
            // exponent bound of the row above, over the quad and the samples
            // beside it, for quads with more than one significant sample
            const uint32_t l = lanes.before(e7), t = lanes.after(e1);
            const uint32_t mid = max(e3, e5);
            const uint32_t m0 = max(max(max(e1, mid), l), 1u), m1 = max(max(max(e7, mid), t), 1u);
            const uint32_t nz = (s | (s >> 1)) & 0x00550055u;
            const uint32_t z0 = nz & 0xFFu, z1 = nz >> 16;
            uq0 += (z0 & (z0 - 1u)) ? m0 : 1u;
            uq1 += (z1 & (z1 - 1u)) ? m1 : 1u;
        }
        const bool over = live && ((mask && uq0 > mmsbp2) || ((mask >> 8) && uq1 > mmsbp2));
        const uint64_t ov = __ballot(over) >> (threadIdx.x & (64u - L));
        if ((uint32_t)ov & ((1u << L) - 1u)) bad = 1;
        const uint32_t code0 = live && !bad ? s & mask & 0xFFu : 0u;
        const uint32_t code1 = live && !bad ? (s >> 16) & (mask >> 8) : 0u;
        // bits per sample, a byte each: U_q, one less where the exponent is known
        const uint4 g0 = s_code[code0], g1 = s_code[code1];
        const uint32_t b0 = (g0.x & (uq0 * 0x01010101u)) - g0.y;
        const uint32_t b1 = (g1.x & (uq1 * 0x01010101u)) - g1.y;
        // running sums, a byte each (at most 124)
        uint32_t a0 = b0 + (b0 << 8), a1 = b1 + (b1 << 8);
        a0 += a0 << 16;
        a1 += a1 << 16;
        const uint32_t t0 = a0 >> 24, tot = t0 + (a1 >> 24);
        const uint32_t incl = lanes.scan(tot);
        const uint32_t at = pos + incl - tot;
        pos += lanes.last(incl);
        // every bit this row reads, and the sign bit that a sample without
        // magnitude bits takes from the position after the last one
        const uint32_t need = on ? pos + 1 : 0;
        if (__any(fill < need)) {
            do {
                const bool act = fill < need;
                uint32_t d0 = raw.x, d1 = raw.y;
                const int32_t over8 = (int32_t)(next + 8 - end);  // bytes past the end
                if (over8 > 0) {
                    d1 |= over8 >= 4 ? 0xFFFFFFFFu : 0xFFFFFFFFu << (32 - 8 * over8);
                    if (over8 > 4) d0 |= over8 >= 8 ? 0xFFFFFFFFu : 0xFFFFFFFFu << (64 - 8 * over8);
                }
                if (act) {
                    next += 8 * L;
                    if (next < end) __builtin_memcpy(&raw, arena + next, 8);
                }
                // bytes that are 0xFF, and those after one
                const uint32_t f0 = bytes_ff(d0), f1 = bytes_ff(d1);
                uint32_t pf = lanes.before(f1);
                if (q == 0) pf = prev;
                uint32_t n0, n1;
                const uint32_t v0 = close_up(d0, __builtin_amdgcn_alignbit(f0, pf, 24) >> 7, n0);
                const uint32_t v1 = close_up(d1, __builtin_amdgcn_alignbit(f1, f0, 24) >> 7, n1);
                const uint32_t sc = lanes.scan(n0 + n1), bits = lanes.last(sc), last = lanes.last(f1);
                const uint32_t wz = (fill >> 5) + 1 + q;
                if (act) {
                    // the words past the partly filled one that this round reaches
                    ring[wz & (kMagRing - 1)] = 0;
                    ring[(wz + L) & (kMagRing - 1)] = 0;
                }
                wave_lds_fence();
                if (act) {
                    const uint32_t b = fill + sc - (n0 + n1), sh = b & 31u, wa = b >> 5;
                    const uint64_t v = (uint64_t)v0 | ((uint64_t)v1 << n0);
                    const uint64_t x = v << sh;
                    const uint32_t y = (uint32_t)(v >> 32) >> 1 >> (31u - sh);
                    atomicOr(&ring[wa & (kMagRing - 1)], (uint32_t)x);
                    atomicOr(&ring[(wa + 1) & (kMagRing - 1)], (uint32_t)(x >> 32));
                    atomicOr(&ring[(wa + 2) & (kMagRing - 1)], y);
                    fill += bits;
                    prev = last;
                }
                wave_lds_fence();
            } while (__any(fill < need));
            ring[kMagRing] = ring[0];
            wave_lds_fence();
        }
        // stream bits at the row's position plus off
        auto window = [&](uint32_t off) -> uint32_t {
            const uint32_t b = at + off, wi = (b >> 5) & (kMagRing - 1);
            return __builtin_amdgcn_alignbit(ring[wi + 1], ring[wi], b & 31u);
        };
        auto offset = [&](uint32_t k) -> uint32_t {  // of sample k in the lane's bits
            return k == 0   ? 0u
                   : k < 4  ? (a0 >> (8 * (k - 1))) & 0xFFu
                   : k == 4 ? t0
                            : t0 + ((a1 >> (8 * (k - 5))) & 0xFFu);
        };
        uint32_t bits[8];
        if constexpr (sizeof(C) == 2) {
            // a coded block of K <= 15 has zblk <= 14 (`on`), so U_q is at most 16 and
            // two samples come from one window
#pragma unroll
            for (uint32_t k = 0; k < 8; k += 2) {
                bits[k] = window(offset(k));
                bits[k + 1] = bits[k] >> (((k < 4 ? b0 : b1) >> (8 * (k & 3u))) & 31u);
            }
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) bits[k] = window(offset(k));
        }
        uint32_t vn[8], mag[8];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            const uint32_t m = ((k < 4 ? b0 : b1) >> (8 * (k & 3u))) & 31u;
            const uint32_t e = ((k < 4 ? g0.z : g1.z) >> (8 * (k & 3u))) & 0xFFu;
            // an insignificant sample has no bits: v is 1, its exponent 0
            vn[k] = __builtin_amdgcn_ubfe(bits[k], 0, m) | (e << m) | 1u;
            mag[k] = __builtin_amdgcn_ubfe((vn[k] + 2) << (p - 1), shift, 31u - shift);
        }
        e1 = 31u - __builtin_clz(vn[1]);
        e3 = 31u - __builtin_clz(vn[3]);
        e5 = 31u - __builtin_clz(vn[5]);
        e7 = 31u - __builtin_clz(vn[7]);
        // rows y and y + 1: signs applied, insignificant samples 0
        uint32_t o0[sizeof(C)], o1[sizeof(C)];
        if constexpr (sizeof(C) == 2) {
            // two samples a dword
            auto pair = [&](uint32_t k, uint32_t sig) -> uint32_t {
                const s16x2 m = __builtin_bit_cast(s16x2, mag[k] | (mag[k + 2] << 16));
                const s16x2 neg = __builtin_bit_cast(
                    s16x2, __builtin_amdgcn_perm(bits[k + 2], bits[k], 0x05040100u) & 0x00010001u);
                const s16x2 x = (m ^ -neg) + neg;
                return __builtin_bit_cast(uint32_t, x) &
                       __builtin_amdgcn_perm(0u, sig, k & 1u ? 0x03030101u : 0x02020000u);
            };
            o0[0] = pair(0, g0.x);
            o0[1] = pair(4, g1.x);
            o1[0] = pair(1, g0.x);
            o1[1] = pair(5, g1.x);
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {
                const uint32_t sgn = (uint32_t)((int32_t)(bits[k] << 31) >> 31);
                const uint32_t sig =
                    (uint32_t)((int32_t)((k < 4 ? g0.x : g1.x) << (31 - 8 * (k & 3u))) >> 31);
                (k & 1u ? o1 : o0)[k >> 1] = ((mag[k] ^ sgn) - sgn) & sig;
            }
        }
        if (live && cols) {
            const bool second = 2 * r + 1 < h;
            if (vec) {
                if constexpr (sizeof(C) == 2) {
                    *reinterpret_cast<uint2 *>(out) = make_uint2(o0[0], o0[1]);
                    if (second) *reinterpret_cast<uint2 *>(out + stride) = make_uint2(o1[0], o1[1]);
                } else {
                    *reinterpret_cast<uint4 *>(out) = make_uint4(o0[0], o0[1], o0[2], o0[3]);
                    if (second)
                        *reinterpret_cast<uint4 *>(out + stride) =
                            make_uint4(o1[0], o1[1], o1[2], o1[3]);
                }
            } else {
                constexpr uint32_t kPer = 4 / sizeof(C);  // samples a dword
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c) {
                    if (c >= cols) break;
                    const uint32_t sh = 16 * (c % kPer);
                    out[c] = (C)(int32_t)(o0[c / kPer] >> sh);
                    if (second) out[stride + c] = (C)(int32_t)(o1[c / kPer] >> sh);
                }
            }
            out += 2 * stride;
        }
    }
    if (bad) {  // a malformed block reads as zeros
        C *o = coef + j.dst + 4 * q;
        for (uint32_t y = 0; y < h; ++y, o += stride)
            for (uint32_t c = 0; c < cols; ++c) o[c] = 0;
    }
    if (valid && q == 0) status[i] = bad ? kCbBad : kCbOk;
}

// ---- refinement passes ---------------------------------------------------------
//
// SigProp (ht_block_decode.rs:1254-1374) is a serial chain per block, over
// significance alone; what it finds and the MagRef bits are then applied to all
// samples in parallel.  After the cleanup a sample is significant exactly when
// it is nonzero (ht_refine.hpp).  Three kernels as for the cleanup; one lane
// per block doing everything, samples included, took 1290 us for 512 tiles of
// 256x256 with both passes in every block; prepare 69, chain 123 and apply 121
// us do the same (the two parallel ones move 200 and 400 MB of samples in rows
// of up to 128 bytes, the chain issues about 12 instructions a sample).

// A refined block's part of its group's workspace; pass count rules of
// decode_impl (:1578-1592).
struct RefWork {
    uint4 *cs, *out, *sp;
};
__device__ __forceinline__ RefWork ref_work(uint4 *work, const RefGroup *groups, uint32_t i) {
    const RefGroup g = groups[i / kHtGroup];
    RefWork w;
    w.cs = work + g.base + i % kHtGroup;
    w.out = w.cs + size_t(kHtGroup) * 2 * g.stripes;
    w.sp = w.out + size_t(kHtGroup) * 4 * g.stripes;
    return w;
}
__device__ __forceinline__ bool ref_runs(const CbJob &j) {
    return !(j.flags & kCbZero) && j.passes >= 2 && j.passes <= 3 && j.lref != 0 && j.zblk < 29 &&
           j.lcup >= 2 && j.w <= 64 && j.h <= 64;
}

// Significance of the cleanup (16 bits per group of 4x4 samples, bit 4 column +
// row; two groups a dword) and the plain SigProp bits: LSB-first, 7 bits after
// 0xFF, zeros past the end.  One block per L lanes, a group a lane.
template <typename C, uint32_t L>
__global__ void __launch_bounds__(kSplitWaves * 64)
sgn_ht_refine_prep(const CbJob *__restrict__ jobs, uint32_t n, const uint8_t *__restrict__ arena,
                   const C *__restrict__ coef, const RefGroup *__restrict__ groups,
                   uint4 *__restrict__ work) {
    __shared__ __attribute__((aligned(16))) uint32_t s_buf[split_blocks(L)][kCleanRing<L>];
    const uint32_t row = threadIdx.x / L, q = threadIdx.x % L;
    const BlockLanes<L> lanes{q};
    const uint32_t i = blockIdx.x * split_blocks(L) + row;
    CbJob j{};
    if (i < n) j = jobs[i];
    const bool on = i < n && ref_runs(j);
    const RefWork w = ref_work(work, groups, i < n ? i : 0);
    // SigProp bytes, eight a lane
    const uint32_t len = on ? min((uint32_t)j.lref, kRefSpBytes) : 0;
    const uint8_t *src = arena + j.src + j.lcup;
    PlainString<L> str(s_buf[row], q, w.sp, (8 * len + 127) >> 7, 0, 0);
    uint32_t prev = 0;
    for (uint32_t at = 0; __any(at < len); at += 8 * L) {
        const uint32_t k = at + 8 * q;
        uint2 d = make_uint2(0, 0);
        if (k < len) {
            __builtin_memcpy(&d, src + k, 8);
            const uint32_t have = (uint32_t)j.lref - k;  // the rest are not of the segment
            if (have < 8) d.y &= have > 4 ? 0xFFFFFFFFu >> (8 * (8 - have)) : 0u;
            if (have < 4) d.x &= 0xFFFFFFFFu >> (8 * (4 - have));
        }
        const uint32_t f0 = bytes_ff(d.x), f1 = bytes_ff(d.y);
        uint32_t pf = lanes.before(f1);
        if (q == 0) pf = prev;
        prev = lanes.last(f1);
        uint32_t n0, n1;
        const uint32_t v0 = close_up(d.x, __builtin_amdgcn_alignbit(f0, pf, 24) >> 7, n0);
        const uint32_t v1 = close_up(d.y, __builtin_amdgcn_alignbit(f1, f0, 24) >> 7, n1);
        str.round(at < len, v0, n0, v1, n1);
    }
    if (on) str.finish();
    // significance
    const bool vec = ((j.dst | j.stride) & 3u) == 0;
    const C *out = coef + j.dst;
    const uint32_t stripes = on ? (j.h + 3u) >> 2 : 0;
    uint16_t *cs = reinterpret_cast<uint16_t *>(w.cs + kHtGroup * (q >> 3)) + (q & 7u);
    for (uint32_t s = 0; s < stripes; ++s) {
        int32_t v[4][4];
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r)
            refine_load<C>(v[r], out, 4 * s + r, 4 * q, j.w, j.h, j.stride, vec);
        cs[s * (kHtGroup * 16)] = (uint16_t)group_sig(v);
        if constexpr (L < 8) cs[s * (kHtGroup * 16) + L] = 0;  // the group beside the last
    }
}

// SigProp of one block per lane: per group the samples that become
// significant and the 16 stream bits that their signs start.  The bits come
// through an LDS ring as in sgn_ht_symbols: four groups take at most 128.
// Full waves, unlike the symbol chain: every lane issues the same instructions
// for every group, so half-filled waves gain nothing at 38000 blocks (125
// against 124 us) and lose at 150000 (341 against 200 us).
__global__ void __launch_bounds__(kSplitWaves * 64)
sgn_ht_sigprop(const CbJob *__restrict__ jobs, uint32_t n, const RefGroup *__restrict__ groups,
               uint4 *__restrict__ work) {
    __shared__ uint32_t s_ring[kSplitWaves][17][64];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t i = blockIdx.x * kSplitWaves * 64 + threadIdx.x;
    const bool valid = i < n;
    uint32_t(*ring)[64] = s_ring[wv];
    CbJob j{};
    if (valid) j = jobs[i];
    const bool on = valid && ref_runs(j);
    if (!on) j.w = j.h = 0;
    const RefWork w = ref_work(work, groups, valid ? i : 0);
    const uint32_t width = j.w, height = j.h, stripes = (height + 3u) >> 2;
    const uint32_t groups_x = (width + 3u) >> 2;
    const bool causal = (j.flags & kCbStripeCausal) != 0;
    const uint32_t last = (8 * min((uint32_t)j.lref, kRefSpBytes) + 127) >> 7;  // zeros from here
    auto unit = [&](uint32_t u) -> uint4 { return w.sp[kHtGroup * min(u, last)]; };
    auto put = [&](uint32_t u, const uint4 &v) {
        const uint32_t s = (u & 3u) * 4u;
        ring[s + 0][lane] = v.x;
        ring[s + 1][lane] = v.y;
        ring[s + 2][lane] = v.z;
        ring[s + 3][lane] = v.w;
        ring[s ? s : 16u][lane] = v.x;
    };
    uint4 pend = make_uint4(0, 0, 0, 0);
    uint32_t res = 4, pos = 0;
    uint32_t cur[9], nxt[9], bot[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) cur[k] = nxt[k] = bot[k] = 0;
    auto load_cs = [&](uint32_t s, uint32_t (&c)[9]) {
        const uint4 a = w.cs[kHtGroup * (2 * s)], b = w.cs[kHtGroup * (2 * s + 1)];
        c[0] = a.x, c[1] = a.y, c[2] = a.z, c[3] = a.w;
        c[4] = b.x, c[5] = b.y, c[6] = b.z, c[7] = b.w;
    };
    if (on) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) put(k, unit(k));
        pend = unit(4);
        load_cs(0, nxt);
    }
    for (uint32_t s = 0; __any(s < stripes); ++s) {
        const bool run = s < stripes;
#pragma unroll
        for (int k = 0; k < 8; ++k) cur[k] = nxt[k];
        if (s + 1 < stripes) {
            load_cs(s + 1, nxt);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) nxt[k] = 0;
        }
        const uint32_t rows = run ? min(4u, height - 4 * s) : 0;
        const uint32_t pattern = 0x1111u * ((1u << rows) - 1u);
        uint32_t prev = 0, found[16];
        uint32_t nbot[8];
#pragma unroll
        for (uint32_t g = 0; g < 16; ++g) {
            found[g] = 0;
            if ((g & 1u) == 0) nbot[g >> 1] = 0;
            if (!__any(run && g < groups_x)) continue;
            if ((g & 3u) == 0 && run && res < (pos >> 7) + 4u) {
                put(res, pend);
                ++res;
                pend = unit(res);
            }
            // this group's 16 bits and the next one's
            auto pair = [&](const uint32_t (&c)[9]) -> uint32_t {
                return g & 1u ? __builtin_amdgcn_alignbit(c[(g >> 1) + 1], c[g >> 1], 16)
                              : c[g >> 1];
            };
            const uint32_t cs = pair(cur), csa = cs & 0xFFFFu;
            // the row above as the reference's prev_row_sig holds it (see
            // rows_refine in ht_refine.hpp), the row below, and the column before
            uint32_t u = (((g ? cs : bot[0]) >> 3) & 0x1111u) | ((pair(bot) >> 3) & 0x11110000u);
            if (!causal) u |= (pair(nxt) & 0x11111111u) << 3;
            uint32_t mbr = cs | ((cs & 0x77777777u) << 1) | ((cs & 0xEEEEEEEEu) >> 1) | u;
            mbr |= (mbr << 4) | (mbr >> 4) | (prev >> 12);
            const uint32_t past = 4 * g + 4 > width ? 4 * g + 4 - width : 0u;  // columns past the block
            const uint32_t inv = run && past < 4 ? ~csa & (pattern >> (4 * past)) : 0u;
            uint32_t cand = mbr & inv, nsig = 0;
            const uint32_t k = (pos >> 5) & 15u;
            uint32_t bits = __builtin_amdgcn_alignbit(ring[k + 1][lane], ring[k][lane], pos & 31u);
            // All 16 places in order, without a branch: a member takes a bit,
            // and a one makes the insignificant samples below and in the next
            // column members too.  A loop over the members alone runs as often
            // as the fullest group of the wave needs and took 2.9 times as long
            // (356 against 123 us for 512 tiles of 256x256, two passes in
            // every block).
            if (__any(cand)) {
#pragma unroll
                for (uint32_t at = 0; at < 16; ++at) {
                    const uint32_t r = at & 3u, is = (cand >> at) & 1u, hit = bits & is;
                    const uint32_t nb = (((2u << r) & 0xFu) | ((((7u << r) >> 1) & 0xFu) << 4))
                                        << (at & ~3u);
                    cand |= (0u - hit) & (inv & nb);
                    nsig |= hit << at;
                    bits >>= is;
                }
            }
            found[g] = nsig | (bits << 16);
            pos += (uint32_t)__builtin_popcount(cand) + (uint32_t)__builtin_popcount(nsig);
            const uint32_t comb = nsig | cs;
            nbot[g >> 1] |= (comb & 0xFFFFu) << (16 * (g & 1u));
            const uint32_t np = comb | ((comb & 0x7777u) << 1) | ((comb & 0xEEEEu) >> 1);
            prev = (np | u) & 0xF000u;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) bot[k] = nbot[k];
        if (run) {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                if (4 * k < groups_x)
                    w.out[kHtGroup * (4 * s + k)] = make_uint4(found[4 * k], found[4 * k + 1],
                                                               found[4 * k + 2], found[4 * k + 3]);
        }
    }
}

// What SigProp found and the MagRef bits (:1377-1432), applied to the samples:
// one block per L lanes, a group a lane.  A sample that SigProp found gets the
// word 3 << (p - 2); MagRef exchanges bit p - 1 of a sample that the cleanup
// found for its bit and sets the midpoint 1 << (p - 2).  MagRef bits run
// backward from the segment's last byte with the VLC stuffing rule, zeros past
// its start, one per such sample in stripe-column order: a group's place is a
// prefix sum of the groups' counts (a stripe takes at most 256 bits).
template <typename C, uint32_t L>
__global__ void __launch_bounds__(kSplitWaves * 64)
sgn_ht_refine_apply(const CbJob *__restrict__ jobs, uint32_t n, const uint8_t *__restrict__ arena,
                    C *__restrict__ coef, const RefGroup *__restrict__ groups,
                    uint4 *__restrict__ work) {
    constexpr uint32_t kRing = 4 * L;  // dwords: a stripe's 16 L bits and a round's 64 L
    __shared__ uint32_t s_ring[split_blocks(L)][kRing + 1];  // and a copy of the first
    const uint32_t row = threadIdx.x / L, q = threadIdx.x % L;
    const BlockLanes<L> lanes{q};
    uint32_t *ring = s_ring[row];
    const uint32_t i = blockIdx.x * split_blocks(L) + row;
    CbJob j{};
    if (i < n) j = jobs[i];
    const bool on = i < n && ref_runs(j);
    if (!on) j.w = j.h = 0;
    const RefWork w = ref_work(work, groups, i < n ? i : 0);
    const bool mag = on && j.passes > 2;
    const uint32_t p = 30u - j.zblk, shift = j.kmax >= 31 ? 0u : 31u - j.kmax;
    const int32_t vnew = on ? (int32_t)((3u << (p - 2)) >> shift) : 0;
    const uint32_t ref0 = on ? ((1u << (p - 1)) | (1u << (p - 2))) >> shift : 0u;  // MagRef bit 0
    const uint32_t ref1 = on ? (1u << (p - 2)) >> shift : 0u;                      // MagRef bit 1
    const bool vec = ((j.dst | j.stride) & 3u) == 0;
    C *out = coef + j.dst;
    const uint32_t stripes = (j.h + 3u) >> 2;
    const uint32_t len = mag ? j.lref : 0, end = j.src + j.lcup + j.lref;
    uint32_t next = 8 * q, carry = 0x80000000u;  // the first byte counts as after one > 0x8F
    uint2 raw = make_uint2(0, 0);
    // bytes next .. next + 7 of the backward stream, the first in bits 0..7
    auto fetch = [&]() {
        raw = make_uint2(0, 0);
        if (next < len) {
            uint64_t x;
            const uint32_t e = end - next;  // one past the first
            if (e >= 8) {
                __builtin_memcpy(&x, arena + e - 8, 8);
            } else {
                __builtin_memcpy(&x, arena, 8);
                x <<= 8 * (8 - e);
            }
            raw.x = __builtin_bswap32((uint32_t)(x >> 32));
            raw.y = __builtin_bswap32((uint32_t)x);
            const uint32_t have = len - next;
            if (have < 8) raw.y &= have > 4 ? 0xFFFFFFFFu >> (8 * (8 - have)) : 0u;
            if (have < 4) raw.x &= 0xFFFFFFFFu >> (8 * (4 - have));
        }
    };
    fetch();
    uint32_t fill = 0, pos = 0;
    if (q == 0) ring[0] = ring[kRing] = 0;
    const uint32_t *found = reinterpret_cast<const uint32_t *>(w.out + kHtGroup * (q >> 2)) + (q & 3u);
    for (uint32_t s = 0; __any(s < stripes); ++s) {
        const bool run = s < stripes && 4 * q < j.w;
        int32_t v[4][4];
        uint32_t f = 0;
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) v[r][c] = 0;
        if (run) {
            f = found[s * (kHtGroup * 16)];
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
                refine_load<C>(v[r], out, 4 * s + r, 4 * q, j.w, j.h, j.stride, vec);
        }
        const uint32_t cs = group_sig(v);
        const uint32_t cnt = mag ? (uint32_t)__builtin_popcount(cs) : 0u;
        const uint32_t incl = lanes.scan(cnt);
        const uint32_t at = pos + incl - cnt;
        pos += lanes.last(incl);
        while (__any(fill < pos)) {
            const bool act = fill < pos;
            const uint32_t g0 = bytes_above(raw.x), g1 = bytes_above(raw.y);
            uint32_t pg = lanes.before(g1);
            if (q == 0) pg = carry;
            const uint32_t last = lanes.last(g1);
            uint32_t n0, n1;
            const uint32_t v0 =
                close_up(raw.x, (bytes_7f(raw.x) & __builtin_amdgcn_alignbit(g0, pg, 24)) >> 7, n0);
            const uint32_t v1 =
                close_up(raw.y, (bytes_7f(raw.y) & __builtin_amdgcn_alignbit(g1, g0, 24)) >> 7, n1);
            const uint32_t sc = lanes.scan(n0 + n1), bits = lanes.last(sc);
            if (act) {
                next += 8 * L;
                fetch();
                const uint32_t z = (fill >> 5) + 1 + q;
                ring[z & (kRing - 1)] = 0;
                ring[(z + L) & (kRing - 1)] = 0;
            }
            wave_lds_fence();
            if (act) {
                const uint32_t b = fill + sc - (n0 + n1), sh = b & 31u, wa = b >> 5;
                const uint64_t x = (uint64_t)v0 | ((uint64_t)v1 << n0), y = x << sh;
                atomicOr(&ring[wa & (kRing - 1)], (uint32_t)y);
                atomicOr(&ring[(wa + 1) & (kRing - 1)], (uint32_t)(y >> 32));
                atomicOr(&ring[(wa + 2) & (kRing - 1)], (uint32_t)(x >> 32) >> 1 >> (31u - sh));
                fill += bits;
                carry = last;
            }
            wave_lds_fence();
            ring[kRing] = ring[0];
            wave_lds_fence();
        }
        if (!run) continue;
        const uint32_t wi = (at >> 5) & (kRing - 1);
        uint32_t mw = __builtin_amdgcn_alignbit(ring[wi + 1], ring[wi], at & 31u);
        uint32_t nsig = f & 0xFFFFu, sg = f >> 16;
        const uint32_t refine = mag ? cs : 0u;
#pragma unroll
        for (uint32_t k = 0; k < 16; ++k) {
            int32_t &x = v[k & 3][k >> 2];
            const uint32_t hit = (refine >> k) & 1u, nw = (nsig >> k) & 1u;
            const uint32_t m = (uint32_t)(x < 0 ? -x : x) ^ ((mw & 1u) ? ref1 : ref0);
            const int32_t changed = x < 0 ? -(int32_t)m : (int32_t)m;
            x = hit ? changed : nw ? ((sg & 1u) ? -vnew : vnew) : x;
            mw >>= hit;
            sg >>= nw;
        }
        if (refine | nsig) {
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
                refine_store<C>(v[r], out, 4 * s + r, 4 * q, j.w, j.h, j.stride, vec);
        }
    }
}

// The same of long lists whose packet headers are parsed on the device (the host
// knows neither which blocks are refined nor their lengths, and reserves no
// workspace for all): all passes of the code-blocks jobs[0 .. n), one block per
// lane, after the cleanup kernels wrote their samples.  A block whose cleanup failed holds zeros or
// partial samples; the passes keep to its rectangle and its refinement
// segment whatever the samples, and its status already reports it.
template <typename C>
__global__ void __launch_bounds__(256)
sgn_ht_refine(const CbJob *__restrict__ jobs, uint32_t n, const uint8_t *__restrict__ arena,
              C *__restrict__ coef) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const CbJob j = jobs[i];
    // pass count rules of decode_impl (ht_block_decode.rs:1578-1592); more
    // than three passes never reach this kernel
    if ((j.flags & kCbZero) || j.passes < 2 || j.passes > 3 || j.lref == 0 || j.zblk >= 29 ||
        j.lcup < 2 || j.w > 64 || j.h > 64)
        return;
    const uint32_t shift = j.kmax >= 31 ? 0u : 31u - j.kmax;
    rows_refine<C>(coef + j.dst, j.w, j.h, j.stride, ((j.dst | j.stride) & 3u) == 0, arena,
                   j.src + j.lcup, j.lref, j.passes, (j.flags & kCbStripeCausal) != 0,
                   30u - j.zblk, shift);
}

}  // namespace sgn
