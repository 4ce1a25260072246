// Classic (EBCOT) code-block decode: the MQ arithmetic decoder (T.800
// Annex C) and the significance-propagation, magnitude-refinement and
// cleanup passes of Annex D, with the code-block styles selective bypass,
// context reset, termination on each pass, vertically causal context and
// segmentation symbols.  Follows
//   crates/signinum-j2k-native/src/j2c/bitplane.rs:90-317, 903-1116,
//   1228-1370 and arithmetic_decoder.rs:42-250, 329-386.
//
// Decomposition: one code-block per lane, a few lanes of each wave.  The MQ
// decoder is one serial chain per block (every decision updates the interval
// and the context the next decision reads), so the parallelism is across
// blocks, and the time is that of the longest chain.  The lanes of a wave run
// one loop whose turn is one decision of each, whatever its pass and kind, as
// straight-line code: a walk over the samples in step would make all lanes wait
// at every sample that any of them decides.
//
// A lane works on a group of eight stripe columns at a time.  Its masks are
// 64-bit strings with six bits a column (the row above, the stripe's four rows,
// the row below) and, where neighbours are needed, a column on either side; the
// pending samples of the pass are a mask as well, whose lowest bit is the next
// one in coding order, and a sample's neighbourhood is a shift of the
// significance string, looked up in a table.  The state of all groups stays in
// LDS (32 bytes a group), magnitude bits leave as one dword per group and pass,
// and the whole wave turns them into samples when its blocks are done.
//
// What bounds it: a turn is about 100 VALU and 50 scalar operations and three
// dependent LDS reads, 475 ns alone on a SIMD, and a 64x64 block of noise takes
// 37,500 of them; with many blocks the VALU.  256 tiles of 256x256 (19,200
// blocks) take 21 ms.  Sixteen lanes walking samples in step, with stripe rows
// fetched from memory and magnitude bits ORed into it one by one, took 50 ms
// (and 8.5 ms more for the 32-wide blocks in a launch of their own).
#include <hip/hip_runtime.h>

#include "../host/plan_types.h"

namespace sgn {

// Table C.2: Qe << 16 | index after an MPS << 8 | index after an LPS << 1 |
// MPS switch (the kernel's table, of both MPS values: see sgn_t1_classic).
__constant__ uint32_t kMqTable[47] = {
    0x56010103u, 0x3401020Cu, 0x18010312u, 0x0AC10418u, 0x0521053Au, 0x02212642u, 0x5601070Du,
    0x5401081Cu, 0x4801091Cu, 0x38010A1Cu, 0x30010B22u, 0x24010C24u, 0x1C010D28u, 0x16011D2Au,
    0x56010F1Du, 0x5401101Cu, 0x5101111Eu, 0x48011220u, 0x38011322u, 0x34011424u, 0x30011526u,
    0x28011626u, 0x24011728u, 0x2201182Au, 0x1C01192Cu, 0x18011A2Eu, 0x16011B30u, 0x14011C32u,
    0x12011D34u, 0x11011E36u, 0x0AC11F38u, 0x09C1203Au, 0x08A1213Cu, 0x0521223Eu, 0x04412340u,
    0x02A12442u, 0x02212544u, 0x01412646u, 0x01112748u, 0x0085284Au, 0x0049294Cu, 0x00252A4Eu,
    0x00152B50u, 0x00092C52u, 0x00052D54u, 0x00012D56u, 0x56012E5Cu,
};

constexpr int kClassicContexts = 19;
constexpr int kCxRunLength = 17, kCxUniform = 18;

// Reads of one codeword segment: absolute arena positions [p, end), bytes
// past `end` read as 0xFF (the MQ decoder's fill, arithmetic_decoder.rs:
// 250-270).  A window of three aligned dwords in registers; the third is
// fetched one dword ahead of use.
struct SegBytes {
    const uint8_t *arena;
    uint32_t end, wpos;  // wpos: arena offset of w0 (multiple of 4)
    uint32_t w0, w1, w2;

    __device__ void start(const uint8_t *a, uint32_t p, uint32_t e) {
        arena = a;
        end = e;
        wpos = p & ~3u;
        const uint32_t *q = reinterpret_cast<const uint32_t *>(a + wpos);
        w0 = q[0];
        w1 = q[1];
        w2 = q[2];
    }
    // byte at p (p >= wpos); slides the window so that p + 1 stays in w0..w1
    __device__ uint32_t at(uint32_t p) {
        if (p + 1 >= wpos + 8) {
            w0 = w1;
            w1 = w2;
            wpos += 4;
            w2 = *reinterpret_cast<const uint32_t *>(arena + wpos + 8);
        }
        const uint32_t rel = p - wpos;
        const uint32_t w = rel < 4 ? w0 : w1;
        const uint32_t b = (w >> ((rel & 3u) * 8u)) & 0xFFu;
        return p < end ? b : 0xFFu;
    }
};

// Raw (bypass) bits with B.10.1 stuffing; past the segment, or a stuffed
// bit that is not 0, yields 1 (bitplane.rs:1339-1370, non-strict).
struct RawBits {
    SegBytes in;
    uint32_t p, bit;  // byte position, bits consumed in it

    __device__ void init(const uint8_t *arena, uint32_t start, uint32_t len) {
        in.start(arena, start, start + len);
        p = start;
        bit = 0;
    }
    __device__ uint32_t get() {
        if (p >= in.end) return 1;
        const uint32_t byte = in.at(p);
        const uint32_t b = (byte >> (7 - bit)) & 1u;
        if (++bit == 8) {
            bit = 0;
            ++p;
        }
        if (bit == 0 && byte == 0xFFu) {  // the next byte's MSB is a stuffed 0
            if (p >= in.end) return 1;
            const uint32_t s = in.at(p) >> 7;
            bit = 1;
            if (s) return 1;
        }
        return b;
    }
};

// Table D.1 from neighbour counts (h, v, d; `swap` for HL, where the roles
// of horizontal and vertical swap; `diag` for HH).
__device__ inline uint32_t zc_label(uint32_t h, uint32_t v, uint32_t d, bool swap, bool diag) {
    if (diag) {
        const uint32_t hv = h + v;
        if (d >= 3) return 8;
        if (d == 2) return hv ? 7 : 6;
        if (d == 1) return hv >= 2 ? 5 : (hv ? 4 : 3);
        return hv >= 2 ? 2 : hv;
    }
    if (swap) {
        const uint32_t t = h;
        h = v;
        v = t;
    }
    if (h == 2) return 8;
    if (h == 1) return v ? 7 : (d ? 6 : 5);
    if (v == 2) return 4;
    if (v == 1) return 3;
    return d >= 2 ? 2 : d;
}

// Masks of a group of eight columns: column c at bits 6 c .. 6 c + 5, bit 0 of
// them the row above the stripe, bits 1-4 its rows, bit 5 the row below.
// `Wide` strings have one more column in front and behind.
constexpr uint64_t kRow0 = 0x0000041041041041ull;  // bit 0 of each column
constexpr uint64_t kRows = kRow0 * 0x1Eull;        // the stripe's rows
constexpr uint32_t kGroupCols = 8;

// Decision tables (bytes): the context of a sample by its neighbourhood index
// (zero coding in LL/LH, HL and HH bands; magnitude refinement, with the
// refined-before bit at 512), then sign coding (context | flip << 5) by sign
// index.
constexpr uint32_t kNbRun = 384, kNbUniform = 385, kNbEntries = 388, kNbRefined = 512;
constexpr uint32_t kTabMr = 3 * kNbEntries, kTabSign = kTabMr + 1024;
constexpr uint32_t kTabBytes = kTabSign + 1024;

// Neighbourhood index of the 15-bit window whose bit 7 is the sample (left
// column bits 0-2, own 6 and 8, right 12-14): right bits move to 3-5.
__device__ __forceinline__ uint32_t nb_index(uint32_t t) {
    return (t & 0x147u) | ((t >> 9) & 0x38u);
}
// Sign index: horizontal and vertical neighbours' significance (bits 1, 4, 6,
// 8) and sign (one above each).
__device__ __forceinline__ uint32_t sign_part(uint32_t t) {
    return (t & 0x142u) | ((t >> 9) & 0x10u);
}

__device__ inline uint8_t classic_table(uint32_t k) {
    if (k >= kTabSign) {
        // Table D.3
        const uint32_t i = k - kTabSign;
        auto contrib = [&](uint32_t b) -> int {
            return (i >> b) & 1u ? ((i >> (b + 1)) & 1u ? -1 : 1) : 0;
        };
        const int hs = contrib(1) + contrib(4), vs = contrib(6) + contrib(8);
        const int H = hs > 0 ? 1 : hs < 0 ? -1 : 0, V = vs > 0 ? 1 : vs < 0 ? -1 : 0;
        if (H == 0) return uint8_t(V == 0 ? 9 : V < 0 ? 10 | 32 : 10);
        return uint8_t((12 + H * V) | (H < 0 ? 32 : 0));
    }
    if (k >= kTabMr) return k - kTabMr >= kNbRefined ? 16 : k > kTabMr ? 15 : 14;
    const uint32_t tab = k / kNbEntries, i = k % kNbEntries;
    if (i == kNbRun) return kCxRunLength;
    if (i >= kNbUniform) return kCxUniform;
    const uint32_t h = ((i >> 1) & 1u) + ((i >> 4) & 1u), v = ((i >> 6) & 1u) + ((i >> 8) & 1u);
    const uint32_t d = (i & 1u) + ((i >> 2) & 1u) + ((i >> 3) & 1u) + ((i >> 5) & 1u);
    return uint8_t(zc_label(h, v, d, tab == 1, tab == 2));
}

// The MQ decoder: C inverted (ITU-T T.88 Annex G conventions), A in the upper
// half, the last byte read, and the next ones in two dwords (the second is
// fetched a dword ahead of its use).  Bytes from `end` on read as 0xFF
// (arithmetic_decoder.rs:250-270).
struct Mq {
    uint32_t c, a, ct, last;
    uint32_t w0, w1, left, pos, end;  // left: bytes in w0; pos: arena offset of w1
    const uint8_t *arena;

    __device__ __forceinline__ uint32_t masked(uint32_t w, uint32_t at) const {
        const int have = (int)(end - at);
        return have >= 4 ? w : have <= 0 ? 0xFFFFFFFFu : w | (0xFFFFFFFFu << (8 * have));
    }
    __device__ __forceinline__ void bytein() {
        const uint32_t b1 = w0 & 0xFFu;
        const bool ff = last == 0xFFu, stop = ff && b1 > 0x8Fu;  // a marker or the end: 1 bits
        c += stop ? 0u : ff ? 0xFE00u - (b1 << 9) : 0xFF00u - (b1 << 8);
        ct = ff && !stop ? 7u : 8u;
        if (!stop) {
            last = b1;
            w0 >>= 8;
            if (--left == 0) {
                w0 = masked(w1, pos);
                left = 4;
                pos += 4;
                w1 = *reinterpret_cast<const uint32_t *>(arena + pos);
            }
        }
    }
    __device__ void init(const uint8_t *ar, uint32_t start, uint32_t len) {
        arena = ar;
        end = start + len;
        const uint32_t a0 = start & ~3u;
        const uint32_t *q = reinterpret_cast<const uint32_t *>(ar + a0);
        w0 = masked(q[0], a0) >> (8 * (start & 3u));
        left = 4 - (start & 3u);
        w1 = q[1];
        pos = a0 + 4;
        last = w0 & 0xFFu;
        c = (last ^ 0xFFu) << 16;
        w0 >>= 8;
        if (--left == 0) {
            w0 = masked(w1, pos);
            left = 4;
            pos += 4;
            w1 = *reinterpret_cast<const uint32_t *>(ar + pos);
        }
        bytein();
        c <<= 7;
        ct -= 7;
        a = 0x80000000u;
    }
    // Decision with the context word *cx: a table entry (Qe << 16 | entry after
    // an MPS << 8 | entry after an LPS << 1 | MPS).
    __device__ __forceinline__ uint32_t decode(uint32_t *cx, const uint32_t *qtab) {
        const uint32_t e = *cx, qe = e & 0xFFFF0000u;
        a -= qe;
        const bool lps = c >= a;
        // conditional exchange (C.3.2): the decision is the LPS, and the state
        // moves on the LPS side, exactly when (a < qe) differs from the
        // sub-interval the code value fell in
        const bool took_lps = (a < qe) != lps;
        c -= lps ? a : 0u;
        a = lps ? qe : a;
        if (!(a & 0x80000000u)) {
            const uint32_t ne = qtab[took_lps ? (e >> 1) & 0x7Fu : (e >> 8) & 0x7Fu];
            uint32_t n = (uint32_t)__builtin_clz(a), sh = min(n, ct);
            a <<= n;
            c <<= sh;
            ct -= sh;
            for (n -= sh; n; n -= sh) {
                bytein();
                sh = min(n, ct);
                c <<= sh;
                ct -= sh;
            }
            *cx = ne;
        }
        return (e & 1u) ^ (took_lps ? 1u : 0u);
    }
};

// Groups a lane keeps in LDS (significance and sign have a stripe of zeros
// above and below), the lanes in use, and whether segments may be raw.
template <int GROUPS, int PADDED, int LANES, bool RAW>
struct ClassicShape {
    static constexpr bool kRaw = RAW;
    static constexpr uint32_t kGroups = GROUPS, kPadded = PADDED, kLanes = LANES;
    static constexpr uint32_t kWords = 2 * (GROUPS + PADDED) * LANES;
};
__host__ __device__ inline uint32_t classic_groups(uint32_t w, uint32_t h) {
    return ((w + kGroupCols - 1) / kGroupCols) * ((h + 3) >> 2);
}
__host__ __device__ inline uint32_t classic_padded(uint32_t w, uint32_t h) {
    return ((w + kGroupCols - 1) / kGroupCols) * (((h + 3) >> 2) + 2);
}
// Dwords of a lane's magnitude bits: per bit-plane and group one of the
// significance passes and one of the refinement.
__host__ __device__ inline uint32_t classic_mag_dwords(uint32_t planes, uint32_t groups) {
    return 2 * planes * groups;
}

// The stripe's rows of a group's mask: four bits a column.
__device__ __forceinline__ uint32_t group_nibbles(uint64_t m) {
    const uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
    uint32_t n = (lo >> 1) & 0xFu;
    n |= ((lo >> 7) & 0xFu) << 4;
    n |= ((lo >> 13) & 0xFu) << 8;
    n |= ((lo >> 19) & 0xFu) << 12;
    n |= ((lo >> 25) & 0xFu) << 16;
    n |= (__builtin_amdgcn_alignbit(hi, lo, 31) & 0xFu) << 20;
    n |= ((hi >> 5) & 0xFu) << 24;
    return n | (((hi >> 11) & 0xFu) << 28);
}

template <class G>
struct ClassicLane {
    // LDS: the groups' masks (significance, sign, visited in this bit-plane's
    // significance pass, refined before) and the 19 contexts, lanes interleaved
    uint64_t *sig, *neg, *vis, *ref;
    uint32_t *cx;
    const uint32_t *qtab;
    const uint8_t *tab, *arena;
    uint32_t *mag;  // this lane's magnitude bits
    const ClassicSeg *segs;
    uint32_t src, len, ns, ng, band, style, planes, nseg, seg, passes;
    Mq mq;
    RawBits rb;
    bool raw;
    uint32_t p, p_end, kind, base;  // pass, end of its segment, pass kind, decision table
    uint32_t s, g;                  // stripe, group
    uint32_t mode;                  // 0 next sample, 1 its sign, 2 and 3 the run's uniform bits
    uint32_t run;
    // Strings of the group, a column in front and behind: significance; signs
    // (refinement: refined before); pending, visited and admitted samples;
    // magnitude bits.  next_*: the next group's first two.
    uint64_t E, N, cand, visited, valid, bits, next_e, next_n;
    uint64_t last_rows, last_cols, below;  // rows of the last stripe, columns of the last group

    __device__ __forceinline__ uint32_t &ctx(uint32_t k) { return cx[k * G::kLanes]; }
    __device__ void reset_contexts() {
        const uint32_t z = qtab[0];
        for (int k = 0; k < kClassicContexts; ++k) ctx(k) = z;
        ctx(0) = qtab[8];
        ctx(kCxRunLength) = qtab[6];
        ctx(kCxUniform) = qtab[92];
    }
    // The block's state before its first pass; false when there is none.
    __device__ bool start(const ClassicJob &j) {
        segs += j.seg;
        src = j.src;
        len = j.len;
        ns = (j.h + 3u) >> 2;
        ng = (j.w + kGroupCols - 1) / kGroupCols;
        band = j.band;
        style = j.style;
        planes = j.planes;
        passes = j.passes;
        nseg = j.nseg;
        below = (style & kCbsCausal) ? 0 : kRow0 << 5;
        last_cols = (1ull << (6 * (j.w - kGroupCols * (ng - 1)))) - 1;
        const uint32_t rows = j.h - 4 * (ns - 1);
        last_rows = 0;
        for (uint32_t r = 0; r < rows; ++r) last_rows |= kRow0 << (r + 1);
        seg = p = mode = run = 0;
        cand = visited = valid = bits = 0;
        reset_contexts();
        if (!open_segment()) return false;
        begin_pass();
        enter_group();
        return true;
    }
    // Opens the next segment with passes; false at the end of the data.
    __device__ bool open_segment() {
        const uint32_t maxp = 1 + 3 * (planes - 1);
        while (seg < max(nseg, 1u)) {
            if (nseg == 0) {
                raw = false;
                p_end = min(passes, maxp);
                mq.init(arena, src, len);
            } else {
                const ClassicSeg sg = segs[seg];
                raw = G::kRaw && sg.raw;
                p_end = min(uint32_t(sg.end), maxp);
                if (raw)
                    rb.init(arena, src + sg.off, sg.len);
                else
                    mq.init(arena, src + sg.off, sg.len);
            }
            ++seg;
            if (p < p_end) return true;
        }
        return false;
    }

    // Mask m of padded group k with the rows above and below.
    __device__ __forceinline__ uint64_t around(const uint64_t *m, uint32_t k) const {
        const uint64_t own = m[(k + ng) * G::kLanes], up = m[k * G::kLanes];
        const uint64_t dn = m[(k + 2 * ng) * G::kLanes];
        return own | ((up >> 4) & kRow0) | ((dn << 4) & below);
    }
    __device__ __forceinline__ void begin_stripe() {
        g = 0;
        next_e = around(sig, s * ng);
        next_n = around(neg, s * ng);
        E = N = 0;  // no column before the first
    }
    __device__ __forceinline__ void begin_pass() {
        kind = p % 3;
        base = kind == 2 ? kTabMr : band == 1 ? kNbEntries : band == 3 ? 2 * kNbEntries : 0u;
        s = 0;
        begin_stripe();
    }
    __device__ __forceinline__ uint32_t decide(uint32_t k) {
        if (G::kRaw && raw) return rb.get();
        return mq.decode(&ctx(k), qtab);
    }

    // Takes group g of the stripe.
    __device__ __forceinline__ void enter_group() {
        const uint32_t k = s * ng + g;
        const bool last = g + 1 == ng;
        const uint64_t le = (E >> 48) & 0x3Fu, ln = (N >> 48) & 0x3Fu;
        const uint64_t seen = vis[k * G::kLanes] << 6, refined = ref[k * G::kLanes] << 6;
        E = (next_e << 6) | le;
        N = (next_n << 6) | ln;
        next_e = next_n = 0;
        if (!last) {
            next_e = around(sig, k + 1);
            next_n = around(neg, k + 1);
        }
        E |= next_e << 54;
        N |= next_n << 54;
        N = kind == 2 ? refined : N;
        valid = ((s + 1 == ns ? last_rows : kRows) & (last ? last_cols : ~0ull)) << 6;
        const uint64_t a = E | (E << 1) | (E >> 1), near = a | (a << 6) | (a >> 6);
        visited = kind == 1 ? 0 : seen;
        cand = (kind == 2 ? E : kind == 1 ? near & ~E : ~E) & valid & ~visited;
        bits = kind == 0 ? E & visited : 0;  // the cleanup adds to what the first pass found
    }

    // The group is done: keeps its masks and takes the next one.  False at the
    // end of the block.
    __device__ __forceinline__ bool advance() {
        const uint32_t k = s * ng + g;
        if (kind == 2) {
            ref[k * G::kLanes] = (E >> 6) & kRows & ~(visited >> 6);
        } else {
            sig[(k + ng) * G::kLanes] = (E >> 6) & kRows;
            neg[(k + ng) * G::kLanes] = (N >> 6) & kRows;
            vis[k * G::kLanes] = kind ? visited >> 6 : 0;
        }
        const uint32_t slot = (p + 2) / 3 * 2 + (kind == 2 ? 1 : 0);
        mag[slot * (ns * ng) + k] = group_nibbles(bits >> 6);
        if (++g == ng) {
            if (++s == ns) {
                if (kind == 0 && (style & kCbsSegSym))  // four symbols, not checked (non-strict)
#pragma unroll 1
                    for (int q = 0; q < 4; ++q) (void)decide(kCxUniform);
                if (style & kCbsReset) reset_contexts();
                if (++p >= p_end && !open_segment()) return false;
                begin_pass();
            } else {
                begin_stripe();
            }
        }
        enter_group();
        return true;
    }

    // One decision of the next pending sample.
    __device__ __forceinline__ void decision() {
        const uint32_t lo = (uint32_t)cand, hi = (uint32_t)(cand >> 32);
        const uint32_t q = lo ? (uint32_t)__builtin_ctz(lo) : 32u + (uint32_t)__builtin_ctz(hi);
        const uint64_t one = 1ull << q;
        const uint32_t t = (uint32_t)(E >> (q - 7)), tn = (uint32_t)(N >> (q - 7));
        const bool sign = mode == 1;
        uint32_t at = base + (nb_index(t) | ((tn << 2) & kNbRefined));
        bool runs = false;
        if (mode != 0 || kind == 0) {
            // run-length mode (D.3.4): a whole column pending in the cleanup
            // pass, nothing significant in it or beside it
            runs = mode == 0 && (t & 0x3FFFFu) == 0 && ((uint32_t)(cand >> q) & 0xFu) == 0xFu &&
                   (one & (kRow0 << 7)) != 0;
            at = runs ? base + kNbRun : at;
            at = mode >= 2 ? base + kNbUniform : at;
            at = sign ? kTabSign + (sign_part(t) | (sign_part(tn) << 1)) : at;
        }
        const uint32_t entry = tab[at];
        uint32_t d = decide(entry & 31u);
        if (!(G::kRaw && raw)) d ^= entry >> 5;  // a raw sign bit is the sign itself
        // a significant sample stays pending for its sign
        const bool found = mode == 0 && kind != 2 && d;
        uint64_t settled = found ? 0 : one;
        uint32_t next = found ? 1 : 0;
        if (runs || mode >= 2) {
            if (runs) {
                settled = d ? 0 : one * 15u;
                next = d ? 2 : 0;
            } else if (mode == 2) {
                settled = 0;
                next = 3;
                run = d << 1;
            } else {
                settled = (one << (run | d)) - one;
                next = 1;
            }
        }
        cand &= ~settled;
        visited |= kind == 1 ? one : 0;
        bits |= sign || (kind == 2 && d) ? one : 0;
        if (sign) {
            E |= one;
            N |= d ? one : 0;
            // samples further on that it makes members
            if (kind == 1) cand |= (0xE2ull << q) & valid & ~E;
        }
        mode = next;
    }
};

// Magnitude bits and signs of block j to samples, a group per lane of the wave.
template <class G>
__device__ void classic_samples(const ClassicJob &j, uint32_t passes, const uint32_t *mag,
                                const uint64_t *neg, int32_t *coef) {
    const uint32_t ng = (j.w + kGroupCols - 1) / kGroupCols, groups = ng * ((j.h + 3u) >> 2);
    for (uint32_t k = threadIdx.x; k < groups; k += 64) {
        uint32_t v[32];
#pragma unroll
        for (int q = 0; q < 32; ++q) v[q] = 0;
        for (uint32_t pl = 0; pl < j.planes; ++pl) {
            if ((pl ? 3 * pl - 2 : 0) >= passes) break;
            uint32_t m = mag[2 * pl * groups + k];
            if (pl && 3 * pl - 1 < passes) m |= mag[(2 * pl + 1) * groups + k];
            const uint32_t bit = j.planes - 1 - pl;
#pragma unroll
            for (int q = 0; q < 32; ++q) v[q] |= ((m >> q) & 1u) << bit;
        }
        const uint32_t nb = group_nibbles(neg[(ng + k) * G::kLanes]);
        const uint32_t x0 = (k % ng) * kGroupCols, y0 = (k / ng) * 4;
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
            if (y0 + r >= j.h) break;
            int32_t *row = coef + j.dst + (y0 + r) * j.stride + x0;
#pragma unroll
            for (uint32_t c = 0; c < kGroupCols; ++c) {
                const int32_t m = (int32_t)v[4 * c + r];
                if (x0 + c < j.w) row[c] = (nb >> (4 * c + r)) & 1u ? -m : m;
            }
        }
    }
}

// One wave per work-group, kLanes of its lanes decoding a block each; a lane
// whose block is done takes the next of the list (*queue, zero at launch, counts
// those taken after the first gridDim.x * kLanes).  Each lane keeps its
// magnitude bits at mag + (blockIdx.x * kLanes + lane) * mag_dwords.
template <class G>
__global__ void __launch_bounds__(64)
sgn_t1_classic(const ClassicJob *__restrict__ jobs, uint32_t n, const uint8_t *__restrict__ arena,
               const ClassicSeg *__restrict__ segs, int32_t *__restrict__ coef,
               uint32_t *__restrict__ mag, uint32_t mag_dwords, uint32_t *queue) {
    __shared__ uint64_t s_mask[G::kWords];  // significance, sign (padded), visited, refined
    __shared__ uint32_t s_cx[kClassicContexts * G::kLanes];
    __shared__ uint32_t s_qtab[94];
    __shared__ uint8_t s_tab[kTabBytes];
    const uint32_t lane = threadIdx.x;
    for (uint32_t k = lane; k < 94; k += 64) {
        // entry 2 i + m: state i with MPS m
        const uint32_t e = kMqTable[k >> 1], m = k & 1u;
        const uint32_t nm = ((e >> 8) & 0x3Fu) * 2 + m;
        const uint32_t nl = ((e >> 1) & 0x7Fu) * 2 + ((e & 1u) ? 1u - m : m);
        s_qtab[k] = (e & 0xFFFF0000u) | (nm << 8) | (nl << 1) | m;
    }
    for (uint32_t k = lane; k < kTabBytes; k += 64) s_tab[k] = classic_table(k);
    const uint32_t me = min(lane, G::kLanes - 1), taken = gridDim.x * G::kLanes;
    uint32_t *const wave_mag = mag + size_t(blockIdx.x) * G::kLanes * mag_dwords;
    ClassicLane<G> L;
    L.sig = s_mask + me;
    L.neg = L.sig + G::kPadded * G::kLanes;
    L.vis = L.neg + G::kPadded * G::kLanes;
    L.ref = L.vis + G::kGroups * G::kLanes;
    L.cx = s_cx + me;
    L.qtab = s_qtab;
    L.tab = s_tab;
    L.arena = arena;
    L.mag = wave_mag + size_t(me) * mag_dwords;
    uint32_t job = lane < G::kLanes ? blockIdx.x * G::kLanes + lane : n;
    bool fresh = job < n, alive = false;
    // every turn ends a block of some lane, so at most n turns
    while (__any(alive || fresh)) {
        for (uint64_t m = __ballot(fresh); m; m &= m - 1) {
            const uint32_t b = (uint32_t)__builtin_ctzll(m);
            for (uint32_t k = lane; k < G::kWords / G::kLanes; k += 64)
                s_mask[k * G::kLanes + b] = 0;
        }
        __syncthreads();
        bool ended = false;
        if (fresh) {
            const ClassicJob j = jobs[job];
            L.segs = segs;
            L.p = 0;
            alive = j.planes && j.passes && L.start(j);
            ended = !alive;
            fresh = false;
        }
        do {
            if (alive && L.cand == 0) {
                alive = L.advance();
                ended = !alive;
            }
            if (alive && L.cand != 0) L.decision();
        } while (!__any(ended));
        __syncthreads();
        for (uint64_t m = __ballot(ended); m; m &= m - 1) {
            const uint32_t b = (uint32_t)__builtin_ctzll(m);
            const uint32_t i = (uint32_t)__builtin_amdgcn_readlane((int)job, (int)b);
            const uint32_t passes = (uint32_t)__builtin_amdgcn_readlane((int)L.p, (int)b);
            classic_samples<G>(jobs[i], passes, wave_mag + size_t(b) * mag_dwords,
                               s_mask + G::kPadded * G::kLanes + b, coef);
        }
        __syncthreads();
        if (ended) {
            job = taken + atomicAdd(queue, 1u);
            fresh = job < n;
        }
    }
}

}  // namespace sgn
