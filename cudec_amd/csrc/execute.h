/* Executing sequences on gfx950: what the LZ4, Snappy and Zstandard decoders
 * share once literals and matches are known. Internal, device code only.
 *
 * A wave holds up to 64 sequences, one a lane, and writes their output
 * through a ring in LDS: literals and independent matches a lane each, the
 * rest in stream order with the wave fanned out over the bytes; whole
 * 16-byte blocks leave with aligned stores. A sequence too long for a group
 * goes global to global. Also here: staging a source range in LDS, the wave
 * scan, and the LDS words that the waves of a block signal through. */
#ifndef CUDEC_AMD_EXECUTE_H
#define CUDEC_AMD_EXECUTE_H

#include "common.h"
#include "ladder.h"

namespace cudec_amd {
namespace {

constexpr uint32_t kRing = 4096;     /* a one-wave decoder's output ring */
constexpr uint32_t kBatchMax = 2048; /* output bytes of one of its groups */
constexpr uint32_t kLaneLit = 64;    /* literal runs copied by their lane */
constexpr uint32_t kLaneMatch = 64;  /* matches copied by their lane (<= 64) */
static_assert(kBatchMax + 32 <= kRing, "ring must hold a batch and a margin");
static_assert(kBatchMax <= 64 * kWave, "CoverLds marks a batch");
static_assert((kRing & (kRing - 1)) == 0, "rings are powers of two");
static_assert(kLaneMatch <= 64, "a lane match copies at most four 16-byte blocks");

/* An output ring of kR bytes (a power of two). */
template <uint32_t kR>
struct alignas(16) RingLds {
    static constexpr uint32_t kSize = kR;
    uint8_t ring[kR];
    uint8_t sink[kWave]; /* stores of lanes with nothing to store */
};
/* Which members of a group cover given bytes of its output: a bit for each
 * member's first byte and, per 64 bytes, the members before them. */
struct alignas(16) CoverLds {
    uint64_t starts[kWave];
    uint8_t before[kWave];
};

template <uint32_t kR = kRing>
__device__ __forceinline__ uint32_t ring_index(uintptr_t dst_addr, uint64_t pos) {
    return (uint32_t)(dst_addr + pos) & (kR - 1);
}

/* ------------------------------------------------------------ staging */

/* Loads compressed bytes [sp, sp + bytes) of the chunk into stage and
 * returns the offset of byte sp inside it. Only aligned 16-byte blocks that
 * hold a byte of [sp, src_size) are read (so none leaves the chunk's
 * pages); later blocks are zero-filled. Every load of the kRounds of 64
 * blocks is issued before the first is stored, with no branch around it
 * (a lane without a block reads the first one again): a load a round took
 * a memory latency a round. Bytes past src_size are never trusted: every
 * member is validated against src_size before anything it read is used. */
template <uint32_t kRounds>
__device__ __forceinline__ uint32_t stage_into(uint8_t* stage, gcu8* src,
                                               uint64_t src_size, uint64_t sp,
                                               uint32_t bytes, uint32_t lane) {
    const uintptr_t a = (uintptr_t)(src + sp);
    const uintptr_t base = a & ~(uintptr_t)15;
    const uintptr_t end = (uintptr_t)src + src_size;
    const uint32_t blocks = (bytes + 30) / 16; /* whatever the alignment of sp */
    uint4 v[kRounds];
    if (sp < src_size) {
#pragma unroll
        for (uint32_t i = 0; i < kRounds; i++) {
            const uint32_t blk = lane + i * kWave;
            const uintptr_t g = base + 16u * blk;
            v[i] = gload16((gcu8*)(blk < blocks && g < end ? g : base));
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < kRounds; i++) {
        const uint32_t blk = lane + i * kWave;
        if (blk < blocks) {
            const bool in = sp < src_size && base + 16u * blk < end;
            *reinterpret_cast<uint4*>(&stage[16u * blk]) = in ? v[i] : make_uint4(0, 0, 0, 0);
        }
    }
    wave_order();
    return (uint32_t)(a - base);
}

/* ------------------------------------------------------------ wave scan */

__device__ __forceinline__ uint32_t wave_inclusive_sum(uint32_t v, uint32_t lane) {
    /* DPP: an inclusive scan inside each row of 16 lanes (row_shr 1, 2, 4,
     * 8; a lane with no source adds the 0 it keeps), then lane 15 of each
     * row into rows 1 and 3 (row_bcast:15) and lane 31 into rows 2 and 3
     * (row_bcast:31). No LDS traffic. */
    (void)lane;
    int x = (int)v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false); /* row_shr:1 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false); /* row_shr:2 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false); /* row_shr:4 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false); /* row_shr:8 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false); /* row_bcast:15 */
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false); /* row_bcast:31 */
    return (uint32_t)x;
}

/* ----------------------------------------------------- ring <-> global */

/* Stores ring bytes of positions [from, to) to dst. Full aligned 16-byte
 * blocks go out as one vector store per lane; the partial blocks at either
 * end (only at the chunk's first byte or its last) as single bytes. */
template <class W>
__device__ __forceinline__ void flush_ring(const W& w, gu8* dst,
                                           uint64_t from, uint64_t to,
                                           uint32_t lane) {
    if (to <= from) {
        return;
    }
    const uintptr_t da = (uintptr_t)dst;
    const uintptr_t a0 = da + from;
    const uintptr_t a1 = da + to;
    uintptr_t b0 = (a0 + 15) & ~(uintptr_t)15;
    uintptr_t b1 = a1 & ~(uintptr_t)15;
    if (b0 > a1) {
        b0 = a1;
    }
    if (b1 < b0) {
        b1 = b0;
    }
    /* head bytes [a0, b0) and tail bytes [b1, a1): fewer than 16 each */
    const uint32_t head = (uint32_t)(b0 - a0);
    const uint32_t tail = (uint32_t)(a1 - b1);
    if (lane < head) {
        const uintptr_t g = a0 + lane;
        *(gu8*)g = w.ring[g & (W::kSize - 1)];
    } else if (lane >= 16 && lane < 16 + tail) {
        const uintptr_t g = b1 + (lane - 16);
        *(gu8*)g = w.ring[g & (W::kSize - 1)];
    }
    const uint32_t blocks = (uint32_t)((b1 - b0) / 16);
    for (uint32_t b = lane; b < blocks; b += kWave) {
        const uintptr_t g = b0 + 16u * b;
        const uint4 v = *reinterpret_cast<const uint4*>(&w.ring[g & (W::kSize - 1)]);
        gstore16((gu8*)g, v);
    }
    wave_order();
}

/* One output byte of history: from the ring when its position is still
 * there, else from global memory (already flushed by this wave). The
 * global read takes the aligned 4-byte word holding the byte: a different
 * load width keeps the compiler from merging the two branches into one
 * flat load, and an aligned word never leaves the page of the byte. */
template <class W>
__device__ __forceinline__ uint8_t history_byte(const W& w, gcu8* dst,
                                                uint64_t y, uint64_t ring_lo) {
    if (y >= ring_lo) {
        return w.ring[ring_index<W::kSize>((uintptr_t)dst, y)];
    }
    const uintptr_t a = (uintptr_t)(dst + y);
    const uint32_t word = *(gcu32*)(a & ~(uintptr_t)3);
    return (uint8_t)(word >> ((a & 3) * 8));
}

/* Byte i (0..15) of a 16-byte register block. */
__device__ __forceinline__ uint32_t block_byte(const uint4& v, uint32_t i) {
    const uint32_t x = (i >> 2) == 0 ? v.x : (i >> 2) == 1 ? v.y : (i >> 2) == 2 ? v.z : v.w;
    return (x >> ((i & 3) * 8)) & 0xFF;
}

/* Exactly n (0..15) bytes of v to ring position r, where they do not wrap:
 * 8/4/2/1-byte stores, so no byte past n is touched. */
template <class W>
__device__ __forceinline__ void ring_tail(W& w, uint32_t r, const uint4& v, uint32_t n) {
    uint8_t* p = &w.ring[r];
    uint64_t lo = ((uint64_t)v.y << 32) | v.x;
    const uint64_t hi = ((uint64_t)v.w << 32) | v.z;
    if (n & 8) {
        __builtin_memcpy(p, &lo, 8);
        p += 8;
        lo = hi;
    }
    if (n & 4) {
        const uint32_t q = (uint32_t)lo;
        __builtin_memcpy(p, &q, 4);
        p += 4;
        lo >>= 32;
    }
    if (n & 2) {
        const uint16_t q = (uint16_t)lo;
        __builtin_memcpy(p, &q, 2);
        p += 2;
        lo >>= 16;
    }
    if (n & 1) {
        *p = (uint8_t)lo;
    }
}

/* Exactly n (0..16) bytes of v to ring position r, wrapping at the ring's
 * end. */
template <class W>
__device__ __forceinline__ void ring_put(W& w, uint32_t r, const uint4& v, uint32_t n) {
    if (n == 0) {
        return;
    }
    if (r + n <= W::kSize) {
        if (n == 16) {
            __builtin_memcpy(&w.ring[r], &v, 16);
        } else {
            ring_tail(w, r, v, n);
        }
        return;
    }
    for (uint32_t i = 0; i < n; i++) {
        w.ring[(r + i) & (W::kSize - 1)] = (uint8_t)block_byte(v, i);
    }
}

/* Four selector bytes (r + i) mod p, i = 0..3, packed, for 3 <= p <= 15 and
 * r < p, given pb = p and cp = 0x80 - p in every byte. A bytewise compare
 * and subtract in one word: every byte stays below 128, so no carry or
 * borrow crosses a byte, and ge * 255 is (ge << 8) - ge modulo 2^32. */
__device__ __forceinline__ uint32_t period_sel(uint32_t r, uint32_t pb, uint32_t cp) {
    const uint32_t sv = __builtin_amdgcn_perm(0u, r, 0u) + 0x03020100u;
    const uint32_t ge = ((sv + cp) >> 7) & 0x01010101u;
    return sv - (((ge << 8) - ge) & pb);
}

/* Bytes of the 16-byte block S picked by four selector bytes (each 0..15). */
__device__ __forceinline__ uint32_t gather16(const uint4& S, uint32_t sel) {
    const uint32_t lo = __builtin_amdgcn_perm(S.y, S.x, sel & 0x07070707u);
    const uint32_t hi = __builtin_amdgcn_perm(S.w, S.z, sel & 0x07070707u);
    const uint32_t pick = 0x03020100u + ((sel >> 1) & 0x04040404u);
    return __builtin_amdgcn_perm(hi, lo, pick);
}

/* Where the last piece of a copy of len bytes starts: copies go out in
 * pieces of 16, 8 or 4 bytes (the largest that fits the length), the last
 * one ending at the copy's end and so overlapping the one before. */
__device__ __forceinline__ uint32_t last_piece(uint32_t len) {
    return len >= 16 ? len - 16 : len >= 8 ? len - 8 : len >= 4 ? len - 4 : 0;
}

/* Four 16-byte global loads of the pieces of a history source of len
 * (1..64) bytes at `at`, issued together: at 0, 16, 32 (or at the last
 * piece where that comes before) and at the last piece, none of which reads
 * more than 15 bytes past the source. Straight-line on purpose: a load under
 * a condition of its own leaves the compiler copying its result where the
 * condition ends, and the copy waits for the load right there. */
struct Period {
    uint4 h0, h1, h2, h3;
};
__device__ __forceinline__ Period load_period(gcu8* at, uint32_t len) {
    const uint32_t last = last_piece(len);
    Period p;
    p.h0 = gload16(at);
    p.h1 = gload16(at + (last < 16u ? last : 16u));
    p.h2 = gload16(at + (last < 32u ? last : 32u));
    p.h3 = gload16(at + last);
    return p;
}
/* What lanes with no history period load instead (never written). */
__device__ __align__(16) uint8_t no_period[16];

/* --------------------------------------------------- global slow path */

/* dst[0, n) = src[0, n), whole wave, global to global. Destination-aligned
 * 16-byte blocks; each lane's source read is an unaligned 16-byte load that
 * stays inside [src, src + n). */
__device__ __forceinline__ void wave_copy_global(gu8* dst, gcu8* src,
                                                 uint64_t n, uint32_t lane) {
    if (n == 0) {
        return;
    }
    const uintptr_t d0 = (uintptr_t)dst;
    uint64_t head = ((d0 + 15) & ~(uintptr_t)15) - d0;
    if (head > n) {
        head = n;
    }
    if (lane < head) {
        dst[lane] = src[lane];
    }
    const uint64_t body = (n - head) / 16;
    /* four loads a lane in flight before their stores: one wave keeps
     * 4 KiB moving, where a load-then-store step waits a full memory
     * latency per KiB (2000 random chunks of up to 4 MiB, each one literal
     * run: 5.0 ms that way, 1.05 ms like this; eight deep: 1.03 ms) */
    constexpr uint32_t kDeep = 4;
    uint64_t b = lane;
    for (; b + (kDeep - 1) * kWave < body; b += kDeep * kWave) {
        uint4 v[kDeep];
#pragma unroll
        for (uint32_t u = 0; u < kDeep; u++) {
            v[u] = gload16(src + head + 16 * (b + u * kWave));
        }
#pragma unroll
        for (uint32_t u = 0; u < kDeep; u++) {
            gstore16(dst + head + 16 * (b + u * kWave), v[u]);
        }
    }
    for (; b < body; b += kWave) {
        gstore16(dst + head + 16 * b, gload16(src + head + 16 * b));
    }
    const uint64_t done = head + 16 * body;
    if (lane < n - done) {
        dst[done + lane] = src[done + lane];
    }
    wave_order();
}

/* Largest period staged in the ring by wave_match_global. */
constexpr uint32_t kStagedPeriod = 1024;
static_assert(kStagedPeriod + 16 <= kRing, "a staged period fits the ring");

/* dst[m + i] = dst[m - off + (i mod off)] for i < len (cap bounds dst),
 * whole wave, in global memory; every source byte precedes m and is final.
 * The ring is free scratch here (everything in it is flushed):
 *  - off >= len: one contiguous copy;
 *  - off < kStagedPeriod: the period, extended by 16 bytes, is staged in
 *    the ring once, then every lane stores 16-byte slices read from it at
 *    (i mod off) -- one global round trip for the whole match, where a
 *    byte-per-lane gather pays one per 64 bytes and whole-period rounds one
 *    per period;
 *  - otherwise: rounds of off (>= kStagedPeriod) bytes. */
template <class W>
__device__ __forceinline__ void wave_match_global(W& w, gu8* dst, uint64_t m,
                                                  uint64_t off, uint64_t len, uint64_t cap,
                                                  uint32_t lane) {
    if (off >= len) {
        wave_copy_global(dst + m, dst + m - off, len, lane);
        return;
    }
    if (off >= kStagedPeriod) {
        for (uint64_t r0 = 0; r0 < len; r0 += off) {
            const uint64_t n = len - r0 < off ? len - r0 : off;
            wave_copy_global(dst + m + r0, dst + m + r0 - off, n, lane);
        }
        return;
    }
    const uint32_t o = (uint32_t)off;
    const uint64_t from = m - o;
    /* the period into ring[0, o): 16-byte loads where the block stays in
     * [0, cap); the bytes a block reads past the period are overwritten by
     * the extension below */
    for (uint32_t b = 16 * lane; b < o; b += 16 * kWave) {
        uint4 v;
        if (from + b + 16 <= cap) {
            v = gload16(dst + from + b);
        } else {
            uint32_t q[4] = {0, 0, 0, 0};
            for (uint32_t i = 0; i < 16 && b + i < o; i++) {
                q[i >> 2] |= (uint32_t)dst[from + b + i] << ((i & 3) * 8);
            }
            v = make_uint4(q[0], q[1], q[2], q[3]);
        }
        __builtin_memcpy(&w.ring[b], &v, 16);
    }
    wave_order();
    /* ring[o + t] = ring[t mod o] for t < 16 */
    if (lane < 16) {
        uint32_t k = lane;
        while (k >= o) {
            k -= o;
        }
        const uint8_t e = w.ring[k];
        w.ring[o + lane] = e;
    }
    wave_order();
    uint32_t r = (16 * lane) % o;
    const uint32_t step = (16 * kWave) % o;
    for (uint64_t b = 16 * lane; b < len; b += 16 * kWave) {
        uint4 v;
        __builtin_memcpy(&v, &w.ring[r], 16);
        if (len - b >= 16) {
            gstore16(dst + m + b, v);
        } else {
            const uint32_t n = (uint32_t)(len - b);
            for (uint32_t i = 0; i < n; i++) {
                dst[m + b + i] = (uint8_t)block_byte(v, i);
            }
        }
        r += step;
        r = r >= o ? r - o : r;
    }
    wave_order();
}

/* ------------------------------------------------- group execution */

/* Clears bit j of a wave-uniform mask in one scalar instruction. */
__device__ __forceinline__ void clear_bit(uint64_t& mask, uint32_t j) {
    asm("s_bitset0_b64 %0, %1" : "+s"(mask) : "s"(j));
}

/* 16 ring bytes from index r, wrapping at the ring's end. */
template <class W>
__device__ __forceinline__ uint4 ring_read16(const W& w, uint32_t r) {
    uint4 v;
    if (r <= W::kSize - 16) {
        __builtin_memcpy(&v, &w.ring[r], 16);
    } else {
        uint32_t q[4] = {0, 0, 0, 0};
        for (uint32_t i = 0; i < 16; i++) {
            q[i >> 2] |= (uint32_t)w.ring[(r + i) & (W::kSize - 1)] << ((i & 3) * 8);
        }
        v = make_uint4(q[0], q[1], q[2], q[3]);
    }
    return v;
}

/* Bytes t < keep of a, the rest of b. */
__device__ __forceinline__ uint4 take_bytes(const uint4& a, const uint4& b, uint32_t keep) {
    if (keep >= 16) {
        return a;
    }
    uint32_t m[4];
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
        const uint32_t c = keep > 4 * q ? keep - 4 * q : 0;
        m[q] = c >= 4 ? 0xFFFFFFFFu : (1u << (8 * c)) - 1u;
    }
    return make_uint4((a.x & m[0]) | (b.x & ~m[0]), (a.y & m[1]) | (b.y & ~m[1]),
                      (a.z & m[2]) | (b.z & ~m[2]), (a.w & m[3]) | (b.w & ~m[3]));
}

/* x mod d for x < 4096 and d >= 1, by the float reciprocal: the quotient
 * x * (1 / d) never exceeds the true one (the reciprocal is within one
 * ulp) and its error stays below one part in 2^11, so it falls short by at
 * most one, and only at exact multiples; one correction suffices. */
__device__ __forceinline__ uint32_t small_mod(uint32_t x, uint32_t d) {
    const float inv = __builtin_amdgcn_rcpf((float)d);
    const uint32_t r = x - __umul24(d, (uint32_t)((float)x * inv));
    return r >= d ? r - d : r;
}

/* The match [m, m + len) with offset o, whole wave, 16 bytes a lane a round
 * of 1024, into the ring, when its period [m - o, m - o + min(o, len))
 * lies in the ring. Match byte i is period byte i mod o, so every lane
 * reads only the period, never bytes this match writes, and the lanes are
 * independent. Lane k's block starts at match byte i0 = 16 k (+ 1024 a
 * round), at period phase s = i0 mod o:
 *  - o >= 16: the block is period bytes s, s + 1, ..., wrapping at most
 *    once, i.e. ring bytes from m - o + s while t < o - s, and from one
 *    period further back, m - 2 o + s, after that: two 16-byte reads and a
 *    byte mask;
 *  - o < 16: the first 16 ring bytes from m - o hold the period, and byte
 *    t is its byte (s + t) mod o, gathered with v_perm selectors (periods
 *    1 and 2 are widened to 4 first).
 * Each block stores exactly its bytes of the match. */
template <class W>
__device__ __forceinline__ void ring_match_wide(W& w, uintptr_t da, uint64_t m, uint32_t o,
                                                uint32_t len, uint32_t lane) {
    const uint32_t rm = ring_index<W::kSize>(da, m);
    const uint32_t rp = ring_index<W::kSize>(da, m - o);
    uint32_t s = small_mod(16 * lane, o);
    const uint32_t step = small_mod(16 * kWave, o);
    if (o >= 16) {
        for (uint32_t i0 = 16 * lane; i0 < len; i0 += 16 * kWave) {
            const uint4 a = ring_read16(w, (rp + s) & (W::kSize - 1));
            const uint4 b = ring_read16(w, (rp + s - o) & (W::kSize - 1));
            const uint32_t n = len - i0 < 16 ? len - i0 : 16;
            ring_put(w, (rm + i0) & (W::kSize - 1), take_bytes(a, b, o - s), n);
            s += step;
            s = s >= o ? s - o : s;
        }
        return;
    }
    uint4 S = ring_read16(w, rp);
    uint32_t p = o;
    if (p <= 2) {
        /* periods 1 and 2 as period 4 */
        S.x = __builtin_amdgcn_perm(0u, S.x, p == 1 ? 0x00000000u : 0x01000100u);
        p = 4;
    }
    const uint32_t pb = __builtin_amdgcn_perm(0u, p, 0u);
    const uint32_t cp = __builtin_amdgcn_perm(0u, 0x80u - p, 0u);
    for (uint32_t i0 = 16 * lane; i0 < len; i0 += 16 * kWave) {
        uint32_t q[4];
        uint32_t r = s;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            q[t] = gather16(S, period_sel(r, pb, cp));
            r += 4;
            r = r >= p ? r - p : r;
            r = r >= p ? r - p : r;
        }
        const uint32_t n = len - i0 < 16 ? len - i0 : 16;
        ring_put(w, (rm + i0) & (W::kSize - 1), make_uint4(q[0], q[1], q[2], q[3]), n);
        s += step;
        s = s >= o ? s - o : s;
    }
}

/* The members of one window that a group executes, as the copy phase needs
 * them: per lane, the member's literal start (window-relative), literal
 * and match lengths, offset and output offset from the group start; and,
 * uniform, how many members run in full, whether member `take` adds its
 * terminal literal only, and the group's output length. */
struct Group {
    uint32_t lit, lit_len, match_len, offset, drel;
    uint32_t take;
    bool terminal;
    uint32_t end_rel;
};

/* LDS bytes by 32-bit LDS address. */
typedef __attribute__((address_space(3))) uint8_t lds_u8;
__device__ __forceinline__ uint32_t lds_address(const uint8_t* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t*)p;
}

/* Exactly len (1..64) bytes to `to`, from `from` (both LDS; `to` is at
 * least 16 bytes, or len, further on: pieces go out in order, so where the
 * copy repeats its source a piece reads what the ones before it wrote) or,
 * where kHist and from_history, from the loaded pieces hp. A
 * lane's copy is at most four 16-byte pieces, or two of 8 or of 4, the last
 * ending at the copy's end (load_period): no tail of 8, 4, 2 and 1 bytes,
 * each under a branch of its own, which took about three times the
 * instructions. */
template <uint32_t kBytes>
struct Piece;
template <>
struct Piece<16> {
    using type = uint4;
    static __device__ __forceinline__ type of(const uint4& v) { return v; }
};
template <>
struct Piece<8> {
    using type = uint2;
    static __device__ __forceinline__ type of(const uint4& v) { return make_uint2(v.x, v.y); }
};
template <>
struct Piece<4> {
    using type = uint32_t;
    static __device__ __forceinline__ type of(const uint4& v) { return v.x; }
};
template <uint32_t kBytes, bool kHist>
__device__ __forceinline__ void put_piece(uint8_t* to, const uint8_t* from, bool from_history,
                                          const uint4& h) {
    typename Piece<kBytes>::type x = Piece<kBytes>::of(h);
    if (!kHist || !from_history) {
        __builtin_memcpy(&x, from, kBytes);
    }
    __builtin_memcpy(to, &x, kBytes);
}
template <bool kHist>
__device__ __forceinline__ void lane_copy(uint8_t* to, const uint8_t* from, uint32_t len,
                                          bool from_history, const Period& hp) {
    const uint32_t last = last_piece(len);
    if (len >= 16) {
        put_piece<16, kHist>(to, from, from_history, hp.h0);
        if (len > 32) {
            put_piece<16, kHist>(to + 16, from + 16, from_history, hp.h1);
        }
        if (len > 48) {
            put_piece<16, kHist>(to + 32, from + 32, from_history, hp.h2);
        }
        put_piece<16, kHist>(to + last, from + last, from_history, hp.h3);
    } else if (len >= 8) {
        put_piece<8, kHist>(to, from, from_history, hp.h0);
        put_piece<8, kHist>(to + last, from + last, from_history, hp.h3);
    } else if (len >= 4) {
        put_piece<4, kHist>(to, from, from_history, hp.h0);
        put_piece<4, kHist>(to + last, from + last, from_history, hp.h3);
    } else {
        /* 1 to 3 bytes: the first, the middle and the last */
        const uint32_t mid = len >> 1, end = len - 1;
        uint8_t a = (uint8_t)hp.h0.x, b = (uint8_t)(hp.h0.x >> (8 * mid)),
                c = (uint8_t)(hp.h0.x >> (8 * end));
        if (!kHist || !from_history) {
            a = from[0];
            b = from[mid];
            c = from[end];
        }
        to[0] = a;
        to[mid] = b;
        to[end] = c;
    }
}

/* One lane's literal of lit_len (1..kLaneLit) bytes, staged at `from`, to
 * the ring at index r0. */
template <class W>
__device__ __forceinline__ void put_literal(W& w, const uint8_t* from, uint32_t lit_len,
                                            uint32_t r0) {
    if (r0 + lit_len <= W::kSize) {
        lane_copy<false>(&w.ring[r0], from, lit_len, false, Period{});
    } else {
        for (uint32_t b = 0; b < lit_len; b++) {
            w.ring[(r0 + b) & (W::kSize - 1)] = from[b];
        }
    }
}

/* How a wave that executes groups stands to the others of its chunk. Alone:
 * it runs every group of the chunk itself, so everything before the group
 * is final. InTurn: the copiers of a pipelined block run consecutive groups
 * at once (below), so what lies between the output position that was final
 * when the group began and the group itself may still be unwritten, and
 * bytes that followers may overwrite in the ring count as gone. */
struct Alone {
    static constexpr bool kInTurn = false;
    static constexpr bool kStrips = true; /* run_strips where it pays */
    __device__ uint64_t final_below(uint64_t d0) const { return d0; }
    __device__ bool wait_turn() const { return true; }
    __device__ void pass(uint64_t) const {} /* the group's bytes are in the ring */
};

/* Lane's members a..b (as a mask) that cover bytes [from, to) of the group,
 * relative to its start, below member `lane`; none for an empty range. Each
 * active lane's member starts at `start` (all different, the first at 0). Two rank queries per lane replace
 * a search over the members. */
__device__ __forceinline__ uint64_t members_covering(CoverLds& c, bool active, uint32_t start,
                                                     uint32_t from, uint32_t to, uint32_t lane) {
    c.starts[lane] = 0;
    wave_order();
    if (active) {
        atomicOr((unsigned long long*)&c.starts[start >> 6], 1ull << (start & 63));
    }
    wave_order();
    const uint32_t mine = (uint32_t)__builtin_popcountll(c.starts[lane]);
    c.before[lane] = (uint8_t)(wave_inclusive_sum(mine, lane) - mine);
    wave_order();
    if (from >= to) {
        return 0;
    }
    const uint32_t last = to - 1;
    const uint64_t upto_a = ~0ull >> (63 - (from & 63)), upto_b = ~0ull >> (63 - (last & 63));
    const uint32_t a = c.before[from >> 6] +
                       (uint32_t)__builtin_popcountll(c.starts[from >> 6] & upto_a) - 1;
    const uint32_t b = c.before[last >> 6] +
                       (uint32_t)__builtin_popcountll(c.starts[last >> 6] & upto_b) - 1;
    const uint64_t below = (1ull << lane) - 1;
    return below & (~0ull << (a & 63)) & (~0ull >> (63 - (b & 63)));
}

/* Matches longer than this go 16 bytes a lane (ring_match_wide) instead of
 * a byte a lane and 64 a step. */
constexpr uint32_t kWideMatch = 256;

/* Output bytes a member from which on members go one by one rather than by
 * strips (run_strips): 312 cycles a member that waits for the one before it,
 * about 700 a strip of 64 bytes. With 16, 24 and 40: 1000 LZ4 chunks of 1 MiB
 * of text 8.7, 7.45 and 7.40 ms, the uneven Snappy batch 12.25, 12.25 and
 * 12.35, Snappy's sparse bytes 2.75, 2.80 and 3.04. */
constexpr uint32_t kStripMember = 24;
constexpr uint32_t kStripAt = 1u << 12, kStripOffset = 1u << 14; /* what its word holds */
static_assert(kBatchMax < kStripAt - 1 && kRing <= kStripOffset && kLaneMatch <= 64,
              "12 bits of a match's start, 14 of its offset, 6 of its length");

/* Many short matches of which each may wait for the one before (columns of
 * numbers, few symbols): by output bytes, 64 at a time, a byte a lane. A
 * byte's source is its member's offset back; where that is a byte of the same
 * strip that is itself still to be copied, it is that byte's source instead,
 * and so on: pointer doubling over the wave, at most six rounds. Every source
 * is then final, and one read and one write copy the strip. `todo` holds the
 * members (matches of up to 64 bytes whose sources lie in the ring); `c` says
 * which member covers a byte.
 *
 * What bounds it is the latency of about four lane shuffles a strip. One chunk
 * of 1 MiB of sorted 64-bit numbers, eight members a strip: 17.2 ms one member
 * after the other, 7.3 so; of text 7.3 and 6.0; 5000 of 64 KiB on a wave each:
 * 2.65 and 1.53 ms, text 1.64 and 1.53. */
template <class W>
__device__ __forceinline__ void run_strips(W& w, const CoverLds& c, uint32_t ring_at,
                                           uint32_t m_rel, uint32_t offset, uint32_t match_len,
                                           uint64_t todo, uint32_t end_rel, uint32_t lane) {
    /* match start, offset and length in one word; none: past every byte */
    constexpr uint32_t kAt = kStripAt - 1;
    const uint32_t info = ((todo >> lane) & 1) != 0
                              ? m_rel | offset << 12 | (match_len - 1) << 26
                              : kAt;
    for (uint32_t s = 0; s < end_rel; s += kWave) {
        const uint64_t starts = c.starts[s / kWave];
        const uint32_t member = c.before[s / kWave] +
                                (uint32_t)__builtin_popcountll(starts & (~0ull >> (63 - lane))) - 1;
        const uint32_t mine = (uint32_t)__shfl((int)info, (int)(member & (kWave - 1)));
        const int pos = (int)(s + lane);
        const int i = pos - (int)(mine & kAt);
        const bool copies = i >= 0 && i <= (int)(mine >> 26);
        int from = copies ? pos - (int)((mine >> 12) & (kStripOffset - 1)) : pos;
        for (;;) {
            const int at = from - (int)s;
            const int further = __shfl(from, at & (int)(kWave - 1));
            const bool moves = at >= 0 && further != from;
            if (__ballot(moves) == 0) {
                break;
            }
            from = moves ? further : from;
        }
        if (copies) {
            w.ring[(ring_at + (uint32_t)pos) & (W::kSize - 1)] =
                w.ring[(ring_at + (uint32_t)from) & (W::kSize - 1)];
        }
        wave_order();
    }
}

/* Executes group g of the window staged at cw into the ring at output
 * positions [dp, dp + g.end_rel), flushes whole 16-byte blocks (all of them
 * when the chunk is done) and advances dp. Returns false only when the
 * wait for its turn was given up.
 *
 * Literals go first, a member a lane. Then the matches that repeat nothing
 * and whose source is final, a member a lane. The others go in stream
 * order, the wave fanned out over the bytes. */
template <class W, class Order>
__device__ __forceinline__ bool execute_group(W& w, CoverLds& cover_lds, const uint8_t* cw,
                                              const Group& g, gu8* dst, uint64_t cap,
                                              uint64_t& dp, uint64_t& flushed, uint64_t ring_lo,
                                              bool done, uint32_t lane, const Order& order) {
    const uintptr_t da = (uintptr_t)dst;
    const uint32_t take = g.take;
    const bool full = lane < take;
    const bool active = full || (g.terminal && lane == take);
    const uint32_t lit = g.lit, lit_len = g.lit_len, match_len = g.match_len,
                   offset = g.offset, drel = g.drel;
    const uint64_t D0 = dp;
    const uint64_t D1 = dp + g.end_rel;
    const uint64_t final_lo = order.final_below(D0);
    uint64_t ring_floor;
    if constexpr (Order::kInTurn) {
        ring_floor = D0 > Order::kHistory ? D0 - Order::kHistory : 0;
    } else {
        ring_floor = D1 + 16 > W::kSize ? D1 + 16 - W::kSize : 0;
    }
    const uint64_t hist_lo = ring_lo > ring_floor ? ring_lo : ring_floor;
    /* positions from here on are 32-bit and relative to the group's start:
     * the group and the ring's history are a few KiB, and a source further
     * back than 2^30 bytes is as good as one that far back */
    const int hist_rel = (int)(hist_lo - D0);
    const int final_rel = (int)(final_lo - D0);
    const uint32_t ring_at = (uint32_t)(da + D0); /* ring index of the group's start, unmasked */
    const uint32_t m_rel = drel + lit_len;
    const int y_rel = offset > 1u << 30 ? -(1 << 30) : (int)(m_rel - offset);
    const uint32_t need = match_len < offset ? match_len : offset;
    const int src_end = y_rel + (int)need;
    const bool has_match = full && match_len != 0;
    const uint32_t rd = (ring_at + m_rel) & (W::kSize - 1);
    const uint32_t ry = (ring_at + m_rel - offset) & (W::kSize - 1);
    const bool short_fit = has_match && match_len <= kLaneMatch && rd + match_len <= W::kSize;
    const bool src_fit = y_rel >= hist_rel && ry + need <= W::kSize;
    /* matches that a lane copies by itself: those that repeat nothing, with
     * a final source, in the ring or in flushed history (whose 16-byte loads
     * may run up to 15 bytes past the source) */
    const bool simple =
        short_fit && offset >= match_len && (src_end <= final_rel || y_rel >= (int)drel);
    const bool from_history = simple && src_end <= hist_rel && hist_lo + 15 <= cap;
    const bool by_lane = from_history || (simple && src_fit);
    /* history periods are loaded now, so the loads overlap the literal
     * phase: every lane loads, with no branch around the loads (whose results
     * would then be copied, waiting for them here); a lane without a
     * history period reads the zero block no_period */
    const Period hp =
        load_period(from_history ? dst + (D0 + m_rel - offset) : (gcu8*)no_period,
                    from_history ? need : 1u);
    /* the literals */
    const bool wide_lit = lit_len > kLaneLit;
    if (active && !wide_lit && lit_len != 0) {
        put_literal(w, cw + lit, lit_len, (ring_at + drel) & (W::kSize - 1));
    }
    for (uint64_t wide = __ballot(active && wide_lit); wide != 0;) {
        const uint32_t j = __builtin_ctzll(wide);
        clear_bit(wide, j);
        const uint32_t jl = __builtin_amdgcn_readlane(lit_len, j);
        const uint32_t jlit = __builtin_amdgcn_readlane(lit, j);
        const uint32_t jr = ring_at + __builtin_amdgcn_readlane(drel, j);
        for (uint32_t i = lane; i < jl; i += kWave) {
            w.ring[(jr + i) & (W::kSize - 1)] = cw[jlit + i];
        }
    }
    wave_order();
    /* the members each of the other matches waits for: those that cover its
     * source between the group's start and its own literals */
    const bool rest = has_match && !by_lane;
    const uint32_t src_from = y_rel > 0 ? (uint32_t)y_rel : 0;
    const uint32_t src_to = !rest || src_end <= 0       ? 0
                            : (uint32_t)src_end < drel ? (uint32_t)src_end
                                                       : drel;
    const uint64_t waits_for =
        members_covering(cover_lds, full, drel, src_from, src_to, lane);
    const bool held = Order::kInTurn && rest && y_rel < 0 && src_end > final_rel;
    if (by_lane) {
        lane_copy<true>(&w.ring[rd], &w.ring[ry], match_len, from_history, hp);
    }
    wave_order();
    /* The common member of a level, a short match (<= 64 bytes) whose period
     * is in the ring and which does not wrap there, is described by its lane
     * up front in two words, so it costs two v_readlane and a byte a lane:
     * fast_a = LDS address of the match (16 bits) and of its period; fast_b
     * = its length (8 bits), o = min(offset, 64) (8 bits) and
     * ceil(4096 / o). Where the match repeats its period, byte i copies
     * period byte i mod offset, which precedes the match, so the lanes do
     * not depend on each other. For i <= 64 the quotient floor(i / o) is
     * (i * ceil(4096 / o)) >> 12: with ceil(4096 / o) = (4096 + e) / o,
     * 0 <= e < o, the scaled product is i / o + i * e / (4096 o), and
     * i * e < 64 * 64 keeps the excess below the 1 / o that separates i / o
     * from the next integer. Two 24-bit multiplies and a shift replace a
     * reciprocal and its correction. */
    const bool fast_member = rest && short_fit && src_fit;
    /* (a source that runs on into the match must not wrap between them) */
    const bool by_pieces = offset >= match_len || (offset >= 16 && ry < rd);
    const uint64_t once_mask = __ballot(fast_member && by_pieces);
    const uint64_t again_mask = __ballot(fast_member && !by_pieces);
    const uint32_t lds_ring = lds_address(w.ring);
    const uint32_t fast_a = (lds_ring + rd) | (lds_ring + ry) << 16;
    const uint32_t fast_o = offset - 1 < kWave ? offset : kWave;
    const uint32_t fast_b = (match_len & 255) | fast_o << 8 | ((4096u + fast_o - 1) / fast_o) << 16;
    const uint32_t sink = lds_address(w.sink) + lane;
    /* lanes past the match write their own sink byte, so no lane is masked */
    auto again_from = [&](uint32_t ja, uint32_t jb) {
        const uint32_t r = __umul24(__umul24(lane, jb >> 16) >> 12, (jb >> 8) & 255);
        return *(lds_u8*)(uintptr_t)((ja >> 16) + lane - r);
    };
    auto put = [&](uint32_t ja, uint32_t jb, uint8_t byte) {
        const uint32_t at = (ja & 0xFFFF) + lane;
        *(lds_u8*)(uintptr_t)(lane < (jb & 255) ? at : sink) = byte;
    };
    uint64_t undone = __ballot(rest);
    /* InTurn: the members that need bytes of groups still running, or of
     * such a member of this group, wait for this group's turn */
    uint64_t later = Order::kInTurn ? __ballot(held) : 0;
    if (Order::kInTurn && later != 0) {
        for (uint64_t more = later;;) {
            more = __ballot(rest && (waits_for & more) != 0) & ~later;
            if (more == 0) {
                break;
            }
            later |= more;
        }
    }
    bool turn = false;
    for (;;) {
        uint64_t todo = undone & ~later;
        /* copies that go by pieces and wait for none: a member a lane
         * where there are several, which costs about what four of them cost
         * one by one */
        const uint64_t lanes =
            todo & once_mask & __ballot((waits_for & undone) == 0);
        if (__builtin_popcountll(lanes) >= 4) {
            if (((lanes >> lane) & 1) != 0) {
                lane_copy<false>(&w.ring[rd], &w.ring[ry], match_len, false, hp);
            }
            todo &= ~lanes;
            undone &= ~lanes;
            wave_order();
        }
        /* the others in stream order, two at a time where the second does
         * not touch the first */
        const uint64_t below = todo & ((1ull << lane) - 1);
        const uint64_t before = below == 0 ? 0 : 1ull << (63 - __builtin_clzll(below));
        const uint64_t tied = __ballot((waits_for & before) != 0) | ~(once_mask | again_mask);
        undone &= ~todo;
        if (Order::kStrips && (todo & ~(once_mask | again_mask)) == 0 &&
            (uint32_t)__builtin_popcountll(todo) * kStripMember > g.end_rel) {
            run_strips(w, cover_lds, ring_at, m_rel, offset, match_len, todo, g.end_rel, lane);
            todo = 0;
        }
        while (todo != 0) {
            const uint32_t j = __builtin_ctzll(todo);
            clear_bit(todo, j);
            const uint32_t a0 = __builtin_amdgcn_readlane(fast_a, j);
            const uint32_t b0 = __builtin_amdgcn_readlane(fast_b, j);
            if ((((once_mask | again_mask) >> j) & 1) != 0) {
                if ((todo & (0 - todo) & ~tied) != 0) {
                    const uint32_t j1 = __builtin_ctzll(todo);
                    clear_bit(todo, j1);
                    const uint32_t a1 = __builtin_amdgcn_readlane(fast_a, j1);
                    const uint32_t b1 = __builtin_amdgcn_readlane(fast_b, j1);
                    const uint8_t x0 = again_from(a0, b0);
                    const uint8_t x1 = again_from(a1, b1);
                    put(a0, b0, x0);
                    put(a1, b1, x1);
                } else {
                    put(a0, b0, again_from(a0, b0));
                }
                wave_order();
                continue;
            }
            const uint32_t jm = __builtin_amdgcn_readlane(match_len, j);
            const uint32_t joff = __builtin_amdgcn_readlane(offset, j);
            const uint64_t jm0 = D0 + __builtin_amdgcn_readlane(m_rel, j);
            const uint64_t jfrom = jm0 - joff;
            if (jm > kWideMatch && jfrom >= hist_lo) {
                ring_match_wide(w, da, jm0, joff, jm, lane);
                wave_order();
                continue;
            }
            /* byte i copies period byte i mod joff, kept per lane as i
             * steps by 64; lane mod joff and 64 mod joff as above (for
             * joff > 64 they are lane and 64) */
            const uint32_t jo = (b0 >> 8) & 255;
            const uint32_t jq = b0 >> 16;
            uint32_t r = lane - __umul24(__umul24(lane, jq) >> 12, jo);
            const uint32_t step =
                joff > kWave ? kWave : kWave - __umul24(__umul24(kWave, jq) >> 12, jo);
            if (jfrom >= hist_lo) {
                const uint32_t jd = (uint32_t)(da + jm0), js = (uint32_t)(da + jfrom);
                for (uint32_t i = lane; i < jm; i += kWave) {
                    w.ring[(jd + i) & (W::kSize - 1)] = w.ring[(js + r) & (W::kSize - 1)];
                    r += step;
                    r = r >= joff ? r - joff : r;
                }
            } else {
                for (uint32_t i = lane; i < jm; i += kWave) {
                    w.ring[ring_index<W::kSize>(da, jm0 + i)] =
                        history_byte(w, dst, jfrom + r, hist_lo);
                    r += step;
                    r = r >= joff ? r - joff : r;
                }
            }
            wave_order();
        }
        if (!Order::kInTurn || turn) {
            break;
        }
        if (!order.wait_turn()) {
            return false;
        }
        if (later == 0) {
            break;
        }
        turn = true;
        later = 0;
    }
    dp = D1;
    order.pass(D1);
    const uintptr_t a_end = done ? da + dp : ((da + dp) & ~(uintptr_t)15);
    const uint64_t to = a_end > da + flushed ? (uint64_t)(a_end - da) : flushed;
    if (to > flushed) {
        flush_ring(w, dst, flushed, to, lane);
        flushed = to;
    }
    return true;
}

/* Largest offset whose period a slow match takes from the ring. */
constexpr uint32_t kSlowRingPeriod = 1024;

/* Executes a sequence the window could not hold (a length with two or more
 * extension bytes, a literal past the window). A literal of at most 64
 * bytes goes into the ring a byte a lane; a longer one runs global to
 * global after the ring is flushed up to it. A match whose period (offset
 * <= kSlowRingPeriod) is in the ring is expanded there 16 bytes a lane
 * (ring_match_wide), in pieces that never lap unflushed bytes or the
 * period, with the finished blocks flushed before each piece; any other
 * match runs global to global (wave_match_global), after everything before
 * it is flushed. On return fewer than 16 bytes are unflushed (none when
 * `done`: the chunk ends here). */
template <class W>
__device__ __forceinline__ void execute_slow(W& w, gcu8* src, gu8* dst,
                                             uint64_t cap, const Lz4Step& q, uint64_t dp_after,
                                             uint64_t& dp,
                                             uint64_t& flushed, uint64_t& ring_lo, bool done,
                                             uint32_t lane) {
    const uintptr_t da = (uintptr_t)dst;
    if (q.lit_len <= kWave) {
        if (lane < q.lit_len) {
            w.ring[ring_index<W::kSize>(da, q.lit_dst + lane)] = src[q.lit_src + lane];
        }
        wave_order();
    } else {
        flush_ring(w, dst, flushed, q.lit_dst, lane);
        wave_copy_global(dst + q.lit_dst, src + q.lit_src, q.lit_len, lane);
        flushed = q.lit_dst + q.lit_len;
        ring_lo = flushed; /* the ring holds none of it */
    }
    if (q.match_len != 0) {
        uint64_t m = q.match_dst;
        const uint32_t o = q.offset;
        const uint64_t floor = m + 16 > W::kSize ? m + 16 - W::kSize : 0;
        if (o <= kSlowRingPeriod && m - o >= (ring_lo > floor ? ring_lo : floor)) {
            /* a piece leaves the period and the (< 16) unflushed bytes
             * below m in place */
            constexpr uint32_t kPiece = W::kSize - kSlowRingPeriod - 32;
            uint64_t left = q.match_len;
            while (left != 0) {
                /* whole blocks below m (compared as addresses: near the
                 * chunk's start the aligned address can precede dst) */
                const uintptr_t a_to = (da + m) & ~(uintptr_t)15;
                if (a_to > da + flushed) {
                    flush_ring(w, dst, flushed, (uint64_t)(a_to - da), lane);
                    flushed = (uint64_t)(a_to - da);
                }
                const uint32_t piece = left < kPiece ? (uint32_t)left : kPiece;
                ring_match_wide(w, da, m, o, piece, lane);
                wave_order();
                m += piece;
                left -= piece;
            }
        } else {
            flush_ring(w, dst, flushed, m, lane);
            wave_match_global(w, dst, m, o, q.match_len, cap, lane);
            flushed = m + q.match_len;
            ring_lo = flushed; /* wave_match_global used the ring as scratch */
        }
    }
    /* leave fewer than 16 unflushed bytes (none when the chunk is done):
     * the next group's output may fill the ring up to its batch limit */
    dp = dp_after;
    const uintptr_t a_end = done ? da + dp : ((da + dp) & ~(uintptr_t)15);
    if (a_end > da + flushed) {
        flush_ring(w, dst, flushed, (uint64_t)(a_end - da), lane);
        flushed = (uint64_t)(a_end - da);
    }
}

/* The waves signal through LDS words (s_sleep between reads). A wait longer
 * than any work could take (2^27 polls: seconds) marks the block broken,
 * and a broken block waits no more. */
typedef __attribute__((address_space(3))) volatile uint32_t lds_flag;
constexpr uint32_t kClaimsOver = 0xFFFFFFFFu; /* in `over`: there is nothing more to wait for */
enum Waited : uint32_t { kReached = 0, kOver = 1, kBroken = 2 };
/* Until *flag is at least `want` (as a signed distance), or, with `over`
 * given, until it says that the claims are over. */
__device__ __forceinline__ Waited await_flag(const lds_flag* flag, uint32_t want,
                                             const lds_flag* over, lds_flag* broken) {
    for (uint32_t i = 0;; i++) {
        /* the end first: `flag` may be the claim itself */
        if (over != nullptr && uniform32(*over) == kClaimsOver) {
            return kOver;
        }
        if ((int32_t)(uniform32(*flag) - want) >= 0) {
            break;
        }
        if (uniform32(*broken) != 0) {
            return kBroken;
        }
        if (i == (1u << 27)) {
            *broken = 1;
            return kBroken;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return kReached;
}
__device__ __forceinline__ void raise_flag(lds_flag* flag, uint32_t value) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    *flag = value;
}

}  // namespace
}  // namespace cudec_amd

#endif /* CUDEC_AMD_EXECUTE_H */
