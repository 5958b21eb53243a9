/* The Zstandard batch decoder for gfx950: a block of two waves per frame,
 * frames taken costliest first (the LZ4 decoder's cost queue: output plus
 * what matches add) by a persistent grid: a frame a block, then from a device
 * counter.
 *
 * The entropy wave walks the frame (zstd_decode.h, walk_frame), builds the
 * FSE tables and decodes the sequences, 64 at a time, into jobs: slots in
 * LDS that the copy wave takes in order. The copy wave decodes the
 * Huffman-coded literals (16 lanes a stream) into the block's 128 KiB slot
 * in global scratch and executes the sequences through an LDS ring
 * (execute.h, the same code that writes LZ4 output). Neither waits for the
 * other beyond the slots, so a frame's time is the longer of the two.
 *
 * What bounds it is the FSE chain: a sequence's three states give the bits
 * that give the next states. The entropy wave spends two lanes on each of the
 * three fields, one on the next state and one on the extra bits: sums over a
 * quad say where each lane's bits end, a shift of the 64 stream bits on top
 * (read while the sums are made) gives them, and one LDS read the next cell,
 * about 36 instructions and 254 cycles a sequence. (Bits read from LDS where
 * the sums say took a second round trip and 388 cycles; every lane keeping
 * the 128 bits on top and choosing words of them, 62 instructions and 338.)
 * Everything that does not feed the next state (code baselines, repeat
 * offsets, limits, positions) is done per 64 sequences, a lane each: 37
 * cycles a sequence, the repeat offsets as a scan over maps of three bytes (one
 * after the other on the scalar unit they took 190 cycles a sequence; as maps
 * that held the distances 8192 frames of 64 KiB took 2.34 ms, and 2.25 so).
 * The copies on the other wave take about 200.
 *
 * One wave a frame with one sequence decoded and executed after the other
 * took 13.72 ms for 8192 frames of 64 KiB and 284 ms for 2000 frames of
 * 1 KiB to 4 MiB; this takes 2.25 and 26.7 ms (4.94 and 56.0 with a lane a
 * Huffman stream). A frame's time is now the entropy wave's: per 64 KiB of
 * text-like data 0.70 M cycles of FSE chain, 0.11 M of tables, 0.10 M of
 * finishing and 0.02 M of staging, against 0.16 M of literals and 0.53 M of
 * copies on the other.
 *
 * The first error in stream order decides a frame: the entropy wave's
 * verdicts travel as jobs, behind the literals that precede them.
 *
 * The content checksum of a frame is checked by a second kernel, four
 * lanes a frame (xxhash.h), over every frame that decoded and carries one:
 * one frame's XXH64 is a serial chain of stripes, so frames in parallel is
 * what fills the device. */
#include <cstddef>
#include <mutex>

#include "common.h"
#include "cudec_zstd.h"
#include "execute.h"
#include "xxhash.h"
#include "zstd_decode.h"

namespace cudec_amd {
namespace {

constexpr int kVerifyBlock = 256;
constexpr uint64_t kPoolKeep = 512ull << 20; /* scratch kept between launches */

/* What the decode leaves for the checksum pass, per frame. */
struct FrameCheck {
    uint64_t written;
    uint32_t checksum;
    uint32_t verify; /* 1: the frame decoded and carries a content checksum */
};

/* What the entropy wave asks of the copy wave, in stream order. */
enum JobKind : uint32_t {
    kJobFrame,     /* a frame begins: chunk index a, output b, capacity c */
    kJobBlock,     /* n output bytes: a copy of a, or (a null) the byte x */
    kJobLiterals,  /* the block's literals: at a, or (a null) n times x */
    kJobHuffman,   /* the block's literals: payload a of b bytes, n symbols */
    kJobSequences, /* n sequences, literals from c on */
    kJobTail,      /* n literals from c on */
    kJobFail,      /* the frame ends with status x */
    kJobEnd,       /* the frame ends: written a, checksum x (y: it has one) */
    kJobQuit,
};
constexpr uint32_t kJobs = 3; /* slots: the entropy wave may run two ahead */
struct alignas(16) Job {
    uint32_t ll[kWave], ml[kWave], off[kWave]; /* kJobSequences, a lane each */
    uint64_t a, b, c;
    uint32_t kind, n, x, y;
};
static_assert(sizeof(Job) % 16 == 0, "slots keep their alignment");

/* An FSE cell of a sequence field in one word: extra bits of the symbol's
 * code (a byte), state bits (a byte, so that a quad's cells add up to a sum
 * of each: at most 63 and 26), symbol (6 bits), next-state base. */
constexpr uint32_t kCellBits = 8, kCellSymbol = 16, kCellBase = 22;
constexpr uint32_t kCellSums = 0xFFFF, kCellExtras = 0xFF;
constexpr uint32_t kCodes = (zstd::kLitLenMax + 1) + (zstd::kMatchLenMax + 1);

/* Staged bitstream of one batch: at most 712 bytes (zstd::kWindowBytes). */
struct alignas(16) EntropyLds {
    uint32_t offset[1u << zstd::kOffsetLog];
    alignas(16) uint8_t window[zstd::kWindowBytes + 16]; /* read with constant offsets, so early */
    uint32_t litlen[1u << zstd::kLitLenLog];
    uint32_t matchlen[1u << zstd::kMatchLenLog];
    uint32_t code[kCodes]; /* baseline, extra bits above it (24) */
    int16_t counts[zstd::kMatchLenMax + 1];
    uint16_t next[zstd::kMatchLenMax + 1];
};
constexpr uint32_t kHeaderStage = 512; /* of the window: table descriptions */
static_assert(kHeaderStage + (1u << zstd::kLitLenLog) <= zstd::kWindowBytes,
              "a field's symbol order lies behind the descriptions");
static_assert(offsetof(EntropyLds, window) >= 712 + 16, "what words_below may read");
static_assert(zstd::kBatch == kWave, "a batch holds a sequence a lane");

struct alignas(16) CopyLds : RingLds<kRing> {
    CoverLds cover;
    alignas(16) uint16_t huffman[zstd::kHufCells];
    /* of a Huffman tree description */
    uint8_t weights[256];
    uint32_t weight_cells[1u << zstd::kWeightLogMax];
    uint32_t first[16]; /* per weight: its next code's cell */
    int16_t counts[zstd::kWeightSymbolMax + 1];
    uint16_t next[zstd::kWeightSymbolMax + 1];
    alignas(16) uint8_t stage[zstd::kWindowBytes + 16]; /* literals of a group; a description */
};
constexpr uint32_t kLitStage = zstd::kWindowBytes - 16; /* literal bytes of a group */

struct alignas(16) FrameLds {
    EntropyLds e;
    CopyLds c;
    Job job[kJobs];
    uint32_t published; /* jobs written */
    uint32_t consumed;  /* jobs done */
    uint32_t unused;
    uint32_t broken;    /* a wait ran out, and no wave waits any more */
    uint32_t begin;     /* the frame the block takes next, kAsk or kNoMore */
    uint32_t after;     /* what `begin` is after the first: kAsk or kNoMore */
};
constexpr uint32_t kAsk = 0xFFFFFFFFu;    /* the launch's counter */
constexpr uint32_t kNoMore = 0xFFFFFFFEu; /* every frame has a block */
static_assert(sizeof(FrameLds) <= 20480, "eight blocks share a CU's 160 KiB");

/* ------------------------------------------------------------ entropy */

typedef __attribute__((address_space(3))) uint32_t lds_u32;
template <class T>
__device__ __forceinline__ uint32_t lds_at(const T* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const T*)p;
}

/* Lane kFrom of every quad, on its whole quad. */
template <uint32_t kFrom>
__device__ __forceinline__ uint32_t quad(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kFrom * 0x55, 0xF, 0xF, true);
}

/* The 128 bits of the staged stream up to the 32-bit word that holds window
 * bit `at` - 1. A stream that ran out (its batch is refused) reads what lies
 * before the window: a batch takes at most 712 bytes, and the tables before
 * it are larger. */
struct Words {
    uint32_t w0, w1, w2, w3;
    int first; /* window bit of w0's lowest */
};
__device__ __forceinline__ Words words_below(uint32_t window, int at) {
    const int word = (at - 1) >> 5;
    const uint32_t a = window + (uint32_t)(4 * word);
    return Words{*(lds_u32*)(uintptr_t)(a - 12), *(lds_u32*)(uintptr_t)(a - 8),
                 *(lds_u32*)(uintptr_t)(a - 4), *(lds_u32*)(uintptr_t)a, 32 * word - 96};
}
/* The three words that hold the 64 bits below window bit `at` and more. */
struct Top {
    uint32_t w0, w1, w2;
    __device__ __forceinline__ uint64_t bits(int at) const {
        return (uint64_t)__builtin_amdgcn_alignbit(w2, w1, (uint32_t)at) << 32 |
               __builtin_amdgcn_alignbit(w1, w0, (uint32_t)at);
    }
};
__device__ __forceinline__ Top top_below(uint32_t window, int at) {
    const uint32_t a = window + (uint32_t)(at >> 3 & ~3);
    return Top{*(lds_u32*)(uintptr_t)(a - 8), *(lds_u32*)(uintptr_t)(a - 4),
               *(lds_u32*)(uintptr_t)a};
}
/* n (0..31) of them from window bit `from` on. */
__device__ __forceinline__ uint32_t bits_of(const Words& w, int from, uint32_t n) {
    const uint32_t p = (uint32_t)(from - w.first);
    const bool far = (p & 64) != 0, odd = (p & 32) != 0;
    const uint32_t a = far ? w.w2 : w.w0, b = far ? w.w3 : w.w1, c = far ? 0u : w.w2;
    return __builtin_amdgcn_ubfe(
        __builtin_amdgcn_alignbit(odd ? c : b, odd ? b : a, p & 31), 0, n);
}

/* Builds a field's cells from counts[0..last] at accuracy `log` (RFC 8878
 * 4.1.1), as zstd::build_fse_table does one cell after the other: "less
 * than one" symbols take the top cells; the others, in symbol order, the
 * cells 0, step, 2 step, ... that lie below those; then, in cell order, each
 * symbol's cells count up from its probability. Cells go 64 at a time: a
 * cell's rank among its symbol's comes from ballots on the symbol's bits.
 * `order` is scratch of 1 << log bytes. False if the counts do not fill the
 * table exactly. */
__device__ __forceinline__ bool build_cells(const int16_t* counts, uint16_t* next,
                                            uint32_t* cells, uint8_t* order, uint32_t last,
                                            uint32_t log, const uint32_t* codes, uint32_t lane) {
    const uint32_t size = 1u << log;
    const uint32_t mask = size - 1;
    const int count = lane <= last ? counts[lane] : 0;
    const uint64_t lows = __ballot(count < 0);
    const uint32_t low = (uint32_t)__builtin_popcountll(lows);
    const uint32_t mine = count > 0 ? (uint32_t)count : 0;
    const uint32_t incl = wave_inclusive_sum(mine, lane);
    const uint32_t placed = uniform32(__builtin_amdgcn_readlane(incl, kWave - 1));
    if (placed + low != size) {
        return false;
    }
    const uint64_t below = (1ull << lane) - 1;
    if (count < 0) {
        cells[size - 1 - (uint32_t)__builtin_popcountll(lows & below)] = lane;
    }
    if (lane <= last) {
        next[lane] = (uint16_t)(count < 0 ? 1 : count);
    }
    for (uint32_t t = 0; t < mine; t++) {
        order[incl - mine + t] = (uint8_t)lane;
    }
    wave_order();
    const uint32_t step = (size >> 1) + (size >> 3) + 3;
    uint32_t run = 0;
    for (uint32_t i0 = 0; i0 < size; i0 += kWave) {
        const uint32_t i = i0 + lane;
        const uint32_t at = (i * step) & mask;
        const bool fits = i < size && at + low < size;
        const uint64_t all = __ballot(fits);
        if (fits) {
            cells[at] = order[run + (uint32_t)__builtin_popcountll(all & below)];
        }
        run += (uint32_t)__builtin_popcountll(all);
    }
    wave_order();
    for (uint32_t c0 = 0; c0 < size; c0 += kWave) {
        const uint32_t c = c0 + lane;
        const uint32_t s = c < size ? cells[c] : 0;
        uint64_t same = __ballot(c < size);
#pragma unroll
        for (uint32_t b = 0; b < 6; b++) {
            const uint64_t set = __ballot(((s >> b) & 1) != 0);
            same &= ((s >> b) & 1) != 0 ? set : ~set;
        }
        const uint32_t first = next[s];
        const uint32_t state = first + (uint32_t)__builtin_popcountll(same & below);
        wave_order();
        if (c < size) {
            if ((same >> lane) == 1) { /* the symbol's last cell here */
                next[s] = (uint16_t)(state + 1);
            }
            const uint32_t bits = log - zstd::high_bit(state);
            const uint32_t extra = codes == nullptr ? s : codes[s] >> 24;
            cells[c] = extra | bits << kCellBits | s << kCellSymbol |
                       ((state << bits) - size) << kCellBase;
        }
        wave_order();
    }
    return true;
}

/* The three repeat offsets after some sequences of a batch, in terms of those
 * before them, a byte each: the offset before that it comes from (0 to 2), or
 * kOwn and the lane of the sequence that brought a distance of its own;
 * beside it, how often code 3 without literals took one off (64 at most). The
 * distances themselves stay where they are, so they may be any of 32 bits:
 * the window of a single-segment frame is its content size, and offset code
 * 31 names distances up to 2^32 - 4 that are decoded. */
struct Repeats {
    uint32_t from, less;
};
static_assert(zstd::kOffsetMax < 32, "every distance fits 32 bits");
constexpr uint32_t kSame = 0x020100, kOwn = 0x80;
/* r after what the lane that DPP pattern kCtrl names has composed so far;
 * unchanged on lanes without one. */
template <int kCtrl, int kRows>
__device__ __forceinline__ Repeats repeats_after(const Repeats& r) {
    const uint32_t from = (uint32_t)__builtin_amdgcn_update_dpp((int)kSame, (int)r.from, kCtrl,
                                                                kRows, 0xF, false);
    const uint32_t less =
        (uint32_t)__builtin_amdgcn_update_dpp(0, (int)r.less, kCtrl, kRows, 0xF, false);
    /* v_perm selectors: the byte of the one before that it comes from, or, of
     * its own, itself (4 to 6) */
    const uint32_t own = __umul24((r.from >> 7) & 0x010101u, 0xFFu);
    const uint32_t pick = (own & 0x060504u) | (~own & r.from);
    return Repeats{__builtin_amdgcn_perm(r.from, from, pick),
                   r.less + __builtin_amdgcn_perm(0u, less, pick)};
}

/* The offset that byte 0 of a map stands for, given those before the batch
 * and, if it is one of the batch's own, that. */
__device__ __forceinline__ uint32_t offset_of(uint32_t from, uint32_t less, uint32_t own,
                                              uint32_t b0, uint32_t b1, uint32_t b2) {
    uint32_t d = b0;
    if ((from & 1) != 0) {
        d = b1;
    }
    if ((from & 2) != 0) {
        d = b2;
    }
    if ((from & kOwn) != 0) {
        d = own;
    }
    return d - (less & 0xFF);
}

/* One sequence field's table. */
struct Field {
    uint32_t* cells;
    const uint32_t* codes; /* null: the offset field, whose extra bits are its symbol */
    uint32_t log;
    bool present;
};

/* walk_frame's flow of the entropy wave. */
struct EntropyFlow {
    FrameLds& l;
    uint32_t lane;
    uint32_t seq;  /* jobs so far */
    bool alive;    /* no wait has run out */
    Field ll, of, ml;
    uint32_t r0, r1, r2; /* the frame's repeat offsets */

    __device__ uint64_t u64(uint64_t v) const { return uniform64(v); }

    /* The next slot, once the copy wave is done with it. */
    __device__ __forceinline__ Job& slot() {
        if (seq >= kJobs && alive) {
            alive = await_flag((const lds_flag*)&l.consumed, seq - kJobs + 1, nullptr,
                               (lds_flag*)&l.broken) == kReached;
        }
        return l.job[seq % kJobs];
    }
    __device__ __forceinline__ void post(Job& j, uint32_t kind, uint32_t n, uint64_t a, uint64_t b,
                                         uint64_t c, uint32_t x, uint32_t y) {
        j.kind = kind;
        j.n = n;
        j.a = a;
        j.b = b;
        j.c = c;
        j.x = x;
        j.y = y;
        seq++;
        raise_flag((lds_flag*)&l.published, seq);
    }
    __device__ __forceinline__ void ask(uint32_t kind, uint32_t n, uint64_t a, uint64_t b,
                                        uint64_t c, uint32_t x, uint32_t y) {
        Job& j = slot();
        post(j, kind, n, a, b, c, x, y);
    }
    __device__ __forceinline__ void begin(uint64_t chunk, gu8* dst, uint64_t cap) {
        ll.present = of.present = ml.present = false;
        r0 = 1;
        r1 = 4;
        r2 = 8;
        ask(kJobFrame, 0, chunk, (uint64_t)(uintptr_t)dst, cap, 0, 0);
    }
    __device__ void block(const ZG uint8_t* from, uint8_t fill, uint64_t n) {
        ask(kJobBlock, (uint32_t)n, (uint64_t)(uintptr_t)from, 0, 0, fill, 0);
    }
    __device__ void literals(const ZG uint8_t* from, uint8_t fill, uint64_t n) {
        ask(kJobLiterals, (uint32_t)n, (uint64_t)(uintptr_t)from, 0, 0, fill, 0);
    }
    __device__ bool huffman(const ZG uint8_t* payload, uint64_t size, uint64_t regen,
                            uint32_t streams, bool treeless) {
        ask(kJobHuffman, (uint32_t)regen, (uint64_t)(uintptr_t)payload, size, 0, streams,
            treeless ? 1u : 0u);
        return true; /* the copy wave refuses it */
    }
    __device__ void tail(uint64_t lp, uint64_t n) {
        if (n != 0) {
            ask(kJobTail, (uint32_t)n, 0, 0, lp, 0, 0);
        }
    }

    /* Loads one field's table (RFC 8878 3.1.1.3.2.1): 0 predefined, 1
     * run-length, 2 an FSE description, 3 repeat; `head` holds the staged
     * section from its current position on, `left` the section's bytes. */
    __device__ __forceinline__ bool load(Field& f, uint32_t mode, const uint8_t* head,
                                         uint64_t left, uint32_t max_symbol, uint32_t log_max,
                                         const int16_t* defaults, uint32_t default_last,
                                         uint32_t default_log, uint32_t& used) {
        used = 0;
        if (mode == 3) {
            return f.present;
        }
        if (mode == 1) {
            const uint32_t s = left == 0 ? 255u : uniform32(head[0]);
            if (s > max_symbol) {
                return false;
            }
            f.cells[0] = s << kCellSymbol | (f.codes == nullptr ? s : f.codes[s] >> 24);
            wave_order();
            f.log = 0;
            f.present = true;
            used = 1;
            return true;
        }
        uint32_t last = default_last, log = default_log;
        if (mode == 0) {
            if (lane <= default_last) {
                l.e.counts[lane] = defaults[lane];
            }
        } else {
            uint64_t u = 0;
            if (!zstd::read_fse_description((const ZL uint8_t*)head, left, max_symbol, log_max,
                                            (ZL int16_t*)l.e.counts, last, log, u)) {
                return false;
            }
            last = uniform32(last);
            log = uniform32(log);
            used = uniform32((uint32_t)u);
        }
        wave_order();
        if (!build_cells(l.e.counts, l.e.next, f.cells, &l.e.window[kHeaderStage], last, log,
                         f.codes, lane)) {
            used = 0;
            return false;
        }
        f.log = log;
        f.present = true;
        return true;
    }

    __device__ int sequences(const ZG uint8_t* sec, uint64_t left, uint32_t modes, uint32_t count,
                             uint64_t regen, uint64_t window, uint64_t cap, uint64_t& lp,
                             uint64_t& o) {
        /* the three descriptions, whose readers stay below kHeaderStage: a
         * field's is at most 53 probabilities of 10 bits and as many 2-bit
         * repeat fields */
        EntropyLds& e = l.e;
        const uint32_t staged = left < kHeaderStage - 16 ? (uint32_t)left : kHeaderStage - 16;
        const uint32_t delta = stage_into<1>(e.window, (gcu8*)sec, staged, 0, staged, lane);
        const uint8_t* head = e.window + delta;
        uint32_t u = 0;
        if (!load(ll, modes >> 6, head, left, zstd::kLitLenMax, zstd::kLitLenLog,
                  zstd::kLitLenDefault, 35, 6, u)) {
            return CUDEC_ERR_CORRUPT_INPUT;
        }
        head += u;
        left -= u;
        sec += u;
        if (!load(of, (modes >> 4) & 3u, head, left, zstd::kOffsetMax, zstd::kOffsetLog,
                  zstd::kOffsetDefault, 28, 5, u)) {
            return CUDEC_ERR_CORRUPT_INPUT;
        }
        head += u;
        left -= u;
        sec += u;
        if (!load(ml, (modes >> 2) & 3u, head, left, zstd::kMatchLenMax, zstd::kMatchLenLog,
                  zstd::kMatchLenDefault, 52, 6, u)) {
            return CUDEC_ERR_CORRUPT_INPUT;
        }
        left -= u;
        sec += u;
        /* the backward bitstream (RFC 8878 4.1): `bits` left of it */
        const uint32_t marker = left == 0 ? 0u : uniform32(sec[left - 1]);
        if (marker == 0) {
            return CUDEC_ERR_CORRUPT_INPUT;
        }
        int bits = 8 * (int)(left - 1) + (int)zstd::high_bit(marker);

        /* this lane's field (0 literal length, 1 match length, 2 offset) and
         * its part of it: lanes 0 to 2 the next state, 4 to 6 the extra bits */
        const uint32_t f = (lane & 3) < 2 ? lane & 3 : 2;
        const bool states = (lane & 4) == 0;
        const uint32_t table = f == 0 ? lds_at(e.litlen) : f == 1 ? lds_at(e.matchlen)
                                                                   : lds_at(e.offset);
        /* what of the three cells' bits lies up to the end of this lane's
         * own: the offset's extra bits come first, then the match length's,
         * then the literal length's, then the states of literal length,
         * match length and offset */
        const uint32_t upto0 = states || f == 0 ? (states ? kCellSums : kCellExtras) : 0;
        const uint32_t upto1 = states    ? (f >= 1 ? kCellSums : kCellExtras)
                               : f <= 1 ? kCellExtras
                                        : 0;
        const uint32_t upto2 = states && f == 2 ? kCellSums : kCellExtras;
        const uint32_t own = states ? kCellBits : 0;
        /* what a value is: 1 << extra bits plus these for the offset, the
         * code above these for the lengths */
        const uint32_t one = f == 2 ? 1 : 0, code = f == 2 ? 0 : 63u << kCellSymbol;
        uint32_t cell = 0; /* of the next sequence */
        int pending = CUDEC_OK; /* the first execution error, reported once
                                   the whole block decodes */
        uint32_t k = 0;
        for (;;) {
            /* stage what the batch reads: its bytes end where `bits` does */
            const uint32_t hi = ((uint32_t)bits + 7) >> 3;
            const uint32_t lo = hi > zstd::kWindowBytes - 32 ? hi - (zstd::kWindowBytes - 32) : 0;
            wave_order();
            const uint32_t skew =
                stage_into<1>(e.window, (gcu8*)sec, hi, lo, hi - lo, lane);
            const uint32_t win = lds_at(e.window);
            const int base = 8 * ((int)skew - (int)lo); /* window bit of stream bit 0 */
            if (k == 0) {
                /* the initial states: literal length, offset, match length */
                const uint32_t n = f == 0 ? ll.log : f == 1 ? ml.log : of.log;
                const uint32_t end = f == 0    ? ll.log
                                     : f == 2 ? ll.log + of.log
                                              : ll.log + of.log + ml.log;
                const uint32_t state =
                    bits_of(words_below(win, base + bits), base + bits - (int)end, n);
                cell = *(lds_u32*)(uintptr_t)(table + 4 * state);
                bits -= (int)(ll.log + of.log + ml.log);
                if (bits < 0) {
                    return CUDEC_ERR_CORRUPT_INPUT;
                }
            }
            const uint32_t cnt = count - k < kWave ? count - k : kWave;
            Job& j = slot();
            /* the extra bits' lanes write; the others to a word of no use */
            uint32_t raw = states ? lds_at(&l.unused) : lds_at(j.ll) + 4 * f;
            const uint32_t stride = states ? 0 : 12;
            int at = base + bits; /* window bit above the next one */
            Top top = top_below(win, at);
            uint32_t end, s = cnt;
            do {
                /* bits from `at` down to the end of this lane's own */
                end = __builtin_amdgcn_sad_u8((quad<0>(cell) & upto0) + (quad<1>(cell) & upto1) +
                                                  (quad<2>(cell) & upto2),
                                              0, 0);
                const uint32_t n = __builtin_amdgcn_ubfe(cell, own, 5);
                uint32_t v = __builtin_amdgcn_ubfe((uint32_t)(top.bits(at) >> ((64 - end) & 63)),
                                                   0, n);
                if (__builtin_expect(__ballot(end > 64) != 0, 0)) {
                    v = bits_of(words_below(win, at), at - (int)end, n);
                }
                at -= (int)__builtin_amdgcn_readlane(end, 2); /* the last of them */
                top = top_below(win, at);
                /* the next cell, its address from the state's lane */
                const uint32_t next = table + 4 * ((cell >> kCellBase) + v);
                const uint32_t word = (cell & code) | ((one << n) + v);
                cell = *(lds_u32*)(uintptr_t)(uint32_t)__builtin_amdgcn_update_dpp(
                    (int)next, (int)next, 0x114, 0xF, 0xA, false); /* row_shr:4 on every other four */
                *(lds_u32*)(uintptr_t)raw = word;
                raw += stride;
            } while (--s != 0);
            if (k + cnt == count) {
                /* no state is read after the block's last sequence */
                at += (int)(__builtin_amdgcn_readlane(end, 2) - __builtin_amdgcn_readlane(end, 4));
            }
            bits = (int)uniform32((uint32_t)(at - base));
            if (bits < 0) {
                return CUDEC_ERR_CORRUPT_INPUT;
            }
            wave_order();
            if (pending == CUDEC_OK) {
                pending = finish_batch(j, cnt, regen, window, cap, lp, o);
            }
            k += cnt;
            if (k == count) {
                break;
            }
        }
        if (bits != 0) {
            return CUDEC_ERR_CORRUPT_INPUT;
        }
        return pending;
    }

    /* A batch's raw values (three words a sequence, in the slot) to lengths
     * and distances, a lane each, with every check of their execution; posts
     * the job, or returns the first error in stream order. */
    __device__ __forceinline__ int finish_batch(Job& j, uint32_t cnt, uint64_t regen,
                                                uint64_t window, uint64_t cap, uint64_t& lp,
                                                uint64_t& o) {
        const uint32_t* raw = j.ll + 3 * lane;
        const uint32_t v0 = raw[0], v1 = raw[1], value = raw[2];
        wave_order();
        const bool in = lane < cnt;
        const uint32_t c0 = v0 >> 16, c1 = v1 >> 16;
        const uint32_t llen =
            in ? (l.e.code[c0 <= zstd::kLitLenMax ? c0 : 0] & 0xFFFFFF) + (v0 & 0xFFFF) : 0;
        const uint32_t mlen =
            in ? (l.e.code[zstd::kLitLenMax + 1 + (c1 <= zstd::kMatchLenMax ? c1 : 0)] & 0xFFFFFF) +
                     (v1 & 0xFFFF)
               : 0;
        /* repeat offsets (RFC 8878 3.1.1.5): each sequence maps the three
         * offsets before it to the three after it, its own distance first;
         * an inclusive scan composes the maps (Repeats). Zero: an error. */
        const uint32_t which = in ? value - 1 + (llen == 0 ? 1u : 0u) : 0;
        const bool own = in && value > 3;
        /* of 0 to 3: the first from {0, 1, 2, 0}, the third from {2, 2, 1, 1}
         * by v_perm, the second 1 or 0 */
        const uint32_t old = __builtin_amdgcn_perm(0x01010202u, 0x00020100u,
                                                   __umul24(which & 3, 0x10001u) + 0x0C040C00u) |
                             (which == 0 ? 0x100u : 0u);
        Repeats r = {own ? 0x010000u | kOwn | lane : old, which == 3 && !own ? 1u : 0u};
        r = repeats_after<0x111, 0xF>(r); /* row_shr:1, 2, 4, 8 */
        r = repeats_after<0x112, 0xF>(r);
        r = repeats_after<0x114, 0xF>(r);
        r = repeats_after<0x118, 0xF>(r);
        r = repeats_after<0x142, 0xA>(r); /* row_bcast:15, 31 */
        r = repeats_after<0x143, 0xC>(r);
        const uint32_t brought = value - 3;
        const uint32_t mine = (uint32_t)__shfl((int)brought, (int)(r.from & (kWave - 1)));
        /* (read before the choice: a choice of members becomes a load at a
         * chosen scratch address, 600 cycles) */
        const uint32_t b0 = uniform32(r0), b1 = uniform32(r1), b2 = uniform32(r2);
        const uint32_t dist = offset_of(r.from, r.less, mine, b0, b1, b2);
        const uint32_t from = uniform32(__builtin_amdgcn_readlane(r.from, kWave - 1));
        const uint32_t less = uniform32(__builtin_amdgcn_readlane(r.less, kWave - 1));
        r0 = offset_of(from, less, __builtin_amdgcn_readlane(brought, from & (kWave - 1)), b0, b1,
                       b2);
        r1 = offset_of(from >> 8, less >> 8,
                       __builtin_amdgcn_readlane(brought, (from >> 8) & (kWave - 1)), b0, b1, b2);
        r2 = offset_of(from >> 16, less >> 16,
                       __builtin_amdgcn_readlane(brought, (from >> 16) & (kWave - 1)), b0, b1, b2);
        /* positions in 32 bits, whatever the lengths claim: a sequence of at
         * most 65536 + 65535 literals and a match of 65539 + 65535 bytes, 64
         * of which stay below 2^25 */
        const uint32_t lit_incl = wave_inclusive_sum(llen, lane);
        const uint32_t out_incl = wave_inclusive_sum(llen + mlen, lane);
        const uint64_t m = o + (out_incl - mlen);
        int ev = CUDEC_OK;
        if (in) {
            if (lit_incl > regen - lp || dist == 0 || dist > m || dist > window) {
                ev = CUDEC_ERR_CORRUPT_INPUT;
            } else if (m > cap || mlen > cap - m) {
                ev = CUDEC_ERR_OUTPUT_TOO_SMALL;
            }
        }
        const uint64_t bad = __ballot(ev != CUDEC_OK);
        if (bad != 0) {
            return (int)uniform32(__builtin_amdgcn_readlane((uint32_t)ev, __builtin_ctzll(bad)));
        }
        j.ll[lane] = llen;
        j.ml[lane] = mlen;
        j.off[lane] = dist;
        post(j, kJobSequences, cnt, 0, 0, lp, 0, 0);
        lp += uniform32(__builtin_amdgcn_readlane(lit_incl, kWave - 1));
        o += uniform32(__builtin_amdgcn_readlane(out_incl, kWave - 1));
        return CUDEC_OK;
    }
};

/* ----------------------------------------------------------- literals */

/* Reads a Huffman tree description (RFC 8878 4.2.1) and fills the decode
 * table, as zstd::read_huffman_table does one step after the other: cell
 * index = the next table_log bits; symbol in the low byte, code length in the
 * high byte. The description is staged; only the FSE-compressed weights are
 * read in sequence. False if it is refused. */
__device__ __forceinline__ bool read_tree(CopyLds& w, gcu8* src, uint64_t size, uint32_t& table_log,
                                          uint32_t& used, uint32_t lane) {
    if (size == 0) {
        return false;
    }
    const uint32_t staged = size < 160 ? (uint32_t)size : 160;
    const uint8_t* head = w.stage + stage_into<1>(w.stage, src, staged, 0, staged, lane);
    const uint32_t header = uniform32(head[0]);
    const uint32_t payload = header >= 128 ? (header - 126) / 2 : header;
    if (payload + 1 > size) {
        return false;
    }
    used = payload + 1;
    uint32_t written = 0;
    if (header >= 128) {
        written = header - 127;
        for (uint32_t i = lane; i < written; i += kWave) {
            const uint32_t b = head[1 + i / 2];
            w.weights[i] = (uint8_t)((i & 1) == 0 ? b >> 4 : b & 15u);
        }
    } else {
        uint32_t last = 0, log = 0;
        uint64_t description = 0;
        if (!zstd::read_fse_description((const ZL uint8_t*)(head + 1), payload,
                                        zstd::kWeightSymbolMax, zstd::kWeightLogMax,
                                        (ZL int16_t*)w.counts, last, log, description)) {
            return false;
        }
        last = uniform32(last);
        log = uniform32(log);
        wave_order();
        if (!build_cells(w.counts, w.next, w.weight_cells, w.stage + 512, last, log, nullptr,
                         lane)) {
            return false;
        }
        const uint32_t from = 1 + uniform32((uint32_t)description);
        const uint32_t mark = from > payload ? 0 : uniform32(head[payload]);
        if (mark == 0) {
            return false;
        }
        /* two states in turn; when a state's update needs more bits than
         * remain, its symbol and the other state's close the list */
        const uint32_t base = lds_at(head + from);
        uint32_t bits = 8 * (payload - from) + zstd::high_bit(mark);
        if (bits < 2 * log) {
            return false;
        }
        const uint32_t a0 = base & ~3u, skew = 8 * (base & 3);
        const auto take = [&](uint32_t n) {
            bits -= n;
            const uint32_t p = bits + skew, a = a0 + (p >> 5 << 2);
            return uniform32(__builtin_amdgcn_ubfe(
                __builtin_amdgcn_alignbit(*(lds_u32*)(uintptr_t)(a + 4), *(lds_u32*)(uintptr_t)a,
                                          p & 31),
                0, n));
        };
        uint32_t one = take(log), other = take(log);
        for (;;) {
            const uint32_t cell = uniform32(w.weight_cells[one]);
            w.weights[written++] = (uint8_t)(cell >> kCellSymbol & 63);
            const uint32_t n = cell >> kCellBits & 15;
            if (written == 255) {
                return false;
            }
            if (n > bits) {
                w.weights[written++] = (uint8_t)(w.weight_cells[other] >> kCellSymbol & 63);
                break;
            }
            one = other;
            other = (cell >> kCellBase) + take(n);
        }
    }
    wave_order();
    /* symbol 64 r + lane on this lane */
    uint32_t weight[4], sum = 0;
    bool over = false;
#pragma unroll
    for (uint32_t r = 0; r < 4; r++) {
        const uint32_t i = r * kWave + lane;
        weight[r] = i < written ? w.weights[i] : 0;
        over |= weight[r] > zstd::kHufLogMax;
        sum += (1u << weight[r]) >> 1;
    }
    if (__ballot(over) != 0) {
        return false;
    }
    const uint32_t total =
        uniform32(__builtin_amdgcn_readlane(wave_inclusive_sum(sum, lane), kWave - 1));
    if (total == 0) {
        return false;
    }
    const uint32_t log = zstd::high_bit(total) + 1;
    if (log > zstd::kHufLogMax) {
        return false;
    }
    const uint32_t rest = (1u << log) - total;
    const uint32_t last_weight = zstd::high_bit(rest) + 1;
    if ((1u << (last_weight - 1)) != rest) {
        return false;
    }
    /* codes of weight 1 (the longest) take the lowest cells, then weight 2,
     * ...; within a weight, symbols in increasing order */
    uint32_t at = 0;
    uint32_t begin = 0; /* of weight `lane` */
    for (uint32_t k = 1; k <= log; k++) {
        uint32_t have = 0;
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) {
            if (r * kWave + lane == written) {
                weight[r] = last_weight;
            }
            have += (uint32_t)__builtin_popcountll(__ballot(weight[r] == k));
        }
        if (k == 1 && have < 2) {
            return false;
        }
        begin = lane == k ? at : begin;
        at += have << (k - 1);
    }
    if (lane < 16) {
        w.first[lane] = begin;
    }
    wave_order();
    const uint64_t below = (1ull << lane) - 1;
#pragma unroll
    for (uint32_t r = 0; r < 4; r++) {
        if (r * kWave > written) {
            break;
        }
        const uint32_t wt = weight[r];
        uint64_t same = ~0ull;
#pragma unroll
        for (uint32_t b = 0; b < 4; b++) {
            const uint64_t set = __ballot(((wt >> b) & 1) != 0);
            same &= ((wt >> b) & 1) != 0 ? set : ~set;
        }
        const uint32_t span = (1u << wt) >> 1;
        const uint32_t to = w.first[wt] + (uint32_t)__builtin_popcountll(same & below) * span;
        wave_order();
        if ((same >> lane) == 1) { /* the weight's last symbol here */
            w.first[wt] = to + span;
        }
        const uint32_t cell = (r * kWave + lane) | (log + 1 - wt) << 8;
        /* short spans by their own lane, long ones by all */
        uint64_t wide = __ballot(span >= 32);
        if (span == 1) {
            w.huffman[to] = (uint16_t)cell;
        } else if (span < 32) {
            for (uint32_t j = 0; j < span; j += 2) {
                *(uint32_t*)&w.huffman[to + j] = cell | cell << 16;
            }
        }
        while (wide != 0) {
            const uint32_t i = (uint32_t)__builtin_ctzll(wide);
            wide &= wide - 1;
            const uint32_t c = __builtin_amdgcn_readlane(cell, i);
            const uint32_t n = __builtin_amdgcn_readlane(span, i);
            const uint32_t t = __builtin_amdgcn_readlane(to, i);
            for (uint32_t j = 2 * lane; j < n; j += 2 * kWave) {
                *(uint32_t*)&w.huffman[t + j] = c | c << 16;
            }
        }
        wave_order();
    }
    table_log = log;
    return true;
}

/* Up to eight codes from stream bit p down. Twelve bytes hold them: 89 bits
 * below p at least, eight codes of 11 bits at most. A stream's first bytes
 * follow a frame's, a block's and a section's header and a tree or a jump
 * table, 14 bytes at least, so the load stays in the frame. */
struct Codes {
    uint64_t acc; /* the next bits on top */
    uint32_t low; /* the bits below, on top */
    uint32_t taken;
    __device__ __forceinline__ void load(gcu8* src, int p) {
        const int end = (p + 7) >> 3;
        uint32_t v[3];
        __builtin_memcpy(v, (const void*)(src + (end - 12)), 12);
        const uint32_t skip = (uint32_t)(8 * end - p);
        const uint64_t tail = (uint64_t)v[0] << skip;
        acc = ((uint64_t)v[2] << 32 | v[1]) << skip | tail >> 32;
        low = (uint32_t)tail;
        taken = 0;
    }
    __device__ __forceinline__ uint32_t index(uint32_t shift) const {
        return (uint32_t)(acc >> 32) >> shift;
    }
    __device__ __forceinline__ void drop(uint32_t n) {
        acc <<= n;
        taken += n;
    }
    /* after four codes: the bits below follow */
    __device__ __forceinline__ void refill() {
        acc |= (uint64_t)low << 32 >> ((64 - taken) & 63);
    }
};

/* From stream bit p code by code until p is `stop` or less; counts them. */
__device__ __forceinline__ int walk_codes(gcu8* src, const uint16_t* table, uint32_t shift, int p,
                                          int stop, uint32_t& count) {
    while (p > stop) {
        Codes c;
        c.load(src, p);
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) {
            if (j == 4) {
                c.refill();
            }
            const uint32_t bits = p > stop ? (uint32_t)table[c.index(shift)] >> 8 : 0;
            count += p > stop ? 1 : 0;
            c.drop(bits);
            p -= (int)bits;
        }
    }
    return p;
}

/* A Huffman-coded literals section's payload (RFC 8878 3.1.1.3.1), as
 * zstd::decode_huffman_section decodes it a lane a stream: the tree
 * description unless treeless (log holds the table of the block before, 0:
 * none), then one or four streams of `regen` symbols in all.
 *
 * A stream is a chain of table lookups, about 110 cycles a symbol. Prefix
 * codes synchronise by themselves: a decoder started at any bit soon finds
 * code boundaries of the real chain. So a stream is cut into 16 segments (64
 * for a single stream), and each lane starts 24 longest codes before its own
 * and walks to its end; then a lane whose start is not where the lane before
 * it ended walks again from there, until all agree. (The first lane is right
 * at once, and each round makes at least one more so; codes that never
 * synchronise take as long as one lane would.) Segments are multiples of
 * table_log, so codes of one length agree at once. Counts give each segment's
 * place, and a second walk writes the symbols, eight a store.
 *
 * A 64 KiB frame's literals took 1.18 M cycles with a lane a stream and the
 * tree read in sequence; 0.16 M so.
 *
 * A stream is right if its chain ends on bit 0 with the symbols it should
 * have: a code that takes bits from below bit 0 ends below it, whatever they
 * are. */
__device__ __forceinline__ bool huffman_section(CopyLds& w, gcu8* payload, uint64_t psize,
                                                uint32_t regen, uint32_t streams, bool treeless,
                                                uint32_t& log, gu8* lits, uint32_t lane) {
    if (!treeless) {
        uint32_t used = 0, tree_log = 0;
        if (!read_tree(w, payload, psize, tree_log, used, lane)) {
            return false;
        }
        log = tree_log;
        payload += used;
        psize -= used;
    } else if (log == 0) {
        return false;
    }
    if (psize == 0) {
        return false;
    }
    const uint32_t lanes = streams == 1 ? kWave : kWave / 4;
    const uint32_t k = lane & (lanes - 1);
    gcu8* src = payload;
    uint32_t size = (uint32_t)psize, n = regen, to = 0;
    if (streams != 1) {
        if (psize < 10 || regen < 6) {
            return false;
        }
        uint32_t jump[3];
        for (uint32_t i = 0; i < 3; i++) {
            jump[i] = uniform32(payload[2 * i] | (uint32_t)payload[2 * i + 1] << 8);
        }
        const uint32_t bytes = (uint32_t)psize - 6;
        if (jump[0] + jump[1] + jump[2] >= bytes) {
            return false;
        }
        const uint32_t g = lane / lanes, seg = (regen + 3) / 4;
        src += 6 + (g > 0 ? jump[0] : 0) + (g > 1 ? jump[1] : 0) + (g > 2 ? jump[2] : 0);
        size = g == 0   ? jump[0]
               : g == 1 ? jump[1]
               : g == 2 ? jump[2]
                        : bytes - jump[0] - jump[1] - jump[2];
        to = g * seg;
        n = g < 3 ? seg : regen - 3 * seg;
    }
    const uint32_t mark = size == 0 ? 0 : src[size - 1];
    if (__ballot(mark == 0) != 0) {
        return false;
    }
    const uint32_t shift = 32 - log;
    const int bits = 8 * (int)(size - 1) + (int)zstd::high_bit(mark);
    const int least = 64 / (int)log + 1;
    int codes = (bits + (int)(lanes * log) - 1) / (int)(lanes * log);
    codes = codes < least ? least : codes;
    const int per = codes * (int)log;
    const int hi = bits - (int)k * per;
    const int lo = hi - per > 0 ? hi - per : 0;
    /* where this lane's codes begin: a guess, but for the first lane */
    int begin = hi + 24 * (int)log < bits ? hi + 24 * (int)log : bits;
    uint32_t count = 0;
    begin = hi <= 0 ? 0 : walk_codes(src, w.huffman, shift, begin, hi, count);
    count = 0;
    int end = walk_codes(src, w.huffman, shift, begin, lo, count);
    for (;;) {
        const int before =
            __builtin_amdgcn_update_dpp(bits, end, 0x138, 0xF, 0xF, false); /* wave_shr:1 */
        const int should = k == 0 ? bits : before;
        if (__ballot(should != begin) == 0) {
            break;
        }
        if (should != begin) {
            begin = should;
            count = 0;
            end = walk_codes(src, w.huffman, shift, begin, lo, count);
        }
    }
    const uint32_t incl = wave_inclusive_sum(count, lane);
    const uint32_t group = lane - k; /* symbols of the streams before */
    const uint32_t earlier = (uint32_t)__shfl((int)(incl - count), (int)group);
    if (__ballot(k == lanes - 1 && (end != 0 || incl - earlier != n)) != 0) {
        return false;
    }
    gu8* out = lits + to + (incl - count - earlier);
    int p = begin;
    while (count != 0) {
        Codes c;
        c.load(src, p);
        uint32_t word[2] = {0, 0};
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) {
            if (j == 4) {
                c.refill();
            }
            const uint32_t cell = w.huffman[c.index(shift)];
            const uint32_t n_bits = j < count ? cell >> 8 : 0;
            word[j / 4] |= (cell & 0xFF) << (8 * (j & 3));
            c.drop(n_bits);
        }
        p -= (int)c.taken;
        if (count >= 8) {
            __builtin_memcpy((void*)out, word, 8);
            out += 8;
            count -= 8;
        } else {
            const uint64_t rest = (uint64_t)word[1] << 32 | word[0];
            for (uint32_t j = 0; j < count; j++) {
                out[j] = (uint8_t)(rest >> (8 * j));
            }
            count = 0;
        }
    }
    wave_order();
    return true;
}

/* ------------------------------------------------------------ copies */

/* The copy wave's place in a frame's output. */
struct CopyState {
    gu8* dst;
    uint64_t cap;
    uint64_t dp;      /* output bytes so far */
    uint64_t flushed; /* of them, in memory */
    uint64_t ring_lo; /* the ring holds none before */
    gcu8* lit;        /* the block's literals */
};

/* n bytes from memory to the output: a few through the ring, more around it. */
__device__ __forceinline__ void copy_bytes(CopyLds& w, CopyState& s, gcu8* from, uint32_t n,
                                           uint32_t lane) {
    const uintptr_t da = (uintptr_t)s.dst;
    if (n <= kBatchMax / 2) {
        for (uint32_t i = lane; i < n; i += kWave) {
            w.ring[ring_index<kRing>(da, s.dp + i)] = from[i];
        }
        wave_order();
        s.dp += n;
        const uintptr_t a_end = (da + s.dp) & ~(uintptr_t)15;
        if (a_end > da + s.flushed) {
            flush_ring(w, s.dst, s.flushed, (uint64_t)(a_end - da), lane);
            s.flushed = (uint64_t)(a_end - da);
        }
        return;
    }
    flush_ring(w, s.dst, s.flushed, s.dp, lane);
    wave_copy_global(s.dst + s.dp, from, n, lane);
    s.dp += n;
    s.flushed = s.dp;
    s.ring_lo = s.dp;
}

/* n times the byte `fill` at `to`. */
__device__ __forceinline__ void fill_bytes(gu8* to, uint32_t fill, uint32_t n, uint32_t lane) {
    const uint32_t word = fill * 0x01010101u;
    const uint4 v = make_uint4(word, word, word, word);
    for (uint32_t i = 16 * lane; i + 16 <= n; i += 16 * kWave) {
        gstore16(to + i, v);
    }
    const uint32_t done = n & ~15u;
    if (lane < n - done) {
        to[done + lane] = (uint8_t)fill;
    }
    wave_order();
}

/* The copy wave's groups go without strips: it is the entropy wave that a
 * frame of short matches waits for, and their registers cost the kernel 3%. */
struct AloneInOrder : Alone {
    static constexpr bool kStrips = false;
};

/* A batch of cnt sequences, as groups that the ring and the literals' stage
 * hold; a sequence that fits neither goes global to global. */
__device__ __forceinline__ void run_sequences(CopyLds& w, CopyState& s, const Job& j, uint32_t cnt,
                                              uint64_t lp, uint32_t lane) {
    const uint32_t ll = j.ll[lane], ml = j.ml[lane], off = j.off[lane];
    for (uint32_t i = 0; i < cnt;) {
        /* sequence i + lane on this lane */
        uint32_t gl = ll, gm = ml, go = off;
        if (i != 0) {
            gl = (uint32_t)__shfl((int)ll, (int)((i + lane) & (kWave - 1)));
            gm = (uint32_t)__shfl((int)ml, (int)((i + lane) & (kWave - 1)));
            go = (uint32_t)__shfl((int)off, (int)((i + lane) & (kWave - 1)));
        }
        const bool in = i + lane < cnt;
        const uint32_t lit = in ? gl : 0, match = in ? gm : 0;
        const uint32_t lit_incl = wave_inclusive_sum(lit, lane);
        const uint32_t out_incl = wave_inclusive_sum(lit + match, lane);
        const uint64_t over = __ballot(!in || lit_incl > kLitStage || out_incl > kBatchMax);
        const uint32_t take = over == 0 ? kWave : (uint32_t)__builtin_ctzll(over);
        if (take == 0) {
            Lz4Step q;
            q.lit_src = lp;
            q.lit_dst = s.dp;
            q.lit_len = uniform32(lit);
            q.match_dst = s.dp + q.lit_len;
            q.match_len = uniform32(match);
            q.offset = uniform32(go);
            execute_slow(w, s.lit, s.dst, s.cap, q, q.match_dst + q.match_len, s.dp, s.flushed,
                         s.ring_lo, false, lane);
            lp += q.lit_len;
            i++;
            continue;
        }
        const uint32_t lits = uniform32(__builtin_amdgcn_readlane(lit_incl, take - 1));
        const uint32_t delta = stage_into<1>(w.stage, s.lit, lp + lits, lp, lits, lane);
        Group g;
        g.lit = lit_incl - lit;
        g.lit_len = lit;
        g.match_len = match;
        g.offset = go;
        g.drel = out_incl - (lit + match);
        g.take = take;
        g.terminal = false;
        g.end_rel = uniform32(__builtin_amdgcn_readlane(out_incl, take - 1));
        execute_group(w, w.cover, w.stage + delta, g, s.dst, s.cap, s.dp, s.flushed, s.ring_lo,
                      false, lane, AloneInOrder{});
        lp += lits;
        i += take;
    }
}

/* Scratch of one launch: the frame counter, the cost order, a FrameCheck
 * per frame, then a literals slot of kBlockCeiling bytes per block of the
 * grid. */
constexpr size_t kCounterBytes = 256;

__global__ void zstd_reset(unsigned long long* counter, unsigned long long first) {
    if (threadIdx.x == 0) {
        *counter = first;
    }
}

constexpr int kFrameBlock = 2 * kWave;
__global__ void __launch_bounds__(kFrameBlock) __attribute__((amdgpu_waves_per_eu(4)))
    zstd_batch(const void* const* srcs, const size_t* sizes, void* const* dsts, const size_t* caps,
               size_t n, cudec_chunk_result* results, unsigned long long* counter,
               const uint32_t* order, FrameCheck* checks, uint8_t* lits_base) {
    __shared__ FrameLds l;
    const uint32_t lane = __lane_id();
    const bool entropy = uniform32(threadIdx.x / kWave) == 0;
    if (entropy) {
        for (uint32_t c = lane; c < kCodes; c += kWave) {
            const uint32_t m = c - (zstd::kLitLenMax + 1);
            l.e.code[c] = c <= zstd::kLitLenMax
                              ? zstd::kLitLenBase[c] | (uint32_t)zstd::kLitLenBits[c] << 24
                              : zstd::kMatchLenBase[m] | (uint32_t)zstd::kMatchLenBits[m] << 24;
        }
        l.published = 0;
        l.consumed = 0;
        l.broken = 0;
        l.begin = blockIdx.x;
        l.after = counter != nullptr ? kAsk : kNoMore;
    }
    __syncthreads();
    if (entropy) {
        EntropyFlow f{l, lane, 0, true,
                      Field{l.e.litlen, l.e.code, 0, false},
                      Field{l.e.offset, nullptr, 0, false},
                      Field{l.e.matchlen, l.e.code + zstd::kLitLenMax + 1, 0, false},
                      1, 4, 8};
        /* every lane issues the atomic (lane 0 adds one, the others zero, so
         * lane 0's old value is the frame's index whatever order the lanes
         * are applied in): a lane-0-only branch here let the compiler's
         * structurizer send lanes 1..63 back to the read without lane 0 */
        while (f.alive) {
            /* a block begins with the frame of its own index, and the counter
             * goes on behind those, if there are any more: a pop takes 12 ns,
             * whoever makes it, and frames by index lie evenly over the CUs
             * (2048 frames of 100 stored bytes: 78 us with a pop for each
             * frame and for each block's end, 45 so; 1000 of 1 MiB of tokens:
             * 8.08 ms and 7.06). What comes next is kept in LDS: held over
             * the frame in registers it costs the FSE loop up to 1%. */
            uint64_t k = uniform32(l.begin);
            if (k == kAsk) {
                const unsigned long long old = atomicAdd(counter, lane == 0 ? 1ull : 0ull);
                k = uniform64(old);
            }
            l.begin = l.after;
            if (k >= n) {
                break;
            }
            const uint64_t i = uniform32(order[k]);
            const ZG uint8_t* src =
                (const ZG uint8_t*)uniform_ptr(static_cast<const uint8_t*>(srcs[i]));
            gu8* dst = global_bytes(dsts[i]);
            const uint64_t size = uniform64(sizes[i]);
            const uint64_t cap = uniform64(caps[i]);
            f.begin(i, dst, cap);
            zstd::FrameEnd end{0, 0, false};
            const int st = (int)uniform32((uint32_t)zstd::walk_frame(f, src, size, cap, end));
            if (st != CUDEC_OK) {
                f.ask(kJobFail, 0, 0, 0, 0, (uint32_t)st, 0);
            } else {
                f.ask(kJobEnd, 0, end.written, 0, 0, end.checksum, end.has_checksum ? 1u : 0u);
            }
        }
        f.ask(kJobQuit, 0, 0, 0, 0, 0, 0);
        return;
    }
    CopyLds& w = l.c;
    gu8* lits = (gu8*)(lits_base + (size_t)blockIdx.x * zstd::kBlockCeiling);
    CopyState s{nullptr, 0, 0, 0, 0, lits};
    uint64_t chunk = 0;
    uint32_t huf_log = 0;
    int status = CUDEC_OK;
    bool open = false; /* a frame has begun and not ended */
    for (uint32_t seq = 0;; seq++) {
        if (await_flag((const lds_flag*)&l.published, seq + 1, nullptr, (lds_flag*)&l.broken) !=
            kReached) {
            if (open) {
                write_result(results, chunk, CUDEC_ERR_CUDA, 0);
                checks[chunk].verify = 0;
            }
            return;
        }
        const Job& j = l.job[seq % kJobs];
        const uint32_t kind = uniform32(j.kind), num = uniform32(j.n), x = uniform32(j.x),
                       y = uniform32(j.y);
        const uint64_t a = uniform64(j.a), b = uniform64(j.b), c = uniform64(j.c);
        if (kind == kJobQuit) {
            return;
        }
        if (kind == kJobFrame) {
            chunk = a;
            s = CopyState{(gu8*)(uintptr_t)b, c, 0, 0, 0, lits};
            huf_log = 0;
            status = CUDEC_OK;
            open = true;
        } else if (kind == kJobFail || kind == kJobEnd) {
            if (kind == kJobFail && status == CUDEC_OK) {
                status = (int)x;
            }
            if (status == CUDEC_OK) {
                flush_ring(w, s.dst, s.flushed, s.dp, lane);
            }
            write_result(results, chunk, status, status == CUDEC_OK ? a : 0);
            FrameCheck fc;
            fc.written = a;
            fc.checksum = x;
            fc.verify = status == CUDEC_OK && y != 0 ? 1u : 0u;
            checks[chunk] = fc;
            open = false;
        } else if (status == CUDEC_OK) {
            if (kind == kJobSequences) {
                run_sequences(w, s, j, num, c, lane);
            } else if (kind == kJobTail) {
                copy_bytes(w, s, s.lit + c, num, lane);
            } else if (kind == kJobLiterals) {
                s.lit = (gcu8*)(uintptr_t)a;
                if (a == 0) {
                    fill_bytes(lits, x, num, lane);
                    s.lit = lits;
                }
            } else if (kind == kJobHuffman) {
                s.lit = lits;
                if (!huffman_section(w, (gcu8*)(uintptr_t)a, b, num, x, y != 0, huf_log, lits,
                                     lane)) {
                    status = CUDEC_ERR_CORRUPT_INPUT;
                }
                status = (int)uniform32((uint32_t)status);
                huf_log = uniform32(huf_log);
                wave_order();
            } else if (a != 0) { /* kJobBlock */
                copy_bytes(w, s, (gcu8*)(uintptr_t)a, num, lane);
            } else {
                flush_ring(w, s.dst, s.flushed, s.dp, lane);
                fill_bytes(s.dst + s.dp, x, num, lane);
                s.dp += num;
                s.flushed = s.dp;
                s.ring_lo = s.dp;
            }
        }
        raise_flag((lds_flag*)&l.consumed, seq + 1);
    }
}

/* Frames that decoded and carry a content checksum: the low 32 bits of the
 * XXH64 (seed 0) of the output must equal it (RFC 8878 3.1.1). */
__global__ void __launch_bounds__(kVerifyBlock)
    zstd_verify(void* const* dsts, size_t n, const FrameCheck* checks,
                cudec_chunk_result* results) {
    const uint32_t lane = __lane_id();
    const uint32_t q = lane % xxh::kGroup;
    constexpr uint32_t kPerBlock = kVerifyBlock / xxh::kGroup;
    const size_t per_grid = (size_t)gridDim.x * kPerBlock;
    for (size_t i = (size_t)blockIdx.x * kPerBlock + threadIdx.x / xxh::kGroup;; i += per_grid) {
        const bool in_range = i < n;
        if (__ballot(in_range) == 0) {
            break;
        }
        const bool live = in_range && checks[i].verify != 0;
        const uint64_t h = xxh::xxh64_group(live ? (gcu8*)dsts[i] : nullptr,
                                            live ? checks[i].written : 0, 0, q, lane - q);
        if (live && q == 0 && (uint32_t)h != checks[i].checksum) {
            write_result(results, i, CUDEC_ERR_CORRUPT_INPUT, 0);
        }
    }
}

std::mutex g_pool_lock;
constexpr int kMaxDevices = 64;
hipMemPool_t g_pool[kMaxDevices];
bool g_pool_tried[kMaxDevices];

/* The device's scratch pool for this decoder, made on first use; it keeps
 * up to kPoolKeep bytes of freed scratch between launches. */
hipMemPool_t zstd_pool(int dev) {
    if (dev < 0 || dev >= kMaxDevices) {
        return nullptr;
    }
    std::lock_guard<std::mutex> hold(g_pool_lock);
    if (!g_pool_tried[dev]) {
        g_pool_tried[dev] = true;
        hipMemPoolProps props = {};
        props.allocType = hipMemAllocationTypePinned;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t pool = nullptr;
        if (hipMemPoolCreate(&pool, &props) == hipSuccess) {
            uint64_t keep = kPoolKeep;
            if (hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep) == hipSuccess) {
                g_pool[dev] = pool;
            } else {
                (void)hipMemPoolDestroy(pool);
            }
        }
        (void)hipGetLastError(); /* a pool that could not be made is not an error */
    }
    return g_pool[dev];
}

}  // namespace

/* tuned.hip: the batch's cost order. */
size_t cost_order_bytes(size_t n);
hipError_t cost_order(const size_t* sizes, const size_t* caps, size_t n, void* work,
                      hipStream_t stream, const uint32_t** order);

hipError_t launch_zstd(const void* const* srcs, const size_t* sizes, void* const* dsts,
                       const size_t* caps, size_t n, cudec_chunk_result* results,
                       hipStream_t stream) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        return e;
    }
    int cus = 0;
    e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) {
        return e;
    }
    /* as many blocks as are resident at once (LDS and registers decide), on
     * every CU */
    int per_cu = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, zstd_batch, kFrameBlock, 0);
    if (e != hipSuccess) {
        return e;
    }
    const size_t blocks = (size_t)(cus > 0 ? cus : 1) * (size_t)(per_cu > 0 ? per_cu : 1);
    const size_t grid = n < blocks ? n : blocks;
    if (n > UINT32_MAX) {
        return hipErrorInvalidValue; /* the cost order indexes frames in 32 bits */
    }
    const size_t order_bytes = (cost_order_bytes(n) + 255) & ~(size_t)255;
    const size_t checks_bytes = (sizeof(FrameCheck) * n + 255) & ~(size_t)255;
    const size_t bytes = kCounterBytes + order_bytes + checks_bytes + grid * zstd::kBlockCeiling;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    e = hipStreamIsCapturing(stream, &capture);
    if (e != hipSuccess) {
        return e;
    }
    hipMemPool_t pool = capture == hipStreamCaptureStatusNone ? zstd_pool(dev) : nullptr;
    void* mem = nullptr;
    e = pool != nullptr ? hipMallocFromPoolAsync(&mem, bytes, pool, stream)
                        : hipMallocAsync(&mem, bytes, stream);
    if (e != hipSuccess) {
        return e;
    }
    uint8_t* base = static_cast<uint8_t*>(mem);
    auto* counter = reinterpret_cast<unsigned long long*>(base);
    void* order_work = base + kCounterBytes;
    auto* checks = reinterpret_cast<FrameCheck*>(base + kCounterBytes + order_bytes);
    uint8_t* lits = base + kCounterBytes + order_bytes + checks_bytes;
    const uint32_t* order = nullptr;
    if (n > grid) {
        hipLaunchKernelGGL(zstd_reset, dim3(1), dim3(kWave), 0, stream, counter,
                           (unsigned long long)grid);
        e = hipGetLastError();
    } else {
        counter = nullptr;
    }
    if (e == hipSuccess) {
        e = cost_order(sizes, caps, n, order_work, stream, &order);
    }
    if (e == hipSuccess) {
        hipLaunchKernelGGL(zstd_batch, dim3((unsigned)grid), dim3(kFrameBlock), 0, stream, srcs, sizes,
                           dsts, caps, n, results, counter, order, checks, lits);
        e = hipGetLastError();
    }
    if (e == hipSuccess) {
        constexpr size_t kPerBlock = kVerifyBlock / xxh::kGroup;
        size_t vgrid = (n + kPerBlock - 1) / kPerBlock;
        vgrid = vgrid > 8192 ? 8192 : vgrid;
        hipLaunchKernelGGL(zstd_verify, dim3((unsigned)vgrid), dim3(kVerifyBlock), 0, stream, dsts,
                           n, checks, results);
        e = hipGetLastError();
    }
    const hipError_t f = hipFreeAsync(mem, stream);
    return e != hipSuccess ? e : f;
}

}  // namespace cudec_amd
