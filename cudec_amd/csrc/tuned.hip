/* The tuned launch form of the LZ4 and Snappy batch decoders for gfx950.
 *
 * Work distribution: three small kernels bin the chunks by decode cost
 * (capacity + (capacity - compressed size), the output plus what matches
 * add to it; four bins per octave) into a device queue. A per-device,
 * per-format decode plan names, for each cost bin, how one of its chunks is
 * decoded: pipelined on a block of four waves (named 128 in the plan) or on
 * one wave (64). The queue holds the pipelined chunks first, then the
 * one-wave ones, each class costliest first. A persistent grid of four-wave
 * blocks pulls chunks from it; once the queue reaches the one-wave class,
 * a block splits into four independent one-wave decoders. A batch without a
 * pipelined chunk goes to a kernel of one-wave decoders alone, and a launch
 * with a resident block for every chunk takes them without the queue.
 *
 * Per chunk, the stream is decoded in windows of source bytes staged in LDS:
 *   1. stage     -- compressed bytes from the window start are loaded as
 *                   aligned 16-byte blocks (a block holding any byte of the
 *                   chunk never leaves the chunk's pages);
 *   2. find      -- where the window's sequences (LZ4) or elements (Snappy),
 *                   its members, start. A pipelined block walks 64 segments
 *                   of the window at once, a lane each ("pipelined blocks"
 *                   below; where their chains do not meet, as a lone wave
 *                   does). A lone wave parses eight candidate positions a
 *                   lane as if a member started there, and follows the true
 *                   chain through their links by pointer doubling: its
 *                   windows hold 512 bytes, and the segment walk there is
 *                   1 to 3% faster on chunks of 64 KiB and 20% slower on
 *                   chunks of 1 to 4 KiB (0.76 against 0.92 ms for 100 003);
 *   3. resolve   -- of 64 members, a lane each: a wavefront prefix sum places
 *                   each member's output and
 *                   the exact validation ladder (src/lz4_block.h:95-258,
 *                   src/snappy_block.h:288-435) runs per lane; the first
 *                   member in stream order that rejects, ends the stream,
 *                   or would overflow the group ends the group, so a chunk's
 *                   status is the sequential ladder's;
 *   4. execute   -- output goes through an LDS ring (execute.h): literals by
 *                   member lanes; matches whose sources are final by member
 *                   lanes (batched 16-byte history loads); the rest in stream
 *                   order with the wave fanned out over the bytes, or, many
 *                   short ones, 64 output bytes at a time;
 *   5. flush     -- completed ring bytes leave as aligned 16-byte stores;
 *                   only a chunk's first and last partial blocks use byte
 *                   stores, so exactly bytes_written bytes are stored.
 * Steps 1-3 read only the source and decide every status; steps 4-5 only
 * write. In a pipelined block one wave runs 1-2 and three take turns at 3-5.
 * A member the window cannot hold (a long run of extension bytes, a Snappy
 * literal over 256 bytes) is decided by the exact scalar ladder and copied
 * wave-wide, global to global.
 */
#include <mutex>

#include "common.h"
#include "cudec_mi355x.h"
#include "execute.h"
#include "ladder.h"
#include "plan.h"

namespace cudec_amd {
namespace {

/* Candidates per lane of the one-wave form: a window spans kCandSplit * 64
 * candidate positions. */
constexpr uint32_t kCandSplit = 8;
/* staged bytes of a window of `window` positions: the window plus
 * the longest candidate that starts in it (an LZ4 sequence with one
 * extension byte per length reads 275 bytes, a Snappy literal window 277),
 * in whole 16-byte blocks. (A 512-byte margin staged 1.5 KiB a window; this
 * one takes the one-wave form 2.8% faster.) */
constexpr uint32_t stage_bytes(uint32_t window) { return window + 304u; }
constexpr uint32_t kStageBuf = stage_bytes(kCandSplit * 64) + 16;
constexpr uint32_t kStop = 0xFFFFu;       /* link of an unresolvable candidate */
static_assert(kBins == kCostBins, "the plan API names every bin");
/* Queue keys: a chunk's class (pipelined first), then its cost bin. */
constexpr int kKeys = 2 * kBins;

static_assert(2 + 269 + 3 <= stage_bytes(0), "a window's last candidate fits the stage");

/* A one-wave decoder's LDS: its ring, the stage of its window and the
 * window's link table (walk_doubling). */
struct alignas(16) WaveLds : RingLds<kRing> {
    uint8_t stage[kStageBuf];
    uint16_t jump[kCandSplit * kWave];
    CoverLds cover;
};
/* A pipelined block's ring, the output bytes of one of its groups (64
 * members of token data give under 2 KiB), and the history before a group
 * that the group may read in the ring. */
constexpr uint32_t kPipeRing = 16384;
constexpr uint32_t kPipeBatch = 2560;
constexpr uint32_t kPipeHistory = kPipeRing - 3 * kPipeBatch - 64;

/* The decode queue hands out positions of the cost-sorted chunk order in
 * up to kSubQueues interleaved sub-queues (of k: sub-queue s holds
 * positions s, s + k, ...), each counter on its own 4 KiB page: the
 * counters' atomics are served in parallel, where one counter for the
 * whole grid serialises every chunk's pop (about 12 ns each, the pace of a
 * batch of many small chunks). A batch of few chunks per wave keeps one
 * queue: its exact costliest-first order matters more there. */
constexpr uint32_t kSubQueues = 8;
constexpr uint32_t kSubStride = 1024; /* uint32 words: 4 KiB apart */

/* A wave's place in the decode queue: the sub-queue it draws from and how
 * many sub-queues it has not yet found drained; of the one queue, the
 * positions before those it hands out, which waves started with. */
struct QueueCursor {
    uint32_t sub;
    uint32_t left;
};

/* Scratch of one tuned launch (stream-ordered allocation). */
struct Queue {
    uint32_t next[kSubQueues * kSubStride];
    uint32_t bin_count[kKeys];
    uint32_t bin_cursor[kKeys];
    uint32_t piped; /* chunks of the pipelined class */
};

/* Loads one dword per lane, `step` bytes apart, of what follows the `bytes`
 * staged at sp (every one inside the source), so that the next window's
 * stage finds those bytes in L2. The caller holds the value until the
 * window is parsed, which keeps the loads off its critical path. */
__device__ __forceinline__ uint32_t touch_ahead(gcu8* src, uint64_t src_size, uint64_t sp,
                                                uint32_t bytes, uint32_t step, uint32_t lane) {
    const uintptr_t base = (uintptr_t)(src + sp) & ~(uintptr_t)15;
    const uintptr_t g = base + 16u * (bytes / 16 + 1) + step * lane;
    const uintptr_t end = (uintptr_t)src + src_size;
    return g + 4 <= end ? *(gcu32*)g : 0u;
}

/* ------------------------------------------------------ candidate parse */

struct Cand {
    uint32_t tok;
    uint32_t lit_len;
    uint32_t lit;    /* stage-relative position of the literals */
    uint32_t offset;
    uint32_t match_len;
    uint32_t next;   /* position after the sequence */
    bool complex;    /* a length needs two or more extension bytes */
};

/* The sequence a token at window position c would encode, assuming at most
 * one extension byte per length. Reads stay below c + 275, inside the
 * stage. (Windows that also held matches with two extension bytes, up to
 * 529 bytes, decoded runs of long short-offset matches 20% faster but token
 * data 2.4% slower: the wider parse cost the kernel registers it spilled.) */
__device__ __forceinline__ Cand parse_candidate(const uint8_t* cw, uint32_t c) {
    /* branch-free: the token and the byte after it, then the three bytes
     * at the offset (offset, match extension); bytes past the sequence are
     * read but never used */
    Cand k;
    k.tok = cw[c];
    const uint32_t e1 = cw[c + 1];
    const uint32_t lh = k.tok >> 4;
    const bool x1 = lh == 15;
    k.lit_len = lh + (x1 ? e1 : 0);
    k.lit = c + 1 + (x1 ? 1 : 0);
    const uint32_t p = k.lit + k.lit_len;
    k.offset = (uint32_t)cw[p] | ((uint32_t)cw[p + 1] << 8);
    const uint32_t e2 = cw[p + 2];
    const uint32_t mh = k.tok & 15;
    const bool x2 = mh == 15;
    k.match_len = mh + 4 + (x2 ? e2 : 0);
    k.next = p + 2 + (x2 ? 1 : 0);
    k.complex = (x1 && e1 == 255) || (x2 && e2 == 255);
    return k;
}

/* ------------------------------------------------- window parse */

/* The chain of links from `start` (members while in the window and under
 * 64; a position with a stop link is no member), by pointer doubling over the window's links in LDS (jump, kC * 64 entries)
 * instead of one dependent step per member. Round r (r = 0..5) has the
 * table map a position to the one 2^r links on: lanes [2^r, 2^(r+1)) take
 * their member from lane (lane - 2^r) with one lookup, then every entry
 * looks itself up to double the reach. A link at or past the window end
 * (kStop included) maps to itself. The rounds stop once the last member
 * found is past the window. `link` is clobbered. */
template <uint32_t kC>
__device__ __forceinline__ uint32_t walk_doubling(uint32_t (&link)[kC], uint32_t start,
                                                  uint16_t* jump, uint32_t& count_out,
                                                  uint32_t& member, uint32_t lane) {
    constexpr uint32_t kW = kC * kWave;
    static_assert(kStop >= kW && kStop <= 0xFFFFu, "a stop link is past every window");
#pragma unroll
    for (uint32_t k = 0; k < kC; k++) {
        jump[k * kWave + lane] = (uint16_t)link[k];
    }
    wave_order();
    uint32_t m = start; /* lane i: member i's position once found */
    uint32_t h = 1;
    for (;;) {
        const uint32_t from = (uint32_t)__shfl((int)m, (int)((lane - h) & (kWave - 1)));
        if (lane >= h && lane < 2 * h) {
            m = from < kW ? jump[from] : from;
        }
        const uint32_t last = uniform32(__builtin_amdgcn_readlane(m, 2 * h - 1));
        if (last >= kW || h == kWave / 2) {
            break;
        }
#pragma unroll
        for (uint32_t k = 0; k < kC; k++) {
            link[k] = link[k] < kW ? jump[link[k]] : link[k];
        }
        wave_order();
#pragma unroll
        for (uint32_t k = 0; k < kC; k++) {
            jump[k * kWave + lane] = (uint16_t)link[k];
        }
        wave_order();
        h *= 2;
    }
    const uint64_t found = 2 * h >= kWave ? ~0ull : (1ull << (2 * h)) - 1;
    const uint64_t past = __ballot(m >= kW) & found;
    uint32_t count, pos;
    if (past != 0) {
        const uint32_t s = (uint32_t)__builtin_ctzll(past);
        pos = __builtin_amdgcn_readlane(m, s);
        count = s;
        if (pos == kStop && s != 0) {
            count = s - 1;
            pos = __builtin_amdgcn_readlane(m, s - 1);
        }
    } else {
        /* 64 members in the window: the table maps 32 links on */
        const uint32_t m64 = jump[uniform32(__builtin_amdgcn_readlane(m, kWave / 2))];
        count = kWave;
        pos = m64;
        if (m64 == kStop) {
            count = kWave - 1;
            pos = __builtin_amdgcn_readlane(m, kWave - 1);
        }
    }
    member = m;
    count_out = uniform32(count);
    return uniform32(pos);
}

/* What resolving up to 64 members of a window decided: status not OK (the
 * chunk fails); slow (the first member is one the window cannot hold); or
 * the group g, whose `g.take` members (and a terminal literal) run, with
 * done when the chunk ends after it. take < count: member take starts the
 * next group. */
struct Resolved {
    int status;
    bool slow;
    bool done;
    Group g;
};

/* The first flagged lane decides the group's end: `cut` (the group's output
 * is full there), `held` (a member the window cannot hold), a status, or the
 * chunk's end. */
struct GroupEnd {
    uint32_t take;
    int status;
    bool slow;
    bool ended;
};
__device__ __forceinline__ GroupEnd group_end(uint32_t count, bool cut, bool hold, int ev,
                                              bool ends) {
    GroupEnd e{count, kOk, false, false};
    const uint64_t flags = __ballot(cut || hold || ev != kOk || ends);
    if (flags != 0) {
        const uint32_t j = __builtin_ctzll(flags);
        e.take = j;
        const uint32_t what =
            uniform32(__builtin_amdgcn_readlane((uint32_t)ev << 2 | (hold ? 2u : 0u) |
                                                    (cut ? 1u : 0u), j));
        if ((what & 2) != 0) {
            e.slow = j == 0;
        } else if ((what >> 2) != 0) {
            e.status = (int)(what >> 2);
        } else if ((what & 1) != 0) {
            e.slow = j == 0;
        } else {
            e.ended = true;
        }
    }
    e.take = uniform32(e.take);
    e.slow = uniform32(e.slow) != 0;
    e.ended = uniform32(e.ended) != 0;
    e.status = (int)uniform32((uint32_t)e.status);
    return e;
}

/* Source bytes from the window start, clamped: no window reaches
 * kMaxWindow, so a position there stands for the source end. */
constexpr uint32_t kMaxWindow = 0x7FFF0000u;
__device__ __forceinline__ uint32_t window_limit(uint64_t src_size, uint64_t base) {
    const uint64_t left = src_size - base;
    return left >= kMaxWindow ? kMaxWindow : (uint32_t)left;
}

/* Extension bytes after the first that a length may have and still be
 * followed in a window: matches of up to 2058 bytes, which a group holds. */
constexpr uint32_t kWalkExtra = 7;
static_assert(4 + 15 + 255 * (kWalkExtra + 1) + 270 <= kPipeBatch, "a group holds any such member");

/* More than a sequence with one extension byte per length (275 bytes) and
 * the margins of every rung reach past its start, and than the margins of
 * the destination. */
constexpr uint32_t kLz4Inside = 320;

/* Resolves the members of an LZ4 window (lane j < count holds member j's
 * position, relative to the window start `base` whose bytes are at cw;
 * kLong: a match length may have up to kWalkExtra + 1 extension bytes): a
 * prefix sum places each member's output from dp on and the exact ladder
 * (src/lz4_block.h:95-258) runs per lane. A group's output stays within
 * `batch` bytes. A position at or past the source end is CORRUPT (nothing
 * at cw is used for it). */
template <bool kLong>
__device__ __forceinline__ Resolved resolve_lz4(const uint8_t* cw, uint32_t member,
                                                uint32_t count, uint64_t base,
                                                uint64_t src_size, uint64_t cap, uint64_t dp,
                                                uint32_t batch, uint32_t lane) {
    const bool is_member = lane < count;
    uint64_t s = base + member; /* absolute source position */
    const bool past = s >= src_size || member >= kMaxWindow;
    Cand c = parse_candidate(cw, is_member && !past ? member : 0);
    /* away from both ends of the chunk only the offset can be wrong */
    const uint32_t last_member = uniform32(__builtin_amdgcn_readlane(member, count - 1));
    const bool inside = last_member < kMaxWindow && src_size - base > last_member + kLz4Inside;
    if (kLong && inside && is_member && c.complex && c.lit_len < 15 + 255) {
        /* a match length of two to kWalkExtra + 1 extension bytes */
        uint32_t q = c.next;
        uint32_t e = 255;
        for (uint32_t i = 0; i < kWalkExtra && e == 255; i++) {
            e = cw[q++];
            c.match_len += e;
        }
        c.complex = e == 255;
    }
    const bool hold = is_member && !past && c.complex;
    const uint32_t out_len = is_member && !hold && !past ? c.lit_len + c.match_len : 0;
    const uint32_t incl = wave_inclusive_sum(out_len, lane);
    const uint32_t drel = incl - out_len;
    const uint64_t d0 = dp + drel; /* absolute destination */
    int ev = kOk;
    bool terminal = false;
    const bool long_match = c.match_len > 4 + 15 + 255 - 1;
    const uint32_t all = uniform32(__builtin_amdgcn_readlane(incl, kWave - 1));
    if (inside && cap - dp > all + kLz4Inside) {
        const uint32_t before = (dp < kMaxWindow ? (uint32_t)dp : kMaxWindow) + drel + c.lit_len;
        if (is_member && !hold && (c.offset == 0 || c.offset > before)) {
            ev = kCorrupt;
        }
    } else if (is_member && !hold && !long_match) {
        if (past) {
            ev = kCorrupt;
        } else {
            s++;
            if ((c.tok >> 4) == 15) {
                if (s + 15 >= src_size) {
                    ev = kCorrupt;
                } else if (15 > cap - d0) {
                    ev = kTooSmall;
                } else {
                    s++;
                    if (s + 15 > src_size) {
                        ev = kCorrupt;
                    }
                }
            }
            const uint64_t L = c.lit_len;
            if (ev == kOk) {
                if (L > src_size - s) {
                    ev = kCorrupt;
                } else if (L > cap - d0) {
                    ev = kTooSmall;
                } else if (cap - d0 - L < kLz4SlackDst || src_size - s - L < kLz4SlackSrc) {
                    if (s + L != src_size) {
                        ev = kCorrupt;
                    } else if (cap == 0 && c.tok != 0) {
                        ev = kCorrupt;
                    } else {
                        terminal = true;
                    }
                } else {
                    const uint64_t dl = d0 + L;
                    uint64_t M = (c.tok & 15) + 4;
                    s += L + 2;
                    if (c.offset == 0 || c.offset > dl) {
                        ev = kCorrupt;
                    } else {
                        if ((c.tok & 15) == 15) {
                            if (s >= src_size) {
                                ev = kCorrupt;
                            } else if (M > cap - dl) {
                                ev = kTooSmall;
                            } else {
                                s++;
                                M = c.match_len;
                                if (s + kLz4MatchMargin > src_size) {
                                    ev = kCorrupt;
                                }
                            }
                        }
                        if (ev == kOk) {
                            if (M > cap - dl) {
                                ev = kTooSmall;
                            } else if (M > cap - dl - kLz4LastLiterals) {
                                ev = kCorrupt;
                            }
                        }
                    }
                }
            }
        }
    }
    const uint32_t mine = terminal ? c.lit_len : out_len;
    /* a full group ends before anything its next member would decide */
    const bool cut = is_member && drel + mine > batch;
    const bool inner = inside && cap - dp > all + kLz4Inside;
    const GroupEnd e = group_end(count, cut, hold || (is_member && long_match && !inner),
                                 cut ? kOk : ev, terminal);
    Resolved r;
    r.status = e.status;
    r.slow = e.slow || count == 0;
    r.done = e.ended;
    r.g.lit = c.lit;
    r.g.lit_len = c.lit_len;
    r.g.match_len = c.match_len;
    r.g.offset = c.offset;
    r.g.drel = drel;
    r.g.take = e.take;
    r.g.terminal = e.ended;
    const uint32_t last = e.ended ? e.take : e.take - 1;
    r.g.end_rel = e.take == 0 && !e.ended
                      ? 0u
                      : uniform32(__builtin_amdgcn_readlane(incl, last) -
                                  (e.ended ? __builtin_amdgcn_readlane(c.match_len, last) : 0));
    return r;
}

/* What parsing one window decided. kGroup: execute `g` (staged at `delta`
 * in the stage buffer) and advance the source by `consumed`. kSlow: one
 * sequence the window cannot hold, by the scalar ladder (`q`, with the
 * cursor after it in sp/dp). kFail: the chunk ends with `status`. */
enum ParseKind : uint32_t { kParseGroup = 0, kParseSlow = 1, kParseFail = 2 };

struct Parsed {
    uint32_t kind;
    int status;
    bool done;        /* the chunk ends after this group / sequence */
    uint32_t delta;
    Group g;
    Lz4Step q;        /* kSlow: the sequence; kGroup with lead: runs first */
    bool lead;        /* kGroup: q precedes the group */
    uint64_t lead_dp; /* output position after q */
};

/* The group a window's chain resolved to, after a possible leading sequence
 * already in `out`; pos: the position after the chain's last member. False
 * when nothing of the window can run (its first member is slow). */
__device__ __forceinline__ bool take_group(const Resolved& r, uint32_t count, uint32_t member,
                                           uint32_t pos, uint64_t base, uint64_t src_size,
                                           uint64_t& sp, uint64_t& dp, Parsed& out) {
    if (r.status != kOk) {
        out.kind = kParseFail;
        out.status = r.status;
        return true;
    }
    if (r.slow || (r.g.take == 0 && !r.done)) {
        return false;
    }
    out.kind = kParseGroup;
    out.g = r.g;
    const uint64_t next_sp =
        r.done ? src_size
               : base + (r.g.take == count ? pos : __builtin_amdgcn_readlane(member, r.g.take));
    sp = uniform64(next_sp);
    dp = uniform64(dp + r.g.end_rel);
    out.done = r.done;
    return true;
}

/* The one-wave form's step: stages the window at sp into `stage`,
 * speculates, walks the chain by pointer doubling over `jump` and resolves
 * it, and advances sp and dp past what it decided. Reads the source only. */
__device__ __forceinline__ Parsed parse_window(uint8_t* stage, uint16_t* jump, gcu8* src,
                                               uint64_t src_size, uint64_t cap, uint64_t& sp,
                                               uint64_t& dp, uint32_t lane,
                                               uint32_t& touch) {
    constexpr uint32_t kC = kCandSplit;
    Parsed out;
    out.kind = kParseFail;
    out.status = kOk;
    out.done = false;
    out.lead = false;
    out.lead_dp = 0;
    const uint64_t base = sp; /* window start; member positions are relative to it */
    out.delta = stage_into<1>(stage, src, src_size, sp, stage_bytes(kC * kWave), lane);
    touch = touch_ahead(src, src_size, sp, stage_bytes(kC * kWave), 16, lane);
    const uint8_t* cw = stage + out.delta;
    /* the scalar ladder reads a sequence's header from the stage while it
     * lies there (an LDS round trip per byte instead of a global one) */
    const StagedBytes staged{src, cw, base, stage_bytes(kC * kWave) + 16 - out.delta};

    /* speculate: the link of each candidate position */
    uint32_t link[kC];
#pragma unroll
    for (uint32_t k = 0; k < kC; k++) {
        const Cand c = parse_candidate(cw, k * kWave + lane);
        link[k] = c.complex ? kStop : c.next;
    }

    /* a window that opens on a sequence it cannot hold: the exact scalar
     * ladder decides that one, and the chain goes on from just past it
     * (the speculated links stay valid) */
    uint32_t start = 0;
    if (uniform32(__builtin_amdgcn_readlane(link[0], 0)) == kStop) {
        Lz4Cursor cur{src, src_size, cap, sp, dp};
        bool last = false;
        const int st = (int)uniform32((uint32_t)lz4_next<true>(cur, out.q, last, staged));
        if (st != kOk) {
            out.status = st;
            return out;
        }
        sp = uniform64(cur.sp);
        dp = uniform64(cur.dp);
        out.lead = true;
        out.lead_dp = dp;
        const uint64_t adv = sp - base;
        if (uniform32(last) != 0 || adv >= kC * kWave) {
            out.kind = kParseSlow;
            out.lead = false;
            out.done = uniform32(last) != 0;
            return out;
        }
        start = (uint32_t)adv;
    }

    /* walk the true chain */
    uint32_t count = 0;
    uint32_t member = 0; /* lane j: position of member j */
    const uint32_t pos = walk_doubling<kC>(link, start, jump, count, member, lane);
    if (count != 0) {
        const Resolved r =
            resolve_lz4<false>(cw, member, count, base, src_size, cap, dp, kBatchMax, lane);
        if (take_group(r, count, member, pos, base, src_size, sp, dp, out)) {
            return out;
        }
    }
    if (out.lead) {
        /* nothing after the leading sequence fits this window */
        out.kind = kParseSlow;
        out.lead = false;
        return out;
    }
    /* one sequence by the exact scalar ladder */
    Lz4Cursor cur{src, src_size, cap, sp, dp};
    bool last = false;
    const int st = (int)uniform32((uint32_t)lz4_next<true>(cur, out.q, last, staged));
    if (st != kOk) {
        out.status = st;
        return out;
    }
    out.kind = kParseSlow;
    out.done = uniform32(last) != 0;
    sp = uniform64(cur.sp);
    dp = uniform64(cur.dp);
    return out;
}

/* ------------------------------------------------- Snappy window parse */

/* Longest literal a Snappy window resolves; longer ones take the scalar
 * ladder. A window literal therefore ends below kC * 64 + 5 + 256. */
constexpr uint32_t kSnappyWinLit = 256;
static_assert(5 + kSnappyWinLit + 16 <= stage_bytes(0) + 16, "stage covers a Snappy window");

/* The element a tag at window position c would encode
 * (src/snappy_block.h:288-435): a literal (lit, lit_len; match_len 0) or a
 * copy-1/2/4 (match_len, offset; lit_len 0). One 8-byte read at the tag. */
__device__ __forceinline__ Cand snappy_element(const uint8_t* cw, uint32_t c) {
    Cand k;
    uint64_t h;
    __builtin_memcpy(&h, cw + c, 8);
    const uint32_t tag = (uint32_t)h & 0xFF;
    k.tok = tag;
    k.complex = false;
    if ((tag & 3) == 0) {
        const uint32_t len6 = tag >> 2;
        uint32_t header = 1;
        uint64_t length = (uint64_t)len6 + 1;
        if (len6 > 59) {
            const uint32_t extra = len6 - 59;
            header += extra;
            const uint64_t bytes = h >> 8;
            length = (extra == 4 ? (bytes & 0xFFFFFFFFull) : (bytes & ((1ull << (8 * extra)) - 1))) + 1;
        }
        if (length > kSnappyWinLit) {
            k.complex = true;
            length = 0;
        }
        k.lit = c + header;
        k.lit_len = (uint32_t)length;
        k.match_len = 0;
        k.offset = 0;
        k.next = c + header + (uint32_t)length;
    } else {
        const uint32_t kind = tag & 3;
        const uint32_t ob = kind == 1 ? 1 : (kind == 2 ? 2 : 4);
        uint32_t offset = (uint32_t)(h >> 8);
        offset &= ob == 1 ? 0xFFu : (ob == 2 ? 0xFFFFu : 0xFFFFFFFFu);
        uint32_t length;
        if (kind == 1) {
            offset |= (tag >> 5) << 8;
            length = 4 + ((tag >> 2) & 7u);
        } else {
            length = (tag >> 2) + 1;
        }
        k.lit = c + 1 + ob;
        k.lit_len = 0;
        k.match_len = length;
        k.offset = offset;
        k.next = c + 1 + ob;
    }
    return k;
}

/* The member a tag at window position c would start: one element, or a
 * literal element fused with the copy element right after it (the pair an
 * LZ4 sequence carries as literals + match), so a window's 64 members hold
 * more of Snappy's short elements. A copy is fused only while its tag lies
 * before the source end (lim = source bytes from the window start). */
__device__ __forceinline__ Cand parse_candidate_snappy(const uint8_t* cw, uint32_t c,
                                                      uint32_t lim) {
    Cand k = snappy_element(cw, c);
    if (k.match_len == 0 && !k.complex && k.next < lim) {
        const Cand m = snappy_element(cw, k.next);
        if (m.match_len != 0) {
            k.match_len = m.match_len;
            k.offset = m.offset;
            k.next = m.next;
        }
    }
    return k;
}

/* More than a literal element with a copy element after it (271 bytes)
 * reaches past its start. */
constexpr uint32_t kSnappyInside = 320;

/* As resolve_lz4, for Snappy elements after the preamble: every member's
 * rungs run in parallel (every reject is CORRUPT_INPUT, so the first
 * failing member in stream order decides), and the member whose position
 * is exactly the end of the source ends the chunk when the output so far
 * equals the declared length. */
__device__ __forceinline__ Resolved resolve_snappy(const uint8_t* cw, uint32_t member,
                                                   uint32_t count, uint64_t base,
                                                   uint64_t src_size, uint64_t declared,
                                                   uint64_t dp, uint32_t lim, uint32_t batch,
                                                   uint32_t lane) {
    const bool is_member = lane < count;
    const uint64_t s = base + member;
    const bool at_end = is_member && (s >= src_size || member >= kMaxWindow);
    const Cand c = parse_candidate_snappy(cw, is_member && !at_end ? member : 0, lim);
    const bool hold = is_member && !at_end && c.complex;
    const uint32_t out_len = is_member && !at_end && !hold ? c.lit_len + c.match_len : 0;
    const uint32_t incl = wave_inclusive_sum(out_len, lane);
    const uint32_t drel = incl - out_len;
    const uint64_t d0 = dp + drel;
    int ev = kOk;
    /* away from both ends of the chunk only the offset can be wrong */
    const uint32_t last_member = uniform32(__builtin_amdgcn_readlane(member, count - 1));
    const uint32_t all = uniform32(__builtin_amdgcn_readlane(incl, kWave - 1));
    if (last_member < kMaxWindow && src_size - base > last_member + kSnappyInside &&
        declared >= dp && declared - dp > all) {
        const uint32_t before = (dp < kMaxWindow ? (uint32_t)dp : kMaxWindow) + drel + c.lit_len;
        if (is_member && !hold && c.match_len != 0 && (c.offset == 0 || c.offset - 1 >= before) &&
            (c.offset == 0 || (uint64_t)c.offset > d0 + c.lit_len)) {
            ev = kCorrupt;
        }
    } else if (is_member && !hold) {
        if (at_end) {
            ev = s == src_size && d0 == declared ? kOk : kCorrupt;
        } else if (d0 > declared) {
            ev = kCorrupt;
        } else if (c.lit_len != 0 || c.match_len == 0) {
            /* a literal element (src/snappy_block.h:345-370), then, in a
             * fused member, the copy element after it at (s2, d2) */
            const uint64_t header = c.lit - member;
            if (header > src_size - s) {
                ev = kCorrupt;
            } else if (c.lit_len > src_size - s - header) {
                ev = kCorrupt;
            } else if (c.lit_len > declared - d0) {
                ev = kCorrupt;
            } else if (c.match_len != 0) {
                const uint64_t s2 = s + header + c.lit_len;
                const uint64_t d2 = d0 + c.lit_len;
                const uint64_t header2 = c.next - (c.lit + c.lit_len);
                if (header2 > src_size - s2) {
                    ev = kCorrupt;
                } else if (c.offset == 0 || (uint64_t)c.offset > d2) {
                    ev = kCorrupt;
                } else if (c.match_len > declared - d2) {
                    ev = kCorrupt;
                }
            }
        } else {
            /* a copy element (src/snappy_block.h:371-435) */
            const uint64_t header = c.lit - member;
            if (header > src_size - s) {
                ev = kCorrupt;
            } else if (c.offset == 0 || (uint64_t)c.offset > d0) {
                ev = kCorrupt;
            } else if (c.match_len > declared - d0) {
                ev = kCorrupt;
            }
        }
    }
    const bool cut = is_member && !at_end && drel + out_len > batch;
    const GroupEnd e = group_end(count, cut, hold, ev, at_end);
    Resolved r;
    r.status = e.status;
    r.slow = e.slow || count == 0;
    r.done = e.ended;
    r.g.lit = c.lit;
    r.g.lit_len = c.lit_len;
    r.g.match_len = c.match_len;
    r.g.offset = c.offset;
    r.g.drel = drel;
    r.g.take = e.take;
    r.g.terminal = false;
    r.g.end_rel =
        e.take == 0 ? 0u : uniform32(__builtin_amdgcn_readlane(incl, e.take - 1));
    return r;
}

/* One Snappy element by the exact scalar ladder, as a sequence of its own. */
__device__ __forceinline__ int snappy_step(SnappyCursor& cur, Lz4Step& q, bool& last) {
    SnappyStep e;
    const int st = (int)uniform32((uint32_t)snappy_next(cur, e, last));
    if (st != kOk) {
        return st;
    }
    q.lit_src = e.is_copy ? 0 : e.from;
    q.lit_dst = e.to;
    q.lit_len = e.is_copy ? 0 : e.length;
    q.match_dst = e.to + (e.is_copy ? 0 : e.length);
    q.match_len = e.is_copy ? e.length : 0;
    q.offset = e.is_copy ? (uint32_t)e.offset : 1u;
    return st;
}

/* As parse_window, for Snappy. */
__device__ __forceinline__ Parsed parse_window_snappy(uint8_t* stage, uint16_t* jump, gcu8* src,
                                                      uint64_t src_size, uint64_t cap,
                                                      uint64_t declared, uint64_t& sp,
                                                      uint64_t& dp, uint32_t lane,
                                                      uint32_t& touch) {
    constexpr uint32_t kC = kCandSplit;
    Parsed out;
    out.kind = kParseFail;
    out.status = kOk;
    out.done = false;
    out.lead = false;
    out.lead_dp = 0;
    const uint64_t base = sp;
    out.delta = stage_into<1>(stage, src, src_size, sp, stage_bytes(kC * kWave), lane);
    touch = touch_ahead(src, src_size, sp, stage_bytes(kC * kWave), 16, lane);
    const uint8_t* cw = stage + out.delta;
    /* a fused copy must start before the source end */
    const uint32_t lim = window_limit(src_size, base);

    uint32_t link[kC];
#pragma unroll
    for (uint32_t k = 0; k < kC; k++) {
        const Cand c = parse_candidate_snappy(cw, k * kWave + lane, lim);
        link[k] = c.complex ? kStop : c.next;
    }
    /* a window that opens on a literal it cannot hold: the scalar ladder
     * decides it and the chain goes on from just past it */
    uint32_t start = 0;
    if (uniform32(__builtin_amdgcn_readlane(link[0], 0)) == kStop) {
        SnappyCursor cur{src, src_size, cap, sp, dp, declared};
        bool last = false;
        const int st = snappy_step(cur, out.q, last);
        if (st != kOk) {
            out.status = st;
            return out;
        }
        sp = uniform64(cur.sp);
        dp = uniform64(cur.dp);
        out.lead = true;
        out.lead_dp = dp;
        const uint64_t adv = sp - base;
        if (uniform32(last) != 0 || adv >= kC * kWave) {
            out.kind = kParseSlow;
            out.lead = false;
            out.done = uniform32(last) != 0;
            return out;
        }
        start = (uint32_t)adv;
    }
    uint32_t count = 0;
    uint32_t member = 0;
    const uint32_t pos = walk_doubling<kC>(link, start, jump, count, member, lane);
    if (count != 0) {
        const Resolved r = resolve_snappy(cw, member, count, base, src_size, declared, dp, lim,
                                          kBatchMax, lane);
        if (take_group(r, count, member, pos, base, src_size, sp, dp, out)) {
            return out;
        }
    }
    if (out.lead) {
        out.kind = kParseSlow;
        out.lead = false;
        return out;
    }
    /* one element by the exact scalar ladder */
    SnappyCursor cur{src, src_size, cap, sp, dp, declared};
    bool last = false;
    const int st = snappy_step(cur, out.q, last);
    if (st != kOk) {
        out.status = st;
        return out;
    }
    out.kind = kParseSlow;
    out.done = uniform32(last) != 0;
    sp = uniform64(cur.sp);
    dp = uniform64(cur.dp);
    return out;
}

/* A window of either format. */
template <int kFormat>
__device__ __forceinline__ Parsed parse_any(uint8_t* stage, uint16_t* jump, gcu8* src,
                                            uint64_t src_size,
                                            uint64_t cap, uint64_t declared, uint64_t& sp,
                                            uint64_t& dp, uint32_t lane,
                                            uint32_t& touch) {
    if (kFormat == kFormatSnappy) {
        return parse_window_snappy(stage, jump, src, src_size, cap, declared, sp, dp, lane,
                                   touch);
    }
    return parse_window(stage, jump, src, src_size, cap, sp, dp, lane, touch);
}

/* Start of a chunk: the Snappy preamble and its declared length against the
 * capacity (src/snappy_block.h:190-263); nothing for LZ4. */
template <int kFormat>
__device__ __forceinline__ int chunk_begin(gcu8* src, uint64_t src_size, uint64_t cap,
                                           uint64_t& sp, uint64_t& declared) {
    sp = 0;
    declared = 0;
    if (kFormat != kFormatSnappy) {
        return kOk;
    }
    SnappyCursor c{src, src_size, cap, 0, 0, 0};
    const int st = (int)uniform32((uint32_t)snappy_begin(c));
    sp = uniform64(c.sp);
    declared = uniform64(c.declared);
    return st;
}

/* ------------------------------------------------- pipelined blocks */

/* A pipelined block decodes one chunk with four waves. Wave 0, the parser,
 * finds where the sequences (LZ4) or elements (Snappy) start, a window of
 * the source at a time, and lists their positions; it decides nothing else.
 * Waves 1 to 3, the copiers, take the listed members 64 at a time, in turn:
 * a group is claimed (resolve_*, which decides every status), then executed
 * while the next copier claims the next one.
 *
 * The parser's walk. A window is 64 segments, one a lane. Every lane first
 * follows the chain from the first byte of its segment as if a member
 * started there, counting members up to where it leaves the segment. Lane
 * i's true entry is where lane i - 1 leaves, so each round hands the exits
 * up one lane and a lane whose entry changed walks again. A wrong start
 * meets the true chain after a few members (18 on 1 MiB LZ4 token chunks, 5
 * to 7 on Snappy's and on 64 KiB ones), so the exits are mostly right at
 * once and few rounds follow. A chain off the true one sometimes takes a
 * byte for a long length and leaves far ahead; a lane takes an entry past
 * its own segment only from a lane that is known to be right, so that such
 * an exit does not cost the lanes behind it their chains. The wave takes 5
 * steps for 64 members of 64 KiB LZ4 token chunks and of Snappy's, 13 on
 * 1 MiB LZ4 token chunks. Speculating on every byte position and then
 * following the links one by one, which this replaced, took 320 vector
 * instructions and 64 dependent scalar steps for the same 64 members.
 *
 * Groups at once. A copier works on group k while groups k - 1 and k - 2
 * are still running. What it needs of them it gets through `done`, the
 * count of groups whose bytes are in the ring, and `done_dp`, the output
 * position they reach; the turn goes on strictly in order. Literals, and
 * matches whose source is final or lies in the group, run before the group's
 * turn; the others wait for it. A group flushes its bytes to memory when its
 * turn has gone on, beside the followers (data whose groups wait for each
 * other, 1 MiB of sorted 64-bit numbers in Snappy: 7.9 ms when the turn went
 * on after the flush, 7.1 so). Three groups of at most kPipeBatch bytes may
 * lie in the ring beside the history that a group reads there (kPipeHistory
 * bytes before its start): a follower can overwrite nothing that a running
 * group reads. Everything older than that history belongs to the fourth group
 * before or an earlier one, whose copier had flushed it when it claimed the
 * group before. Only a member outside the ring's rules waits until the groups
 * before are in memory (`landed`). */
constexpr uint32_t kCopiers = kPipeWaves - 1;
constexpr int kPipeBlock = kPipeWaves * kWave;
static_assert(kPipeHistory >= kCopiers * kPipeBatch + 16,
              "what a group reads from memory lies before the third group before it");
static_assert(kPipeBatch < kStripAt && kPipeHistory + kPipeBatch < kStripOffset,
              "run_strips packs a member into a word");
static_assert(kPipeHistory + kCopiers * kPipeBatch + 64 <= kPipeRing &&
                  (kCopiers - 1) * kPipeBatch <= kPipeHistory,
              "running groups and their history share the ring");
static_assert(kPipeBatch <= 64 * kWave, "CoverLds marks a batch");

/* Bytes of a lane's segment: the window is 64 of them. A window takes as
 * many steps as the longest wrong chain in it (about 85 members of LZ4 token
 * data), whatever its size, so a wider one is parsed faster by the byte: one
 * 1 MiB chunk in 2.32 ms with segments of 64, 1.44 with 128, 1.30 with 192
 * and 1.28 with 320 (the copiers bound it then). LDS sets the line: four
 * blocks a CU at 128, three at 192, and a full chip needs the fourth (the
 * uneven LZ4 batch: 17.5 ms, 20.1 with 192 and 21.7 with 64 and three waves
 * on five blocks). So LZ4 launches that have a block of three a CU for every
 * chunk take 192 (16 chunks of 4 KiB to 1 MiB: 1.46 -> 1.34 ms; 700 of 256
 * KiB: 0.57 -> 0.52), all others 128. Snappy's chains meet sooner and gain
 * nothing (700 of 256 KiB: 0.79 ms, 0.82 with 192). A chunk's first window,
 * and one after a window cut short, is a small one, so that its members
 * reach the copiers early. */
constexpr uint32_t kSegment = 128;
constexpr uint32_t kSegmentWide = 192;
constexpr uint32_t kSegmentFirst = 32;
constexpr uint32_t stage_rounds(uint32_t bytes) { return (bytes / 16 + 1 + kWave - 1) / kWave; }
constexpr uint32_t kStageRoundsUsual = stage_rounds(stage_bytes(kSegment * kWave));
constexpr uint32_t kStageRoundsFirst = stage_rounds(stage_bytes(kSegmentFirst * kWave));
static_assert(stage_rounds(stage_bytes(kCandSplit * kWave)) == 1, "one-wave stage");
/* Members listed of one window; a window that holds more ends there. */
constexpr uint32_t list_max(uint32_t segment) { return 10 * segment; }
constexpr uint32_t kListEnd = 0xFFFFu; /* a listed position at the source end */

struct PipeWindow {
    uint64_t base;   /* source position of the window */
    uint32_t count;  /* listed members */
    uint32_t delta;  /* where the window starts in its stage */
    uint32_t staged; /* staged bytes from the window start */
};

/* The claims' state: where the next group starts. */
struct PipeClaim {
    uint64_t dp;      /* output position */
    uint64_t flushed; /* everything below is in memory (groups flush what follows) */
    uint64_t ring_lo; /* the ring holds nothing below */
    uint32_t win;     /* window, kNoWindow before the first */
    uint32_t idx;     /* next member of it */
};
constexpr uint32_t kNoWindow = 0xFFFFFFFFu;

template <uint32_t kSeg>
struct alignas(16) PipeLds {
    static constexpr uint32_t kSegment = kSeg;
    union {
        struct {
            RingLds<kPipeRing> w;
            alignas(16) uint8_t stage[2][stage_bytes(kSeg * kWave) + 16];
            uint16_t list[2][list_max(kSeg) + 2];
            CoverLds cover[kCopiers];
        } pipe;                       /* pipelined */
        WaveLds split[kPipeWaves];    /* one chunk a wave, once the block splits */
    };
    PipeWindow window[2];
    PipeClaim next;
    uint64_t declared;    /* Snappy's preamble */
    int32_t begun;        /* its verdict */
    uint32_t chunk_idx;
    uint32_t published;   /* windows listed */
    uint32_t retired;     /* windows whose members are all claimed */
    uint32_t retired_k[2];/* the groups claimed by then */
    uint32_t claim;       /* the group to be claimed next, or kClaimsOver */
    uint32_t done;        /* groups whose bytes are in the ring */
    uint32_t done_dp;     /* output position they reach (low 32 bits) */
    uint32_t landed[kCopiers]; /* per copier: its last group in memory, and one */
    uint32_t broken;      /* a wait ran out, and no wave waits any more */
};
static_assert(sizeof(PipeLds<kSegment>) <= 40960, "four blocks share a CU's 160 KiB");
static_assert(sizeof(PipeLds<kSegmentWide>) <= 54608, "three blocks");

/* A copier's group among the groups at once (execute_group's Order). */
template <class L>
struct InTurn {
    static constexpr bool kInTurn = true;
    static constexpr bool kStrips = true;
    static constexpr uint32_t kHistory = kPipeHistory;
    L& l;
    uint32_t k;
    /* everything below is final, in the ring or in memory: done_dp is at most
     * two groups behind */
    __device__ uint64_t final_below(uint64_t d0) const {
        const uint32_t reached = uniform32(*(const lds_flag*)&l.done_dp);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        return d0 - (uint32_t)((uint32_t)d0 - reached);
    }
    __device__ bool wait_turn() const {
        return await_flag((const lds_flag*)&l.done, k, nullptr, (lds_flag*)&l.broken) == kReached;
    }
    /* the turn goes on: the group's bytes up to dp are in the ring */
    __device__ void pass(uint64_t dp) const {
        raise_flag((lds_flag*)&l.done_dp, (uint32_t)dp);
        *(lds_flag*)&l.done = k + 1;
    }
    /* the group's bytes are in memory, and it reads the ring no more */
    __device__ void finish() const { raise_flag((lds_flag*)&l.landed[k % kCopiers], k + 1); }
    /* until the groups before have got that far */
    __device__ bool wait_landed() const {
        bool ok = true;
        for (uint32_t i = 1; i < kCopiers; i++) {
            ok = ok && (k < i || await_flag((const lds_flag*)&l.landed[(k - i) % kCopiers],
                                            k - i + 1, nullptr, (lds_flag*)&l.broken) == kReached);
        }
        return ok;
    }
};

/* The position after the member at window position p, or kWalkStop | p
 * where it cannot be told from the window: an LZ4 length of more than
 * kWalkExtra + 1 extension bytes or one that runs past the stage (`limit`
 * bytes from the window start), a Snappy literal past the window's
 * longest. Positions past the source end (lim) are not walked from. */
constexpr uint32_t kWalkStop = 0x80000000u;
__device__ __forceinline__ uint32_t walk_long_lz4(const uint8_t* cw, uint32_t p, uint32_t limit) {
    const uint32_t tok = cw[p];
    uint32_t q = p + 1;
    uint32_t lit = tok >> 4;
    bool stop = false;
    if (lit == 15) {
        uint32_t e = 255;
        for (uint32_t i = 0; i <= kWalkExtra && e == 255 && q < limit; i++) {
            e = cw[q++];
            lit += e;
        }
        stop = e == 255;
    }
    q += lit + 2;
    if ((tok & 15) == 15) {
        uint32_t e = 255;
        for (uint32_t i = 0; i <= kWalkExtra && e == 255 && q < limit; i++) {
            e = cw[q++];
        }
        stop = stop || e == 255;
    }
    return stop ? kWalkStop | p : q;
}
__device__ __forceinline__ uint32_t walk_step_lz4(const uint8_t* cw, uint32_t p, uint32_t limit) {
    /* lengths of at most one extension byte without a branch, in two LDS
     * round trips; bytes that are none are read but never used */
    const uint32_t tok = cw[p];
    const uint32_t e1 = cw[p + 1];
    const bool x1 = tok >= 0xF0;
    const uint32_t q = p + 3 + (x1 ? 16 + e1 : tok >> 4);
    const uint32_t e2 = cw[q];
    const bool x2 = (tok & 15) == 15;
    uint32_t next = q + (x2 ? 1 : 0);
    if ((x1 && e1 == 255) || (x2 && e2 == 255)) {
        next = walk_long_lz4(cw, p, limit);
    }
    return next;
}
template <int kFormat>
__device__ __forceinline__ uint32_t walk_step(const uint8_t* cw, uint32_t p, uint32_t limit,
                                              uint32_t lim) {
    if (kFormat == kFormatSnappy) {
        const Cand c = parse_candidate_snappy(cw, p, lim);
        return c.complex ? kWalkStop | p : c.next;
    }
    return walk_step_lz4(cw, p, limit);
}

/* Data whose chains do not meet. Lengths that repeat (columns of integers, a
 * period in Snappy's elements of 64 bytes) or two or three bytes a sequence
 * keep a wrong chain wrong for all of a window, and then every round moves
 * most lanes on by one segment: 64 rounds, 2700 steps a window and as many
 * LDS reads on every lane (1000 LZ4 chunks of 1 MiB of two symbols: 76.8 ms).
 * Chains that do meet take few rounds (1 window in 80 of 1 MiB LZ4 tokens
 * takes more than 8, 1 in 650 more than 10 and 1 in 6000 more than 12; of text,
 * tables and sorted numbers 1 in 100 more than 5). So after kWalkRounds the rest
 * of the window is walked as the one-wave form walks (walk_dense), from every
 * byte position, and so are the next kDenseWindows. Those cost a chunk whose
 * chains do meet 0.3 ms, and a launch waits for its slowest chunk, so the line
 * lies where no such window comes: with 12 rounds 1500 token chunks of 4 KiB to
 * 1 MiB took 1.87 ms, and 1.76 with 16 and 20. (Smaller segments take more
 * rounds of fewer steps, and are left to it.) */
constexpr uint32_t kWalkRounds = 20;
constexpr uint32_t kDenseWindows = 15;
/* walk_dense's link table lies behind the positions it lists. */
constexpr uint32_t kDenseTable = kCandSplit * kWave;
constexpr uint32_t dense_max(uint32_t most) { return most - kDenseTable; }
/* Marks of a link there: out of the walk's range, or a member whose end the
 * window cannot tell. */
constexpr uint32_t kLinkOut = 0x4000u, kLinkStop = 0x8000u, kLinkAt = 0x3FFFu;
static_assert(kCandSplit * kWave + 4 + 15 + 255 * (kWalkExtra + 2) < kLinkAt, "links fit");

/* Lists the chain's members from window position `from` to `end`, 64 at a
 * time, behind the `count` listed so far, and returns as walk_window does.
 * Every position is a candidate, eight a lane, and pointer doubling follows
 * the chain through their links. */
template <int kFormat, uint32_t kMost>
__device__ __forceinline__ uint32_t walk_dense(const uint8_t* cw, uint32_t from, uint32_t end,
                                               uint32_t limit, uint32_t lim, uint16_t* list,
                                               uint32_t& count, uint32_t lane) {
    uint16_t* jump = list + dense_max(kMost);
    while (from < end && count + kWave <= dense_max(kMost)) {
        const uint32_t range = end - from;
        uint32_t link[kCandSplit];
#pragma unroll
        for (uint32_t k = 0; k < kCandSplit; k++) {
            const uint32_t c = k * kWave + lane;
            const uint32_t next = walk_step<kFormat>(cw, c < range ? from + c : from, limit, lim);
            const uint32_t to = (next & ~kWalkStop) - from;
            link[k] = (next & kWalkStop) != 0 ? kLinkStop | c
                      : to >= range           ? kLinkOut | to
                                              : to;
        }
        uint32_t found = 0, member = 0;
        const uint32_t next = walk_doubling<kCandSplit>(link, 0, jump, found, member, lane);
        if (lane < found) {
            list[count + lane] = (uint16_t)(from + member);
        }
        count += found;
        if ((next & kLinkStop) != 0) {
            return kWalkStop | (from + (next & kLinkAt));
        }
        from += next & kLinkAt;
    }
    return from;
}

/* Walks the window's chain (see above) from its first byte and lists its
 * members; returns where it goes on: a window position, or kWalkStop | the
 * last listed member, whose end the window cannot tell. `dense`: windows
 * still to be walked from every position. */
template <int kFormat, uint32_t kMost>
__device__ __forceinline__ uint32_t walk_window(const uint8_t* cw, uint32_t segment,
                                                uint32_t limit, uint32_t lim, uint16_t* list,
                                                uint32_t& count, uint32_t& dense, uint32_t lane) {
    const uint32_t start = lane * segment;
    const uint32_t end = start + segment < lim ? start + segment : lim;
    uint32_t entry = start;
    uint32_t exit, mine;
    bool moves = true;
    /* from where on the chain is walked from every position */
    uint32_t rest = dense != 0 ? 0u : kWalkStop;
    if (dense != 0) {
        dense--;
        entry = lim;
        exit = 0;
        mine = 0;
    }
    for (uint32_t round = 0; rest != 0; round++) {
        if (moves) {
            mine = 0;
            exit = entry;
            while (exit < end) {
                exit = walk_step<kFormat>(cw, exit, limit, lim);
                mine++;
            }
        }
        const uint32_t before =
            (uint32_t)__builtin_amdgcn_update_dpp(0, (int)exit, 0x138, 0xF, 0xF, false);
        uint32_t from = lane == 0 ? 0 : before;
        const uint64_t moved = __ballot(from != entry);
        if (moved == 0) {
            break;
        }
        /* up to the first lane that moves, entries and exits are final, and
         * so is where the chain goes from there */
        const uint32_t first = (uint32_t)__builtin_ctzll(moved);
        const uint32_t reached = uniform32(__builtin_amdgcn_readlane(from, first));
        if (reached >= lim || (round >= kWalkRounds && segment >= kSegment)) {
            /* the chain stops, or leaves the source, before that lane (or the
             * rest is for walk_dense) */
            rest = reached;
            dense = reached < lim ? kDenseWindows : 0;
            if (lane >= first) {
                entry = lim;
                exit = reached;
                mine = 0;
            }
            break;
        }
        const bool sure = lane >= first && reached >= start;
        from = sure ? reached : from;
        moves = from != entry && (sure || from < end);
        entry = moves ? from : entry;
    }
    const uint32_t incl = wave_inclusive_sum(mine, lane);
    const uint32_t total = uniform32(__builtin_amdgcn_readlane(incl, kWave - 1));
    uint32_t i = incl - mine;
    uint32_t p = entry;
    uint32_t next = 0; /* the member after a full list, on its lane */
    while (p < end) {
        if (i < kMost) {
            list[i] = (uint16_t)p;
        } else if (i == kMost) {
            next = p;
        }
        i++;
        p = walk_step<kFormat>(cw, p, limit, lim);
    }
    if (total > kMost) {
        count = kMost;
        const uint64_t holder = __ballot(incl - mine <= kMost && kMost < incl);
        return uniform32(__builtin_amdgcn_readlane(next, __builtin_ctzll(holder)));
    }
    count = total;
    if (rest < lim) {
        return walk_dense<kFormat, kMost>(cw, rest, segment * kWave < lim ? segment * kWave : lim,
                                          limit, lim, list, count, lane);
    }
    return uniform32(__builtin_amdgcn_readlane(exit, kWave - 1));
}

/* The parser's side of a chunk: window after window into the two window
 * slots, a slot again once the groups of its window have finished. */
template <int kFormat, class L>
__device__ __forceinline__ void run_parser(L& l, gcu8* src, uint64_t src_size, uint64_t cap,
                                           uint32_t lane) {
    constexpr uint32_t kSeg = L::kSegment;
    constexpr uint32_t kStageRounds = stage_rounds(stage_bytes(kSeg * kWave));
    uint64_t base = 0;
    if (kFormat == kFormatSnappy) {
        uint64_t declared = 0;
        const int begun = chunk_begin<kFormat>(src, src_size, cap, base, declared);
        l.declared = declared;
        l.begun = begun;
        if (begun != kOk) {
            raise_flag((lds_flag*)&l.published, 1);
            return;
        }
    }
    uint32_t segment = kSegmentFirst;
    uint32_t dense = 0;
    for (uint32_t w = 0;; w++) {
        const uint32_t b = w & 1;
        const lds_flag* over = (const lds_flag*)&l.claim;
        lds_flag* broken = (lds_flag*)&l.broken;
        if (w >= 2) {
            if (await_flag((const lds_flag*)&l.retired, w - 1, over, broken) != kReached) {
                return;
            }
            const uint32_t groups = uniform32(*(const lds_flag*)&l.retired_k[b]);
            if (await_flag((const lds_flag*)&l.done, groups, over, broken) != kReached) {
                return;
            }
        }
        uint8_t* stage = l.pipe.stage[b];
        uint16_t* list = l.pipe.list[b];
        const uint32_t lim = window_limit(src_size, base);
        /* what is left of a short source is spread over the lanes */
        const uint32_t spread = lim / kWave + 1;
        segment = spread < segment ? spread : segment;
        const uint32_t limit = stage_bytes(segment * kWave);
        const uint32_t delta =
            kSeg > kSegment && segment > kSegment
                ? stage_into<kStageRounds>(stage, src, src_size, base, limit, lane)
            : segment > kSegmentFirst
                ? stage_into<kStageRoundsUsual>(stage, src, src_size, base, limit, lane)
                : stage_into<kStageRoundsFirst>(stage, src, src_size, base, limit, lane);
        const uint32_t touch = touch_ahead(src, src_size, base, limit, kSeg, lane);
        const uint8_t* cw = stage + delta;
        uint32_t count = 0;
        const uint32_t next =
            walk_window<kFormat, list_max(kSeg)>(cw, segment, limit, lim, list, count, dense, lane);
        bool last = false;
        uint64_t next_base = base + next;
        /* a wide window only behind one that was not cut short: what it stages
         * past a cut is staged in vain */
        segment = segment < kSegment ? kSegment : kSeg;
        if ((next & kWalkStop) != 0) {
            /* only where the member ends matters here (the copiers decide
             * what it is worth): the exact ladder, with room for any output */
            const uint64_t at = base + (next & ~kWalkStop);
            const uint64_t room = 1ull << 62;
            bool ends = false;
            int st;
            Lz4Step q;
            if (kFormat == kFormatSnappy) {
                SnappyCursor cur{src, src_size, room, at, room / 2, room};
                st = snappy_step(cur, q, ends);
                next_base = uniform64(cur.sp);
            } else {
                Lz4Cursor cur{src, src_size, room, at, room / 2};
                const StagedBytes staged{src, cw, base, limit};
                st = (int)uniform32((uint32_t)lz4_next<true>(cur, q, ends, staged));
                next_base = uniform64(cur.sp);
            }
            last = st != kOk || uniform32(ends) != 0;
            segment = kSegmentFirst;
        } else if (next >= lim) {
            last = true;
        }
        if (last) {
            /* whatever comes after the last member lies at the source end */
            list[count] = (uint16_t)kListEnd;
            count++;
        }
        l.window[b].base = base;
        l.window[b].count = count;
        l.window[b].delta = delta;
        l.window[b].staged = limit;
        raise_flag((lds_flag*)&l.published, w + 1);
        asm volatile("" ::"v"(touch));
        if (last) {
            return;
        }
        base = next_base;
    }
}

/* A copier's side of a chunk: claims every kCopiers-th group, from group
 * `c` on, and executes it. The copier whose claim decides the chunk's end
 * returns true, with the status and the bytes produced. kParseOnly: claims
 * only. */
template <int kFormat, bool kParseOnly, class L>
__device__ __forceinline__ bool run_copier(L& l, uint32_t c, gcu8* src, uint64_t src_size, gu8* dst,
                                           uint64_t cap, int& status, uint64_t& produced,
                                           uint32_t lane) {
    lds_flag* broken = (lds_flag*)&l.broken;
    lds_flag* claim = (lds_flag*)&l.claim;
    for (uint32_t k = c;; k += kCopiers) {
        produced = 0;
        const Waited got = await_flag(claim, k, claim, broken);
        if (got == kOver) {
            return false;
        }
        if (got == kBroken) {
            status = CUDEC_ERR_CUDA;
            return true;
        }
        const InTurn<L> turn{l, k};
        uint64_t dp = uniform64(l.next.dp);
        uint64_t flushed = uniform64(l.next.flushed);
        uint64_t ring_lo = uniform64(l.next.ring_lo);
        uint32_t win = uniform32(l.next.win);
        uint32_t idx = uniform32(l.next.idx);
        if (win == kNoWindow || idx == uniform32(l.window[win & 1].count)) {
            if (win != kNoWindow) {
                l.retired_k[win & 1] = k;
                raise_flag((lds_flag*)&l.retired, win + 1);
            }
            win++;
            idx = 0;
            if (await_flag((const lds_flag*)&l.published, win + 1, nullptr, broken) != kReached) {
                status = CUDEC_ERR_CUDA;
                return true;
            }
            if (kFormat == kFormatSnappy && win == 0 &&
                uniform32((uint32_t)l.begun) != (uint32_t)kOk) {
                status = (int)uniform32((uint32_t)l.begun);
                raise_flag(claim, kClaimsOver);
                return true;
            }
        }
        const uint32_t b = win & 1;
        const uint64_t base = uniform64(l.window[b].base);
        const uint32_t listed = uniform32(l.window[b].count);
        const uint8_t* cw = l.pipe.stage[b] + uniform32(l.window[b].delta);
        const uint32_t lim = window_limit(src_size, base);
        const uint32_t left = listed - idx;
        const uint32_t count = left < kWave ? left : kWave;
        uint32_t member = lane < count ? (uint32_t)l.pipe.list[b][idx + lane] : 0;
        member = member == kListEnd ? lim : member;
        const uint64_t declared = kFormat == kFormatSnappy ? uniform64(l.declared) : 0;
        const Resolved r =
            kFormat == kFormatSnappy
                ? resolve_snappy(cw, member, count, base, src_size, declared, dp, lim, kPipeBatch,
                                 lane)
                : resolve_lz4<true>(cw, member, count, base, src_size, cap, dp, kPipeBatch, lane);
        if (r.status != kOk) {
            status = r.status;
            raise_flag(claim, kClaimsOver);
            return true;
        }
        if (!r.slow) {
            if (r.done) {
                raise_flag(claim, kClaimsOver);
            } else {
                l.next.dp = dp + r.g.end_rel;
                l.next.flushed = flushed;
                l.next.ring_lo = ring_lo;
                l.next.win = win;
                l.next.idx = idx + r.g.take;
                raise_flag(claim, k + 1);
            }
            bool ran;
            if (kParseOnly) {
                dp += r.g.end_rel;
                ran = turn.wait_turn();
                turn.pass(dp);
            } else {
                /* what precedes the group is flushed by then, up to the last
                 * whole 16 bytes */
                const uint64_t whole = (((uintptr_t)dst + dp) & ~(uintptr_t)15) - (uintptr_t)dst;
                if ((int64_t)whole > (int64_t)flushed) {
                    flushed = whole;
                }
                ran = execute_group(l.pipe.w, l.pipe.cover[c], cw, r.g, dst, cap, dp, flushed, ring_lo, r.done,
                                    lane, turn);
            }
            if (!ran) {
                status = CUDEC_ERR_CUDA;
                return true;
            }
            turn.finish();
            if (r.done) {
                status = kOk;
                produced = dp;
                return true;
            }
            continue;
        }
        /* a member the window cannot hold: the exact scalar ladder, then the
         * slow copies, alone in the block (they use the ring as they like) */
        Lz4Step q;
        bool last = false;
        int st;
        const uint64_t at = base + uniform32(__builtin_amdgcn_readlane(member, 0));
        uint64_t dp_after;
        if (kFormat == kFormatSnappy) {
            SnappyCursor cur{src, src_size, cap, at, dp, declared};
            st = snappy_step(cur, q, last);
            dp_after = uniform64(cur.dp);
        } else {
            Lz4Cursor cur{src, src_size, cap, at, dp};
            const StagedBytes staged{src, cw, base, uniform32(l.window[b].staged)};
            st = (int)uniform32((uint32_t)lz4_next<true>(cur, q, last, staged));
            dp_after = uniform64(cur.dp);
        }
        if (st != kOk) {
            status = st;
            raise_flag(claim, kClaimsOver);
            return true;
        }
        last = uniform32(last) != 0;
        if (!turn.wait_turn() || !turn.wait_landed()) {
            status = CUDEC_ERR_CUDA;
            return true;
        }
        if (kParseOnly) {
            dp = dp_after;
        } else {
            const uint64_t whole = (((uintptr_t)dst + dp) & ~(uintptr_t)15) - (uintptr_t)dst;
            if ((int64_t)whole > (int64_t)flushed) {
                flushed = whole;
            }
            execute_slow(l.pipe.w, src, dst, cap, q, dp_after, dp, flushed, ring_lo, last, lane);
        }
        turn.pass(dp);
        turn.finish();
        if (last) {
            raise_flag(claim, kClaimsOver);
            status = kOk;
            produced = dp;
            return true;
        }
        l.next.dp = dp;
        l.next.flushed = flushed;
        l.next.ring_lo = ring_lo;
        l.next.win = win;
        l.next.idx = idx + 1;
        raise_flag(claim, k + 1);
    }
}

/* ------------------------------------------------------------- one wave */

struct ChunkOut {
    int status;
    uint64_t produced;
};

/* One wave per chunk: parse a window, then execute it, in turn.
 * kParseOnly: parse only (statuses and sizes, no output bytes). */
template <int kFormat, bool kParseOnly>
__device__ __forceinline__ ChunkOut decode_chunk(WaveLds& w, gcu8* src,
                                                 uint64_t src_size, gu8* dst, uint64_t cap,
                                                 uint32_t lane) {
    uint64_t sp = 0, declared = 0, pdp = 0, dp = 0, flushed = 0, ring_lo = 0;
    uint64_t fuel = src_size == UINT64_MAX ? UINT64_MAX : src_size + 2;
    int status = chunk_begin<kFormat>(src, src_size, cap, sp, declared);
    while (status == kOk) {
        if (fuel-- == 0) {
            status = kCorrupt;
            break;
        }
        uint32_t touch = 0;
        const Parsed pr =
            parse_any<kFormat>(w.stage, w.jump, src, src_size, cap, declared, sp, pdp, lane, touch);
        if (pr.kind == kParseFail) {
            status = pr.status;
            break;
        }
        if (kParseOnly) {
            dp = pdp;
        } else if (pr.kind == kParseGroup) {
            if (pr.lead) {
                execute_slow(w, src, dst, cap, pr.q, pr.lead_dp, dp, flushed, ring_lo, false,
                             lane);
            }
            execute_group(w, w.cover, w.stage + pr.delta, pr.g, dst, cap, dp, flushed, ring_lo, pr.done,
                          lane, Alone{});
        } else {
            execute_slow(w, src, dst, cap, pr.q, pdp, dp, flushed, ring_lo, pr.done, lane);
        }
        /* the look-ahead loads land by now */
        asm volatile("" ::"v"(touch));
        if (pr.done) {
            break;
        }
    }
    ChunkOut r;
    r.status = status;
    r.produced = dp;
    return r;
}

/* ------------------------------------------------------------ kernels */

__global__ void queue_reset(Queue* q) {
    const uint32_t t = threadIdx.x;
    if (t < kKeys) {
        q->bin_count[t] = 0;
        q->bin_cursor[t] = 0;
    }
    if (t < kSubQueues) {
        q->next[t * kSubStride] = 0;
    }
}

/* Bin of a chunk by its decode cost, compressed size plus capacity: a
 * chunk's time follows the bytes it produces (a 4 MiB run of short-offset
 * matches compresses to a few hundred KiB yet decodes as long as 4 MiB of
 * literals and far matches). Four bins per octave; larger cost, smaller
 * bin, decoded first. */
__device__ __forceinline__ uint32_t cost_bin(uint64_t src_size, uint64_t cap) {
    const uint64_t lim = 1ull << 61;
    const uint64_t a = src_size < lim ? src_size : lim;
    const uint64_t b = cap < lim ? cap : lim;
    /* the output, plus what matches add to it (capacity - compressed):
     * match bytes cost the decode its time, literal bytes are a copy */
    const uint64_t cost = b + (b > a ? b - a : 0);
    return kBins - 1 - cost_key(cost);
}

/* Queue key of a chunk: its class under the plan, then its bin. */
__device__ __forceinline__ uint32_t queue_key(const Plan& plan, uint64_t src_size, uint64_t cap) {
    const uint32_t bin = cost_bin(src_size, cap);
    return plan_pipes(plan, bin) ? bin : kBins + bin;
}

/* Chunks per cost bin. A block counts its chunks in LDS and adds one
 * global atomic per bin it holds: a batch of like chunks (one bin) would
 * otherwise serialise one atomic per chunk on that bin's counter. */
__global__ void queue_count(const size_t* sizes, const size_t* caps, size_t n, Queue* q,
                            Plan plan) {
    __shared__ uint32_t local[kKeys];
    for (uint32_t t = threadIdx.x; t < kKeys; t += blockDim.x) {
        local[t] = 0;
    }
    __syncthreads();
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        atomicAdd(&local[queue_key(plan, sizes[i], caps[i])], 1u);
    }
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < kKeys; t += blockDim.x) {
        if (local[t] != 0) {
            atomicAdd(&q->bin_count[t], local[t]);
        }
    }
}

constexpr int kFillBlock = 256;
static_assert(kKeys == 2 * kFillBlock, "a thread of queue_fill adds up two keys");

/* Each chunk's place in the order: its bin's base, the block's range in
 * that bin (one global atomic per bin the block holds) and its rank in the
 * block (an LDS atomic). Every block adds the counts up for itself: a kernel
 * that did it once, on one thread, took 7 us and the gap to the next one. */
__global__ void __launch_bounds__(kFillBlock)
    queue_fill(const size_t* sizes, const size_t* caps, size_t n, Queue* q, uint32_t* order,
               Plan plan) {
    __shared__ uint32_t local[kKeys];
    __shared__ uint32_t range[kKeys];
    __shared__ uint32_t waves[kFillBlock / kWave];
    const uint32_t k = 2 * threadIdx.x;
    const uint32_t c0 = q->bin_count[k], c1 = q->bin_count[k + 1];
    const uint32_t incl = wave_inclusive_sum(c0 + c1, __lane_id());
    if (__lane_id() == kWave - 1) {
        waves[threadIdx.x / kWave] = incl;
    }
    local[k] = 0;
    local[k + 1] = 0;
    __syncthreads();
    uint32_t base = incl - c0 - c1; /* of key k */
    for (uint32_t w = 0; w < threadIdx.x / kWave; w++) {
        base += waves[w];
    }
    if (blockIdx.x == 0 && k == (uint32_t)kBins) {
        q->piped = base;
    }
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t b = 0, rank = 0;
    if (i < n) {
        b = queue_key(plan, sizes[i], caps[i]);
        rank = atomicAdd(&local[b], 1u);
    }
    __syncthreads();
    if (local[k] != 0) {
        range[k] = base + atomicAdd(&q->bin_cursor[k], local[k]);
    }
    if (local[k + 1] != 0) {
        range[k + 1] = base + c0 + atomicAdd(&q->bin_cursor[k + 1], local[k + 1]);
    }
    __syncthreads();
    if (i < n) {
        order[range[b] + rank] = (uint32_t)i;
    }
}

/* The next queue position for this wave from kSubs sub-queues (1: the
 * single counter; 0: no queue, the launch has a place for every chunk and
 * gives each wave or block its own, `own`), or at least n once every one is
 * drained (n < 2^32).
 * Every lane takes part in the atomic and only lane 0 adds: a
 * lane-0-only branch at a persistent loop's top and bottom lets the
 * compiler fold both into an exec-masked inner loop that only lane 0 can
 * leave. */
template <uint32_t kSubs>
__device__ __forceinline__ uint32_t queue_pop(Queue* q, size_t n, QueueCursor& c,
                                              uint32_t lane, uint64_t own) {
    if (kSubs == 0) {
        const bool first = c.left == 0;
        c.left = 1;
        return first && own < n ? (uint32_t)own : (uint32_t)n;
    }
    if (kSubs == 1) {
        return c.sub >= n ? (uint32_t)n
                          : uniform32(c.sub + atomicAdd(&q->next[0], lane == 0 ? 1u : 0u));
    }
    while (c.left != 0) {
        const uint32_t i =
            uniform32(atomicAdd(&q->next[c.sub * kSubStride], lane == 0 ? 1u : 0u));
        const uint64_t pos = (uint64_t)c.sub + (uint64_t)kSubs * i;
        if (pos < n) {
            return (uint32_t)pos;
        }
        c.sub = (c.sub + 1) % (kSubs == 0 ? 1 : kSubs);
        c.left--;
    }
    return (uint32_t)n;
}

/* The chunk at a queue position: the cost order's, or, with no queue, the
 * position itself. */
template <uint32_t kSubs>
__device__ __forceinline__ uint64_t chunk_at(const uint32_t* order, uint32_t idx) {
    return kSubs == 0 ? idx : order[idx];
}

/* One chunk a wave, from queue position idx on, until the queue is dry. */
template <int kFormat, uint32_t kSubs, bool kParseOnly>
__device__ __forceinline__ void decode_alone(WaveLds& w, uint32_t idx, const void* const* srcs,
                                             const size_t* src_sizes, void* const* dsts,
                                             const size_t* caps, size_t n,
                                             cudec_chunk_result* results, Queue* q,
                                             const uint32_t* order, QueueCursor& cursor,
                                             uint32_t lane) {
    while (idx < n) {
        const uint64_t chunk = chunk_at<kSubs>(order, idx);
        gcu8* src = global_bytes(srcs[chunk]);
        gu8* dst = global_bytes(dsts[chunk]);
        const uint64_t src_size = uniform64(src_sizes[chunk]);
        const uint64_t cap = uniform64(caps[chunk]);
        const ChunkOut o = decode_chunk<kFormat, kParseOnly>(w, src, src_size, dst, cap, lane);
        write_result(results, chunk, (int)uniform32((uint32_t)o.status), uniform64(o.produced));
        idx = queue_pop<kSubs>(q, n, cursor, lane, n);
    }
}


/* Whether a queued batch has no chunk that its plan pipelines: the queue
 * holds those first. */
__device__ __forceinline__ bool none_piped(const Queue* q) {
    return uniform32(q->piped) == 0;
}

/* The persistent decoder. A block takes the queue's pipelined chunks first,
 * all four waves on one chunk (above); a barrier opens every chunk, so that
 * no control word is reset while another wave may still read it. The queue
 * holds every pipelined chunk before the others, so once a block meets one
 * of the others it splits for good into four one-wave decoders.
 *
 * Four blocks fill a CU's LDS, sixteen waves at 128 VGPRs each (three with
 * kSegmentWide, twelve waves). kSubs:
 * decode sub-queues, kSubQueues for launches of many chunks per wave, 0 for
 * launches with a resident block for every chunk, else 1 (the single
 * counter, whose code keeps the fewest scalar registers live). */
template <int kFormat, uint32_t kSubs, bool kParseOnly, uint32_t kSeg = kSegment>
__global__ void __launch_bounds__(kPipeBlock)
    __attribute__((amdgpu_waves_per_eu(kSeg == kSegment ? 4 : 3)))
    piped_batch(const void* const* srcs, const size_t* src_sizes, void* const* dsts,
                const size_t* caps, size_t n, cudec_chunk_result* results, Queue* q,
                const uint32_t* order, Plan plan) {
    __shared__ PipeLds<kSeg> l;
    const uint32_t lane = __lane_id();
    const uint32_t wave = uniform32(threadIdx.x / kWave);
    /* Of the one queue, every block starts with its own position. Of a CU's
     * four blocks the first to come is the fastest (1.76 us a KiB of a 1 MiB
     * chunk, 2.05 on the third), and where blocks took the positions as they
     * reached the counter, an unrelated change to the code before it gave the
     * largest chunks to late ones (3000 chunks of 4 KiB to 1 MiB: 1.79 -> 2.14
     * ms; 1.80 so. The uneven LZ4 batch takes 1% longer than without it). */
    QueueCursor cursor{kSubs == 0   ? 0
                       : kSubs == 1 ? gridDim.x
                                    : blockIdx.x % (kSubs == 0 ? 1 : kSubs),
                       kSubs};
    uint32_t start = kSubs == 1 ? blockIdx.x : (uint32_t)n;
    uint32_t idx;
    if (kSubs != 0 && none_piped(q)) {
        return; /* alone_batch follows and takes them all */
    }
    if (wave == 0 && lane == 0) {
        l.broken = 0;
    }
    for (;;) {
        /* every wave is done with the previous chunk's control words */
        __syncthreads();
        if (wave == 0) {
            l.chunk_idx = start < n ? start : queue_pop<kSubs>(q, n, cursor, lane, blockIdx.x);
            start = (uint32_t)n;
            l.next.dp = 0;
            l.next.flushed = 0;
            l.next.ring_lo = 0;
            l.next.win = kNoWindow;
            l.next.idx = 0;
            l.published = 0;
            l.retired = 0;
            l.claim = 0;
            l.done = 0;
            l.done_dp = 0;
            for (uint32_t i = 0; i < kCopiers; i++) {
                l.landed[i] = 0;
            }
        }
        __syncthreads();
        idx = uniform32(l.chunk_idx);
        if (idx >= n) {
            return;
        }
        const uint64_t chunk = chunk_at<kSubs>(order, idx);
        gcu8* src = global_bytes(srcs[chunk]);
        gu8* dst = global_bytes(dsts[chunk]);
        const uint64_t src_size = uniform64(src_sizes[chunk]);
        const uint64_t cap = uniform64(caps[chunk]);
        if (!plan_pipes(plan, cost_bin(src_size, cap))) {
            break;
        }
        if (wave == 0) {
            run_parser<kFormat>(l, src, src_size, cap, lane);
        } else {
            int status = kOk;
            uint64_t produced = 0;
            if (run_copier<kFormat, kParseOnly>(l, wave - 1, src, src_size, dst, cap, status,
                                                produced, lane)) {
                write_result(results, chunk, (int)uniform32((uint32_t)status),
                             uniform64(produced));
            }
        }
    }
    /* no barrier follows; the first wave decodes the chunk in hand */
    if (wave != 0) {
        idx = queue_pop<kSubs>(q, n, cursor, lane, n);
    }
    decode_alone<kFormat, kSubs, kParseOnly>(l.split[wave], idx, srcs, src_sizes, dsts, caps, n,
                                             results, q, order, cursor, lane);
}

/* The persistent decoder of launches where every chunk runs on one wave:
 * those are bound by throughput and gain from a fifth wave per SIMD (96
 * VGPRs): 16 384 token chunks of 64 KiB in 2.69 ms against 3.05 by
 * piped_batch's split blocks, and 2.62 now. Only the queue build knows whether
 * a batch has chunks to pipeline, so it `follows` a piped_batch that leaves
 * batches without one untouched, and leaves the others to that: an empty launch
 * is about 2 us, and up to 8 with the gap before the next. (With that launch, a
 * kernel to add the queue's counts up and 5120 waves whatever the batch, 1500
 * chunks of 512 bytes took 113 us, 2500 of 64 KiB 816 and 20 000 of 512 bytes
 * 329; they take 46, 686 and 273. Before there were two kernels: 88, 856 and
 * 310.) */
constexpr int kAloneBlock = kAloneWaves * kWave;
template <int kFormat, uint32_t kSubs, bool kParseOnly>
__global__ void __launch_bounds__(kAloneBlock) __attribute__((amdgpu_waves_per_eu(5)))
    alone_batch(const void* const* srcs, const size_t* src_sizes, void* const* dsts,
                const size_t* caps, size_t n, cudec_chunk_result* results, Queue* q,
                const uint32_t* order, bool follows) {
    __shared__ WaveLds w[kAloneWaves];
    const uint32_t lane = __lane_id();
    QueueCursor cursor{kSubs == 0 ? 0 : blockIdx.x % (kSubs == 0 ? 1 : kSubs), kSubs};
    const uint32_t wave = uniform32(threadIdx.x / kWave);
    if (follows && !none_piped(q)) {
        return;
    }
    const uint64_t own = (uint64_t)blockIdx.x * kAloneWaves + wave;
    uint32_t idx;
    if (kSubs == 1) {
        /* of the one queue, every wave starts with a position of its own: up
         * to 5120 pops of about 12 ns each fewer at one counter, and none at
         * all where every chunk has a wave */
        idx = own < n ? (uint32_t)own : (uint32_t)n;
        cursor.sub = gridDim.x * kAloneWaves;
    } else {
        idx = queue_pop<kSubs>(q, n, cursor, lane, own);
    }
    decode_alone<kFormat, kSubs, kParseOnly>(w[wave], idx, srcs,
                                             src_sizes, dsts, caps, n, results, q, order, cursor,
                                             lane);
}

/* Launch geometry and a scratch pool, per device, set up on first use. The
 * pool keeps freed scratch (release threshold at its maximum) so that a
 * stream of launches does not return memory to the driver between them. */
struct DeviceState {
    int cus = 0;
    int pipe_blocks_per_cu[2] = {0, 0};  /* piped_batch, per format */
    int wide_blocks_per_cu = 0;          /* LZ4's piped_batch in kSegmentWide's windows */
    int alone_blocks_per_cu[2] = {0, 0}; /* alone_batch */
    DecodePlan plan[2];          /* per format (kFormatLz4, kFormatSnappy) */
    hipMemPool_t pool = nullptr; /* made on the first allocating launch */
    bool pool_tried = false;
    void* fixed = nullptr;       /* this device's address of fixed_scratch */
    hipError_t fixed_status = hipErrorNotReady;
    bool ready = false;
};
constexpr int kMaxDevices = 64;

/* Scratch of the allocation-free launch (launch_tuned_fixed): the queue and
 * the order of up to kFixedMaxChunks chunks (4.04 MiB), one copy per device
 * for the life of the process. Host code never passes this name to a
 * kernel or a copy: on the host it is a stand-in, and each device's
 * address of its own copy comes from hipGetSymbolAddress
 * (DeviceState::fixed). */
constexpr size_t kFixedMaxChunks = CUDEC_MI355X_NOALLOC_MAX_CHUNKS;
constexpr size_t kFixedBytes = sizeof(Queue) + sizeof(uint32_t) * kFixedMaxChunks;
static __device__ __align__(256) uint8_t scratch[kFixedBytes];

DeviceState g_devices[kMaxDevices];
std::mutex g_devices_lock;

hipError_t device_state(DeviceState** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        return e;
    }
    if (dev < 0 || dev >= kMaxDevices) {
        return hipErrorInvalidDevice;
    }
    std::lock_guard<std::mutex> hold(g_devices_lock);
    DeviceState& d = g_devices[dev];
    if (!d.ready) {
        e = hipDeviceGetAttribute(&d.cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) {
            return e;
        }
        const void* kernels[2][2] = {
            {reinterpret_cast<const void*>(&piped_batch<kFormatLz4, 1, false>),
             reinterpret_cast<const void*>(&alone_batch<kFormatLz4, 1, false>)},
            {reinterpret_cast<const void*>(&piped_batch<kFormatSnappy, 1, false>),
             reinterpret_cast<const void*>(&alone_batch<kFormatSnappy, 1, false>)}};
        for (int f = 0; f < 2; f++) {
            int per = 0;
            e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernels[f][0], kPipeBlock, 0);
            if (e != hipSuccess) {
                return e;
            }
            d.pipe_blocks_per_cu[f] = per > 0 ? per : 1;
            e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernels[f][1], kAloneBlock, 0);
            if (e != hipSuccess) {
                return e;
            }
            d.alone_blocks_per_cu[f] = per > 0 ? per : 1;
        }
        int wide = 0;
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &wide,
            reinterpret_cast<const void*>(&piped_batch<kFormatLz4, 0, false, kSegmentWide>),
            kPipeBlock, 0);
        if (e != hipSuccess) {
            return e;
        }
        d.wide_blocks_per_cu = wide > 0 ? wide : 1;
        for (int f = 0; f < 2; f++) {
            d.plan[f] = DecodePlan::usual(f);
        }
        /* this device is current: its own copy of the fixed scratch */
        d.fixed_status = hipGetSymbolAddress(&d.fixed, HIP_SYMBOL(scratch));
        if (d.fixed_status != hipSuccess) {
            d.fixed = nullptr;
            (void)hipGetLastError(); /* only the allocation-free entry needs it */
        }
        d.ready = true;
    }
    *out = &d;
    return hipSuccess;
}

/* The device's scratch pool, made on first use. It keeps freed scratch up
 * to kPoolKeep bytes, so that a stream of launches does not return memory
 * to the driver between them, while one very large batch's scratch is
 * given back once it is freed. */
constexpr uint64_t kPoolKeep = 64ull << 20;
hipMemPool_t scratch_pool(DeviceState& d, int dev) {
    std::lock_guard<std::mutex> hold(g_devices_lock);
    if (!d.pool_tried) {
        d.pool_tried = true;
        hipMemPoolProps props = {};
        props.allocType = hipMemAllocationTypePinned;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t pool = nullptr;
        if (hipMemPoolCreate(&pool, &props) == hipSuccess) {
            uint64_t keep = kPoolKeep;
            if (hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep) == hipSuccess) {
                d.pool = pool;
            } else {
                (void)hipMemPoolDestroy(pool);
            }
        }
        (void)hipGetLastError(); /* a pool that could not be made is not an error */
    }
    return d.pool;
}

}  // namespace

hipError_t set_pipe_min_cost(int format, uint64_t min_cost) {
    DeviceState* dev = nullptr;
    const hipError_t e = device_state(&dev);
    if (e != hipSuccess) {
        return e;
    }
    std::lock_guard<std::mutex> hold(g_devices_lock);
    dev->plan[format].set_threshold(min_cost);
    return hipSuccess;
}

hipError_t get_pipe_min_cost(int format, uint64_t* min_cost) {
    DeviceState* dev = nullptr;
    const hipError_t e = device_state(&dev);
    if (e != hipSuccess) {
        return e;
    }
    std::lock_guard<std::mutex> hold(g_devices_lock);
    *min_cost = dev->plan[format].min_cost;
    return hipSuccess;
}

hipError_t set_decode_plan(int format, const uint16_t* lanes) {
    DeviceState* dev = nullptr;
    const hipError_t e = device_state(&dev);
    if (e != hipSuccess) {
        return e;
    }
    std::lock_guard<std::mutex> hold(g_devices_lock);
    dev->plan[format].set_bins(lanes);
    return hipSuccess;
}

bool read_plan(int format, DecodePlan* plan) {
    DeviceState* dev = nullptr;
    if (device_state(&dev) != hipSuccess) {
        return false;
    }
    std::lock_guard<std::mutex> hold(g_devices_lock);
    *plan = dev->plan[format];
    return true;
}

bool write_plan(int format, const DecodePlan& plan) {
    DeviceState* dev = nullptr;
    if (device_state(&dev) != hipSuccess) {
        return false;
    }
    std::lock_guard<std::mutex> hold(g_devices_lock);
    dev->plan[format] = plan;
    return true;
}

hipError_t get_decode_plan(int format, uint16_t* lanes) {
    DeviceState* dev = nullptr;
    const hipError_t e = device_state(&dev);
    if (e != hipSuccess) {
        return e;
    }
    Plan p;
    {
        std::lock_guard<std::mutex> hold(g_devices_lock);
        p = dev->plan[format].plan;
    }
    for (int b = 0; b < kBins; b++) {
        lanes[b] = plan_pipes(p, (uint32_t)b) ? 128 : 64;
    }
    return hipSuccess;
}

uint32_t host_cost_bin(uint64_t src_size, uint64_t cap) {
    const uint64_t lim = 1ull << 61;
    const uint64_t a = src_size < lim ? src_size : lim;
    const uint64_t b = cap < lim ? cap : lim;
    const uint64_t cost = b + (b > a ? b - a : 0);
    return kBins - 1 - cost_key(cost);
}

namespace {

/* How a launch of n chunks runs now. */
Launch launch_of(const DeviceState& dev, int f, size_t n) {
    const size_t cus = (size_t)dev.cus;
    const Resident at{cus * (size_t)dev.pipe_blocks_per_cu[f],
                      f == 0 ? cus * (size_t)dev.wide_blocks_per_cu : 0,
                      cus * (size_t)dev.alone_blocks_per_cu[f]};
    std::lock_guard<std::mutex> hold(g_devices_lock);
    return plan_launch(dev.plan[f], at, n);
}

/* Launches the persistent decoder on `stream`; parse_only launches its
 * parse-only build. Unless the launch is direct, the batch is first binned
 * into the queue held by `work` (a Queue, then order[n]). */
hipError_t queue_and_decode(const Launch& launch, int format, const void* const* srcs,
                            const size_t* src_sizes, void* const* dsts, const size_t* caps,
                            size_t n, cudec_chunk_result* results, void* work,
                            hipStream_t stream, bool parse_only) {
    const Plan plan = launch.plan;
    Queue* q = static_cast<Queue*>(work);
    uint32_t* order = launch.direct ? nullptr : reinterpret_cast<uint32_t*>(q + 1);
    if (!launch.direct) {
        const unsigned tb = kFillBlock;
        const unsigned nb = (unsigned)((n + tb - 1) / tb);
        hipLaunchKernelGGL(queue_reset, dim3(1), dim3(kKeys), 0, stream, q);
        hipLaunchKernelGGL(queue_count, dim3(nb), dim3(tb), 0, stream, src_sizes, caps, n, q,
                           plan);
        hipLaunchKernelGGL(queue_fill, dim3(nb), dim3(tb), 0, stream, src_sizes, caps, n, q,
                           order, plan);
    }
    /* pipelined blocks, each of which splits into one-wave decoders when it
     * meets a one-wave chunk, unless the batch has no other; or, where it has
     * none or the plan pipelines no chunk, the one-wave kernel */
    const int f = format == kFormatSnappy ? 1 : 0;
    for (int pass = 0; pass < (launch.alone_grid != 0 ? 2 : 1); pass++) {
        const bool follows = pass != 0, pipes = launch.pipes && !follows;
        const int waves = (int)(pipes ? kPipeWaves : kAloneWaves);
        const size_t grid = follows ? launch.alone_grid : launch.grid;
        const dim3 gd((unsigned)grid), bd((unsigned)(waves * (int)kWave));
        const int subs = launch.wide ? 3 : launch.direct ? 2 : launch.many ? 1 : 0;
        const int shape = (parse_only ? 16 : 0) | (f ? 8 : 0) | (pipes ? 0 : 4) | subs;
        switch (shape) {
#define CUDEC_PIPED(kShape, kFmt, kS, kP)                                                 \
    case kShape:                                                                          \
        hipLaunchKernelGGL((piped_batch<kFmt, kS, kP>), gd, bd, 0, stream, srcs,          \
                           src_sizes, dsts, caps, n, results, q, order, plan);            \
        break;                                                                            \
    case kShape + 4:                                                                      \
        hipLaunchKernelGGL((alone_batch<kFmt, kS, kP>), gd, bd, 0, stream, srcs,          \
                           src_sizes, dsts, caps, n, results, q, order, follows);         \
        break;
#define CUDEC_WIDE(kShape, kP)                                                            \
    case kShape:                                                                          \
        hipLaunchKernelGGL((piped_batch<kFormatLz4, 0, kP, kSegmentWide>), gd, bd, 0,     \
                           stream, srcs, src_sizes, dsts, caps, n, results, q, order,     \
                           plan);                                                         \
        break;
            CUDEC_WIDE(3, false)
            CUDEC_WIDE(19, true)
#undef CUDEC_WIDE
            CUDEC_PIPED(0, kFormatLz4, 1, false)
            CUDEC_PIPED(1, kFormatLz4, kSubQueues, false)
            CUDEC_PIPED(2, kFormatLz4, 0, false)
            CUDEC_PIPED(8, kFormatSnappy, 1, false)
            CUDEC_PIPED(9, kFormatSnappy, kSubQueues, false)
            CUDEC_PIPED(10, kFormatSnappy, 0, false)
            CUDEC_PIPED(16, kFormatLz4, 1, true)
            CUDEC_PIPED(17, kFormatLz4, kSubQueues, true)
            CUDEC_PIPED(18, kFormatLz4, 0, true)
            CUDEC_PIPED(24, kFormatSnappy, 1, true)
            CUDEC_PIPED(25, kFormatSnappy, kSubQueues, true)
            CUDEC_PIPED(26, kFormatSnappy, 0, true)
#undef CUDEC_PIPED
            default:
                return hipErrorInvalidValue;
        }
    }
    return hipGetLastError();
}

}  // namespace

size_t cost_order_bytes(size_t n) {
    return sizeof(Queue) + sizeof(uint32_t) * n;
}

/* The order of a batch by decode cost, costliest first, for a decoder
 * outside this kernel family (the Zstandard frames, whose time also follows
 * the output plus what matches add): the same queue build with every chunk
 * in one class. `work` holds cost_order_bytes(n) bytes; *order points into
 * it (u32 chunk indices, n <= UINT32_MAX). */
hipError_t cost_order(const size_t* sizes, const size_t* caps, size_t n, void* work,
                      hipStream_t stream, const uint32_t** order) {
    if (n > UINT32_MAX) {
        return hipErrorInvalidValue;
    }
    const Plan plan{};
    Queue* q = static_cast<Queue*>(work);
    uint32_t* out = reinterpret_cast<uint32_t*>(q + 1);
    const unsigned tb = kFillBlock;
    const unsigned nb = (unsigned)((n + tb - 1) / tb);
    hipLaunchKernelGGL(queue_reset, dim3(1), dim3(kKeys), 0, stream, q);
    hipLaunchKernelGGL(queue_count, dim3(nb), dim3(tb), 0, stream, sizes, caps, n, q, plan);
    hipLaunchKernelGGL(queue_fill, dim3(nb), dim3(tb), 0, stream, sizes, caps, n, q, out, plan);
    *order = out;
    return hipGetLastError();
}

hipError_t launch_tuned(int format, const void* const* srcs, const size_t* src_sizes,
                        void* const* dsts, const size_t* caps, size_t n,
                        cudec_chunk_result* results, hipStream_t stream, bool parse_only) {
    if (n > UINT32_MAX) {
        /* the queue indexes chunks in 32 bits; larger batches take the
         * plain form, which has no such limit (and no parse-only build) */
        return parse_only ? hipErrorInvalidValue
                          : launch_plain(format, srcs, src_sizes, dsts, caps, n, results, stream);
    }
    DeviceState* dev = nullptr;
    hipError_t e = device_state(&dev);
    if (e != hipSuccess) {
        return e;
    }
    int id = 0;
    e = hipGetDevice(&id);
    if (e != hipSuccess) {
        return e;
    }
    const int f = format == kFormatSnappy ? kFormatSnappy : kFormatLz4;
    const Launch launch = launch_of(*dev, f, n);
    if (launch.direct) {
        return queue_and_decode(launch, format, srcs, src_sizes, dsts, caps, n, results, nullptr,
                                stream, parse_only);
    }
    hipMemPool_t pool = scratch_pool(*dev, id);
    const size_t bytes = sizeof(Queue) + sizeof(uint32_t) * n;
    /* under stream capture the scratch becomes a graph allocation node of
     * the device's default pool; eager launches use the keeping pool */
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    e = hipStreamIsCapturing(stream, &capture);
    if (e != hipSuccess) {
        return e;
    }
    void* mem = nullptr;
    e = pool != nullptr && capture == hipStreamCaptureStatusNone
            ? hipMallocFromPoolAsync(&mem, bytes, pool, stream)
            : hipMallocAsync(&mem, bytes, stream);
    if (e != hipSuccess) {
        return e;
    }
    e = queue_and_decode(launch, format, srcs, src_sizes, dsts, caps, n, results, mem, stream,
                         parse_only);
    const hipError_t freed = hipFreeAsync(mem, stream);
    return e != hipSuccess ? e : freed;
}

hipError_t launch_tuned_fixed(int format, const void* const* srcs, const size_t* src_sizes,
                              void* const* dsts, const size_t* caps, size_t n,
                              cudec_chunk_result* results, hipStream_t stream) {
    if (n > kFixedMaxChunks) {
        return hipErrorInvalidValue; /* the entry point refuses this first */
    }
    DeviceState* dev = nullptr;
    hipError_t e = device_state(&dev);
    if (e != hipSuccess) {
        return e;
    }
    if (dev->fixed == nullptr) {
        return dev->fixed_status != hipSuccess ? dev->fixed_status : hipErrorInvalidSymbol;
    }
    const int f = format == kFormatSnappy ? kFormatSnappy : kFormatLz4;
    return queue_and_decode(launch_of(*dev, f, n), format, srcs, src_sizes, dsts, caps, n,
                            results, dev->fixed, stream, false);
}

}  // namespace cudec_amd
