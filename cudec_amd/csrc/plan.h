/* Decode plans: how the chunks of each cost bin are decoded. Internal, host
 * code but for the cost's key. */
#ifndef CUDEC_AMD_PLAN_H
#define CUDEC_AMD_PLAN_H

#include <stddef.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define CUDEC_HD __host__ __device__
#else
#define CUDEC_HD
#endif

namespace cudec_amd {

constexpr uint32_t kOctaveBits = 2; /* cost bins per octave: 4 */
constexpr int kBins = 64 << kOctaveBits;

/* Default plans (LZ4, Snappy): chunks costing at least this (capacity +
 * capacity - compressed) are pipelined. */
constexpr uint64_t kDefaultPipeMinCost[2] = {128u << 10, 64u << 10};
/* ... and in launches of few chunks: below this one wave is as fast (a 4 KiB
 * token page alone: 36 us on one wave, 40 pipelined). */
constexpr uint64_t kFewPipeMinCost = 8u << 10;

/* Order-preserving key of a cost below 2^63: the octave and the next
 * kOctaveBits bits below its leading one (costs below 2^kOctaveBits are
 * their own key). */
CUDEC_HD inline uint32_t cost_key(uint64_t cost) {
    if (cost < (1u << kOctaveBits)) {
        return (uint32_t)cost;
    }
    const uint32_t lg = 63u - (uint32_t)__builtin_clzll(cost);
    return lg << kOctaveBits |
           (uint32_t)((cost >> (lg - kOctaveBits)) & ((1u << kOctaveBits) - 1));
}

/* A decode plan: bit b (of word b / 64) set when cost bin b decodes on
 * a pipelined block, clear for one wave. Passed to the kernels by value. */
struct Plan {
    uint64_t pipes[kBins / 64];
};

CUDEC_HD inline bool plan_pipes(const Plan& p, uint32_t bin) {
    return ((p.pipes[bin >> 6] >> (bin & 63)) & 1u) != 0;
}

/* The plan that pipelines chunks costing at least min_cost: every
 * bin up to the bin of a chunk whose cost is exactly min_cost (costlier
 * bins have smaller numbers). 0 takes every bin, UINT64_MAX none. */
inline Plan plan_from_threshold(uint64_t min_cost) {
    Plan p = {};
    const int32_t last = min_cost == 0 ? kBins - 1
                         : min_cost == UINT64_MAX ? -1
                                                  : (int32_t)(kBins - 1 - cost_key(min_cost));
    for (int32_t b = 0; b <= last; b++) {
        p.pipes[b >> 6] |= 1ull << (b & 63);
    }
    return p;
}

/* A format's plan on one device. */
struct DecodePlan {
    Plan plan;
    uint64_t min_cost; /* the threshold last set */
    bool chosen;       /* the caller (or a tuner for it) has set a plan */

    static DecodePlan usual(int format) {
        return {plan_from_threshold(kDefaultPipeMinCost[format]), kDefaultPipeMinCost[format],
                false};
    }
    void set_threshold(uint64_t cost) {
        plan = plan_from_threshold(cost);
        min_cost = cost;
        chosen = true;
    }
    void set_bins(const uint16_t* lanes) {
        plan = {};
        for (int b = 0; b < kBins; b++) {
            if (lanes[b] == 128) {
                plan.pipes[b >> 6] |= 1ull << (b & 63);
            }
        }
        chosen = true;
    }
    /* What a launch of n chunks follows. A launch of few chunks leaves most
     * of the chip idle whatever it does, and takes as long as its largest
     * chunk: unless a plan was chosen, all its chunks from kFewPipeMinCost on
     * are pipelined (16 token chunks of 4 KiB to 1 MiB: 1.45 ms, against 2.38
     * with the threshold alone), up to two chunks a resident block. A chosen
     * plan is followed as it is, also one that equals the default. */
    Plan of_launch(size_t n, size_t blocks) const {
        return !chosen && n <= 2 * blocks ? plan_from_threshold(kFewPipeMinCost) : plan;
    }
};

/* Waves of a block of piped_batch and of alone_batch (tuned.hip). */
constexpr uint32_t kPipeWaves = 4;
constexpr uint32_t kAloneWaves = 2;

/* Blocks that a device holds at once, on all its CUs together. */
struct Resident {
    size_t piped; /* of piped_batch */
    size_t wide;  /* of its build for wide windows; 0: the format has none */
    size_t alone; /* of alone_batch */
};

/* Chunks per wave from which the queue hands out its order through
 * sub-queues (tuned.hip). */
constexpr uint64_t kSubQueueMinPerWave = 16;

/* How one launch runs: its plan, whether any chunk may be pipelined, its
 * grid, and whether every chunk has a resident block (or wave) of its own,
 * so that it needs no queue and no scratch. */
struct Launch {
    Plan plan;
    bool pipes;
    bool direct;
    bool wide;         /* direct and pipelined: in kSegmentWide's windows */
    bool many;         /* through sub-queues */
    size_t grid;
    size_t alone_grid; /* of the one-wave kernel that follows, or 0 */
};

/* The queue's three kernels and the scratch allocation cost about 25 us, so a
 * launch that has a resident block for each chunk takes them in their own
 * order. The one-wave kernel that follows has no more waves than there are
 * chunks: a wave that finds nothing costs the others a pop's time. Whether
 * the order goes through sub-queues is settled for both kernels by the first
 * one's waves, which are the fewer (65 536 chunks on 256 CUs): by its own
 * 5120 the second would leave 65 536 to 81 919 small chunks to one counter
 * (80 000 of 512 bytes: 1014 us, 346 so). */
inline Launch plan_launch(const DecodePlan& set, const Resident& at, size_t n) {
    Launch r;
    r.plan = set.of_launch(n, at.piped);
    bool all = true;
    r.pipes = false;
    for (int w = 0; w < kBins / 64; w++) {
        r.pipes = r.pipes || r.plan.pipes[w] != 0;
        all = all && r.plan.pipes[w] == ~0ull;
    }
    const size_t per = r.pipes ? 1 : kAloneWaves; /* chunks a block starts with */
    const size_t blocks = r.pipes ? at.piped : at.alone;
    const size_t wanted = (n + per - 1) / per;
    r.direct = wanted <= blocks;
    r.wide = r.pipes && r.direct && n <= at.wide;
    r.grid = r.direct ? wanted : blocks;
    r.many = (uint64_t)n >=
             kSubQueueMinPerWave * (r.pipes ? kPipeWaves : kAloneWaves) * (uint64_t)r.grid;
    const size_t pairs = (n + kAloneWaves - 1) / kAloneWaves;
    r.alone_grid = !r.pipes || all || r.direct ? 0 : pairs < at.alone ? pairs : at.alone;
    return r;
}

/* The current device's plan of a format, whole, for a tuner that puts it
 * back; false when there is no device (tuned.hip). */
bool read_plan(int format, DecodePlan* plan);
bool write_plan(int format, const DecodePlan& plan);

}  // namespace cudec_amd

#endif /* CUDEC_AMD_PLAN_H */
