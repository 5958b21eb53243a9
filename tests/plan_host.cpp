/* cudec_amd/csrc/plan.h built for the CPU: TEST INFRASTRUCTURE ONLY. */
#include "plan.h"

#include <cstring>

extern "C" {

/* The plan (kBins / 64 words) that a launch of n chunks follows on a device
 * of `blocks` resident blocks; how: 0 nothing set, 1 a threshold, 2 the bins
 * that this threshold gives. */
void host_plan(int format, int how, uint64_t threshold, uint64_t n, uint64_t blocks,
               uint64_t* words, uint64_t* min_cost) {
    using namespace cudec_amd;
    DecodePlan d = DecodePlan::usual(format);
    if (how == 1) {
        d.set_threshold(threshold);
    } else if (how == 2) {
        const Plan p = plan_from_threshold(threshold);
        uint16_t lanes[kBins];
        for (int b = 0; b < kBins; b++) {
            lanes[b] = plan_pipes(p, (uint32_t)b) ? 128 : 64;
        }
        d.set_bins(lanes);
    }
    const Plan p = d.of_launch(n, blocks);
    std::memcpy(words, p.pipes, sizeof(p.pipes));
    *min_cost = d.min_cost;
}

/* How a launch of n chunks runs under the default plan (threshold 1) or one
 * by threshold, on a device of these resident blocks. */
void host_launch(int format, uint64_t threshold, uint64_t n, uint64_t piped, uint64_t wide,
                 uint64_t alone, uint64_t* grids, int* flags) {
    using namespace cudec_amd;
    DecodePlan d = DecodePlan::usual(format);
    if (threshold != 1) {
        d.set_threshold(threshold);
    }
    const Launch r = plan_launch(d, Resident{piped, wide, alone}, n);
    grids[0] = r.grid;
    grids[1] = r.alone_grid;
    flags[0] = r.pipes;
    flags[1] = r.direct;
    flags[2] = r.wide;
    flags[3] = r.many;
}

}  // extern "C"
