/*
 * Sizes and rules of the work splits that are host arithmetic alone, without
 * GPU calls or types.
 */
#ifndef GGDMC_WORK_SPLIT_H
#define GGDMC_WORK_SPLIT_H

#include <algorithm>
#include <cstdint>

namespace ggdmc {

constexpr int kBlock = 256;        /* threads per workgroup of the sweep kernels */
constexpr int kWaves = kBlock / 64;
constexpr int kChunk = 128;        /* trials per canonical chunk sum */

/* In a launch of every chain group (or of several iterations) a workgroup
 * polls flags of its subject and gives up kSpinLimit polls, about 0.4 s, after
 * the polled flag last advanced. A flag advances once an iteration, so what
 * has to stay far below that is one iteration of the longest subject: its G
 * groups in a row, k chains each, or a ring of ring_chains steps. A chunk of a
 * chain takes a wave about 4 us with 2 accumulators when every SIMD has 4
 * waves, three times that in FP64. */
constexpr double kMaxIterationUs = 5e4;
inline double iteration_us(int64_t ntrial, int n_acc, bool fp64, int G, int k, int ring_chains) {
    const double chunk_us = 2.0 * n_acc * (fp64 ? 3.0 : 1.0);
    const double rounds = (double)((ntrial + kChunk * kWaves - 1) / (kChunk * kWaves));
    return rounds * chunk_us * (double)std::max((int64_t)G * k, (int64_t)ring_chains);
}
inline bool waits_fit(int64_t ntrial, int n_acc, bool fp64, int G, int k, int ring_chains) {
    return iteration_us(ntrial, n_acc, fp64, G, k, ring_chains) < kMaxIterationUs;
}

} // namespace ggdmc

#endif
