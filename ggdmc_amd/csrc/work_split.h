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

/* Items that span every chain group wait for items of their subject with higher
 * workgroup ids too. Those lie within min(8, subjects) x ranges consecutive
 * ids, behind phi_wgs population workgroups; launches of other threads'
 * sessions may hold every other slot while they wait for the same reason. As
 * many launches as a process has hardware queues (4) cannot stop each other
 * while each of them may hold a subject's items: then one of them has all of a
 * subject's. Mode 3, whose items wait for lower ids only, needs no such bound
 * (8 waves, 4 x 768: 23.2 us an iteration, mode 4 22.3). */
inline bool span_beside_others(int64_t phi_wgs, int64_t subjects, int64_t ranges, int64_t slots) {
    return 4 * (phi_wgs + std::min<int64_t>(8, subjects) * ranges) <= slots;
}

/* The split of a likelihood call of n vectors over nj chunks on `cus` CUs: k
 * vectors and jper chunks per workgroup of `threads`, its trials staged in LDS
 * or not. Per workgroup the constants take about 4 us whatever k, a chunk of
 * one vector about 3 us of one wave; about 3 workgroups of 4 waves are resident
 * on a CU. Times of whole calls, about 50 us of each outside the kernel:
 *   - few vectors and chunks (at most 8 chunks per CU): one workgroup of 8
 *     waves per vector and 8 chunks, one chunk a wave, so that the call is one
 *     set-up and one chunk long (1 x 768: 55.5 us, 4 waves in two rounds 60.6);
 *   - two vectors per CU or more: 4 waves and whole vectors, k of them together
 *     while a wave has less than 6 chunks and 3.5 workgroups per CU remain, for
 *     one set-up per k (8190 x 768: k = 1 176 us, 2 159, 4 153; 2000 x 768: 84,
 *     80, 82; 624 x 768: 65, 66, 69; 1000 x 2047 of 4 accumulators: 93, 99,
 *     114);
 *   - a long subject under few vectors: 4 waves and 16 chunks (4 a wave), fewer
 *     by fours, down to one a wave, while that leaves less than 3 workgroups per
 *     CU (33 x 100608 of 4 accumulators: 4 chunks 197 us, 8 to 24 181, 48 198,
 *     one workgroup per vector 804; 4 x 100608: 4 and 8 chunks 132, 16 138, 32
 *     150; 200 x 1634: 1 chunk 71, 4 60, 8 60, 12 63; 64 x 5090: 1 79, 4 61, 16
 *     63), spread evenly over a vector's workgroups (500 x 2146, 17 chunks: 16
 *     and 1 76 us, 12 and 5 70; 400 x 1250, 10 chunks: 8 and 2 65, 5 and 5 62).
 *     Below 7 chunks a second workgroup would be a set-up for 2 at most (400 x
 *     610: 4 and 1 61 us, together 59).
 * The first stages its trials in LDS with the set-up's loads; the others read
 * them from L2 as they go (staged: 1000 x 2047 93 us instead of 90). */
struct LoglikeShape {
    int k, threads, jper;
    bool stage;
};
inline LoglikeShape loglike_shape(int64_t n, int nj, int64_t cus, bool may_split) {
    LoglikeShape s{1, 256, nj, false};
    if (may_split && n * ((nj + 7) / 8) <= cus) {
        s.jper = std::min(nj, 8);
        s.threads = nj > 4 ? 512 : 256;
        s.stage = true;
    } else if (n >= 2 * cus || !may_split) {
        while (s.k < 4 && s.k * nj < 24 && n / (s.k + 1) >= 7 * cus / 2) ++s.k;
    } else if (nj >= 7) {
        s.jper = 16;
        while (s.jper > 4 && n * ((nj + s.jper - 1) / s.jper) < 3 * cus) s.jper -= 4;
        const int parts = (nj + s.jper - 1) / s.jper;
        s.jper = (nj + parts - 1) / parts;
    }
    return s;
}

} // namespace ggdmc

#endif
