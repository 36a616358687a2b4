// hy_rules.hpp -- which kernel a batch takes, where that depends on sizes alone: plain host
// functions, each with the measurements that put its line where it is.
#pragma once
#include <stdint.h>

#include "hy_moe.h"

namespace hy {

// largest batch the one-launch decode routing takes; the decode GEMV takes at least
// these in AUTO mode
constexpr uint32_t GEMV_MAX_TOKENS = 16;

// AUTO mode, expert products of quantized weights: the decode GEMV (true) or the stream over
// the weights on the int8 matrix cores (hy_mfma_few.hip).
//
// Few pairs per expert belong to the GEMV, many to the stream: 3 and 5 (Q4_0), 2 and 2.5
// (Q8_0).  Between these the GEMV reads a layer once per four pairs of every expert, the
// stream once per 32, but a stream wave walks a whole reduction alone: with fewer waves than
// the chip has SIMDs (1024) a launch takes that walk's latency, whatever the batch, and the
// GEMV keeps batches whose passes over the layer stay below a + b / waves.  Widths without
// the GEMV's ring (blocks of a row not a multiple of 8) count double.  a and b are a fit of
// both kernels' times over 34 layers and T = 17..96, at most 8 % off the faster one, as us of
// GEMV / stream (H x I, E, K):
//   Q4_0 4096 x 3072, 64, 8: T = 28 324 / 298, 40 438 / 332; 8, 1: 28 93 / 94, 40 119 / 95
//        2048 x 1536, 8, 1: 28 51 / 62, 40 57 / 61; 32, 4: 28 76 / 68, 40 79 / 75
//        1024 x 768, 16, 2: 28 38 / 46, 40 42 / 45; 1024 x 1408, 16, 2: 28 62 / 52
//   Q8_0 4096 x 3072, 64, 8: T = 17 437 / 403; 8, 1: 17 90 / 110; 2048 x 1536, 16, 2: 17 57 / 62;
//        1024 x 768, 32, 4: 17 39 / 45; 1024 x 1408, 32, 4: 17 69 / 55
inline bool gemv_batch(int wt, uint32_t T, int K, int E, int H, int I, int has_shared) {
    if (T <= GEMV_MAX_TOKENS) return true;
    if (wt != HY_TYPE_Q4_0 && wt != HY_TYPE_Q8_0) return false;
    const bool q4 = wt == HY_TYPE_Q4_0;
    const uint64_t pairs2 = 2 * (uint64_t)T * (uint64_t)K, e = (uint64_t)E;
    if (pairs2 <= (q4 ? 6 : 4) * e) return true;
    if (pairs2 > (q4 ? 10 : 5) * e) return false;
    const int64_t mats = E + has_shared, waves = mats * (2 * I / 64);
    if (waves >= 1024) return false;
    // four pairs a pass, a routed expert's last one 3/8 empty on average
    const double passes = T * (double)K / 4 + 0.375 * E + (has_shared ? T / 4.0 : 0.0);
    const bool ring = H % 256 == 0 && I % 256 == 0;
    return passes / mats * (ring ? 1 : 2) <= (q4 ? 0.95 + 750.0 / waves : 0.65 + 700.0 / waves);
}

}  // namespace hy
