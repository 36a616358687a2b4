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

// The grouped GEMM's batches that the stream of hy_mfma_few.hip takes (cached: its
// gate/up weights fit the Infinity Cache).
//
// It wins while most experts fit one of its 32-pair tiles, as a second tile streams the weights
// again.  H 4096, I 3072, E 64, K 8, stream against the tall shape: T = 208 (26 pairs per
// expert) Q4_0 381 / 483 us, Q8_0 533 / 578; T = 240 444 / 494 and 640 / 592.  (Q4_0 alone would
// cross past 30 pairs; one line serves both.)  Where the weights are cached a second tile finds
// them there: up to 64 pairs, past which the tall shape too has a second tile.  Q8_0 between 32
// and 60 pairs, where evenly routed experts fill two of the stream's tiles and one of the tall
// shape's, gains only while the stream's waves leave the chip idle (3 per SIMD are resident,
// the line is at nine tenths): E 16, K 4, 2048 x 1536 T = 200 (1880 waves) 93 / 110, E 8, K 1,
// 4096 x 3072 T = 400 (2690) 175 / 188; with more E 32, K 4, 2048 x 1536 T = 300 (2980)
// 155 / 136, T = 448 158 / 137, but T = 496 165 / 164; E 64, K 8, 1024 x 768 T = 400 (3460)
// 105 / 92, T = 496 109 / 110.  (Skewed routing gains from the stream at these sizes too,
// 145 / 169 and 90 / 95 at T = 400; the rule goes by even routing.)  Q4_0, with half the bytes,
// gains throughout: E 32, K 4, 2048 x 1536 T = 400 127 / 134, E 64, K 8, 1024 x 768 90 / 95.
inline bool few_batch(int wt, int64_t T, int K, int E, int I, int has_shared, bool cached) {
    const int64_t pairs = T * K;
    if (pairs <= 26 * (int64_t)E) return true;
    if (!cached || pairs > 64 * (int64_t)E) return false;
    if (wt == HY_TYPE_Q4_0 || pairs <= 32 * (int64_t)E || pairs > 60 * (int64_t)E) return true;
    const int64_t tiles = pairs / 32 + E / 2 + (has_shared ? T / 32 : 0);  // half an expert's last tile empty
    return tiles * (2 * I / 64) <= 1024 * 3 * 9 / 10;
}

// RMSNorm rows read by four waves each, whole rows in registers (rms_norm_w_reg_kernel),
// against one wave per row: ahead while the rows are long or few.  us, four waves / one:
// H 4096 T = 1 6 / 11, 1000 7 / 25, 8192 40 / 59; H 1536 T = 4096 10 / 13; H 1024 T = 2000 6.4 / 6.4,
// 4096 8.1 / 7.7; H 256 T = 2000 6.2 / 6.3, 8192 10.9 / 6.2.
constexpr int RMSW_MAX_CHUNKS = 16;  // of 256 floats
inline bool norm_in_registers(int T, int H) {
    return H % 256 == 0 && H <= 256 * RMSW_MAX_CHUNKS && (H > 1024 || T <= 2048);
}

// The stand-alone fp32 product (hy_lm_head_f32): sizes of 64 to 1023 tiles of 128 x 128, which
// cut tiles between work groups and are refused under stream capture; and those of them that
// use the shared scratch -- not the decode-sized ones, a stream over W without pieces.
constexpr int GEMM_GEMV_ROWS = 16;
inline bool gemm_mid_size(int M, int N, int K) {
    const int64_t tiles = (int64_t)((M + 127) / 128) * ((N + 127) / 128);
    return K % 32 == 0 && tiles >= 64 && tiles < 1024 && tiles * (K / 32) >= 2048;
}
inline bool gemm_takes_scratch(int M, int N, int K) { return M > GEMM_GEMV_ROWS && gemm_mid_size(M, N, K); }

}  // namespace hy
