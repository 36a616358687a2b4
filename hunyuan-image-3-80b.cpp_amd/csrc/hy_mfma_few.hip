// hy_mfma_few.hip -- grouped expert GEMMs on the int8 matrix cores while experts see few
// tokens: hy_mfma.hip's products, bit for bit, as a stream over the weights.
//
// Tiles of up to 32 pairs of one expert (or 32 tokens of the shared one).  A wave takes
// one 64-row group of the weights times the whole tile over all of K, by itself: weights,
// activations and scales go from memory straight into registers in MFMA operand order,
// FEW_D blocks ahead, with no LDS and no barrier, and Q4_0 nibbles become int8 in
// registers (every weight is used by one wave only).  Per 32-wide block the wave issues the
// same two block-dot MFMAs, the same two rank-1 scale MFMAs and the same ordered fmas.
//
// Bound: HBM (each expert's weights once), with the rescale's 64 vector operations per block
// and wave close behind.  H 4096, I 3072, E 64, K 8, T = 48: Q4_0 337 us a layer (1.38 GB of
// weights, 1.43 GB through the memory fabric by the counters; the LDS-staged 64-pair tiles
// 455), Q8_0 471 (2.6 GB; 536).  One tile's results
// at a time keep three waves on a SIMD: three of them four blocks deep run Q4_0 in 354 us
// where two eight deep take 371.  Non-temporal weight loads take Q8_0 from 525 to 471 and
// Q4_0 from 354 to 337; where a launch's weights fit the Infinity Cache they stay cached
// (H 2048, I 1536, E 16: 71 us, non-temporal 79).
#include <utility>

#include "hy_mfma.hpp"

namespace hy {

constexpr int FEW_D = 4;  // blocks in registers, one of them in use

template <int WT, int MODE, bool NT>
__global__ __launch_bounds__(256, 3) void moe_few_kernel(MmArgs a) {
    constexpr bool Q4 = WT == HY_TYPE_Q4_0;
    constexpr int BPB = Q4 ? 16 : 32, D = FEW_D;
    const int tid = threadIdx.x, lane = tid % WAVE, lr = lane % 32, lg = lane / 32;
    const int wv = __builtin_amdgcn_readfirstlane(tid / WAVE);
    // consecutive work groups take consecutive row blocks of a tile: a tile's weights
    // spread over all XCDs, so that these end together whatever the tile count; its
    // activations (32 rows) are small enough for every XCD to fetch them
    const int tile = (int)blockIdx.x / a.nrb, grp = (int)blockIdx.x % a.nrb * 4 + wv;  // grp: 64-row group
    if (tile >= a.R.meta[1] || grp * 64 >= (MODE == 0 ? 2 * a.I : a.H)) return;
    const int e = a.R.tile_e[tile], start = a.R.tile_start[tile], n = a.R.tile_n[tile];
    const int nb = a.Kdim / QK;
    const uint32_t n_slots = (uint32_t)(a.T * a.K + a.T);
    // the tile's pairs are consecutive rows of the slot-ordered operands and of y; lanes
    // past the last pair repeat it
    const int slot = (e == a.E ? a.T * a.K : a.R.off[e]) + start + min(lr, n - 1);

    // block b: a wave-uniform base and a lane offset
    const uint8_t* const wq = a.W.qs + (size_t)e * a.W.qs_stride + (size_t)grp * nb * (64 * BPB);
    const uint16_t* const ws = a.W.sc + (size_t)e * a.W.sc_stride + (size_t)grp * nb * 64;
    const uint32_t w_off = (uint32_t)(lr * BPB + (Q4 ? 0 : 16 * lg));
    const uint32_t x_off = (uint32_t)slot * 32u + 16u * (uint32_t)lg;

    struct Blk {
        v4i_t w0, w1, x;  // rows lr and 32 + lr (Q4_0: both lane halves the raw nibbles), token lr
        uint32_t dw;      // lane l: scale of row l
        float dx;         // scale of token lr
    };
    Blk bk[D];
    auto load = [&](int b, Blk& d) {
        const uint8_t* q = wq + (size_t)b * (64 * BPB);
        const v4i_t *r0 = reinterpret_cast<const v4i_t*>(q + w_off),
                    *r1 = reinterpret_cast<const v4i_t*>(q + 32 * BPB + w_off);
        d.w0 = NT ? __builtin_nontemporal_load(r0) : *r0;
        d.w1 = NT ? __builtin_nontemporal_load(r1) : *r1;
        d.dw = ws[(size_t)b * 64 + lane];
        d.x = *reinterpret_cast<const v4i_t*>(reinterpret_cast<const uint8_t*>(a.aq) + (size_t)b * n_slots * 32 + x_off);
        d.dx = (a.ad + (size_t)b * n_slots)[slot];
    };
    float acc0[16], acc1[16];  // rows 0-31 / 32-63 of the group
#pragma unroll
    for (int v = 0; v < 16; v++) acc0[v] = acc1[v] = 0.0f;
    // rank-1 scale operands {d, 0, 0, ...}: rows 0-31 use k-slot 0 of the lower lane half,
    // rows 32-63 that of the upper one, where dw lies; the other half is zero in both
    const uint32_t lo = lg ? 0u : ~0u, hi = ~lo;
    v4i_t xa = {}, xb = {};
    const uint32_t sh = 4u - 4u * (uint32_t)lg;
    auto step = [&](const Blk& d) {
        const uint32_t dx = (uint32_t)__builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(d.dx, 0.0f));  // exact
        const v16f_t zf = {};
        auto tile = [&](v4i_t w, uint32_t half, float (&acc)[16]) {
            if constexpr (Q4) {
#pragma unroll
                for (int i = 0; i < 4; i++) w[i] = unpack_q4x16(w[i], sh);
            }
            xa[0] = (int)(d.dw & half);
            xb[0] = (int)(dx & half);
            const v16i_t S = block_dot_tile(w, d.x);
            const v16f_t C = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h_t, xa),
                                                                    __builtin_bit_cast(v8h_t, xb), zf, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] = fmaf((float)S[v], C[v], acc[v]);
            __builtin_amdgcn_sched_barrier(0);  // one tile's results live at a time
        };
        tile(d.w0, lo, acc0);
        tile(d.w1, hi, acc1);
    };
#pragma unroll
    for (int i = 0; i < D - 1; i++) load(min(i, nb - 1), bk[i]);
    for (int b0 = 0; b0 < nb; b0 += D)
#pragma unroll
        for (int i = 0; i < D; i++) {
            load(min(b0 + i + D - 1, nb - 1), bk[(i + D - 1) % D]);  // past the last block: that one again
            __builtin_amdgcn_sched_barrier(0);                       // the refill goes out ahead of the math
            if (b0 + i < nb) step(bk[i]);
        }
    if constexpr (Q4) {
#pragma unroll
        for (int v = 0; v < 16; v++) {
            acc0[v] *= 0.0625f;
            acc1[v] *= 0.0625f;
        }
    }
    if (lr >= n) return;
    if (MODE == 0)
        mm_store_h(a, acc0, acc1, grp, slot, lg);
    else
        mm_store_y(a, acc0, acc1, grp * 64, slot, lg);
}

template <int WT, int MODE>
static hipError_t few_launch(MmArgs a, int n_tiles_bound, int rows, hipStream_t s) {
    a.nrb = (rows / 64 + 3) / 4;
    const dim3 grid((unsigned)(n_tiles_bound * a.nrb));
    if (a.W.qs_stride * (size_t)a.W.n_mats > INFINITY_CACHE)
        hipLaunchKernelGGL((moe_few_kernel<WT, MODE, true>), grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((moe_few_kernel<WT, MODE, false>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_up_few(int wtype, int n_tiles_bound, const MmArgs& a, hipStream_t s) {
    return wtype == HY_TYPE_Q4_0 ? few_launch<HY_TYPE_Q4_0, 0>(a, n_tiles_bound, 2 * a.I, s)
                                 : few_launch<HY_TYPE_Q8_0, 0>(a, n_tiles_bound, 2 * a.I, s);
}
hipError_t launch_down_few(int wtype, int n_tiles_bound, const MmArgs& a, hipStream_t s) {
    return wtype == HY_TYPE_Q4_0 ? few_launch<HY_TYPE_Q4_0, 1>(a, n_tiles_bound, a.H, s)
                                 : few_launch<HY_TYPE_Q8_0, 1>(a, n_tiles_bound, a.H, s);
}

}  // namespace hy
