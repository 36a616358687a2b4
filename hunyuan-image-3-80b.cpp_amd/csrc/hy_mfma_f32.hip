// hy_mfma_f32.hip -- expert products of batches with F32 weights on the fp32 matrix cores.
//
// v_mfma_f32_16x16x4f32 computes each output as the chain
//   d = fmaf(a3, b3, fmaf(a2, b2, fmaf(a1, b1, fmaf(a0, b0, c))))
// with one rounding per fma (compared bit for bit on the device over four exponent
// ranges, denormals among them), so walking k in ascending fours gives exactly the
// per-row chain acc = fmaf(w_k, x_k, acc) of the decode GEMV and the oracle.
//
// Work item = (tile of up to TOK = 64 or 32 (token, expert) pairs, 128 weight rows).  A work group of
// four waves copies, per 32-wide block, its two 64-row groups (the resident quad-major
// blocks, 8 KB each) and the tile's activation rows into a ring of LDS stages
// (buffer_load ... lds, one barrier per stage); the activations land quad-major too, so an
// operand read (lane l: row or token l % 16, element l / 16 of the quad) is 256 contiguous
// bytes.  Wave w takes rows 16 p .. + 15 and 32 + 16 p .. + 15 (p = w % 2) of row group
// w / 2 -- in the packed gate_up order the gate rows and their matching up rows -- times
// the tile's active 16-token groups.
#include <utility>

#include "hy_device.hpp"
#include "hy_launch.hpp"
#include "hy_layout.hpp"
#include "hy_lds.hpp"

// Bound: HBM (each expert's weights once per tile) while tiles hold up to ~32 pairs, the
// fp32 matrix cores beyond.  Whole layers of 16 experts of top-4 and the shared one,
// 4096 x 3072 (2.57 GB; T = 96 fetches 2.66 GB): T = 32 522 us, T = 96 558 us (both products
// 537 at best, 5.0 TB/s), T = 512 1.85 ms (105 TFLOP/s).  The decode GEMV, which took these
// batches before, reads the weights once per four pairs: 910 us, 2.06 ms, 10.6 ms.
namespace hy {

constexpr int MF_RING = 3;  // stages of one block: two in flight while one is consumed
constexpr int MF_A = 2 * 64 * QK * 4;  // bytes of the two row groups' block

struct MfArgs {
    MatView W;
    Routing R;
    const float* x;  // activation rows of Kd floats: x by token (mode 0), h by slot (mode 1)
    int T, E, K;
    int Kd;          // reduction length
    int n_groups;    // 64-row groups of the weight matrix
    int nrb;         // work groups per tile
    int tiles;       // tile bound (sizes the grid)
    int ld;          // row length of out
    float* out;      // mode 0: h [slots][I]; mode 1: y [slots][H]
};

template <int MODE, int TOK>
__global__ __launch_bounds__(256, 2) void moe_mfma_f32_kernel(MfArgs a) {
    constexpr int STAGE = MF_A + TOK * QK * 4;
    constexpr int XL = TOK / 32;      // activation copies per wave and stage
    constexpr int LOADS = 4 + XL;
    constexpr int NG = TOK / 16;      // 16-token groups
    __shared__ __attribute__((aligned(1024))) uint8_t ring[MF_RING][STAGE];
    __shared__ int slot_s[TOK], row_s[TOK];
    // the shared expert's tiles (the list's last, with the most tokens) start first
    const int tile = a.tiles - 1 - (int)blockIdx.x / a.nrb, rb = (int)blockIdx.x % a.nrb;
    if (tile >= a.R.meta[1]) return;
    const int e = a.R.tile_e[tile], start = a.R.tile_start[tile], n = a.R.tile_n[tile];
    const int tid = threadIdx.x, lane = tid % WAVE;
    const int wv = __builtin_amdgcn_readfirstlane(tid / WAVE);
    if (tid < TOK) {
        // positions past n repeat the tile's first pair (read, never stored)
        const int i = tid < n ? tid : 0;
        const bool shared = e == a.E;
        const int slot = shared ? a.T * a.K + start + i : a.R.off[e] + start + i;
        slot_s[tid] = slot;
        row_s[tid] = MODE == 1 ? slot : shared ? start + i : a.R.srt_tok[slot];
    }
    __syncthreads();

    const int nb = a.Kd / QK, p = wv % 2, G = 2 * rb + wv / 2;
    // copies: wave w moves quads 4 p .. 4 p + 3 of its row group (1 KB each) and quads
    // 2 w, 2 w + 1 of the activations (TOK tokens of 16 bytes each: one copy per quad, or
    // one for both); a group past the matrix repeats the last
    const __amdgpu_buffer_rsrc_t rw =
        buf_rsrc(a.W.qs + (size_t)e * a.W.qs_stride + (size_t)min(G, a.n_groups - 1) * nb * 64 * QK * 4);
    const __amdgpu_buffer_rsrc_t rx = buf_rsrc(a.x);
    const uint32_t w_off = (uint32_t)(4096 * p + 16 * lane);
    const uint32_t x_off =
        (uint32_t)row_s[lane % TOK] * (uint32_t)a.Kd * 4u + 32u * (uint32_t)wv + 16u * (uint32_t)(lane / TOK);
    auto issue = [&](int s) {
        uint8_t* st = ring[s % MF_RING];
        uint8_t* aw = st + (wv / 2) * 8192 + 4096 * p;
#pragma unroll
        for (int c = 0; c < 4; c++) b2l(rw, aw + 1024 * c, w_off + 1024u * c, (uint32_t)s * 8192u);
        uint8_t* bx = st + MF_A + 2 * TOK * 16 * wv;
#pragma unroll
        for (int c = 0; c < XL; c++) b2l(rx, bx + 1024 * c, x_off + 16u * c, (uint32_t)s * 128u);
    };
    const uint32_t ring0 = lds_off(ring[0]);
    const uint32_t a_lane = ring0 + (uint32_t)((wv / 2) * 8192 + (16 * p + lane % 16) * 16 + (lane / 16) * 4);
    const uint32_t b_lane = ring0 + (uint32_t)(MF_A + (lane % 16) * 16 + (lane / 16) * 4);
    const int ng = (n + 15) / 16;  // active 16-token groups (wave-uniform)
    v4f_t acc[NG][2];
#pragma unroll
    for (int g = 0; g < NG; g++) acc[g][0] = acc[g][1] = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};

#pragma unroll
    for (int s = 0; s < MF_RING - 1; s++)
        if (s < nb) issue(s);
    uint32_t soff = 0;
    for (int s = 0; s < nb; s++) {
        soff = __builtin_amdgcn_readfirstlane(soff);
        wait_copies<LOADS, MF_RING - 2>(nb - 1 - s);
        __builtin_amdgcn_s_barrier();
        // the slot read in iteration s - 1, which every wave finished before this barrier
        if (s + MF_RING - 1 < nb) issue(s + MF_RING - 1);
        const uint32_t al = a_lane + soff, bl = b_lane + soff;
        uint32_t wr[2][8], xr[2][8];  // [row half][quad]; [group parity][quad]
        auto load_x = [&]<int GI, int... C>(std::integral_constant<int, GI>, std::integer_sequence<int, C...>) {
            ((xr[GI & 1][C] = lds_b32_at<C * TOK * 16 + GI * 256>(bl)), ...);
        };
        [&]<int... C>(std::integer_sequence<int, C...>) {
            ((wr[0][C] = lds_b32_at<C * 1024>(al)), ...);
            ((wr[1][C] = lds_b32_at<C * 1024 + 512>(al)), ...);
        }(std::make_integer_sequence<int, 8>{});
        load_x(std::integral_constant<int, 0>{}, std::make_integer_sequence<int, 8>{});
        lds_wait();
#pragma unroll
        for (int c = 0; c < 8; c++) {
            lds_pin(wr[0][c]);
            lds_pin(wr[1][c]);
        }
        auto group = [&]<int GI>(std::integral_constant<int, GI>) {
            if (GI >= ng) return;
#pragma unroll
            for (int c = 0; c < 8; c++) lds_pin(xr[GI & 1][c]);
            if constexpr (GI < NG - 1) load_x(std::integral_constant<int, GI + 1>{}, std::make_integer_sequence<int, 8>{});
#pragma unroll
            for (int c = 0; c < 8; c++)
#pragma unroll
                for (int r = 0; r < 2; r++)
                    acc[GI][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        __uint_as_float(wr[r][c]), __uint_as_float(xr[GI & 1][c]), acc[GI][r], 0, 0, 0);
            lds_wait();  // the next group's reads
        };
        group(std::integral_constant<int, 0>{});
        group(std::integral_constant<int, 1>{});
        if constexpr (NG == 4) {
            group(std::integral_constant<int, 2>{});
            group(std::integral_constant<int, 3>{});
        }
        soff = soff + STAGE == (uint32_t)(MF_RING * STAGE) ? 0u : soff + STAGE;
    }

    if (G >= a.n_groups) return;
    const int r4 = 16 * p + 4 * (lane / 16);  // result register v: row r4 + v (and 32 + r4 + v) of the group
#pragma unroll
    for (int g = 0; g < NG; g++) {
        const int j = 16 * g + lane % 16;
        if (j >= n) continue;
        float* o = a.out + (size_t)slot_s[j] * a.ld;
        const v4f_t u = acc[g][0], v = acc[g][1];
        if (MODE == 0) {
            *reinterpret_cast<float4*>(o + 32 * G + r4) =
                make_float4(swiglu(u[0], v[0]), swiglu(u[1], v[1]), swiglu(u[2], v[2]), swiglu(u[3], v[3]));
        } else {
            *reinterpret_cast<v4f_t*>(o + 64 * G + r4) = u;
            *reinterpret_cast<v4f_t*>(o + 64 * G + 32 + r4) = v;
        }
    }
}

// 32-pair tiles while experts see up to 32 pairs each.  Layers of 16 experts of top-4, 32- against
// 64-pair tiles: T = 96 558 / 600 us, 128 716 / 707, 160 899 / 780, 512 1981 / 1845.
int mfma_f32_tokens(int T, int K, int E) { return (int64_t)T * K <= 32 * (int64_t)E ? 32 : 64; }

// The decode GEMV (4 pairs per pass over an expert's weights) stays the better one up to about
// 3 pairs per expert.  Layers of 4096 x 3072, GEMV against these products: 64 experts of top-8
// T = 16 1.43 / 1.48 ms; 16 of top-4 T = 16 554 / 514 us, T = 32 910 / 522, T = 96 2062 / 558.
// Past 32 tokens the shared expert alone takes the GEMV nine passes, and these win however few
// pairs the routed ones see: 2048 x 1536, 64 experts of top-1 T = 33 210 / 207 us, 48 231 / 221,
// 16 of top-1 T = 33 193 / 142 (a tie again at T = 64 of 64: 274 / 281).
bool mfma_f32_ok(int T, int K, int E, int H, int I) {
    if (T <= 32 && (int64_t)T * K <= 3 * (int64_t)E) return false;
    // the activation rows are addressed with 32-bit byte offsets
    const uint64_t lim = 1ull << 32;
    return (uint64_t)T * H * 4 < lim && (uint64_t)T * (K + 1) * I * 4 < lim;
}

template <int MODE>
static hipError_t launch_mode_f32(MfArgs a, hipStream_t s) {
    a.nrb = (a.n_groups + 1) / 2;
    const dim3 grid((unsigned)a.tiles * (unsigned)a.nrb);
    if (mfma_f32_tokens(a.T, a.K, a.E) == 32)
        hipLaunchKernelGGL((moe_mfma_f32_kernel<MODE, 32>), grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((moe_mfma_f32_kernel<MODE, 64>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_ffn_up_mfma_f32(int n_tiles_bound, const MatView& W, const Routing& R, const float* x, int T, int H,
                                  int I, int E, int K, float* hf, hipStream_t s) {
    return launch_mode_f32<0>(MfArgs{W, R, x, T, E, K, H, 2 * I / 64, 0, n_tiles_bound, I, hf}, s);
}

hipError_t launch_ffn_down_mfma_f32(int n_tiles_bound, const MatView& W, const Routing& R, const float* hf, int T,
                                    int H, int I, int E, int K, float* y, hipStream_t s) {
    return launch_mode_f32<1>(MfArgs{W, R, hf, T, E, K, I, H / 64, 0, n_tiles_bound, H, y}, s);
}

}  // namespace hy
