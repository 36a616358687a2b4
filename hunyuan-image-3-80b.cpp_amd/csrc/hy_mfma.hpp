// hy_mfma.hpp -- what the two grouped GEMMs on the int8 matrix cores share (hy_mfma.hip,
// hy_mfma_few.hip): arguments, block products, Q4_0 unpack, epilogues.
#pragma once
#include "hy_device.hpp"
#include "hy_launch.hpp"
#include "hy_layout.hpp"
#include "hy_lds.hpp"

namespace hy {

typedef int v16i_t __attribute__((ext_vector_type(16)));
typedef float v16f_t __attribute__((ext_vector_type(16)));
typedef _Float16 v8h_t __attribute__((ext_vector_type(8)));

struct MmArgs {
    MatView W;
    Routing R;
    const int8_t* aq;   // activations int8, block-major in slot order [Kdim/32][slots][32]: the
                        // gathered x (mode 0, gather_act_kernel) or h (mode 1)
    const float* ad;    // their scales (exact fp16 values) [Kdim/32][slots]
    int T, H, I, E, K;
    int Kdim;           // reduction length (H for mode 0, I for modes 1/2)
    int nrb;            // row blocks of the weight matrix
    int tiles_pad;      // tile bound rounded up to a multiple of MM_XCD x the shape's GROUP (sizes the grid)
    int8_t* hq;         // mode 0 outputs
    float* hd;
    int* hs;
    float* y;           // mode 1 output
    int* ctr;           // MM_CTR_INTS work counters, zeroed by gather_act_kernel before the gate/up launch
};

// A weight n - 8 is left in the high nibble of its byte, as the int8 value 16 (n - 8)
// (n with its top bit flipped is n - 8 in two's complement): a shift and one
// three-input logic operation per four weights.  Block dots and accumulators come out 16
// times too large, exactly -- a block dot is at most 16 x 8 x 127 x 32 < 2^24, and the
// accumulator chain scales by a power of two (its values are multiples of 2^-48, far
// from denormals) -- and the epilogue multiplies by 1/16.  Against n - 8 itself (five
// operations per four weights): Q4_0 layers of T = 48 465 -> 454 us, 4096 skewed tokens
// 3.94 -> 3.92 ms, a decoder layer of T = 300 906 -> 895 us (same box).
template <bool PLAIN = false>
__device__ __forceinline__ int unpack_q4x16(int v, uint32_t sh) {
    uint32_t n = ((uint32_t)v << sh) & 0xF0F0F0F0u;
    if constexpr (PLAIN) asm("" : "+v"(n));  // keeps the two operations apart
    return (int)(n ^ 0x80808080u);
}

// The exact int32 dots of one 32-wide GGUF block over a 32x32 tile (K = 32 is one
// block): v_mfma_i32_32x32x32_i8 with a zero accumulator.
__device__ __forceinline__ v16i_t block_dot_tile(v4i_t A, v4i_t B) {
    const v16i_t zero = {};
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B, zero, 0, 0, 0);
}

// the products of tiles of up to FEW_TOK pairs (hy_mfma_few.hip)
constexpr int FEW_TOK = 32;
constexpr size_t INFINITY_CACHE = (size_t)256 << 20;
hipError_t launch_up_few(int wtype, int n_tiles_bound, const MmArgs& a, hipStream_t s);
hipError_t launch_down_few(int wtype, int n_tiles_bound, const MmArgs& a, hipStream_t s);

// Epilogues for the two 32-row results of a 64-row slab, one token per lane (result
// register v: row 8 (v / 4) + 4 lg + v % 4 of each).

// gate (ag) and matching up rows (au) of slab `slab`: h = silu(g) * u and its Q8_0
// quantization, block-major (block plane `slab`, row `slot`)
__device__ __forceinline__ void mm_store_h(const MmArgs& a, const float (&ag)[16], const float (&au)[16], int slab,
                                           int slot, int lg) {
    float h[16];
    float amax = 0.0f;
#pragma unroll
    for (int v = 0; v < 16; v++) {
        h[v] = swiglu(ag[v], au[v]);
        amax = fmaxf(amax, fabsf(h[v]));
    }
    amax = fmaxf(amax, __shfl_xor(amax, 32, WAVE));
    const float d = amax / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    int qsum = 0;
    int packed[4];
#pragma unroll
    for (int g = 0; g < 4; g++) {
        uint32_t p = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int q = (int)__builtin_roundf(h[4 * g + i] * id);
            qsum += q;
            p |= ((uint32_t)(q & 0xff)) << (8 * i);
        }
        packed[g] = (int)p;
    }
    qsum += __shfl_xor(qsum, 32, WAVE);
    const size_t hi = (size_t)slab * (size_t)(a.T * a.K + a.T) + (size_t)slot;
    int8_t* dst = a.hq + hi * QK;
#pragma unroll
    for (int g = 0; g < 4; g++) *reinterpret_cast<int*>(dst + 8 * g + 4 * lg) = packed[g];
    if (lg == 0) {
        a.hd[hi] = h2f(f2h(d));
        a.hs[hi] = qsum;
    }
}

// rows r0 .. + 31 and r0 + 32 .. of y's row `slot`
__device__ __forceinline__ void mm_store_y(const MmArgs& a, const float (&ag)[16], const float (&au)[16], int r0,
                                           int slot, int lg) {
    float* yr = a.y + (size_t)slot * a.H + r0;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const int r = 8 * g + 4 * lg;
        *reinterpret_cast<float4*>(yr + r) = make_float4(ag[4 * g], ag[4 * g + 1], ag[4 * g + 2], ag[4 * g + 3]);
        *reinterpret_cast<float4*>(yr + 32 + r) = make_float4(au[4 * g], au[4 * g + 1], au[4 * g + 2], au[4 * g + 3]);
    }
}

}  // namespace hy
