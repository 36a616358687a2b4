// hy_split.hpp -- fp32 products on the bf16 matrix cores, shared by the GEMMs and the
// prompt attention.
//
// Every fp32 operand is split exactly into three bf16 pieces, x = hi + mid + lo (8 + 8 + 8
// significand bits, round to nearest at each step, both remainders exact in fp32; bf16
// has fp32's exponent range and the matrix cores keep bf16 denormals), and a product is
// the sum of the six piece products of weight 2^-16 and above,
//   hi hi + hi mid + mid hi + mid mid + hi lo + lo hi,
// accumulated in fp32 by v_mfma_f32_32x32x16_bf16.  What is left out, mid lo + lo mid +
// lo lo, is below 2^-24 of the product: no more than one fp32 rounding of it.  Six
// bf16 MFMAs of 16 k-steps take 6 x 32 cycles where eight fp32 MFMAs of 2 take 8 x 64.
//
// These instructions cut the low bits of what they add towards minus infinity (measured: a
// mean error of -0.21 of the rms error, whatever the result's sign; the fp32 MFMAs show
// none), and a later average over rows, as in attention, keeps such a mean while it thins
// out the rest.  So the accumulators hold the sum and its negative in turns (flip_at),
// with the pieces of A negated alike, and the mean cancels.
//
// The split is exact down to 2^-110, and below wherever the last pieces' bits end at bf16's
// smallest denormal, 2^-133 (zeros, values that were bf16 or fp16 before).  Any other
// operand leaves a remainder that is no bf16 value, which split2 records: its users compute
// such products on the fp32 matrix cores instead.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

#include "hy_lds.hpp"

namespace hy {

// f(integral_constant 0), ..., f(integral_constant N - 1): loops whose index is a constant
// (LDS offsets in instructions, register arrays)
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (f(std::integral_constant<int, I>{}), ...);
    }(std::make_integer_sequence<int, N>{});
}

typedef float v16f_t __attribute__((ext_vector_type(16)));
typedef float v2f_t __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf_t __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf_t __attribute__((ext_vector_type(8)));

// two floats -> their three bf16 pieces, packed (v_cvt_pk_bf16_f32, round to nearest even)
struct Split2 {
    uint32_t p[3];
};
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
    const v2f_t f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, v2bf_t));
}
// lost gathers the last remainders' bits; lost_bits(lost) once a split was not exact (a bf16
// value has the low half of its fp32 bits clear): one operation for two operands, eleven
// for their split (77 x 6144 x 4096: 165 -> 167 us; 4096 rows: 1.03 ms with and without)
__device__ __forceinline__ bool lost_bits(uint32_t lost) { return (lost & 0xffffu) != 0; }
__device__ __forceinline__ Split2 split2(float a, float b, uint32_t& lost) {
    Split2 s;
    s.p[0] = pk_bf16(a, b);
    a -= __uint_as_float(s.p[0] << 16);
    b -= __uint_as_float(s.p[0] & 0xffff0000u);
    s.p[1] = pk_bf16(a, b);
    a -= __uint_as_float(s.p[1] << 16);
    b -= __uint_as_float(s.p[1] & 0xffff0000u);
    s.p[2] = pk_bf16(a, b);
    lost |= __float_as_uint(a) | __float_as_uint(b);
    asm("" : "+v"(lost));  // formed here: the compiler would gather many remainders first, in registers
    return s;
}
__device__ __forceinline__ v16f_t mfma_bf16(v4i_t a, v4i_t b, v16f_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf_t, a), __builtin_bit_cast(v8bf_t, b), c, 0,
                                                   0, 0);
}
// Sign turns: PERIOD stages of one sign, the first one half as long, so that the growing
// means of neighbouring turns cancel.  flip_at: stage d of a range opens a turn;
// turn_sign: its sign.
template <int PERIOD>
__device__ __forceinline__ bool flip_at(int d) { return d % PERIOD == PERIOD / 2; }
template <int PERIOD>
__device__ __forceinline__ float turn_sign(int d) { return (d + PERIOD / 2) / PERIOD % 2 ? -1.0f : 1.0f; }
// finite iff x - x == 0
__device__ __forceinline__ bool non_finite(float x) { return !(x - x == 0.0f); }

}  // namespace hy
