// hy_gemm.hip -- fp32 matrix products C[M][N] = (R[M][N] +) A[M][K] . W[N][K]^T on the
// bf16 matrix cores, with fp32 accuracy.
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
// Infinities and NaNs have no such split (inf - inf), and a value that rounds up to
// infinity in bf16 neither: a wave whose accumulators hold a non-finite value after its
// k-range computes that range again on the fp32 matrix cores (segment_f32), so such
// inputs give what the fp32 product gives.
#include <utility>

#include "hy_device.hpp"
#include "hy_launch.hpp"
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
__device__ __forceinline__ Split2 split2(float a, float b) {
    Split2 s;
    s.p[0] = pk_bf16(a, b);
    a -= __uint_as_float(s.p[0] << 16);
    b -= __uint_as_float(s.p[0] & 0xffff0000u);
    s.p[1] = pk_bf16(a, b);
    a -= __uint_as_float(s.p[1] << 16);
    b -= __uint_as_float(s.p[1] & 0xffff0000u);
    s.p[2] = pk_bf16(a, b);
    return s;
}
__device__ __forceinline__ v16f_t mfma_bf16(v4i_t a, v4i_t b, v16f_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf_t, a), __builtin_bit_cast(v8bf_t, b), c, 0,
                                                   0, 0);
}
// finite iff x - x == 0
__device__ __forceinline__ bool non_finite(float x) { return !(x - x == 0.0f); }

// ---------------------------------------------------------------- small batches (M <= 128)
// A stream over W: a work group of four waves takes all M rows of A (MT tiles of 32) times
// 128 rows of W, 32 per wave.  A wave loads its W rows straight into registers in MFMA
// operand order, SK_D stages of 32 floats ahead, and splits each element once; A is split
// by the work group into a double-buffered LDS stage the four waves share (one barrier
// per stage).  The tiles x stages units are cut into G equal contiguous ranges (stream-K,
// one per work group): a tile cut between ranges leaves partial tiles in slots 2 g (the
// range's first piece) and 2 g + 1, which gemm_small_sum_kernel adds in k order.
//
// Bound: HBM (W once) up to M = 64, then the stage loop's LDS and splitting work.  The
// 4096 -> 6144 and 6144 -> 4096 projections (168 MB of W), both products with their sums:
// M = 20 55 us, 50 70 us, 77 80 us, 128 95 us; one wave per 64 x 64 fp32 MFMA tile, which
// these batches took before, ran 552 us at M = 77 (96 waves for 256 CUs).  Two stages of W
// in flight beat four (M = 128: 40 against 44 us a product) and six; 512 work groups beat
// 256 and 384, and 768 lose more in the sums than they gain.  Against 64 bits the results
// are three times closer than the fp32 MFMA's (M = 77: 6.4e-7 against 2.0e-6 of the whole
// attention's output): K / 16 x 6 roundings instead of K.
constexpr int SK_BN = 128;  // W rows per work group
constexpr int SK_KC = 32;   // floats of K per stage
constexpr int SK_D = 2;     // stages of W in flight

struct GemmSmallArgs {
    const float* A;
    const float* W;
    const float* R;  // optional: C = R + A.W^T
    float* C;
    int M, N, K;
    int G;           // work groups; G = tiles: one whole tile each
    int qd, rem;     // tiles x stages = G qd + rem: the first rem ranges take qd + 1 units
    float* part;     // 2 G slots of MT x 32 x 128 floats (unused when G = tiles)
};

// first unit of range g, and the range unit u falls in
__device__ __forceinline__ int gs_lo(const GemmSmallArgs& p, int g) { return g * p.qd + min(g, p.rem); }
__device__ __forceinline__ int gs_owner(const GemmSmallArgs& p, int u) {
    const int big = p.rem * (p.qd + 1);
    return u < big ? u / (p.qd + 1) : p.rem + (u - big) / p.qd;
}

// LDS of one A stage: three pieces of 4 k-chunks of 8 (chunk 2 u + h holds floats
// 16 u + 4 h .. + 3 and 16 u + 8 + 4 h .. + 3 of a row, the k-slots of MFMA lane half h
// in sub-step u), each 32 MT rows of 16 bytes.  The 128 bytes between chunks put the four
// chunks a wave stores at once (8 rows x 8 float4) on different banks.
template <int MT>
struct SkLds {
    static constexpr int CHUNK = MT * 32 * 16 + 128;
    static constexpr int PIECE = 4 * CHUNK;
    static constexpr int BYTES = 3 * PIECE;
};

template <int MT>
__global__ __launch_bounds__(256, 2) void gemm_small_kernel(GemmSmallArgs p) {
    using L = SkLds<MT>;
    __shared__ __attribute__((aligned(16))) uint8_t abuf[2][L::BYTES];
    const int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE;
    const int lr = lane % 32, h = lane / 32;
    const int M = p.M, N = p.N, K = p.K;
    const int nst = K / SK_KC;

    // A: thread tid copies float4 k4 of rows ar + 32 i of every stage
    const int k4 = tid % 8, ar = tid / 8;
    const uint32_t a_dst = lds_off(abuf[0]) + (uint32_t)((2 * (k4 / 4) + k4 % 2) * L::CHUNK + ar * 16 + 8 * ((k4 / 2) % 2));
    const uint32_t a_src = lds_off(abuf[0]) + (uint32_t)(h * L::CHUNK + lr * 16);
    const float* arow[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) arow[i] = p.A + (size_t)min(ar + 32 * i, M - 1) * K + 4 * k4;

    // stages [s0, s1) of tile t on the fp32 matrix cores (non-finite operands)
    auto segment_f32 = [&](int t, int s0, int s1, v16f_t (&acc)[MT]) {
        const float* w = p.W + (size_t)min(t * SK_BN + 32 * wv + lr, N - 1) * K + h;
#pragma unroll
        for (int i = 0; i < MT; i++) acc[i] = v16f_t{};
        for (int k = s0 * SK_KC; k < s1 * SK_KC; k += 2) {
            const float b = w[k];
#pragma unroll
            for (int i = 0; i < MT; i++)
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(p.A[(size_t)min(32 * i + lr, M - 1) * K + k + h], b,
                                                              acc[i], 0, 0, 0);
        }
    };
    auto segment = [&](int t, int s0, int s1, v16f_t (&acc)[MT]) {
        const float* w = p.W + (size_t)min(t * SK_BN + 32 * wv + lr, N - 1) * K + 4 * h;
        v4f_t wb[SK_D][4];  // [stage][2 u + q]: floats 16 u + 8 q + 4 h .. + 3
        v4f_t ab[MT];
        auto load_w = [&](int s, v4f_t (&d)[4]) {
            const float* src = w + (size_t)min(s, s1 - 1) * SK_KC;
#pragma unroll
            for (int j = 0; j < 4; j++) d[j] = *reinterpret_cast<const v4f_t*>(src + 8 * j);
        };
        auto load_a = [&](int s) {
            const size_t k0 = (size_t)min(s, s1 - 1) * SK_KC;
#pragma unroll
            for (int i = 0; i < MT; i++) ab[i] = *reinterpret_cast<const v4f_t*>(arow[i] + k0);
        };
#pragma unroll
        for (int i = 0; i < MT; i++) acc[i] = v16f_t{};
        load_a(s0);
#pragma unroll
        for (int d = 0; d < SK_D - 1; d++) load_w(s0 + d, wb[d]);
        auto stage = [&](auto dc, int s) {
            constexpr int D = decltype(dc)::value;
            constexpr int BUF = (D & 1) * L::BYTES;  // SK_D is even: D & 1 == (s - s0) & 1
            // A(s) -> LDS; its buffer was last read in stage s - 2, which every wave had
            // finished before the barrier of stage s - 1
            static_for<MT>([&](auto ic) {
                constexpr int I = decltype(ic)::value;
                const Split2 x = split2(ab[I][0], ab[I][1]), y = split2(ab[I][2], ab[I][3]);
                static_for<3>([&](auto qc) {
                    constexpr int Q = decltype(qc)::value;
                    lds_st64_at<BUF + Q * L::PIECE + I * 512>(a_dst, x.p[Q], y.p[Q]);
                });
            });
            load_a(s + 1);
            load_w(s + SK_D - 1, wb[(D + SK_D - 1) % SK_D]);
            __builtin_amdgcn_sched_barrier(0);  // the refills go out ahead of the math
            lds_wait();
            __builtin_amdgcn_s_barrier();
            static_for<2>([&](auto uc) {
                constexpr int UU = decltype(uc)::value;
                v4i_t af[MT][3];
                static_for<MT>([&](auto ic) {
                    static_for<3>([&](auto qc) {
                        constexpr int I = decltype(ic)::value, Q = decltype(qc)::value;
                        af[I][Q] = lds_b128_at<BUF + Q * L::PIECE + 2 * UU * L::CHUNK + I * 512>(a_src);
                    });
                });
                v4i_t wf[3];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const v4f_t v = wb[D][2 * UU + j / 2];
                    const Split2 x = split2(v[2 * (j % 2)], v[2 * (j % 2) + 1]);
#pragma unroll
                    for (int q = 0; q < 3; q++) wf[q][j] = (int)x.p[q];
                }
                lds_wait();
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int q = 0; q < 3; q++) lds_pin(af[i][q]);
                // the small products first
                constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PW[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                for (int c = 0; c < 6; c++)
#pragma unroll
                    for (int i = 0; i < MT; i++) acc[i] = mfma_bf16(af[i][PA[c]], wf[PW[c]], acc[i]);
                __builtin_amdgcn_sched_barrier(0);  // one sub-step's operands live at a time
            });
        };
        for (int sb = s0; sb < s1; sb += SK_D)
            static_for<SK_D>([&](auto dc) {
                if (sb + decltype(dc)::value < s1) stage(dc, sb + decltype(dc)::value);
            });
        bool bad = false;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) bad |= non_finite(acc[i][v]);
        if (__any(bad)) segment_f32(t, s0, s1, acc);
        __builtin_amdgcn_s_barrier();  // every wave is done with the A stages
    };

    v16f_t acc[MT];
    auto store = [&](int t) {
        const int col = t * SK_BN + 32 * wv + lr;
        if (col >= N) return;
        int r0 = 4 * h;
        lds_pin(r0);  // the 16 MT row offsets are formed here, not kept across the stage loop
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int row = 32 * i + 8 * (v / 4) + r0 + v % 4;
                if (row >= M) continue;
                const size_t o = (size_t)row * N + col;
                p.C[o] = p.R ? p.R[o] + acc[i][v] : acc[i][v];
            }
    };
    const int g = blockIdx.x;
    const int lo = gs_lo(p, g), hi = gs_lo(p, g + 1);
    for (int u = lo; u < hi;) {
        const int t = u / nst, s0 = u - t * nst, s1 = min(nst, s0 + (hi - u));
        segment(t, s0, s1, acc);
        if (s0 == 0 && s1 == nst) {
            store(t);
        } else {
            float* slot = p.part + (size_t)(2 * g + (u == lo ? 0 : 1)) * (MT * 32 * SK_BN) + tid;
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int v = 0; v < 16; v++) slot[(i * 16 + v) * 256] = acc[i][v];
        }
        u += s1 - s0;
    }
}

// Sum of the pieces of every cut tile, in k order (+ R): work group (t, y) takes values
// 4 y .. 4 y + 3 (value 16 i + v) of every thread of tile t.
template <int MT>
__global__ __launch_bounds__(256) void gemm_small_sum_kernel(GemmSmallArgs p) {
    const int nst = p.K / SK_KC;
    const int t = blockIdx.x;
    const int u0 = t * nst, u1 = u0 + nst - 1;
    const int g0 = gs_owner(p, u0), g1 = gs_owner(p, u1);
    if (g0 == g1) return;
    const int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE, lr = lane % 32, h = lane / 32;
    // the first piece is g0's last one unless g0's range starts at this tile
    const int slot0 = 2 * g0 + (gs_lo(p, g0) == u0 ? 0 : 1);
    const float* __restrict__ part = p.part + (size_t)blockIdx.y * 4 * 256 + tid;
    constexpr size_t SLOT = MT * 32 * SK_BN;
    float sum[4];
#pragma unroll
    for (int j = 0; j < 4; j++) sum[j] = part[slot0 * SLOT + j * 256];
    for (int g = g0 + 1; g <= g1; g++)
#pragma unroll
        for (int j = 0; j < 4; j++) sum[j] += part[2 * (size_t)g * SLOT + j * 256];
    const int col = t * SK_BN + 32 * wv + lr;
    const int i = blockIdx.y / 4;
    if (col >= p.N) return;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int row = 32 * i + 8 * (blockIdx.y % 4) + 4 * h + j;
        if (row >= p.M) break;
        const size_t o = (size_t)row * p.N + col;
        p.C[o] = p.R ? p.R[o] + sum[j] : sum[j];
    }
}

bool gemm_small_ok(int M, int N, int K) {
    // 32-bit unit counts
    return M > 16 && M <= 128 && K % SK_KC == 0 && (int64_t)(N + SK_BN) / SK_BN * (K / SK_KC) < (1 << 30);
}

template <int MT>
static hipError_t gemm_small_launch(const GemmSmallArgs& p, int tiles, hipStream_t s) {
    hipLaunchKernelGGL(gemm_small_kernel<MT>, dim3(p.G), dim3(256), 0, s, p);
    // ranges that are whole tiles leave no pieces
    if (tiles % p.G != 0) hipLaunchKernelGGL(gemm_small_sum_kernel<MT>, dim3(tiles, 4 * MT), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_gemm_small(const float* A, const float* W, const float* R, float* C, int M, int N, int K,
                             hipStream_t s, float* ws) {
    const int tiles = (N + SK_BN - 1) / SK_BN, U = tiles * (K / SK_KC);
    // with scratch: two work groups per CU, four stages each at least
    const int G = !ws ? tiles : U < 4 * GEMM_SK_GROUPS ? (U + 3) / 4 : GEMM_SK_GROUPS;
    const GemmSmallArgs p{A, W, R, C, M, N, K, G, U / G, U % G, ws};
    switch ((M + 31) / 32) {
    case 1: return gemm_small_launch<1>(p, tiles, s);
    case 2: return gemm_small_launch<2>(p, tiles, s);
    case 3: return gemm_small_launch<3>(p, tiles, s);
    default: return gemm_small_launch<4>(p, tiles, s);
    }
}

}  // namespace hy
