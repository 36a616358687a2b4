// hy_gemm.hip -- fp32 matrix products C[M][N] = (R[M][N] +) A[M][K] . W[N][K]^T on the
// bf16 matrix cores, with fp32 accuracy.
//
// Operands are split into three bf16 pieces each and the six significant piece products
// summed, with the accumulators' sign in turns: hy_split.hpp.
//
// Infinities and NaNs have no such split (inf - inf), and a value that rounds up to
// infinity in bf16 neither: a wave whose accumulators hold a non-finite value after its
// k-range computes that range again on the fp32 matrix cores (segment_f32), so such
// inputs give what the fp32 product gives.  So does a work group that met an operand too
// small for an exact split (most of them below 2^-110).
#include "hy_device.hpp"
#include "hy_launch.hpp"
#include "hy_lds.hpp"
#include "hy_split.hpp"

namespace hy {

// Both products cut their tiles x stages units into p.G contiguous ranges of p.qd units, the
// first p.rem of one more: first unit of range g, and the range that unit u falls in.
template <class P>
__device__ __forceinline__ int gs_lo(const P& p, int g) {
    return g * p.qd + min(g, p.rem);
}
template <class P>
__device__ __forceinline__ int gs_owner(const P& p, int u) {
    const int big = p.rem * (p.qd + 1);
    return u < big ? u / (p.qd + 1) : p.rem + (u - big) / p.qd;
}

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
constexpr int SK_TURN = 4;  // stages of one accumulator sign
static_assert(SK_TURN / 2 % SK_D == 0, "signs turn between unrolled rounds");

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
    __shared__ int lost_at;  // first unit of the last range that held an inexact split
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
        const float* w = p.W + (size_t)min(t * SK_BN + 32 * wv + lr, N - 1) * K + 4 * h;
        const float* arow[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) {
            arow[i] = p.A + (size_t)min(32 * i + lr, M - 1) * K + 4 * h;
            acc[i] = v16f_t{};
        }
        for (int k = s0 * SK_KC; k < s1 * SK_KC; k += 8) {
            const v4f_t b = *reinterpret_cast<const v4f_t*>(w + k);
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const v4f_t a = *reinterpret_cast<const v4f_t*>(arow[i] + k);
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[j], acc[i], 0, 0, 0);
            }
        }
    };
    if (tid == 0) lost_at = -1;
    auto segment = [&](int u, int t, int s0, int s1, v16f_t (&acc)[MT]) {
        uint32_t lost = 0;
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
        auto negate = [&] {
#pragma unroll
            for (int i = 0; i < MT; i++) acc[i] = -acc[i];
        };
        auto stage = [&](auto dc, int s) {
            constexpr int D = decltype(dc)::value;
            constexpr int BUF = (D & 1) * L::BYTES;  // SK_D is even: D & 1 == (s - s0) & 1
            const float sgn = turn_sign<SK_TURN>(s - s0);
            // A(s) -> LDS; its buffer was last read in stage s - 2, which every wave had
            // finished before the barrier of stage s - 1
            static_for<MT>([&](auto ic) {
                constexpr int I = decltype(ic)::value;
                const Split2 x = split2(sgn * ab[I][0], sgn * ab[I][1], lost),
                             y = split2(sgn * ab[I][2], sgn * ab[I][3], lost);
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
                    const Split2 x = split2(v[2 * (j % 2)], v[2 * (j % 2) + 1], lost);
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
        for (int sb = s0; sb < s1; sb += SK_D) {
            if (flip_at<SK_TURN>(sb - s0)) negate();
            static_for<SK_D>([&](auto dc) {
                if (sb + decltype(dc)::value < s1) stage(dc, sb + decltype(dc)::value);
            });
        }
        if (turn_sign<SK_TURN>(s1 - 1 - s0) < 0.0f) negate();
        bool bad = false;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) bad |= non_finite(acc[i][v]);
        if (lost_bits(lost)) lost_at = u;
        __syncthreads();  // every wave is done with the A stages; the next write follows a later barrier
        if (__any(bad) || lost_at == u) segment_f32(t, s0, s1, acc);
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
        segment(u, t, s0, s1, acc);
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

size_t gemm_small_ws_bytes(int max_rows) {
    return max_rows <= 16 ? 0 : (size_t)2 * GEMM_SK_GROUPS * (32 * min((max_rows + 31) / 32, 4)) * SK_BN * 4;
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

// ---------------------------------------------------------------- larger batches (M > 128)
// Work groups of eight waves take tiles of bm <= 64 MT rows of A times 256 rows of W:
// wave (wm, wn) owns the 32-row subtiles 2 i + wm of A (i < MT) times 64 rows of W.  K
// advances in stages of 16 floats: every thread loads its float4s of a stage one stage
// ahead, splits each element once and stores the pieces into a double-buffered LDS stage,
// so a tile's elements are fetched and split once per work group.  A stage runs in MT
// groups of 12 MFMAs (one subtile of A, two of W); the next group's operands are read, a
// share of the next stage is split and stored, under the current group's MFMAs.  The one
// barrier of a stage stands before its last group, under which the next stage's first
// operands are read.
//
// The tiles x stages units are cut into G equal contiguous ranges as above; an XCD's work
// groups take neighbouring ranges, and tiles run through eight row tiles of A before the
// next tile of W, so an XCD's L2 holds what its work groups share.  M is spread evenly over
// its row tiles (bm a multiple of 32), so no tile is mostly padding.
//
// Bound: the bf16 matrix cores at the rate this card sustains.  4096 x 6144 x 4096: 1.01 ms
// = 203 TFLOP/s, 1.22 PFLOP/s of bf16 (a library product of 8192^3: 1.26); the LDS-staged
// fp32 MFMA kernel it replaced took 1.58 ms, and 186 us against 106 at 300 rows.  At 96 and
// 128 rows gemm_small_kernel is still ahead (whole attention, T = 77: 100 against 110 us,
// 128: 121 against 126).
constexpr int GS_BN = 256;  // W rows per work group
constexpr int GS_KC = 16;   // floats of K per stage
constexpr int GS_THREADS = 512;
constexpr int GS_TURN = 8;  // stages of one accumulator sign (a multiple of 4)

struct GemmSplitArgs {
    const float* A;
    const float* W;
    const float* R;  // optional: C = R + A.W^T
    float* C;
    int M, N, K;
    int bm;          // rows of A per tile (a multiple of 32)
    int mt, nt;      // tiles along M and N
    int G;           // work groups; G = tiles: one whole tile each
    int qd, rem;     // tiles x stages = G qd + rem: the first rem ranges take qd + 1 units
    float* part;     // 2 G slots of MT x 64 x 256 floats (unused when G = tiles)
};
// row and column tile of tile t
__device__ __forceinline__ void gs_tile(const GemmSplitArgs& p, int t, int& m, int& n) {
    const int sg = t / (8 * p.nt), r = t - sg * 8 * p.nt, mw = min(8, p.mt - 8 * sg);
    m = 8 * sg + r % mw;
    n = r / mw;
}

// LDS of one stage: for A and W three pieces of two k-chunks of 8 (chunk h: floats
// 4 h .. + 3 and 8 + 4 h .. + 3 of a row, the k-slots of MFMA lane half h), each one
// 16-byte slot per row; the 64 bytes between chunks put the two chunks a wave stores at
// once on different banks.
template <int MT>
struct GsLds {
    static constexpr int CHUNK_A = MT * 64 * 16 + 64, PIECE_A = 2 * CHUNK_A;
    static constexpr int CHUNK_W = GS_BN * 16 + 64, PIECE_W = 2 * CHUNK_W;
    static constexpr int OFF_W = 3 * PIECE_A;
    static constexpr int BYTES = OFF_W + 3 * PIECE_W;
    static constexpr int NA = (MT + 1) / 2;  // float4s of A per thread and stage (the last may be half)
    static constexpr int NC = NA + 2;        // and of A and W
};

template <int MT>
__global__ __launch_bounds__(GS_THREADS, 2) void gemm_split_kernel(GemmSplitArgs p) {
    using L = GsLds<MT>;
    __shared__ __attribute__((aligned(1024))) uint8_t buf[2][L::BYTES];
    __shared__ int lost_at;  // first unit of the last range that held an inexact split
    const int tid = threadIdx.x, lane = tid % WAVE;
    const int wv = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int wm = wv / 4, wn = wv % 4;  // waves w and w + 4 share a SIMD: one of each wm
    const int lr = lane % 32, h = lane / 32;
    const int M = p.M, N = p.N, K = p.K;
    const int nst = K / GS_KC;
    const int mv = (p.bm / 32 - wm + 1) / 2;  // this wave's subtiles of A: MT or MT - 1

    // float4 i of a stage: floats 4 (tid % 4) .. + 3 of tile row 128 i + tid / 4 (A) or
    // 128 (i - NA) + tid / 4 (W)
    const int k4 = tid % 4, cr = tid / 4;
    const int dst = (k4 % 2 ? 1 : 0), sub = 8 * (k4 / 2);
    uint8_t* const wr_a = buf[0] + dst * L::CHUNK_A + cr * 16 + sub;
    uint8_t* const wr_w = buf[0] + L::OFF_W + dst * L::CHUNK_W + cr * 16 + sub;
    const uint8_t* const rd_a = buf[0] + h * L::CHUNK_A + (32 * wm + lr) * 16;
    const uint8_t* const rd_w = buf[0] + L::OFF_W + h * L::CHUNK_W + (64 * wn + lr) * 16;
    const bool a_last = 128 * (L::NA - 1) + 16 * wv < p.bm;  // this wave copies the last float4 of A

    // stages [s0, s1) of the tile at (m0, n0) on the fp32 matrix cores (non-finite operands)
    auto segment_f32 = [&](int m0, int n0, int s0, int s1, v16f_t (&acc)[MT][2]) {
        const float* w[2];
#pragma unroll
        for (int j = 0; j < 2; j++) w[j] = p.W + (size_t)min(n0 + 64 * wn + 32 * j + lr, N - 1) * K + 4 * h;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = v16f_t{};
        for (int k = s0 * GS_KC; k < s1 * GS_KC; k += 8) {
            const v4f_t b[2] = {*reinterpret_cast<const v4f_t*>(w[0] + k), *reinterpret_cast<const v4f_t*>(w[1] + k)};
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const v4f_t a = *reinterpret_cast<const v4f_t*>(
                    p.A + (size_t)min(m0 + 32 * (2 * i + wm) + lr, M - 1) * K + k + 4 * h);
#pragma unroll
                for (int c = 0; c < 4; c++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[c], b[j][c], acc[i][j], 0, 0, 0);
            }
        }
    };
    if (tid == 0) lost_at = -1;
    auto segment = [&](int u, int m0, int n0, int s0, int s1, v16f_t (&acc)[MT][2]) {
        uint32_t lost = 0;
        const uint8_t* const ab = reinterpret_cast<const uint8_t*>(p.A + (size_t)m0 * K);
        const uint8_t* const wb = reinterpret_cast<const uint8_t*>(p.W + (size_t)n0 * K);
        uint32_t off[L::NC];
        static_for<L::NC>([&](auto fc) {
            constexpr int F = decltype(fc)::value;
            const int r = F < L::NA ? min(128 * F + cr, M - 1 - m0) : min(128 * (F - L::NA) + cr, N - 1 - n0);
            off[F] = ((uint32_t)r * (uint32_t)K + 4u * (uint32_t)k4) * 4u;
        });
        v4f_t x[L::NC];
        auto load = [&](auto fc, int s) {
            constexpr int F = decltype(fc)::value;
            if (F == L::NA - 1 && !a_last) return;
            const uint8_t* base = (F < L::NA ? ab : wb) + (size_t)min(s, s1 - 1) * (GS_KC * 4);
            x[F] = *reinterpret_cast<const v4f_t*>(base + off[F]);
        };
        auto put = [&](auto fc, auto bc, int s) {  // split float4 F of stage s into buffer B
            constexpr int F = decltype(fc)::value, B = decltype(bc)::value;
            if (F == L::NA - 1 && !a_last) return;
            if constexpr (F < L::NA) x[F] *= turn_sign<GS_TURN>(s - s0);
            const Split2 a = split2(x[F][0], x[F][1], lost), b = split2(x[F][2], x[F][3], lost);
#pragma unroll
            for (int q = 0; q < 3; q++) {
                uint8_t* d = F < L::NA ? wr_a + B * L::BYTES + q * L::PIECE_A + F * 2048
                                       : wr_w + B * L::BYTES + q * L::PIECE_W + (F - L::NA) * 2048;
                *reinterpret_cast<uint2*>(d) = make_uint2(a.p[q], b.p[q]);
            }
        };
        v4i_t af[2][3], wf[2][2][3];  // [parity][piece], [parity][subtile][piece]
        auto read_a = [&](auto ic, auto bc, auto pc) {
            constexpr int I = decltype(ic)::value, B = decltype(bc)::value, P = decltype(pc)::value;
#pragma unroll
            for (int q = 0; q < 3; q++)
                af[P][q] = *reinterpret_cast<const v4i_t*>(rd_a + B * L::BYTES + q * L::PIECE_A + I * 1024);
        };
        auto read_w = [&](auto bc) {
            constexpr int B = decltype(bc)::value;
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int q = 0; q < 3; q++)
                    wf[B][j][q] = *reinterpret_cast<const v4i_t*>(rd_w + B * L::BYTES + q * L::PIECE_W + j * 512);
        };
        using C0 = std::integral_constant<int, 0>;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = v16f_t{};
        static_for<L::NC>([&](auto fc) { load(fc, s0); });
        __syncthreads();  // every wave is done with the last segment's stages
        static_for<L::NC>([&](auto fc) {
            put(fc, C0{}, s0);
            load(fc, s0 + 1);
        });
        __syncthreads();
        read_w(C0{});
        read_a(C0{}, C0{}, C0{});
        auto stage = [&](auto bc, int s) {
            constexpr int B = decltype(bc)::value, NB = 1 - B;  // buffer of stage s: s - s0 is even <=> B = 0
            static_for<MT>([&](auto ic) {
                constexpr int I = decltype(ic)::value;
                constexpr int P = (B * MT + I) & 1;  // parity of this group's A operands
                if constexpr (I == MT - 1) {
                    __syncthreads();  // stage s + 1 is in LDS, stage s is read out
                    read_w(std::integral_constant<int, NB>{});
                    read_a(C0{}, std::integral_constant<int, NB>{}, std::integral_constant<int, 1 - P>{});
                } else {
                    read_a(std::integral_constant<int, I + 1>{}, bc, std::integral_constant<int, 1 - P>{});
                    // this group's share of the next stage
                    static_for<L::NC>([&](auto fc) {
                        constexpr int F = decltype(fc)::value;
                        if constexpr (F * (MT - 1) / L::NC == I) {
                            put(fc, std::integral_constant<int, NB>{}, s + 1);
                            load(fc, s + 2);
                        }
                    });
                }
                // the small products first
                constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PW[6] = {0, 2, 1, 0, 1, 0};
                if (I < MT - 1 || mv == MT) {
#pragma unroll
                    for (int c = 0; c < 6; c++)
#pragma unroll
                        for (int j = 0; j < 2; j++) acc[I][j] = mfma_bf16(af[P][PA[c]], wf[B][j][PW[c]], acc[I][j]);
                }
                __builtin_amdgcn_sched_barrier(0);  // one group's operands and stores at a time
            });
        };
        auto negate = [&] {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = -acc[i][j];
        };
        for (int s = s0; s < s1; s += 2) {
            if (flip_at<GS_TURN>(s - s0)) negate();
            stage(C0{}, s);
            if (s + 1 < s1) stage(std::integral_constant<int, 1>{}, s + 1);
        }
        if (turn_sign<GS_TURN>(s1 - 1 - s0) < 0.0f) negate();
        bool bad = false;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) bad |= non_finite(acc[i][j][v]);
        if (lost_bits(lost)) lost_at = u;
        __syncthreads();  // the next write follows a later barrier
        if (__any(bad) || lost_at == u) segment_f32(m0, n0, s0, s1, acc);
    };

    v16f_t acc[MT][2];
    auto store = [&](int m0, int n0) {
        int r0 = m0 + 4 * h;
        lds_pin(r0);  // the row offsets are formed here, not kept across the stage loop
#pragma unroll
        for (int i = 0; i < MT; i++) {
            if (i >= mv) break;  // wave-uniform: the next tile's rows
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int col = n0 + 64 * wn + 32 * j + lr;
                if (col >= N) continue;
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int row = 32 * (2 * i + wm) + 8 * (v / 4) + r0 + v % 4;
                    if (row >= M) continue;
                    const size_t o = (size_t)row * N + col;
                    p.C[o] = p.R ? p.R[o] + acc[i][j][v] : acc[i][j][v];
                }
            }
        }
    };
    // an XCD (work groups go round robin over the eight) takes neighbouring ranges
    const int g = p.G % 8 ? (int)blockIdx.x : (int)(blockIdx.x % 8) * (p.G / 8) + (int)blockIdx.x / 8;
    const int lo = gs_lo(p, g), hi = gs_lo(p, g + 1);
    for (int u = lo; u < hi;) {
        const int t = u / nst, s0 = u - t * nst, s1 = min(nst, s0 + (hi - u));
        int m, n;
        gs_tile(p, t, m, n);
        segment(u, m * p.bm, n * GS_BN, s0, s1, acc);
        if (s0 == 0 && s1 == nst) {
            store(m * p.bm, n * GS_BN);
        } else {
            float* slot = p.part + (size_t)(2 * g + (u == lo ? 0 : 1)) * (MT * 64 * GS_BN) + tid;
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int v = 0; v < 16; v++) slot[((i * 2 + j) * 16 + v) * GS_THREADS] = acc[i][j][v];
        }
        u += s1 - s0;
    }
}

// Sum of the pieces of every cut tile, in k order (+ R): work group (t, y) takes values
// 4 y .. 4 y + 3 (value 32 i + 16 j + v) of every thread of tile t.
template <int MT>
__global__ __launch_bounds__(GS_THREADS) void gemm_split_sum_kernel(GemmSplitArgs p) {
    const int nst = p.K / GS_KC;
    const int t = blockIdx.x;
    const int u0 = t * nst, u1 = u0 + nst - 1;
    const int g0 = gs_owner(p, u0), g1 = gs_owner(p, u1);
    if (g0 == g1) return;
    const int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE, wm = wv / 4, wn = wv % 4;
    const int lr = lane % 32, h = lane / 32;
    const int i = blockIdx.y / 8, j = blockIdx.y / 4 % 2;
    if (2 * i + wm >= p.bm / 32) return;
    // the first piece is g0's last one unless g0's range starts at this tile
    const int slot0 = 2 * g0 + (gs_lo(p, g0) == u0 ? 0 : 1);
    const float* __restrict__ part = p.part + (size_t)blockIdx.y * 4 * GS_THREADS + tid;
    constexpr size_t SLOT = MT * 64 * GS_BN;
    float sum[4];
#pragma unroll
    for (int v = 0; v < 4; v++) sum[v] = part[slot0 * SLOT + v * GS_THREADS];
    for (int g = g0 + 1; g <= g1; g++)
#pragma unroll
        for (int v = 0; v < 4; v++) sum[v] += part[2 * (size_t)g * SLOT + v * GS_THREADS];
    int m, n;
    gs_tile(p, t, m, n);
    const int col = n * GS_BN + 64 * wn + 32 * j + lr;
    if (col >= p.N) return;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int row = m * p.bm + 32 * (2 * i + wm) + 8 * (blockIdx.y % 4) + 4 * h + v;
        if (row >= p.M) break;
        const size_t o = (size_t)row * p.N + col;
        p.C[o] = p.R ? p.R[o] + sum[v] : sum[v];
    }
}

template <int MT>
static hipError_t gemm_split_launch(const GemmSplitArgs& p, hipStream_t s) {
    hipLaunchKernelGGL(gemm_split_kernel<MT>, dim3(p.G), dim3(GS_THREADS), 0, s, p);
    // ranges that are whole tiles leave no pieces
    if (p.mt * p.nt % p.G != 0)
        hipLaunchKernelGGL(gemm_split_sum_kernel<MT>, dim3(p.mt * p.nt, 8 * MT), dim3(GS_THREADS), 0, s, p);
    return hipGetLastError();
}

// rows of A per tile: up to 256; half that where whole tiles have to fill the chip and would
// not twice over
static int gs_rows(int M, int N, bool ws) {
    return !ws && (int64_t)((M + 255) / 256) * ((N + GS_BN - 1) / GS_BN) < 2 * GEMM_SPLIT_GROUPS ? 128 : 256;
}

bool gemm_split_ok(int M, int N, int K, bool ws) {
    const int rows = gs_rows(M, N, ws);
    const int64_t tiles = (int64_t)((M + rows - 1) / rows) * ((N + GS_BN - 1) / GS_BN);
    // 32-bit unit counts and row offsets
    if (M <= 64 || K % GS_KC != 0 || K > (1 << 20) || tiles * (K / GS_KC) >= (1 << 30)) return false;
    return ws || tiles >= GEMM_SPLIT_GROUPS;
}

hipError_t launch_gemm_split(const float* A, const float* W, const float* R, float* C, int M, int N, int K,
                             hipStream_t s, float* ws) {
    const int rows = gs_rows(M, N, ws != nullptr);
    int mt = (M + rows - 1) / rows;
    const int nt = (N + GS_BN - 1) / GS_BN;
    const int sub = (M + 32 * mt - 1) / (32 * mt);  // 32-row subtiles of a tile
    mt = (M + 32 * sub - 1) / (32 * sub);
    const int tiles = mt * nt, U = tiles * (K / GS_KC);
    // with scratch: one work group per CU, eight stages each at least
    const int G = !ws ? tiles : U < 8 * GEMM_SPLIT_GROUPS ? (U + 7) / 8 : GEMM_SPLIT_GROUPS;
    const GemmSplitArgs p{A, W, R, C, M, N, K, 32 * sub, mt, nt, G, U / G, U % G, ws};
    switch ((sub + 1) / 2) {  // more than 64 rows: three subtiles at least
    case 2: return gemm_split_launch<2>(p, s);
    case 3: return gemm_split_launch<3>(p, s);
    default: return gemm_split_launch<4>(p, s);
    }
}

size_t gemm_split_ws_bytes(int max_rows) {
    // slots of 64 MT rows, MT pairs of 32-row subtiles (launch_gemm_split)
    const int mt = max_rows <= 64 ? 0 : max_rows > 192 ? 4 : max_rows > 128 ? 3 : 2;
    return (size_t)2 * GEMM_SPLIT_GROUPS * (64 * mt) * GS_BN * 4;
}

}  // namespace hy
