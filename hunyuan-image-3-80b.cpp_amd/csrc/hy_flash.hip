// hy_flash.hip -- attention of a prompt (more than a few queries) with online softmax, its
// two products on the bf16 matrix cores with fp32 accuracy (hy_split.hpp).
//
// One work group of eight waves per (64-query tile, kv group[, key chunk]): wave w takes
// query half w / 4 (32 queries) of head w % 4 of the group.  Blocks of 32 keys: every
// thread loads its share of a block of K and V one block ahead, splits it once and stores
// the pieces to LDS, K as it is and V transposed, both in MFMA operand order.  Scores are
// computed transposed, S^T = K Q^T (keys on MFMA rows, queries on the lanes), so a query's
// softmax statistics stay in its lane pair and the probabilities, split in registers, are
// the operand of O^T += V^T P^T as they lie.
//
// The two waves of a SIMD (the two query halves) run half a block apart: half 1 multiplies
// block kb - 1's probabilities with V while half 0 is at block kb's scores, so one's
// softmax and splits run under the other's matrix instructions.  V is kept for three
// blocks for that, K for two (126 KB of LDS at head_dim 128).
//
// Bound: the bf16 matrix cores at the rate this card sustains.  T = 4096, 32 / 8 heads of 128,
// causal: 0.68 ms, 1.2 PFLOP/s of bf16; four waves per 32 queries on the fp32 MFMAs took
// 1.19 ms.  T = 1000: 64 us (109).  Up to about 100 keys a launch is 10 us of start-up
// (code and operands fetched once) and 2 to 4 per block.
//
// Values without a split (infinities, NaNs, values that round up to infinity in bf16)
// leave a non-finite sum: such a wave computes its keys again on the fp32 matrix cores.
// So do the waves that met a q, k or v too small for an exact split.  The probabilities
// are taken 2^40 times too large, which keeps the split of each of them exact (they are 0 or
// at least 2^-126, the split needs 2^-110); the sum of the values and the sum of the
// probabilities carry the factor alike.
#include "hy_device.hpp"
#include "hy_launch.hpp"
#include "hy_lds.hpp"
#include "hy_split.hpp"

namespace hy {

constexpr int FS_TURN = 4;  // key blocks of one accumulator sign
constexpr float FS_PSCALE = 0x1p40f;  // of the probabilities

template <int HD>
struct FsLds {
    // K: per piece HD / 8 chunks (chunk 2 c + h: floats 16 c + 4 h .. + 3 and 16 c + 8 +
    // 4 h .. + 3, the k-slots of MFMA lane half h in step c) of 32 keys x 16 bytes; the 32
    // bytes between chunks put the chunks a wave stores at once on different banks
    static constexpr int CHUNK_K = 32 * 16 + 32, PIECE_K = HD / 8 * CHUNK_K, BUF_K = 3 * PIECE_K;
    // V: per piece 4 chunks (2 c + h: keys in the same order) of HD dims x 16 bytes
    static constexpr int CHUNK_V = HD * 16, PIECE_V = 4 * CHUNK_V, BUF_V = 3 * PIECE_V;
    static constexpr int OFF_V = 2 * BUF_K;
    static constexpr int BYTES = OFF_V + 3 * BUF_V;
};

template <int HD>
__global__ __launch_bounds__(512, 2) void flash_split_kernel(FlashArgs a) {
    using L = FsLds<HD>;
    constexpr int NC = HD / 16;  // k-steps of the scores
    constexpr int ND = HD / 32;  // 32-dim tiles of the output
    constexpr int NK = HD / 64;  // float4s of K, and dims of V, per thread and block
    __shared__ __attribute__((aligned(1024))) uint8_t lds[L::BYTES];
    __shared__ int lost_s;  // an inexact split of K or V
    const int tid = threadIdx.x, lane = tid % WAVE;
    const int wv = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int lr = lane % 32, h = lane / 32;
    const int half = wv / 4, hw = wv % 4;  // waves w and w + 4 share a SIMD
    const int n_qt = (a.T + 63) / 64;
    // chunk-major, and inside a chunk the longest (causal) query tiles first
    const int per_chunk = n_qt * a.nkv;
    const int chunk = (int)blockIdx.x / per_chunk, rem = (int)blockIdx.x % per_chunk;
    const int qt = n_qt - 1 - rem / a.nkv, g = rem % a.nkv;
    const int head = g * 4 + hw;
    const int qw = qt * 64 + half * 32;  // this wave's first query
    const int qrow = min(qw + lr, a.T - 1);

    // key blocks the 32 queries from q0 see: all, or (causal) keys <= q_pos0 + q
    auto blocks = [&](int q0) {
        const int end = a.causal ? min(a.kv_len, a.q_pos0 + min(q0 + 31, a.T - 1) + 1) : a.kv_len;
        return q0 < a.T ? (end + 31) / 32 : 0;
    };
    const int nblk = max(blocks(qt * 64), blocks(qt * 64 + 32)), my_nblk = blocks(qw);
    // this work group's blocks: all of them, or chunk `chunk` of cb blocks; the wave's part
    const int kb0 = a.cb ? chunk * a.cb : 0, kb1 = a.cb ? min(nblk, kb0 + a.cb) : nblk;
    if (kb0 >= nblk) return;  // whole work group: the tile has fewer chunks
    const int my_kb1 = min(my_nblk, kb1);

    // K: float4 4 (tid % (HD / 4)) of keys tid / (HD / 4) + KR i; V: keys 4 vg .. + 3 of
    // dims vd + 32 i
    constexpr int KR = 512 / (HD / 4);
    const float* const kg = a.k + (size_t)g * a.L * HD;
    const float* const vg_ = a.v + (size_t)g * a.L * HD;
    const int k4 = tid % (HD / 4), kr = tid / (HD / 4);
    const int vch = wv % 4, vsub = lane / 32, vd = NK * 32 * (wv / 4) + lane % 32;
    const int vkey = 16 * (vch / 2) + 8 * vsub + 4 * (vch % 2);
    uint8_t* const k_dst = lds + (2 * (k4 / 4) + k4 % 2) * L::CHUNK_K + kr * 16 + 8 * (k4 / 2 % 2);
    uint8_t* const v_dst = lds + L::OFF_V + vch * L::CHUNK_V + vd * 16 + 8 * vsub;
    v4f_t kx[NK], vx[NK];
    auto load_k = [&](int kb) {
#pragma unroll
        for (int i = 0; i < NK; i++) {
            const int key = min(kb * 32 + kr + KR * i, a.kv_len - 1);  // in bounds
            kx[i] = *reinterpret_cast<const v4f_t*>(kg + (size_t)key * HD + 4 * k4);
        }
    };
    auto load_v = [&](int kb) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float* row = vg_ + (size_t)min(kb * 32 + vkey + j, a.kv_len - 1) * HD + vd;
#pragma unroll
            for (int i = 0; i < NK; i++) vx[i][j] = row[32 * i];
        }
    };
    uint32_t lost = 0;
    if (tid == 0) lost_s = 0;
    auto put = [&](uint8_t* dst, int piece, v4f_t x) {
        const Split2 s = split2(x[0], x[1], lost), t = split2(x[2], x[3], lost);
#pragma unroll
        for (int q = 0; q < 3; q++) *reinterpret_cast<uint2*>(dst + q * piece) = make_uint2(s.p[q], t.p[q]);
    };
    auto put_k = [&](int kb) {
        uint8_t* const d = k_dst + (kb & 1) * L::BUF_K;
#pragma unroll
        for (int i = 0; i < NK; i++) put(d + KR * 16 * i, L::PIECE_K, kx[i]);
    };
    auto put_v = [&](int kb) {
        const float sgn = turn_sign<FS_TURN>(kb - kb0);
        uint8_t* const d = v_dst + (kb % 3) * L::BUF_V;
#pragma unroll
        for (int i = 0; i < NK; i++) put(d + 512 * i, L::PIECE_V, vx[i] * sgn);
    };

    load_k(kb0);
    load_v(kb0);
    __builtin_amdgcn_sched_barrier(0);  // in flight while Q is read and split

    // Q: lane (query lr, half h) holds the pieces of floats 16 c + 4 h .. + 3 and 16 c + 8 +
    // 4 h .. + 3, pre-multiplied by scale * log2(e): the scores come out in the base-2
    // domain, where the softmax uses the hardware 2^x (2^-inf = 0 serves the masked keys)
    const float qscale = a.scale * 1.4426950408889634f;
    const float* const qp = a.q + ((size_t)qrow * a.nh + head) * HD;
    v4i_t qf[NC][3];
    uint32_t q_lost = 0;
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const v4f_t x = *reinterpret_cast<const v4f_t*>(qp + 16 * c + 8 * u + 4 * h) * qscale;
            const Split2 s = split2(x[0], x[1], q_lost), t = split2(x[2], x[3], q_lost);
#pragma unroll
            for (int q = 0; q < 3; q++) {
                qf[c][q][2 * u] = (int)s.p[q];
                qf[c][q][2 * u + 1] = (int)t.p[q];
            }
        }

    v16f_t o[ND];
    float m_run, l_run;
    const int my_q = a.q_pos0 + qw + lr;  // key index of this lane's query (causal bound)
    constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};  // the small products first
    v4i_t pf[2][3];  // the probabilities' pieces, keys 16 c .. in step c

    auto mask = [&](int kb, v16f_t& s) {
        // only blocks that reach past the wave's first query or past kv_len
        if (kb * 32 + 31 >= a.kv_len || (a.causal && kb * 32 + 31 > a.q_pos0 + qw)) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int key = kb * 32 + 8 * (v / 4) + 4 * h + v % 4;
                if (key >= a.kv_len || (a.causal && key > my_q)) s[v] = -INFINITY;
            }
        }
    };
    // online softmax over this lane pair's 32 keys; s becomes the probabilities times pscale
    auto softmax = [&](v16f_t& s, float pscale) {
        float mloc = s[0];
#pragma unroll
        for (int v = 1; v < 16; v++) mloc = fmaxf(mloc, s[v]);
        mloc = fmaxf(mloc, __shfl_xor(mloc, 32, WAVE));
        // every processed block leaves at least one visible key per query: m_new is finite
        const float m_new = fmaxf(m_run, mloc);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);  // 0 for the first block
        float psum = 0.0f;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            s[v] = __builtin_amdgcn_exp2f(s[v] - m_new) * pscale;
            psum += s[v];
        }
        psum += __shfl_xor(psum, 32, WAVE);
        l_run = l_run * alpha + psum;
        m_run = m_new;
        return alpha;
    };
    auto rescale = [&](float alpha) {
        if (__ballot(alpha != 1.0f)) {  // the running max moved for some query
#pragma unroll
            for (int d = 0; d < ND; d++) o[d] *= alpha;
        }
    };
    // scores of block kb and its probabilities' pieces; returns the factor of o
    auto scores = [&](int kb) {
        const uint8_t* const kb_ = lds + (kb & 1) * L::BUF_K + h * L::CHUNK_K + lr * 16;
        v4i_t kf[2][3];  // the next step's reads run under this one's products
        auto read = [&](int c) {
#pragma unroll
            for (int q = 0; q < 3; q++)
                kf[c & 1][q] = *reinterpret_cast<const v4i_t*>(kb_ + q * L::PIECE_K + 2 * c * L::CHUNK_K);
        };
        v16f_t s = v16f_t{};
        read(0);
#pragma unroll
        for (int c = 0; c < NC; c++) {
            if (c + 1 < NC) read(c + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 6; i++) s = mfma_bf16(kf[c & 1][PA[i]], qf[c][PB[i]], s);
            __builtin_amdgcn_sched_barrier(0);
        }
        mask(kb, s);
        const float alpha = softmax(s, FS_PSCALE);
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                uint32_t none = 0;  // exact
                const Split2 t = split2(s[8 * c + 2 * j], s[8 * c + 2 * j + 1], none);
#pragma unroll
                for (int q = 0; q < 3; q++) pf[c][q][j] = (int)t.p[q];
            }
        return alpha;
    };
    auto values = [&](int kb, float alpha) {
        if (flip_at<FS_TURN>(kb - kb0)) alpha = -alpha;  // V's sign turned with block kb
        rescale(alpha);
        const uint8_t* const vb = lds + L::OFF_V + (kb % 3) * L::BUF_V + h * L::CHUNK_V + lr * 16;
        v4i_t vf[2][3];
        auto read = [&](int i) {  // dims 32 (i % ND) .. of step i / ND
#pragma unroll
            for (int q = 0; q < 3; q++)
                vf[i & 1][q] = *reinterpret_cast<const v4i_t*>(vb + q * L::PIECE_V + 2 * (i / ND) * L::CHUNK_V +
                                                               512 * (i % ND));
        };
        read(0);
#pragma unroll
        for (int i = 0; i < 2 * ND; i++) {
            if (i + 1 < 2 * ND) read(i + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 6; j++) o[i % ND] = mfma_bf16(vf[i & 1][PA[j]], pf[i / ND][PB[j]], o[i % ND]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto reset = [&] {
#pragma unroll
        for (int d = 0; d < ND; d++) o[d] = v16f_t{};
        m_run = -INFINITY;
        l_run = 0.0f;
    };

    reset();
    put_k(kb0);
    load_k(kb0 + 1);  // blocks past the last key re-read it
    float alpha = 1.0f;
    for (int kb = kb0; kb < kb1; kb++) {
        put_v(kb);
        load_v(kb + 1);
        __syncthreads();  // block kb is in LDS; K of block kb - 1 and V of kb - 2 are read out
        if (half == 1 && kb > kb0 && kb - 1 < my_kb1) values(kb - 1, alpha);
        if (kb < my_kb1) alpha = scores(kb);
        if (kb + 1 < kb1) put_k(kb + 1);
        load_k(kb + 2);
        if (half == 0 && kb < my_kb1) values(kb, alpha);
    }
    if (lost_bits(lost)) lost_s = 1;
    __syncthreads();
    if (kb0 >= my_kb1) return;
    if (half == 1 && my_kb1 == kb1) values(kb1 - 1, alpha);
    if (turn_sign<FS_TURN>(my_kb1 - 1 - kb0) < 0.0f) {
#pragma unroll
        for (int d = 0; d < ND; d++) o[d] = -o[d];
    }
    bool bad = non_finite(l_run) || lost_bits(q_lost) || lost_s;
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
        for (int v = 0; v < 16; v++) bad |= non_finite(o[d][v]);
    float unscale = 1.0f / FS_PSCALE;
    if (__any(bad)) {  // again on the fp32 matrix cores, K and V straight from memory
        unscale = 1.0f;
        reset();
        for (int kb = kb0; kb < my_kb1; kb++) {
            const float* const k = kg + (size_t)min(kb * 32 + lr, a.kv_len - 1) * HD + 4 * h;
            v16f_t s = v16f_t{};
            for (int d = 0; d < HD; d += 8) {
                const v4f_t kx = *reinterpret_cast<const v4f_t*>(k + d);
                const v4f_t qx = *reinterpret_cast<const v4f_t*>(qp + d + 4 * h) * qscale;
#pragma unroll
                for (int j = 0; j < 4; j++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[j], qx[j], s, 0, 0, 0);
            }
            mask(kb, s);
            rescale(softmax(s, 1.0f));
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int key = min(kb * 32 + 8 * (v / 4) + 4 * h + v % 4, a.kv_len - 1);
#pragma unroll
                for (int d = 0; d < ND; d++)
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vg_[(size_t)key * HD + 32 * d + lr], s[v], o[d], 0, 0,
                                                                0);
            }
        }
    }
    if (a.cb && my_nblk > a.cb) {
        // partial result of this chunk: unnormalised O^T, running max and sum
        float* pp = a.part + ((size_t)(((2 * qt + half) * a.nch + chunk) * a.nkv + g) * 4 + hw) * (HD * 32 + 128);
#pragma unroll
        for (int d = 0; d < ND; d++)
#pragma unroll
            for (int v = 0; v < 16; v++) pp[(d * 16 + v) * 64 + lane] = o[d][v] * unscale;
        pp[HD * 32 + lane] = m_run;
        pp[HD * 32 + 64 + lane] = l_run * unscale;
        return;
    }
    if (qw + lr >= a.T) return;
    const float inv = 1.0f / l_run;
    float* op = a.out + ((size_t)(qw + lr) * a.nh + head) * HD;
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
        for (int v = 0; v < 4; v++)
            *reinterpret_cast<float4*>(op + 32 * d + 8 * v + 4 * h) = make_float4(
                o[d][4 * v] * inv, o[d][4 * v + 1] * inv, o[d][4 * v + 2] * inv, o[d][4 * v + 3] * inv);
}

hipError_t launch_flash_split(const FlashArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)((a.T + 63) / 64 * a.nkv * a.nch));
    if (a.hd == 128)
        hipLaunchKernelGGL(flash_split_kernel<128>, grid, dim3(512), 0, s, a);
    else if (a.hd == 64)
        hipLaunchKernelGGL(flash_split_kernel<64>, grid, dim3(512), 0, s, a);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace hy
