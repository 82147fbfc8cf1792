// Causal attention of a batch of prompt tokens against the KV cache (query m attends to cache rows 0 .. pos0 + m), for
// heads of 64, 128 and 256 dimensions and contexts of any length: one pass over the keys with a running maximum.
//
// Rounding points of the reference (llama2_q4.cu:410-427) that survive the one pass: scores are rounded to fp16, sums of
// exponentials and of P V are fp32, the output is fp16.  The probability itself is rounded to fp16 before the division by
// the row's sum instead of after it (the same relative step; small probabilities no longer become fp16 denormals).
// One that does not: below 1024 positions the reference, and with it the token-by-token path, starts a row's maximum from 0
// (the lanes of its block that hold no score).  Exponentials of a row whose scores all lie below -87 are then fp32 denormals,
// below about -104 all zero and the output 0 / 0; here the maximum is that of the scores, and such rows
// come out as any other.
#include <atomic>

#include "common.hpp"
#include "gemm_tile.hpp"

typedef short s16x4 __attribute__((ext_vector_type(4)));

namespace pfa {

// Eight halves of a column: two transposed reads of 4 rows each.  ds_read_b64_tr_b16 hands lane l of a group of 16
// column l of the 4 x 16 block whose row i / 4 the group's lanes i name, four columns a lane.
__device__ __forceinline__ h16x8 read_tr8(const uint16_t* p0, const uint16_t* p1) {
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)p0);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)p1);
    return __builtin_bit_cast(h16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// One query by one wave, for blocks with values that are not finite: only the keys it sees take part.  Bound by the round trips
// of its loads; with 16 bytes of a key a lane and 8 value rows in flight, a 2000-token pass over two 7B layers whose every value
// row is infinite somewhere takes 12.7 ms (46.6 with 2 bytes at a time; 1.9 where all values are finite).
// FRAG: `out` is the whole block in fragment order (gemm_tile.hpp) of `tiles` 32-row tiles, in which the query's columns are those
// of row `row` from `col0` on.
template <int HS, bool FRAG>
__device__ __forceinline__ void attn_row(uint16_t* out, const uint16_t* q, const uint16_t* kh, const uint16_t* vh, size_t kv_dim,
                                         int keys, float alpha, int out_perm, int row, int col0, int tiles) {
    constexpr int D = HS / 64;
    const int lane = threadIdx.x & 63;
    float o[D], m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int d = 0; d < D; d++) o[d] = 0.0f;
#pragma unroll 1
    for (int t0 = 0; t0 < keys; t0 += 64) {
        float s = 0.0f;
        const uint16_t* k = kh + (size_t)min(t0 + lane, keys - 1) * kv_dim;
#pragma unroll 4
        for (int i = 0; i < HS; i += 8) {
            const u32x4 qv = *reinterpret_cast<const u32x4*>(q + i), kv = *reinterpret_cast<const u32x4*>(k + i);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const h16x2 a = as_h2(qv[e]), b = as_h2(kv[e]);
                s = fmaf((float)a[0], (float)b[0], s);
                s = fmaf((float)a[1], (float)b[1], s);
            }
        }
        s = t0 + lane < keys ? half_bits_to_float(float_to_half_bits(s * alpha)) : -INFINITY;
        const float m_new = fmaxf(m, wave_max(s));
        const float f = m_new == -INFINITY ? 1.0f : expf(m - m_new);
        const float e = expf(s - (m_new == -INFINITY ? 0.0f : m_new));
        m = m_new;
        l = fmaf(l, f, wave_sum(e));
        const float p = half_bits_to_float(float_to_half_bits(e));
#pragma unroll
        for (int d = 0; d < D; d++) o[d] *= f;
#pragma unroll 1
        for (int i = 0; i < 64 && t0 + i < keys; i += 8) {
            uint16_t v[8][D];
#pragma unroll
            for (int j = 0; j < 8; j++)
#pragma unroll
                for (int d = 0; d < D; d++) v[j][d] = vh[(size_t)min(t0 + i + j, keys - 1) * kv_dim + d * 64 + lane];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float pi = __shfl(p, i + j);
                if (t0 + i + j < keys) {
#pragma unroll
                    for (int d = 0; d < D; d++) o[d] = fmaf(pi, half_bits_to_float(v[j][d]), o[d]);
                }
            }
        }
    }
    const int at = out_perm ? (lane & 56) | ((lane & 3) << 1) | ((lane >> 2) & 1) : lane;  // (0,4,1,5,2,6,3,7)
#pragma unroll
    for (int d = 0; d < D; d++) {
        out[FRAG ? pf::fragment_offset(row, col0 + d * 64 + at, tiles) : d * 64 + at] = float_to_half_bits(o[d] / l);
    }
}

// A workgroup owns 32 * QW consecutive query tokens of one head: wave (qs, ks) takes the qs-th 32 queries and, of every
// tile of 32 * NSUB * KW keys, the ks-th NSUB blocks of 32.
//  * S^T = K Q^T: with the queries as columns a lane holds 16 scores of ONE query, so the row statistics are in-lane
//    reductions and one half swap, and the probabilities leave the exponential as the second product's operand: the key
//    order of an accumulator (8 (j/4) + 4 (lane/32) + j%4) is taken for the contraction, and the value fragments are read
//    from LDS in that order, transposed by the LDS itself.
//  * The accumulated output is rescaled only when some row's maximum grows by more than 5 (a factor of e^5 is nothing to
//    fp16 or fp32): rarely after the first tiles where scores are within a few units of each other, again and again where
//    they spread over tens.
//  * K and V tiles travel through registers into LDS one tile ahead (BUF buffers; rows padded so that fragment reads and
//    transposed reads are free of bank conflicts).
//  * The matrix product gives queries zero times the values past them, which is NaN where such a value is not finite: blocks
//    that staged one past their first query do their queries one by one instead (attn_row).  Looking for them costs 512
//    tokens x 32 heads 14.2 -> 15.1 us (under the profiler).
//  * KW > 1: the key slices' (maximum, sum, output) meet in LDS at the end.
// What bounds it: the vector instructions between the two products (about 10 per score, an exponential among them, against
// two matrix instructions per 16 scores of a lane); with two workgroups per compute unit one's products run under the
// other's exponentials.  The form before this one held whole score rows in LDS (three passes, 32 queries per workgroup, at
// most 1920 keys): 512 tokens x 32 heads 17.3 -> 13.2 us, 1920 tokens 97 us for the last 512 alone -> 63 us for all 2000;
// heads of 64 and 256 dimensions ran without matrix cores (700 tokens x 32 heads of 64: 278 -> 12.3 us).
template <int HS, int QW, int KW, int NSUB, int BUF, bool FRAG>
__global__ __launch_bounds__(QW * KW * 64, HS == 256 ? 1 : 2) void attn_kernel(uint16_t* out, const uint16_t* q, const uint16_t* key_cache,
                                                                             const uint16_t* value_cache, int num_heads, int kv_mul, int M,
                                                                             int pos0, int out_perm, int tiles) {
    constexpr int NT = QW * KW * 64;
    constexpr int TK = 32 * NSUB * KW;
    constexpr int KS = HS + 8, VS = HS + 16;  // halves per tile row: row strides of 4 and 8 dwords modulo the 32 banks
    constexpr int NP = TK * HS / 8 / NT;      // 16-byte pieces of each tile per thread
    constexpr int NB = HS / 32;
    constexpr float LOG2E = 1.4426950408889634f;
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    uint16_t* Kt = smem;                  // [BUF][TK][KS]
    uint16_t* Vt = smem + BUF * TK * KS;  // [BUF][TK][VS]

    // All query blocks of a head run on one XCD (workgroup ids go round-robin over the 8), neighbouring heads (which share
    // K and V under grouped queries) too.  Blocks go longest first; where all of an XCD's blocks are resident at once the
    // second half goes shortest first, so that a compute unit's two are one long and one short.
    const int nqb = (M + 32 * QW - 1) / (32 * QW), hpx = (num_heads + 7) >> 3;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int rank = slot / hpx, h = xcd * hpx + slot % hpx;
    if (h >= num_heads) return;
    const int qb = (hpx * nqb <= 64 && rank * 2 >= nqb) ? rank - (nqb + 1) / 2 : nqb - 1 - rank;
    const int mq0 = qb * 32 * QW;
    const int nk = pos0 + min(mq0 + 32 * QW, M);  // keys visible to the block's last query
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qs = wave % QW, ks = wave / QW;
    const int l32 = lane & 31, lh = lane >> 5;
    const size_t kv_dim = (size_t)num_heads / kv_mul * HS;
    const float alpha = (float)(1.0 / sqrt((double)HS));
    const uint16_t* kh = key_cache + (size_t)(h / kv_mul) * HS;
    const uint16_t* vh = value_cache + (size_t)(h / kv_mul) * HS;

    const int mq = mq0 + qs * 32;             // the wave's first query
    const bool live = mq < M;                 // (the others only help to stage)
    const int qpos = pos0 + mq + l32;         // the lane's query position
    const int qlast = pos0 + min(mq + 31, M - 1);

    u32x4 kr[NP], vr[NP];
    auto load = [&](int t0) {  // unconditional, rows past the end clamped
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int idx = i * NT + tid;
            const size_t row = (size_t)min(t0 + idx / (HS / 8), nk - 1) * kv_dim + (idx % (HS / 8)) * 8;
            kr[i] = *reinterpret_cast<const u32x4*>(kh + row);
            vr[i] = *reinterpret_cast<const u32x4*>(vh + row);
        }
    };
    uint32_t wild = 0;  // bits 15 and 31: a value that is not finite (an exponent of all ones carries) in a tile on the diagonal
    auto store = [&](int t0, int buf) {
#pragma unroll
        for (int i = 0; i < NP; i++) {
            const int idx = i * NT + tid;
            const int row = idx / (HS / 8), c = idx % (HS / 8);
            *reinterpret_cast<u32x4*>(Kt + (buf * TK + row) * KS + c * 8) = kr[i];
            *reinterpret_cast<u32x4*>(Vt + (buf * TK + row) * VS + c * 8) = vr[i];
        }
        if (t0 + TK > pos0 + mq0) {
#pragma unroll
            for (int i = 0; i < NP; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) wild |= (vr[i][e] & 0x7C007C00u) + 0x04000400u;
        }
    };
    load(0);
    h16x8 qf[HS / 16];
    {
        const uint16_t* qrow = q + ((size_t)min(mq + l32, M - 1) * num_heads + h) * HS + lh * 8;
#pragma unroll
        for (int f = 0; f < HS / 16; f++) qf[f] = *reinterpret_cast<const h16x8*>(qrow + f * 16);
    }
    f32x16 o[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int j = 0; j < 16; j++) o[b][j] = 0.0f;
    float m_ref = -INFINITY, l = 0.0f;  // l: the lane's own share of the row's sum (its half of each block's keys)

    auto compute = [&](int t0, int buf) {
        const int kb = ks * NSUB * 32;  // the wave's first row of the tile
        if (!live || t0 + kb > qlast) return;
        const uint16_t* kt = Kt + (buf * TK + kb + l32) * KS + lh * 8;
        f32x16 s[NSUB];
#pragma unroll
        for (int u = 0; u < NSUB; u++) {
#pragma unroll
            for (int j = 0; j < 16; j++) s[u][j] = 0.0f;
#pragma unroll
            for (int f = 0; f < HS / 16; f++) {
                const h16x8 kf = *reinterpret_cast<const h16x8*>(kt + u * 32 * KS + f * 16);
                s[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[f], s[u], 0, 0, 0);
            }
        }
        float tmax = -INFINITY;
#pragma unroll
        for (int u = 0; u < NSUB; u++)
#pragma unroll
            for (int j = 0; j < 16; j++) s[u][j] = (float)(h16_t)(s[u][j] * alpha);
        if (t0 + kb + 32 * NSUB - 1 > pos0 + mq) {  // some key of the block lies past some query
#pragma unroll
            for (int u = 0; u < NSUB; u++)
#pragma unroll
                for (int j = 0; j < 16; j++)
                    if (t0 + kb + u * 32 + (j >> 2) * 8 + lh * 4 + (j & 3) > qpos) s[u][j] = -INFINITY;
        }
#pragma unroll
        for (int u = 0; u < NSUB; u++)
#pragma unroll
            for (int j = 0; j < 16; j++) tmax = fmaxf(tmax, s[u][j]);
        float other = tmax;
        swap32(tmax, other);
        tmax = fmaxf(tmax, other);
        if (__builtin_amdgcn_ballot_w64(tmax > m_ref + 5.0f)) {
            const float m_new = fmaxf(m_ref, tmax);
            const float f = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f((m_ref - m_new) * LOG2E);
            m_ref = m_new;
            l *= f;
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int j = 0; j < 16; j++) o[b][j] *= f;
        }
        const float mL = m_ref == -INFINITY ? 0.0f : m_ref * LOG2E;  // (a row that has seen no key yet: all scores are -inf)
        h16x8 p[NSUB][2];
#pragma unroll
        for (int u = 0; u < NSUB; u++)
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const float e = __builtin_amdgcn_exp2f(fmaf(s[u][j], LOG2E, -mL));
                l += e;
                p[u][j >> 3][j & 7] = (h16_t)e;
            }
        const uint16_t* vt = Vt + (buf * TK + kb + lh * 4 + ((lane & 15) >> 2)) * VS + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
#pragma unroll
        for (int u = 0; u < NSUB; u++)
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    const uint16_t* p0 = vt + (u * 32 + t * 16) * VS + b * 32;
                    o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(read_tr8(p0, p0 + 8 * VS), p[u][t], o[b], 0, 0, 0);
                }
    };

    const int ntiles = (nk + TK - 1) / TK;
    store(0, 0);
    __syncthreads();
    for (int it = 0; it < ntiles; it++) {
        const int t0 = it * TK;
        load(t0 + TK);  // (past the end: the last row again)
        if (BUF == 2) {
            compute(t0, it & 1);
            store(t0 + TK, (it + 1) & 1);
        } else {
            compute(t0, 0);
            __syncthreads();
            store(t0 + TK, 0);
        }
        __syncthreads();
    }
    if (__syncthreads_or((wild & 0x80008000u) != 0)) {
        for (int m = mq0 + wave; m < min(mq0 + 32 * QW, M); m += QW * KW)
            attn_row<HS, FRAG>(FRAG ? out : out + ((size_t)m * num_heads + h) * HS, q + ((size_t)m * num_heads + h) * HS, kh, vh, kv_dim, pos0 + m + 1, alpha, out_perm,
                               m, h * HS, tiles);
        return;
    }
    {
        float other = l;
        swap32(l, other);
        l += other;
    }
    if (KW > 1) {
        // every slice but the first hands over (o, maximum, sum) through the idle tiles, a register of all lanes per row
        constexpr int W = NB * 16 + 2;
        float* meet = reinterpret_cast<float*>(smem) + lane;
        if (ks > 0) {
            float* mine = meet + ((ks - 1) * QW + qs) * W * 64;
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int j = 0; j < 16; j++) mine[(b * 16 + j) * 64] = o[b][j];
            mine[NB * 16 * 64] = m_ref;
            mine[(NB * 16 + 1) * 64] = l;
        }
        __syncthreads();
        if (ks > 0) return;
        float m_all = m_ref;
#pragma unroll
        for (int k = 1; k < KW; k++) m_all = fmaxf(m_all, meet[(((k - 1) * QW + qs) * W + NB * 16) * 64]);
        // (the first slice of a live row always saw key 0, so m_all is finite there)
        float f = __builtin_amdgcn_exp2f((m_ref - m_all) * LOG2E);
        l *= f;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int j = 0; j < 16; j++) o[b][j] *= f;
#pragma unroll
        for (int k = 1; k < KW; k++) {
            const float* theirs = meet + ((k - 1) * QW + qs) * W * 64;
            f = __builtin_amdgcn_exp2f((theirs[NB * 16 * 64] - m_all) * LOG2E);
            l = fmaf(theirs[(NB * 16 + 1) * 64], f, l);
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int j = 0; j < 16; j++) o[b][j] = fmaf(theirs[(b * 16 + j) * 64], f, o[b][j]);
        }
    }
    if (!live || mq + l32 >= M) return;
    // A lane holds 4 of every 8 output dimensions of its query, lane ^ 32 the other 4: one half swap leaves each with whole
    // pieces of 8 (the even ones in the lower half of the wave, the odd ones in the upper).
    const float inv = 1.0f / l;
    uint16_t* orow = out + ((size_t)(mq + l32) * num_heads + h) * HS + lh * 8;
    auto pack2 = [&](float a, float b) {
        h16x2 r;
        r[0] = (h16_t)(a * inv);
        r[1] = (h16_t)(b * inv);
        return __builtin_bit_cast(float, r);
    };
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int g = 0; g < 4; g += 2) {
            float x0 = pack2(o[b][4 * g], o[b][4 * g + 1]), x1 = pack2(o[b][4 * g + 2], o[b][4 * g + 3]);
            float y0 = pack2(o[b][4 * g + 4], o[b][4 * g + 5]), y1 = pack2(o[b][4 * g + 6], o[b][4 * g + 7]);
            swap32(x0, y0);
            swap32(x1, y1);
            const uint32_t a0 = __builtin_bit_cast(uint32_t, x0), a1 = __builtin_bit_cast(uint32_t, x1);
            const uint32_t b0 = __builtin_bit_cast(uint32_t, y0), b1 = __builtin_bit_cast(uint32_t, y1);
            u32x4 r;
            if (out_perm) {  // (0,4,1,5,2,6,3,7)
                r[0] = __builtin_amdgcn_perm(b0, a0, 0x05040100u);
                r[1] = __builtin_amdgcn_perm(b0, a0, 0x07060302u);
                r[2] = __builtin_amdgcn_perm(b1, a1, 0x05040100u);
                r[3] = __builtin_amdgcn_perm(b1, a1, 0x07060302u);
            } else {
                r = u32x4{a0, a1, b0, b1};
            }
            *reinterpret_cast<u32x4*>(FRAG ? out + pf::fragment_offset(mq + l32, h * HS + lh * 8 + b * 32 + g * 8, tiles) : orow + b * 32 + g * 8) = r;
        }
}

template <int HS, int QW, int KW, int NSUB, int BUF, bool FRAG>
int launch(awq_ctx* ctx, uint16_t* out, const uint16_t* q, const uint16_t* kc, const uint16_t* vc, int nh, int kv_mul, int M, int pos0,
           int out_perm, int tiles) {
    constexpr int TK = 32 * NSUB * KW;
    constexpr int staged = BUF * TK * (2 * HS + 24) * 2;
    constexpr int meet = (KW - 1) * QW * (HS / 2 + 2) * 256;
    constexpr int lds = staged > meet ? staged : meet;
    static std::atomic<bool> raised[64];  // per device: the kernel may take more than the default 64 KB of LDS
    if (lds > 64 * 1024 && !(ctx->device < 64 && raised[ctx->device].load(std::memory_order_relaxed))) {
        const hipError_t e = hipFuncSetAttribute((const void*)attn_kernel<HS, QW, KW, NSUB, BUF, FRAG>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) {
            awq_set_error("hipFuncSetAttribute(attn_prefill) failed: %s", hipGetErrorString(e));
            return AWQ_ERR_HIP;
        }
        if (ctx->device < 64) raised[ctx->device].store(true, std::memory_order_relaxed);
    }
    const int nqb = div_up(M, 32 * QW), hpx = (nh + 7) / 8;
    hipLaunchKernelGGL((attn_kernel<HS, QW, KW, NSUB, BUF, FRAG>), dim3(8 * hpx * nqb), dim3(QW * KW * 64), lds, ctx->stream, out, q, kc, vc, nh,
                       kv_mul, M, pos0, out_perm, tiles);
    return awq_check_launch("attn_prefill");
}

}  // namespace pfa

// tiles: 32-row tiles of an output in fragment order, 0: rows
int awq_launch_attn_prefill(awq_ctx* ctx, uint16_t* out, const uint16_t* q, const uint16_t* kc, const uint16_t* vc, int nh, int hs,
                            int kv_mul, int M, int pos0, int out_perm, int tiles) {
#define AWQ_FORM(HS, QW, KW, NSUB, BUF)                                                                                      \
    return tiles ? pfa::launch<HS, QW, KW, NSUB, BUF, true>(ctx, out, q, kc, vc, nh, kv_mul, M, pos0, out_perm, tiles)      \
                 : pfa::launch<HS, QW, KW, NSUB, BUF, false>(ctx, out, q, kc, vc, nh, kv_mul, M, pos0, out_perm, 0)
    // Measured, us (128 queries x all keys | 64 queries x 2 key slices | 32 queries x 4 key slices, per workgroup):
    //   32 heads of 128: 512 tokens 16.9 | 13.2 | 14.1;  2000 tokens 62.6 | 68.5 | 99;  37 tokens 4.9 | 6.5 | 6.9, behind
    //   1500 cached ones 38 | 28 | 24;  64 heads: 650 tokens 24.9 | 26.0 | 36.6, 150 behind 650 24.2 | 18.8 | 22.5
    //   32 heads of 64: 700 tokens 15.6 | 12.3 | 12.0, 1500 tokens 32.5 | 27.9 | 30.0
    // Hence: the widest form where it alone gives every compute unit a workgroup (each K and V tile then serves 128
    // queries) and where all keys are one tile; the four-slice form where queries are few and keys many; the middle one
    // otherwise.  256-wide heads have registers for the middle form with one block per wave only (4 x 1: 30.5, 2 x 2: 23.1
    // for 8 heads, 500 tokens).
    const bool one_tile = pos0 + M <= 64;
    const bool few = nh * div_up(M, 64) <= ctx->cus / 4 && pos0 + M >= 512;
    if (hs == 128) {
        if (one_tile || nh * div_up(M, 128) >= ctx->cus) AWQ_FORM(128, 4, 1, 2, 2);
        if (few) AWQ_FORM(128, 1, 4, 1, 1);
        AWQ_FORM(128, 2, 2, 2, 1);
    }
    if (hs == 64) {
        if (one_tile) AWQ_FORM(64, 4, 1, 2, 2);
        if (few) AWQ_FORM(64, 1, 4, 1, 1);
        AWQ_FORM(64, 2, 2, 2, 1);
    }
    if (hs == 256) AWQ_FORM(256, 2, 2, 1, 2);
#undef AWQ_FORM
    awq_set_error("prefill attention: head_size %d unsupported", hs);
    return AWQ_ERR_SHAPE;
}
