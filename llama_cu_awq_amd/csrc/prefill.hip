// Multi-token prefill: every projection of M prompt tokens as one int4-weight x fp16-activation GEMM on the
// fp16 matrix cores, with batched RMSNorm and RoPE around it (most forms of the GEMM are in gemm_rows.hip, the causal
// attention in prefill_attention.hip).
//
// The reference has no such path: it feeds prompt tokens through its matrix-VECTOR kernels one at a time
// (llama2_q4.cu:716-735).  The contract here is therefore the result of that token-by-token run: after
// awq_transformer_prefill(t, M, gen) the KV cache rows, the logits of the last token, the token list and the
// position equal what M calls of awq_transformer_forward would leave, up to fp32 summation order and one rounding:
// q/k/v, scores, attention output, residual stream and hidden vector are rounded to fp16 where the reference kernels
// round them, probabilities before their division by the row's sum instead of after it.  The attention differs in one
// more point, which shows only where all scores of a query lie below about -87 (prefill_attention.hip).
//
// Dequantised weights are bit-exact: w16 = half_rne((q - z) * s) computed as an exact fp16 integer (q - z)
// times the fp16 scale in one rounding.
#include <string.h>

#include <mutex>

#include "common.hpp"
#include "gemm_tile.hpp"

namespace pf {

// A tile's 128 columns are four blocks of 32 weight rows.  Which matrix a block belongs to and its first row:
// single / QKV: consecutive rows of one matrix; FFN: blocks alternate gate, up over the same 32 row indices, so that a
// wave (two adjacent blocks) holds a gate column and its up column in the same lane.
struct BlockMap {
    int mat, row0;
};

__device__ __forceinline__ BlockMap block_map(const GemmParams& p, int tile, int b) {
    BlockMap m;
    if (p.epi == EPI_FFN) {
        m.mat = b & 1;
        m.row0 = tile * 64 + (b >> 1) * 32;
        return m;
    }
    int mat = 0, tt = tile;
    if (p.epi == EPI_QKV) {
        const int t0 = p.N[0] / BN, t1 = p.N[1] / BN;
        if (tt >= t0 + t1) {
            mat = 2;
            tt -= t0 + t1;
        } else if (tt >= t0) {
            mat = 1;
            tt -= t0;
        }
    }
    m.mat = mat;
    m.row0 = tt * BN + b * 32;
    return m;
}

constexpr int A_STAGES = 3;                   // activation tiles in the LDS ring (2 steps ahead)
constexpr int W_STAGES = 3;                   // pairs of steps (one quantisation group) of packed weights in the LDS ring
constexpr int TILE_BYTES = BM * BK * 2;       // 16 KB
constexpr int W_WAVE_BYTES = 32 * 64 + 256 + 256;  // per wave and pair of steps: 32 rows x 64 packed bytes, zeros, scales
constexpr int W_STAGE_BYTES = 4 * W_WAVE_BYTES;
constexpr int GEMM_LDS_BYTES = A_STAGES * TILE_BYTES + W_STAGES * W_STAGE_BYTES;

// C[m][n] = sum_k A[m][k] * half((q[n][k] - z) * s), tile 128 x 128, K step 64.
//  * Workgroup = 4 waves; wave w owns tile columns 32w .. 32w+31 and all 128 rows: four 32x32x16 fp16 MFMA
//    accumulators.  A lane's MFMA operand for the weights is 8 consecutive K of one weight row = one packed dword, so
//    dequantised weights never pass through LDS: lane (row l % 32, half l / 32) takes its row's 16 packed bytes of
//    the step and dequantises a dword right before the MFMAs that use it (bit-exact half((q-z)*s)).
//  * Every global load is a direct global -> LDS load.  The activation tile (16 KB, natural order, read by every
//    wave as fragments) travels two steps ahead into a ring of three tiles.  Packed weights travel per pair of steps
//    (128 K = one quantisation group: 64 contiguous bytes per row, one zero-point dword and one scale) two pairs
//    ahead into a ring that only the loading wave reads back, so they need no barrier.  LDS is the prefetch ring: no
//    register carries a load across iterations and one hand-counted s_waitcnt per step covers everything.
//  * One barrier per step.  The loop body has no conditional around its loads (steps past the end are requested too), so
//    the number of loads between a request and its use is constant.
// Workgroup ids are mapped so that the M tiles sharing a weight tile run on one XCD (ids go round-robin over the 8
// XCDs), which reads the weights from HBM once.
//
// APERM: every 16-byte chunk of A holds its 8 activations in the order (0,4,1,5,2,6,3,7), the order in which a packed
// dword dequantises.  Both MFMA operands contract over K, so any order they agree on gives the same products; with A
// already in that order the weights go into the MFMA as they come out of the dequantisation.  The prefill path writes
// its intermediate activations that way; the public entry points take A in natural order.
// WHOLE: K is a multiple of 128.  Otherwise activations past K are zeros that the loads fetch in their place: what lies there
// is the next row (or the end of the allocation), and a zero scale does not make a product with infinity zero.
template <bool APERM, bool WHOLE>
__global__ __launch_bounds__(256, 2) void gemm_int4_kernel(const GemmParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_bytes[];  // [A ring][W ring]; nothing else is in LDS
    constexpr uint32_t W_RING = A_STAGES * TILE_BYTES;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int per_tile = p.mtiles * p.ksplit;
    const int tile = (slot / per_tile) * 8 + xcd;
    if (tile >= p.ntiles) return;
    const int m_index = (slot % per_tile) / p.ksplit, ks = (slot % per_tile) % p.ksplit;
    const int m0 = m_index * BM;

    // activation loader: wave w, instruction q covers tile rows (4w + q) * 8 .. + 8 (8 lanes x 16 bytes per row);
    // the lane's LDS chunk is lane & 7, so it fetches the source chunk that the swizzle maps there
    uint32_t a_off[4];  // byte offsets from p.A (a chunk of activations is far below 4 GB)
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int r = (wave * 4 + q) * 8 + (lane >> 3);
        const int c = (lane & 7) ^ lds_key(r);
        a_off[q] = (uint32_t)(((size_t)min(m0 + r, p.M - 1) * p.lda + c * 8) * 2);  // rows past M are computed, never stored
    }
    // weight loader: instruction q of a pair of steps covers the wave's rows 16q .. 16q+15, 4 lanes x 16 bytes per
    // row; 16-byte unit u of a row's 64 bytes sits at LDS unit u ^ ((row >> 1) & 3) (bank spread for the reads below)
    const BlockMap wb = block_map(p, tile, wave);
    const uint32_t* wmat = (wb.mat == 0 ? p.w[0] : (wb.mat == 1 ? p.w[1] : p.w[2]));
    const uint32_t* zmat = (wb.mat == 0 ? p.z[0] : (wb.mat == 1 ? p.z[1] : p.z[2]));
    const uint16_t* smat = (wb.mat == 0 ? p.s[0] : (wb.mat == 1 ? p.s[1] : p.s[2]));
    const uint32_t* w_src[2];
    int w_unit[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int r = 16 * q + (lane >> 2);
        w_unit[q] = (lane & 3) ^ ((r >> 1) & 3);
        w_src[q] = wmat + (size_t)(wb.row0 + r) * (p.C * 4);
    }
    // consumer side: this lane's weight row and which 32-element half of a step it multiplies
    const int lrow = lane & 31, lhalf = lane >> 5;
    const uint32_t* zrow = zmat + (size_t)(wb.row0 + lrow) * p.pzh;
    const size_t s_row = (size_t)(wb.row0 + lrow) * p.sh;  // index of the row's first scale (scales travel as aligned dwords)
    const int n_groups = p.sh;

    uint32_t magic = 0x64006400u;
    asm("" : "+v"(magic));
    f32x16 acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 16; j++) acc[i][j] = 0.0f;

    const int nsteps = (p.K + BK - 1) / BK;
    // split K: the halves meet at an even step, so that both start on a quantisation group
    const int s_split = (nsteps / 2) & ~1;
    const int s_begin = ks ? s_split : 0;
    const int s_end = (p.ksplit == 2 && ks == 0) ? s_split : nsteps;
    auto load_a = [&](int step) {  // 4 loads
        const uint32_t dst = (uint32_t)((step % A_STAGES) * TILE_BYTES + wave * 4096);
        if (WHOLE) {
            const uint16_t* base = p.A + min(step, nsteps - 1) * BK;
#pragma unroll
            for (int q = 0; q < 4; q++) dma16(base, a_off[q], dst + q * 1024);
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = (wave * 4 + q) * 8 + (lane >> 3);
                const int k = step * BK + ((lane & 7) ^ lds_key(r)) * 8;
                const void* src = reinterpret_cast<const uint8_t*>(p.A) + a_off[q] + (size_t)step * (BK * 2);
                dma16(k < p.K ? src : (const void*)zeros16, dst + q * 1024);
            }
        }
    };
    auto load_w = [&](int pair) {  // 4 loads: K range [128 * pair, 128 * pair + 128) of the wave's 32 rows
        const uint32_t dst = W_RING + (uint32_t)((pair % W_STAGES) * W_STAGE_BYTES + wave * W_WAVE_BYTES);
#pragma unroll
        for (int q = 0; q < 2; q++) dma16(w_src[q] + (size_t)min(pair * 4 + w_unit[q], p.C - 1) * 4, dst + q * 1024);
        const int g = min(pair, n_groups - 1);
        dma4(zrow + (g >> 3), dst + 2048);
        dma4(smat + ((s_row + g) & ~(size_t)1), dst + 2304);
    };
    // K mapping of the four MFMAs of a step: MFMA j multiplies K chunk j (lanes 0-31) and chunk 4 + j (lanes 32-63),
    // i.e. dword j of each lane's 16 bytes against the matching 8 activations.
    auto compute = [&](int step) {
        const uint16_t* at = reinterpret_cast<const uint16_t*>(lds_bytes + (step % A_STAGES) * TILE_BYTES);
        const int pair = step >> 1;
        const uint8_t* ws = lds_bytes + W_RING + (pair % W_STAGES) * W_STAGE_BYTES + wave * W_WAVE_BYTES;
        const int unit = (step & 1) * 2 + lhalf;
        const u32x4 wq = *reinterpret_cast<const u32x4*>(ws + lrow * 64 + ((unit ^ ((lrow >> 1) & 3)) << 4));
        const uint32_t zw = *reinterpret_cast<const uint32_t*>(ws + 2048 + lane * 4);
        const uint32_t sw = *reinterpret_cast<const uint32_t*>(ws + 2304 + lane * 4);
        const int g = min(pair, n_groups - 1);
        const uint32_t z = (zw >> (4 * (g & 7))) & 0xFu;
        const uint16_t sbits = (uint16_t)(((s_row + g) & 1) ? (sw >> 16) : (sw & 0xFFFFu));
        const bool live = step * BK + lhalf * 32 < p.K;  // past K: zero scale, zero products
        const Group gc = group_consts(z, live ? sbits : (uint16_t)0);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const u32x4 dq = dequant8(wq[j], gc, magic);
            const h16x8 bf = __builtin_bit_cast(h16x8, APERM ? dq : unpermute8(dq));
            const int chunk = j + 4 * lhalf;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const h16x8 af = *reinterpret_cast<const h16x8*>(&at[lds_off(i * 32 + (lane & 31), chunk)]);
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf, acc[i], 0, 0, 0);
            }
        }
    };

    // Prologue: the first two activation tiles and weight pairs.
    load_a(s_begin);
    load_a(s_begin + 1);
    load_w(s_begin >> 1);
    load_w((s_begin >> 1) + 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (int step = s_begin; step < s_end; step += 2) {
        // even step: request activation tile step+2 and weight pair (step/2)+2, then multiply
        load_a(step + 2);  // into the slot that step-1 multiplied: every wave is past the barrier that ended it
        load_w((step >> 1) + 2);  // into the slot this wave finished reading at the end of the previous iteration
        compute(step);
        // needed next: activation tile step+1, requested in the previous iteration's odd half, followed by 4 + 4
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        __syncthreads();
        // odd step
        load_a(step + 3);
        compute(step + 1);
        // needed next: activation tile step+2 (followed by 4 + 4 loads) and weight pair (step/2)+1 (older still)
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        __syncthreads();
    }

    if (p.ksplit == 2) {
        // The two halves of K meet here.  Each workgroup writes its fp32 partial tile through to memory and counts
        // itself in; the first to arrive leaves, the second adds the other's partial to its own (a two-term fp32 sum
        // does not depend on which one that is) and goes on to the epilogue.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct-to-LDS load is still on its way
        __syncthreads();
        const size_t tile_id = (size_t)tile * p.mtiles + m_index;
        float* mine = p.part + (tile_id * 2 + ks) * (size_t)(BM * BN);
        const float* other = p.part + (tile_id * 2 + (ks ^ 1)) * (size_t)(BM * BN);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 16; j++)
                __hip_atomic_store(&mine[((wave * 4 + i) * 16 + j) * 64 + lane], acc[i][j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        unsigned int* arrival = reinterpret_cast<unsigned int*>(lds_bytes);
        if (tid == 0) *arrival = __hip_atomic_fetch_add(&p.part_counter[tile_id], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*arrival == 0u) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (tid == 0) p.part_counter[tile_id] = 0;  // ready for the next launch
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 16; j++) acc[i][j] += other[((wave * 4 + i) * 16 + j) * 64 + lane];
    }

    // ---- epilogue.  acc[i][j] is D[row = 32*i + 8*(j/4) + 4*(lane/32) + j%4][col = lane%32] of the wave's 32 columns:
    // a lane holds one column, so stored from registers every value would be a 2-byte access of its own (measured: 15 us
    // for the RoPE form, 12 for SiLU, 5 for the residual form, of a 50 us K loop).  The four waves therefore pass their
    // accumulators through the now idle LDS rings as one fp32 tile [wave][128 rows][32 columns], and every lane then
    // owns 8 consecutive columns of a row: one 16-byte store (and one 16-byte load of the old values, the rotation
    // factors or the partner columns) per 8 results.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct-to-LDS load is still on its way
    __syncthreads();
    float* tile_f = reinterpret_cast<float*>(lds_bytes);
    {
        float* mine = tile_f + wave * 4096 + (lane >> 5) * 128 + (lane & 31);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 16; j++) mine[(i * 32 + (j >> 2) * 8 + (j & 3)) * 32] = acc[i][j];
    }
    __syncthreads();
    const int chunk = lane & 3, rsub = lane >> 2;  // 8 columns of row rsub, rsub + 16, ...
    auto read8 = [&](int w, int row, float (&v)[8]) {
        const f32x4* src = reinterpret_cast<const f32x4*>(tile_f + w * 4096 + row * 32 + chunk * 8);
        const f32x4 a = src[0], b = src[1];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e] = a[e];
            v[4 + e] = b[e];
        }
    };
    auto pack8 = [](const float (&v)[8]) {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (uint32_t)float_to_half_bits(v[2 * e]) | ((uint32_t)float_to_half_bits(v[2 * e + 1]) << 16);
        return o;
    };
    if (p.epi == EPI_FFN) {
        // waves 0, 2 hold gate columns, waves 1, 3 the up columns of the same weight rows: the two waves of a pair take
        // 64 tile rows each
        const int wg = wave & ~1;
        const int n0 = block_map(p, tile, wg).row0 + chunk * 8;
        uint16_t* o = p.out[0] + (size_t)p.out_off[0] + n0;
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const int row = (wave & 1) * 64 + it * 16 + rsub;
            const int m = m0 + row;
            float g[8], u[8], v[8];
            read8(wg, row, g);
            read8(wg + 1, row, u);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float s = g[e] * (1.0f / (1.0f + expf(-g[e])));
                v[e] = s * u[e];
            }
            if (p.out_perm) {  // (0,4,1,5,2,6,3,7): the order a permuted-A GEMM reads
                const float t[8] = {v[0], v[4], v[1], v[5], v[2], v[6], v[3], v[7]};
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = t[e];
            }
            if (m < p.M) *reinterpret_cast<u32x4*>(o + (size_t)m * p.ldo[0]) = pack8(v);
        }
        return;
    }
    const int mat = wb.mat;
    uint16_t* o = (mat == 0 ? p.out[0] : (mat == 1 ? p.out[1] : p.out[2])) +
                  (size_t)(mat == 0 ? p.out_off[0] : (mat == 1 ? p.out_off[1] : p.out_off[2])) + wb.row0 + chunk * 8;
    const size_t ld = (size_t)(mat == 0 ? p.ldo[0] : (mat == 1 ? p.ldo[1] : p.ldo[2]));
    if (p.rope && mat < 2) {
        // The tile is one head: column c < 64 rotates with column c + 64, which the wave two further on holds.  Values
        // are rounded to fp16 first and rotated in fp32, as the separate kernel does on the stored q and k
        // (gpu_kernels.h:351-361).  (cos, sin) of 8 consecutive pairs are 64 contiguous bytes of the table.
        const int pair0 = (wave & 1) * 32 + chunk * 8;  // 0 .. 63
#pragma unroll
        for (int it = 0; it < 8; it++) {
            const int row = it * 16 + rsub;
            const int m = m0 + row;
            const f32x4* cs = reinterpret_cast<const f32x4*>(p.rope + (size_t)(p.rope_pos0 + min(m, p.M - 1)) * 64 + pair0);
            const f32x4 c0 = cs[0], c1 = cs[1], c2 = cs[2], c3 = cs[3];
            const float cosv[8] = {c0[0], c0[2], c1[0], c1[2], c2[0], c2[2], c3[0], c3[2]};
            const float sinv[8] = {c0[1], c0[3], c1[1], c1[3], c2[1], c2[3], c3[1], c3[3]};
            float a[8], b[8], v[8];
            read8(wave, row, a);
            read8(wave ^ 2, row, b);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float own = half_bits_to_float(float_to_half_bits(a[e]));
                const float other = half_bits_to_float(float_to_half_bits(b[e]));
                // columns below 64 are the first elements of their pairs, the others the second
                float r0, r1;
                if (wave < 2) rope_rotate(own, other, cosv[e], sinv[e], r0, r1);
                else rope_rotate(other, own, cosv[e], sinv[e], r0, r1);
                v[e] = wave < 2 ? r0 : r1;
            }
            if (m < p.M) *reinterpret_cast<u32x4*>(o + (size_t)m * ld) = pack8(v);
        }
        return;
    }
    // plain and residual forms; the old values of all 8 row passes are requested before the first is used
    u32x4 old[8];
    if (p.epi == EPI_RESID) {
#pragma unroll
        for (int it = 0; it < 8; it++)
            old[it] = *reinterpret_cast<const u32x4*>(o + (size_t)min(m0 + it * 16 + rsub, p.M - 1) * ld);
    }
#pragma unroll
    for (int it = 0; it < 8; it++) {
        const int row = it * 16 + rsub;
        const int m = m0 + row;
        float v[8];
        read8(wave, row, v);
        if (p.epi == EPI_RESID) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[2 * e] += half_bits_to_float((uint16_t)(old[it][e] & 0xFFFFu));
                v[2 * e + 1] += half_bits_to_float((uint16_t)(old[it][e] >> 16));
            }
        }
        if (m < p.M) *reinterpret_cast<u32x4*>(o + (size_t)m * ld) = pack8(v);
    }
}

// ---------------------------------------------------------------- row-wise helpers
__global__ __launch_bounds__(256) void embed_rows_kernel(uint16_t* x, const uint16_t* table, int dim, const int* tokens, int pos0) {
    const int m = blockIdx.x;
    const int token = tokens[pos0 + m];
    const u32x4* src = reinterpret_cast<const u32x4*>(table + (size_t)token * dim);
    u32x4* dst = reinterpret_cast<u32x4*>(x + (size_t)m * dim);
    for (int i = threadIdx.x; i < (dim >> 3); i += 256) dst[i] = src[i];
}

// o[m] = half(x[m] * (rsqrt(mean(x[m]^2) + 1e-5) * w))  (gpu_kernels.h:72-105, one workgroup per token row).
// 16-byte pieces; up to 4 per thread stay in registers between the two passes (rows of up to 8192), longer rows
// re-read the rest.
// perm: every 8 outputs are stored in the order (0,4,1,5,2,6,3,7) (what a permuted-A GEMM reads).  tiles: 32-row tiles of an
// output in fragment order (the few-row GEMM's), 0: rows.
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(uint16_t* o, const uint16_t* x, const uint16_t* weight, int size, int perm, int tiles) {
    __shared__ float red[4];
    constexpr int NP = 4;
    const int tid = threadIdx.x;
    const int n8 = size >> 3;
    const u32x4* xr = reinterpret_cast<const u32x4*>(x + (size_t)blockIdx.x * size);
    const u32x4* wr = reinterpret_cast<const u32x4*>(weight);
    auto orow = [&](int e) -> u32x4& {
        return *reinterpret_cast<u32x4*>(o + (tiles ? fragment_offset(blockIdx.x, e * 8, tiles) : (size_t)blockIdx.x * size + e * 8));
    };
    u32x4 v[NP], w[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int e = min(i * 256 + tid, n8 - 1);
        v[i] = xr[e];
        w[i] = wr[e];
    }
    auto sumsq = [](const u32x4 p, float part) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const h16x2 h = as_h2(p[k]);
            part = fmaf((float)h[0], (float)h[0], part);
            part = fmaf((float)h[1], (float)h[1], part);
        }
        return part;
    };
    auto scale = [perm](const u32x4 p, const u32x4 wv, float ss) {
        u32x4 r;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const h16x2 h = as_h2(p[k]), hw = as_h2(wv[k]);
            h16x2 q;
            q[0] = (h16_t)((float)h[0] * (ss * (float)hw[0]));
            q[1] = (h16_t)((float)h[1] * (ss * (float)hw[1]));
            r[k] = as_u32(q);
        }
        return perm ? permute8(r) : r;
    };
    float part = 0.0f;
#pragma unroll
    for (int i = 0; i < NP; i++)
        if (i * 256 + tid < n8) part = sumsq(v[i], part);
    for (int e = NP * 256 + tid; e < n8; e += 256) part = sumsq(xr[e], part);
    part = wave_sum(part);
    if ((tid & 63) == 0) red[tid >> 6] = part;
    __syncthreads();
    float ss = (red[0] + red[1]) + (red[2] + red[3]);
    ss /= (float)size;
    ss += 1e-5f;
    ss = 1.0f / sqrtf(ss);
#pragma unroll
    for (int i = 0; i < NP; i++)
        if (i * 256 + tid < n8) orow(i * 256 + tid) = scale(v[i], w[i], ss);
    for (int e = NP * 256 + tid; e < n8; e += 256) orow(e) = scale(xr[e], wr[e], ss);
}

// x[m] += the fp32 partial sums of a product over x's columns (added up in order, one rounding, as the product's own epilogue
// does it), then o[m] = the RMSNorm of x[m] as above.  Bound by latency: one workgroup per row, every load of a thread
// requested at once (4 columns a piece; two pieces, rows of up to 8192, stay in registers).  FRAG: the output goes in fragment
// order of `tiles` tiles (asked at run time, 700 rows of 2048 in four parts took 8.84 us instead of 8.59).
template <int PARTS, bool FRAG>
__global__ __launch_bounds__(1024) void rmsnorm_parts_kernel(uint16_t* o, uint16_t* x, const float* part, const uint16_t* weight, int size,
                                                           int perm, int tiles) {
    __shared__ float red[16];
    constexpr int NP = 2;
    const int tid = threadIdx.x;
    const int n4 = size >> 2;
    u32x2* xr = reinterpret_cast<u32x2*>(x + (size_t)blockIdx.x * size);
    const u32x2* wr = reinterpret_cast<const u32x2*>(weight);
    const f32x4* pr = reinterpret_cast<const f32x4*>(part + (size_t)blockIdx.x * size);
    const size_t stride = (size_t)gridDim.x * n4;  // from one part to the next
    struct Piece {
        u32x2 x, w;
        f32x4 p[PARTS];
    };
    auto load = [&](Piece& v, int e) {
        v.x = xr[e];
        v.w = wr[e];
#pragma unroll
        for (int k = 0; k < PARTS; k++) v.p[k] = pr[(size_t)k * stride + e];
    };
    auto sum = [&](Piece& v) {  // the new x, rounded, in v.x; its squares
        f32x4 t = v.p[0];
#pragma unroll
        for (int k = 1; k < PARTS; k++) t += v.p[k];
        float sq = 0.0f;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            h16x2 h = as_h2(v.x[k]);
            h[0] = (h16_t)(t[2 * k] + (float)h[0]);
            h[1] = (h16_t)(t[2 * k + 1] + (float)h[1]);
            v.x[k] = as_u32(h);
            sq = fmaf((float)h[0], (float)h[0], sq);
            sq = fmaf((float)h[1], (float)h[1], sq);
        }
        return sq;
    };
    auto put = [&](const Piece& v, int e, float ss) {
        u32x2 r;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const h16x2 h = as_h2(v.x[k]), hw = as_h2(v.w[k]);
            h16x2 q;
            q[0] = (h16_t)((float)h[0] * (ss * (float)hw[0]));
            q[1] = (h16_t)((float)h[1] * (ss * (float)hw[1]));
            r[k] = as_u32(q);
        }
        if (perm) {  // lanes 2i and 2i + 1 hold columns 0..3 and 4..7 of eight: (0,4)(1,5) to the one, (2,6)(3,7) to the other
            const bool odd = e & 1;
            const uint32_t give = odd ? r[0] : r[1];
            const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
            const uint32_t lo = odd ? got : r[0], hi = odd ? r[1] : got;
            r[0] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
            r[1] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
        }
        *reinterpret_cast<u32x2*>(o + (FRAG ? fragment_offset(blockIdx.x, e * 4 & ~7, tiles) + (e & 1) * 4 : (size_t)blockIdx.x * size + e * 4)) = r;
    };
    Piece v[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) load(v[i], min(i * 1024 + tid, n4 - 1));
    float sq = 0.0f;
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const float s = sum(v[i]);
        if (i * 1024 + tid < n4) {
            sq += s;
            xr[i * 1024 + tid] = v[i].x;
        }
    }
    for (int e = NP * 1024 + tid; e < n4; e += 1024) {
        Piece u;
        load(u, e);
        sq += sum(u);
        xr[e] = u.x;
    }
    sq = wave_sum(sq);
    if ((tid & 63) == 0) red[tid >> 6] = sq;
    __syncthreads();
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) ss += red[i];
    ss /= (float)size;
    ss += 1e-5f;
    ss = 1.0f / sqrtf(ss);
#pragma unroll
    for (int i = 0; i < NP; i++)
        if (i * 1024 + tid < n4) put(v[i], i * 1024 + tid, ss);
    for (int e = NP * 1024 + tid; e < n4; e += 1024) {
        Piece u;
        u.x = xr[e];
        u.w = wr[e];
        put(u, e, ss);
    }
}

// RoPE of q rows [M][heads*hs] and of the K cache rows pos0..pos0+M-1 (gpu_kernels.h:340-363 per position).
__global__ void rope_rows_kernel(uint16_t* q, uint16_t* kcache_layer, int num_heads, int num_kv_heads, int head_size, int pos0,
                                 float rope_theta, const float2* table) {
    const int m = blockIdx.y;
    const int h = blockIdx.x;
    const int i = threadIdx.x;
    const int pos = pos0 + m;
    const int half_size = head_size >> 1;
    float fcr, fci;
    if (table) {  // (cos, sin) per position and pair, computed once at load time with the formula below
        const float2 cs = table[(size_t)pos * half_size + i];
        fcr = cs.x;
        fci = cs.y;
    } else {
        const int head_dim = (i * 2) % head_size;
        const float freq = 1.0f / powf(rope_theta, head_dim / (float)head_size);
        const float val = pos * freq;
        fcr = cosf(val);
        fci = sinf(val);
    }
    uint16_t* qh = q + ((size_t)m * num_heads + h) * head_size;
    const float q0 = half_bits_to_float(qh[i]);
    const float q1 = half_bits_to_float(qh[i + half_size]);
    float r0, r1;
    rope_rotate(q0, q1, fcr, fci, r0, r1);
    qh[i] = float_to_half_bits(r0);
    qh[i + half_size] = float_to_half_bits(r1);
    if (h < num_kv_heads) {
        uint16_t* k = kcache_layer + ((size_t)pos * num_kv_heads + h) * head_size;
        const float k0 = half_bits_to_float(k[i]);
        const float k1 = half_bits_to_float(k[i + half_size]);
        rope_rotate(k0, k1, fcr, fci, r0, r1);
        k[i] = float_to_half_bits(r0);
        k[i + half_size] = float_to_half_bits(r1);
    }
}

__global__ void set_pos_kernel(int* pos_dev, volatile int* pos_host, int value) {
    *pos_dev = value;
    *pos_host = value;
}

__global__ __launch_bounds__(256) void copy_row_kernel(uint16_t* dst, const uint16_t* src, int n8) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n8) reinterpret_cast<u32x4*>(dst)[i] = reinterpret_cast<const u32x4*>(src)[i];
}

}  // namespace pf

// ---------------------------------------------------------------- split-K workspace that needs no allocation
// awq_gemm_int4_static keeps the split-K workspace (fp32 partial tiles, then the per-tile arrival counters) in this
// file-scope device array instead of memory obtained with hipMalloc.  Every GPU the library runs on holds its own copy
// at its own address until the process ends.  In host code the array's name is only a stand-in for the symbol: the
// device address is looked up once per device with hipGetSymbolAddress and kept in g_scratch_ptr, and that pointer is
// what kernels and clears receive.
constexpr size_t kScratchBytes = kPartBytes + kPartTiles * sizeof(unsigned int);
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices];    // device address of `scratch` on each device, null until looked up
static bool g_gemm_lds_raised[kMaxDevices];  // the GEMM kernel's dynamic LDS limit has been raised on the device

namespace pf {
__global__ void clear_words_kernel(unsigned int* words, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) words[i] = 0u;
}
}  // namespace pf

// Once per device, with that device current: raise the GEMM kernel's LDS limit and look up the address of `scratch`.
// Called when a context is created, so that the entry points themselves do no set-up work.
int awq_gemm_device_setup(int device) {
    if (device < 0 || device >= kMaxDevices) {
        awq_set_error("device ordinal %d out of range", device);
        return AWQ_ERR_ARG;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_gemm_lds_raised[device]) {
        const void* kernels[3] = {(const void*)pf::gemm_int4_kernel<true, true>, (const void*)pf::gemm_int4_kernel<false, true>,
                                  (const void*)pf::gemm_int4_kernel<false, false>};
        for (const void* k : kernels) {
            const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, pf::GEMM_LDS_BYTES);
            if (e != hipSuccess) {
                awq_set_error("hipFuncSetAttribute(gemm_int4) failed: %s", hipGetErrorString(e));
                return AWQ_ERR_HIP;
            }
        }
        if (int r = awq_gemm_rows_setup()) return r;
        if (int r = awq_gemm_few_setup()) return r;
        g_gemm_lds_raised[device] = true;
    }
    if (!g_scratch_ptr[device]) {
        void* ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            awq_set_error("hipGetSymbolAddress(scratch) failed on device %d: %s", device, hipGetErrorString(e));
            return AWQ_ERR_HIP;
        }
        g_scratch_ptr[device] = ptr;
    }
    return AWQ_OK;
}

// ---------------------------------------------------------------- launchers (internal)
// The context's split-K workspace, allocated whole the first time.  Its counters are cleared ahead of every product, also
// where the context's stream is being recorded: what is recorded there runs when the graph does, and an eager product may
// come first, so that they are cleared at once on a stream of their own.
int awq_reserve_gemm_workspace(awq_ctx* ctx) {
    if (ctx->gemm_part) return AWQ_OK;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &capturing) != hipSuccess) (void)hipGetLastError();
    void* block = nullptr;
    if (const hipError_t e = hipMalloc(&block, kScratchBytes); e != hipSuccess) {
        (void)hipGetLastError();  // a caller that goes on without it must not find this behind its next launch
        awq_set_error("split-K workspace allocation failed: %s", hipGetErrorString(e));
        return AWQ_ERR_HIP;
    }
    unsigned int* counter = reinterpret_cast<unsigned int*>(static_cast<uint8_t*>(block) + kPartBytes);
    const bool recorded = capturing != hipStreamCaptureStatusNone;
    hipStream_t stream = ctx->stream;
    hipError_t e = recorded ? hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) : hipSuccess;
    if (e == hipSuccess) {
        hipLaunchKernelGGL(pf::clear_words_kernel, dim3(1), dim3(kPartTiles), 0, stream, counter, kPartTiles);
        e = hipGetLastError();
        if (recorded) {
            if (e == hipSuccess) e = hipStreamSynchronize(stream);
            (void)hipStreamDestroy(stream);
        }
    }
    if (e != hipSuccess) {
        (void)hipFree(block);
        awq_set_error("clearing the split-K counters failed: %s", hipGetErrorString(e));
        return AWQ_ERR_HIP;
    }
    ctx->gemm_part = static_cast<float*>(block);
    return AWQ_OK;
}

// The split-K workspace of a launch over `tiles` output tiles: the file-scope device array (static_ws; no allocation) or
// the context's, allocated whole on first use, so that it never moves.
static int bind_workspace(awq_ctx* ctx, pf::GemmParams& p, int tiles, bool static_ws, const char* what) {
    if (static_ws) {
        unsigned char* ws = static_cast<unsigned char*>(g_scratch_ptr[ctx->device]);
        if (!ws) {
            awq_set_error("%s: the static workspace was not set up on device %d", what, ctx->device);
            return AWQ_ERR_HIP;
        }
        p.part = reinterpret_cast<float*>(ws);
        p.part_counter = reinterpret_cast<unsigned int*>(ws + kPartBytes);
        // the array keeps whatever the previous call on this GPU left: the arrival counters must start at zero
        // (a fill kernel rather than a memset node, so that the call can be recorded into a graph)
        hipLaunchKernelGGL(pf::clear_words_kernel, dim3(div_up(tiles, 256)), dim3(256), 0, ctx->stream, p.part_counter, tiles);
        return awq_check_launch("clear_words");
    }
    if (int r = awq_reserve_gemm_workspace(ctx)) return r;
    p.part = ctx->gemm_part;
    p.part_counter = reinterpret_cast<unsigned int*>(reinterpret_cast<uint8_t*>(ctx->gemm_part) + kPartBytes);
    return AWQ_OK;
}

// Expected time of the 128 x 128 kernel, to be weighed against the forms of gemm_rows.hip (147 of 159 products within 15 %).
// It is as good as any of them where about one of its workgroups comes to a compute unit and K is long: weights from memory,
// 512 x 11008 x 4096 in two parts 67 us, 128 x 256 in four parts 64, 64 x 256 in four 70, 64 x 128 71; 77 x 5120 x 13824 in
// two parts 37.5 us, 96 x 256 in four 34, 32 x 64 36, 64 x 128 36.  At K = 4096 it is not (512 x 4096 x 4096: 32 us, 64 x 128 28).
static float general_us(int cus, long long tiles, int K, int ksplit) {
    const float split = ksplit > 1 ? 2.0f + 0.5e-6f * tiles * ksplit * (pf::BM * pf::BN * sizeof(float)) : 0.0f;
    return awq_gemm_us(cus, 2, tiles * ksplit, div_up(div_up(K, pf::BK), ksplit), awq_step_us{0.52f, 0.58f, 1.1f}) + split;
}

// How a product over `ntiles` tiles of 128 weight rows runs.
struct GemmRoute {
    int form;    // of gemm_rows.hip; -1: the 128 x 128 kernel
    int ksplit;  // workgroups per tile along K
    float us;    // what the launch is expected to take
};
// The 128 x 128 kernel gives a single matrix with fewer tiles than compute units two workgroups per tile, each half of K.
static bool general_splits(int M, int K, int ntiles, bool single) {
    return single && (long long)div_up(M, pf::BM) * ntiles < 256 && K >= 8 * pf::BK;
}
// single: one matrix (plain or residual form); the QKV and gate/up products split K in the row forms only
static GemmRoute route_gemm(int cus, int M, int K, int ntiles, bool single) {
    const int ksplit = general_splits(M, K, ntiles, single) ? 2 : 1;
    const awq_rows_plan plan = awq_plan_gemm_rows(cus, M, K, ntiles * 2, ksplit == 2 || !single);
    const float general = general_us(cus, (long long)div_up(M, pf::BM) * ntiles, K, ksplit);
    if (plan.form >= 0 && plan.us < general) return GemmRoute{plan.form, plan.ksplit, plan.us};
    return GemmRoute{-1, ksplit, general};
}

static int gemm_ready(awq_ctx* ctx, const pf::GemmParams& p, const char* what) {
    // the kernels' LDS exceeds the default dynamic limit; raised per device when a context is created
    // (contexts on a caller's stream included), here only for a device that was missed
    if (ctx->device < 0 || ctx->device >= kMaxDevices || !g_gemm_lds_raised[ctx->device]) {
        if (int r = awq_gemm_device_setup(ctx->device)) return r;
    }
    if ((size_t)p.M * (size_t)p.lda * 2 >= ((size_t)1 << 32)) {  // the kernels address A by 32-bit byte offsets
        awq_set_error("%s: activation block of %d x %d halves exceeds 4 GB", what, p.M, p.lda);
        return AWQ_ERR_SHAPE;
    }
    return AWQ_OK;
}

// static_ws: take the split-K workspace from the file-scope device array (no allocation) instead of the context's.
// a_perm: A holds every 8 activations in the order (0,4,1,5,2,6,3,7).
// *rotated (QKV): whether the epilogue did what p.rope asks for.
static int launch_gemm(awq_ctx* ctx, pf::GemmParams& p, int ntiles, const char* what, bool a_perm, bool static_ws = false,
                       bool* rotated = nullptr) {
    if (int r = gemm_ready(ctx, p, what)) return r;
    const bool single = p.epi == pf::EPI_STORE || p.epi == pf::EPI_RESID;
    // reserved by every product of few tiles, whether its form splits K or not: a smaller one of the same weights, which
    // may be recorded into a graph where nothing can be allocated, may split
    if (general_splits(p.M, p.K, ntiles, single) && !static_ws)
        if (int r = awq_reserve_gemm_workspace(ctx)) return r;
    const GemmRoute route = route_gemm(ctx->cus, p.M, p.K, ntiles, single);
    p.mtiles = div_up(p.M, pf::BM);
    p.ntiles = ntiles;
    p.ksplit = route.ksplit;
    if (p.ksplit > 1)
        if (int r = bind_workspace(ctx, p, route.form >= 0 ? kPartTiles : p.mtiles * ntiles, static_ws, what)) return r;
    if (route.form >= 0) return awq_launch_gemm_rows(ctx, p, ntiles * 2, route.form, route.ksplit, a_perm, what);
    if (p.rope && p.head_size != 128) {
        p.rope = nullptr;
        *rotated = false;
    }
    // ids go round-robin over the 8 XCDs; each XCD takes every 8th weight tile with all of its M tiles (and K halves)
    const int grid = 8 * p.mtiles * p.ksplit * div_up(ntiles, 8);
    if (a_perm)  // (K a multiple of 128, as in every model that prefills)
        hipLaunchKernelGGL((pf::gemm_int4_kernel<true, true>), dim3(grid), dim3(256), pf::GEMM_LDS_BYTES, ctx->stream, p);
    else if ((p.K & 127) == 0)
        hipLaunchKernelGGL((pf::gemm_int4_kernel<false, true>), dim3(grid), dim3(256), pf::GEMM_LDS_BYTES, ctx->stream, p);
    else
        hipLaunchKernelGGL((pf::gemm_int4_kernel<false, false>), dim3(grid), dim3(256), pf::GEMM_LDS_BYTES, ctx->stream, p);
    return awq_check_launch(what);
}

static void set_mat(pf::GemmParams& p, int i, const awq_qweight* w, int N, uint16_t* out, long long ldo, long long off) {
    p.w[i] = w->weight;
    p.z[i] = w->zeros;
    p.s[i] = w->scales;
    p.N[i] = N;
    p.out[i] = out;
    p.ldo[i] = ldo;
    p.out_off[i] = off;
}

static void gemm_common(pf::GemmParams& p, const uint16_t* A, int lda, int M, int K, int epi) {
    memset(&p, 0, sizeof(p));
    p.A = A;
    p.lda = lda;
    p.M = M;
    p.K = K;
    p.C = div_up(K, 32);
    p.pzh = packed_zeros_height(K);
    p.sh = scales_height(K);
    p.epi = epi;
}

int awq_launch_gemm_single(awq_ctx* ctx, uint16_t* out, long long ldo, const uint16_t* A, int lda, int M, const awq_qweight* w,
                           int K, int N, int accum, bool static_ws, bool a_perm) {
    pf::GemmParams p;
    gemm_common(p, A, lda, M, K, accum ? pf::EPI_RESID : pf::EPI_STORE);
    set_mat(p, 0, w, N, out, ldo, 0);
    return launch_gemm(ctx, p, N / pf::BN, "gemm_int4", a_perm, static_ws);
}

int awq_launch_rmsnorm_rows(awq_ctx* ctx, uint16_t* o, const uint16_t* x, const uint16_t* w, int size, int M, int perm, int tiles);

// Whether a pass of M rows goes through a layer in the few-row form: its four products hand each other activations in
// fragment order, so that they are weighed together.  Inside a pass the sum of their estimates counts for kFewWeight (by 32-row
// tiles) of the row forms': they start and end faster, and what they read of weights and activations overlaps better, the more so the
// fewer the rows.  Four layers and the logits, us, row forms | few-row form, by key and value columns, at 4, 32, 33 and 64 rows:
// dim 2048 (256) by 5632 246 | 207, 266 | 226, 270 | 246, 277 | 250; 4096 (4096) by 11008 361 | 327, 375 | 339, 422 | 372, 429 | 392;
// 6656 (6656) by 17920 595 | 549, 641 | 592, 718 | 657, 743 | 698; 8192 (8192) by 22016 651 | 646, 695 | 686, 804 | 757, 826 | 811;
// 8192 (1024) by 28672 666 | 647, 718 | 719, 778 | 826, 807 | 891; 8192 (8192) by 28672 728 | 714, 786 | 777, 866 | 890, 897 | 957.
// At 65, 96, 97 and 128 rows: 2048 300 | 273, 299 | 278, 307 | 289, 311 | 301; 4096 517 | 439, 522 | 452, 523 | 511, 534 | 534; 5120
// (5120) by 13824 637 | 544, 651 | 568, 655 | 609, 670 | 636; 6656 907 | 792, 916 | 826, 971 | 963, 984 | 1009; 8192 (1024) by 28672
// 1004 | 994, 1019 | 1046, 1079 | 1137, 1102 | 1192; 8192 (8192) by 28672 1109 | 1080, 1135 | 1141, 1244 | 1306, 1267 | 1376.  The estimates
// are too high for narrow products of several row tiles: 1536 (256) by 4096 stays with the row forms past 64 rows (288 | 265 at 65,
// 275 | 267 at 128).
bool awq_prefill_takes_few(awq_ctx* ctx, int M, int dim, int kv_dim, int hidden) {
    if (M > kFewRows) return false;
    constexpr float kFewWeight[4] = {0.75f, 0.89f, 1.05f, 1.06f};
    const auto few = [&](int K, int N, bool split) { return awq_plan_gemm_few(ctx->cus, M, K, N, split).us; };
    const auto rows = [&](int K, int N, bool single) {
        const float us = route_gemm(ctx->cus, M, K, N / pf::BN, single).us;
        if (!single) return us;
        const awq_rows_plan parts = awq_plan_gemm_rows(ctx->cus, M, K, N / 64, true, true);
        return parts.form >= 0 && parts.us < us ? parts.us : us;
    };
    return kFewWeight[(M - 1) / 32] * (few(dim, dim + 2 * kv_dim, false) + few(dim, dim, true) + few(dim, 2 * hidden, false) + few(hidden, dim, true)) <
           rows(dim, dim + 2 * kv_dim, false) + rows(dim, dim, true) + rows(dim, 2 * hidden, false) + rows(hidden, dim, true);
}

// x += A . W, or (parts > 0) its partial sums in ctx->gemm_part, [part][M][N], for awq_launch_rmsnorm_parts to add to x (with no
// other product of the context in between: its parts may take the same place).  Where K is split, parts that meet in the launch cost it 6 to 8 us (written through, counted in, read back).  7B shape, us with
// the parts in the launch -> left to the norm: 37 tokens O 14.2 -> 9.9, down 20.4 -> 16.7 (norm 4.0 -> 4.8), 512 tokens down
// 67 -> 55 (norm 5.1 -> 9.1).
int awq_launch_gemm_resid(awq_ctx* ctx, uint16_t* x, const uint16_t* A, int lda, int M, const awq_qweight* w, int K, int N, int* parts) {
    *parts = 0;
    const GemmRoute route = route_gemm(ctx->cus, M, K, N / pf::BN, true);
    const awq_rows_plan plan = awq_plan_gemm_rows(ctx->cus, M, K, N / 64, true, true);
    if (plan.form >= 0 && plan.ksplit > 1 && plan.us < route.us && awq_reserve_gemm_workspace(ctx) == AWQ_OK) {
        pf::GemmParams p;
        gemm_common(p, A, lda, M, K, pf::EPI_PART);
        set_mat(p, 0, w, N, x, N, 0);
        p.part = ctx->gemm_part;
        if (int r = gemm_ready(ctx, p, "gemm_int4")) return r;
        *parts = plan.ksplit;
        return awq_launch_gemm_rows(ctx, p, N / 64, plan.form, plan.ksplit, true, "gemm_int4");
    }
    return awq_launch_gemm_single(ctx, x, N, A, lda, M, w, K, N, 1, false, true);
}

// The same in the few-row form, A in fragment order.
int awq_launch_gemm_few_resid(awq_ctx* ctx, uint16_t* x, const uint16_t* A, int M, const awq_qweight* w, int K, int N, int* parts) {
    pf::GemmParams p;
    gemm_common(p, A, K, M, K, pf::EPI_RESID);
    set_mat(p, 0, w, N, x, N, 0);
    awq_few_plan plan = awq_plan_gemm_few(ctx->cus, M, K, N, true);
    if (plan.ksplit > 1 && awq_reserve_gemm_workspace(ctx) != AWQ_OK) plan = awq_plan_gemm_few(ctx->cus, M, K, N, false);
    *parts = 0;
    if (plan.ksplit > 1) {
        p.epi = pf::EPI_PART;
        p.part = ctx->gemm_part;
        *parts = plan.ksplit;
    }
    return awq_launch_gemm_few(ctx, p, N, plan, "gemm_few");
}

// o = RMSNorm of x, M rows of `size`; parts > 0: after adding those of the last awq_launch_gemm_resid to x; tiles > 0: o in
// fragment order
int awq_launch_rmsnorm_parts(awq_ctx* ctx, uint16_t* o, uint16_t* x, const uint16_t* w, int size, int M, int perm, int parts, int tiles) {
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(M), dim3(1024), 0, ctx->stream, o, x, ctx->gemm_part, w, size, perm, tiles); };
    switch (parts) {
        case 0: return awq_launch_rmsnorm_rows(ctx, o, x, w, size, M, perm, tiles);
        case 2: tiles ? go(pf::rmsnorm_parts_kernel<2, true>) : go(pf::rmsnorm_parts_kernel<2, false>); break;
        case 3: tiles ? go(pf::rmsnorm_parts_kernel<3, true>) : go(pf::rmsnorm_parts_kernel<3, false>); break;
        case 4: tiles ? go(pf::rmsnorm_parts_kernel<4, true>) : go(pf::rmsnorm_parts_kernel<4, false>); break;
        default: awq_set_error("rmsnorm: %d parts", parts); return AWQ_ERR_ARG;
    }
    return awq_check_launch("rmsnorm_parts");
}
int awq_launch_rmsnorm_parts(awq_ctx* ctx, uint16_t* o, uint16_t* x, const uint16_t* w, int size, int M, int perm, int parts) {
    return awq_launch_rmsnorm_parts(ctx, o, x, w, size, M, perm, parts, 0);
}

int awq_launch_rope_rows(awq_ctx* ctx, uint16_t* q, uint16_t* kcache_layer, int nh, int nkv, int hs, int pos0, float theta, int M,
                         const float2* table);

// q rows and K, V cache rows of M positions from pos0 on, q and k rotated
int awq_launch_gemm_qkv(awq_ctx* ctx, uint16_t* q, uint16_t* kcache_layer, uint16_t* vcache_layer, const uint16_t* A, int lda, int M,
                        const awq_qweight* qw, const awq_qweight* kw, const awq_qweight* vw, int K, int Nq, int Nkv, int head_size,
                        const float2* rope, float theta, int pos0, bool a_perm, bool few) {
    pf::GemmParams p;
    gemm_common(p, A, lda, M, K, pf::EPI_QKV);
    bool rotated = rope != nullptr && (head_size == 64 || head_size == 128 || head_size == 256);
    p.rope = rotated ? rope : nullptr;
    p.head_size = head_size;
    p.rope_pos0 = pos0;
    set_mat(p, 0, qw, Nq, q, Nq, 0);
    set_mat(p, 1, kw, Nkv, kcache_layer, Nkv, (long long)pos0 * Nkv);
    set_mat(p, 2, vw, Nkv, vcache_layer, Nkv, (long long)pos0 * Nkv);
    if (few) {
        if (int r = awq_launch_gemm_few(ctx, p, Nq + 2 * Nkv, awq_plan_gemm_few(ctx->cus, M, K, Nq + 2 * Nkv, false), "gemm_few_qkv")) return r;
    } else if (int r = launch_gemm(ctx, p, (Nq + 2 * Nkv) / pf::BN, "gemm_int4_qkv", a_perm, false, &rotated)) return r;
    return rotated ? AWQ_OK : awq_launch_rope_rows(ctx, q, kcache_layer, Nq / head_size, Nkv / head_size, head_size, pos0, theta, M, rope);
}

int awq_launch_gemm_ffn(awq_ctx* ctx, uint16_t* hb, const uint16_t* A, int lda, int M, const awq_qweight* gate_w,
                        const awq_qweight* up_w, int K, int N, bool a_perm, bool out_perm, bool few) {
    pf::GemmParams p;
    gemm_common(p, A, lda, M, K, pf::EPI_FFN);
    p.out_perm = out_perm;
    set_mat(p, 0, gate_w, N, hb, N, 0);
    set_mat(p, 1, up_w, N, hb, N, 0);
    if (few) return awq_launch_gemm_few(ctx, p, 2 * N, awq_plan_gemm_few(ctx->cus, M, K, 2 * N, false), "gemm_few_ffn");
    return launch_gemm(ctx, p, N / 64, "gemm_int4_ffn", a_perm);
}

int awq_launch_embed_rows(awq_ctx* ctx, uint16_t* x, const uint16_t* table, int dim, const int* tokens, int pos0, int M) {
    hipLaunchKernelGGL(pf::embed_rows_kernel, dim3(M), dim3(256), 0, ctx->stream, x, table, dim, tokens, pos0);
    return awq_check_launch("embed_rows");
}

int awq_launch_rmsnorm_rows(awq_ctx* ctx, uint16_t* o, const uint16_t* x, const uint16_t* w, int size, int M, int perm, int tiles) {
    hipLaunchKernelGGL(pf::rmsnorm_rows_kernel, dim3(M), dim3(256), 0, ctx->stream, o, x, w, size, perm, tiles);
    return awq_check_launch("rmsnorm_rows");
}

int awq_launch_rope_rows(awq_ctx* ctx, uint16_t* q, uint16_t* kcache_layer, int nh, int nkv, int hs, int pos0, float theta, int M,
                         const float2* table) {
    hipLaunchKernelGGL(pf::rope_rows_kernel, dim3(nh, M), dim3(hs / 2), 0, ctx->stream, q, kcache_layer, nh, nkv, hs, pos0, theta,
                       table);
    return awq_check_launch("rope_rows");
}

int awq_launch_set_pos(awq_ctx* ctx, int* pos_dev, volatile int* pos_host, int value) {
    hipLaunchKernelGGL(pf::set_pos_kernel, dim3(1), dim3(1), 0, ctx->stream, pos_dev, pos_host, value);
    return awq_check_launch("set_pos");
}

int awq_launch_copy_row(awq_ctx* ctx, uint16_t* dst, const uint16_t* src, int n) {
    hipLaunchKernelGGL(pf::copy_row_kernel, dim3(div_up(n >> 3, 256)), dim3(256), 0, ctx->stream, dst, src, n >> 3);
    return awq_check_launch("copy_row");
}

extern "C" {

int awq_gemm_int4(awq_ctx* ctx, uint16_t* out, int ldo, const uint16_t* a, int lda, int M, const awq_qweight* w, int K, int N,
                  int accum) {
    if (int r = awq_bind(ctx)) return r;
    AWQ_REQUIRE(out && a && w && w->weight && w->zeros && w->scales, AWQ_ERR_ARG, "null pointer");
    if (M <= 0 || K <= 0 || N <= 0 || (K & 31) || (N & 127) || (lda & 7)) {
        awq_set_error("awq_gemm_int4: needs M > 0, K %% 32 == 0, N %% 128 == 0, lda %% 8 == 0 (got M=%d K=%d N=%d lda=%d)", M, K, N, lda);
        return AWQ_ERR_SHAPE;
    }
    return awq_launch_gemm_single(ctx, out, ldo, a, lda, M, w, K, N, accum, false, false);
}

int awq_gemm_int4_static(awq_ctx* ctx, uint16_t* out, int ldo, const uint16_t* a, int lda, int M, const awq_qweight* w, int K,
                         int N, int accum) {
    if (int r = awq_bind(ctx)) return r;
    AWQ_REQUIRE(out && a && w && w->weight && w->zeros && w->scales, AWQ_ERR_ARG, "null pointer");
    if (M <= 0 || K <= 0 || N <= 0 || (K & 31) || (N & 127) || (lda & 7)) {
        awq_set_error("awq_gemm_int4_static: needs M > 0, K %% 32 == 0, N %% 128 == 0, lda %% 8 == 0 (got M=%d K=%d N=%d lda=%d)", M, K, N,
                      lda);
        return AWQ_ERR_SHAPE;
    }
    AWQ_REQUIRE(ctx->device >= 0 && ctx->device < kMaxDevices && g_scratch_ptr[ctx->device] && g_gemm_lds_raised[ctx->device],
                AWQ_ERR_HIP, "the static workspace was not set up on this device when the context was created");
    return awq_launch_gemm_single(ctx, out, ldo, a, lda, M, w, K, N, accum, true, false);
}

int awq_gemm_int4_form(int compute_units, int M, int K, int N, int form[4]) {
    AWQ_REQUIRE(form && compute_units > 0, AWQ_ERR_ARG, "null form or no compute units");
    if (M <= 0 || K <= 0 || N <= 0 || (K & 31) || (N & 127)) {
        awq_set_error("awq_gemm_int4_form: needs M > 0, K %% 32 == 0, N %% 128 == 0 (got M=%d K=%d N=%d)", M, K, N);
        return AWQ_ERR_SHAPE;
    }
    const GemmRoute route = route_gemm(compute_units, M, K, N / pf::BN, true);
    form[0] = pf::BM;
    form[1] = pf::BN;
    form[2] = 1;
    if (route.form >= 0) awq_rows_form(route.form, form);
    form[3] = route.ksplit;
    return AWQ_OK;
}

}  // extern "C"
