#include <type_traits>

#include "common.hpp"
#include "gemm_tile.hpp"

namespace pf {

// A wave's 64 columns are two blocks of 32 weight rows whose results meet in the epilogue: consecutive rows (plain forms,
// V), the gate and up rows of the same indices (FFN), or the two halves of rotation pairs (Q and K with RoPE).
struct ColGroup {
    int mat0, mat1, row0, row1;
};

__device__ __forceinline__ ColGroup col_group(const GemmParams& p, int g) {
    if (p.epi == EPI_FFN) return ColGroup{0, 1, g * 32, g * 32};
    int mat = 0;
    if (p.epi == EPI_QKV) {
        const int t0 = p.N[0] >> 6, t1 = p.N[1] >> 6;
        if (g >= t0 + t1) {
            mat = 2;
            g -= t0 + t1;
        } else if (g >= t0) {
            mat = 1;
            g -= t0;
        }
        if (p.rope && mat < 2) {
            const int per_head = p.head_size >> 6;
            const int row = (g / per_head) * p.head_size + (g % per_head) * 32;
            return ColGroup{mat, mat, row, row + (p.head_size >> 1)};
        }
    }
    return ColGroup{mat, mat, g * 64, g * 64 + 32};
}

// The activation tile in LDS is [rows][64 halves], 16-byte chunks XOR-ed with a key of the row: the 32 rows of a fragment
// read spread over all banks.
__device__ __forceinline__ int rows_key(int row) { return (row ^ ((row & 31) >> 3)) & 7; }

template <int MT_, int NW_, int KW_, int AS_, int WS_>
struct RowsForm {
    static constexpr int MT = MT_, NW = NW_, KW = KW_;  // row blocks per wave; waves along columns, K
    static constexpr int AS = AS_, WS = WS_;            // slots of the activation (steps) and weight (pairs of steps) rings
    static constexpr int WAVES = NW * KW;
    static constexpr int BMR = MT * 32;        // tile rows
    static constexpr int A_BYTES = BMR * 128;  // activation tile of a step and K slice
    static constexpr int W_BYTES = 4096;       // packed weights of 64 rows for a pair of steps
    static constexpr int ZS_BYTES = 6 * 256;   // scales (5 dwords a row) and zeros (one) of 64 rows for 8 pairs
    static constexpr int A_RING = AS * A_BYTES, W_RING = WS * W_BYTES + 2 * ZS_BYTES;
    static constexpr int LDS = KW * (A_RING + NW * W_RING);
    static constexpr int PER_CU = 160 * 1024 / LDS, WAVES_PER_SIMD = PER_CU * WAVES / 4 > 0 ? PER_CU * WAVES / 4 : 1;
    static constexpr int RB = WAVES * MT * 8192 <= LDS ? MT : (MT % 2 == 0 ? MT / 2 : 1);  // row blocks per epilogue round
    static constexpr int ROUNDS = MT / RB;
    static_assert(WAVES * RB * 8192 <= LDS && MT % RB == 0, "the accumulators pass through LDS");
    // an epilogue item is 8 columns of a row in both blocks of a wave's columns; PER of them per lane and round
    static constexpr int ITEMS = RB * 128, PER = (ITEMS + 64 * KW - 1) / (64 * KW);
    static constexpr int PART_FLOATS = ROUNDS * PER * 16 * WAVES * 64;  // a workgroup's partial tile
};

// C[m][n] = sum_k A[m][k] * half((q[n][k] - z) * s): prefill.hip's product, rounding points and epilogues, in tiles whose
// waves own 64 columns, so that an activation fragment read from LDS feeds two matrix instructions (in the 128 x 128
// kernel's waves of 32 columns it feeds one, which takes the LDS's whole bandwidth at full matrix rate).
//  * A wave's tile is 32 MT rows x 64 columns; NW waves side by side make the workgroup's tile and KW such groups take a
//    slice of K each and meet in LDS at the end (few rows: the chip is filled along K without partial tiles in memory).
//  * Activations and packed weights travel global -> LDS directly into rings of AS steps and WS pairs of steps; the rings
//    are as short as two workgroups per compute unit need (128 x 256: two slots each, 76 KB; what a third slot would hide,
//    the other workgroup hides).  One barrier per step where waves share a tile, none where they do not.
//  * Weights are dequantised from the wave's own packed dwords, one matrix fragment ahead of the products that use it; the
//    last products of a step run behind its barrier, under the first reads of the next.
//  * Scales and zeros come for eight groups at a time.
// What bounds it: many rows, the matrix cores at the clock they leave (1.0 PFLOP/s of the 1.65 the instruction alone
// reaches; per step of a 128 x 256 tile 32 matrix instructions, 104 dequantising ones and 16 KB of fragments a wave); few
// rows, the serial chain of a step (request, read, dequantise, multiply) at four to eight waves per compute unit:
// weights from memory or from cache take the same time.
// Measured, us, the 128 x 128 kernel -> this one: 7B shape, 64 rows QKV 38.6 -> 17.8, O 24.5 -> 14.2, gate/up 39.8 -> 30.2,
// down 54.3 -> 20.1; 300 rows gate/up 105 -> 76; 2000 rows QKV 233 -> 194, O 81 -> 74, gate/up 415 -> 358, down 213 ->
// 184; 70B shape, 2000 rows gate/up 2102 -> 1624.
// APERM: A's chunks of 8 are in the order a packed dword dequantises in; WHOLE: K is a multiple of 128 (nothing to mask).
template <class F, bool APERM, bool WHOLE>
__global__ __launch_bounds__(F::WAVES * 64, F::WAVES_PER_SIMD) void gemm_rows_kernel(const GemmParams p) {
    constexpr int MT = F::MT, NW = F::NW, KW = F::KW, AS = F::AS, WS = F::WS;
    constexpr int NT = F::WAVES * 64;
    constexpr int AL = 4 * MT / NW;           // activation loads per wave and step
    constexpr int WL = 4;                     // weight loads per wave and pair of steps
    constexpr bool SHARED = NW > 1;           // waves read what other waves loaded: a barrier per step
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_bytes[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / NW, nw = wave % NW;
    // Workgroup ids go round-robin over the 8 XCDs; each XCD takes an eighth of the workgroups, in an order that keeps the
    // row tiles and K parts of a weight tile together (its rows leave memory once).  Whole weight tiles per XCD would
    // leave some XCDs a round more than the others (44 tiles of 11 row tiles, 64 places per XCD: 62 us instead of 41).
    const int per_tile = p.mtiles * p.ksplit, total = p.ntiles * per_tile, per_xcd = (total + 7) >> 3;
    const int id = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || id >= total) return;
    const int tile = id / per_tile;
    const int m_index = (id % per_tile) / p.ksplit, ks = (id % per_tile) % p.ksplit;
    const int m0 = m_index * F::BMR;
    const ColGroup cg = col_group(p, tile * NW + nw);

    const uint32_t a_ring = (uint32_t)(kw * F::A_RING);
    const uint32_t w_ring = (uint32_t)(KW * F::A_RING + (kw * NW + nw) * F::W_RING);

    // activation loader: instruction q of the slice's wave nw covers tile rows (nw * AL + q) * 8 .. + 8, 8 lanes x 16 bytes
    // per row; the lane's LDS chunk is lane & 7, so it fetches the source chunk that the swizzle maps there
    uint32_t a_off[AL];  // byte offset from p.A of the lane's chunk in the first step
#pragma unroll
    for (int q = 0; q < AL; q++) {
        const int r = (nw * AL + q) * 8 + (lane >> 3);
        a_off[q] = (uint32_t)(((size_t)min(m0 + r, p.M - 1) * p.lda + ((lane & 7) ^ rows_key(r)) * 8) * 2);  // rows past M are computed, never stored
    }
    // weight loader: 16 rows of a block per instruction, 4 lanes x 16 bytes per row; 16-byte unit u of a row's 64 bytes
    // sits at LDS unit u ^ ((row >> 1) & 3)
    auto mat_of = [&](int mat, const auto* const(&a)[3]) { return mat == 0 ? a[0] : (mat == 1 ? a[1] : a[2]); };
    const uint32_t* wblk[2] = {uniform_ptr(mat_of(cg.mat0, p.w) + (size_t)cg.row0 * (p.C * 4)),
                               uniform_ptr(mat_of(cg.mat1, p.w) + (size_t)cg.row1 * (p.C * 4))};
    uint32_t w_off[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int r = 16 * q + (lane >> 2);
        w_off[q] = (uint32_t)((r * p.C + ((lane & 3) ^ ((r >> 1) & 3))) * 16);
    }
    const int lrow = lane & 31, lhalf = lane >> 5;
    auto row_of = [&](int r) { return (r < 32 ? cg.row0 : cg.row1 - 32) + r; };  // r: row of the wave's 64
    auto mat_row = [&](int r) { return r < 32 ? cg.mat0 : cg.mat1; };

    uint32_t magic = 0x64006400u;
    asm("" : "+v"(magic));
    f32x16 acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 16; j++) acc[i][0][j] = acc[i][1][j] = 0.0f;

    // This wave's K range, in pairs of steps (a pair is one quantisation group).
    const int npairs = p.sh, slices = KW * p.ksplit, slice = ks * KW + kw;
    const int p_begin = (int)((long long)slice * npairs / slices), p_end = (int)((long long)(slice + 1) * npairs / slices);
    const int trips = (SHARED && KW > 1) ? (npairs + slices - 1) / slices : p_end - p_begin;
    auto load_a = [&](int step) {
        const uint32_t dst = a_ring + (uint32_t)((step % AS) * F::A_BYTES + nw * (AL * 1024));
        if (WHOLE) {
            const uint16_t* base = p.A + min(step, 2 * npairs - 1) * BK;
#pragma unroll
            for (int q = 0; q < AL; q++) dma16(base, a_off[q], dst + q * 1024);
        } else {  // chunks past K are zero
#pragma unroll
            for (int q = 0; q < AL; q++) {
                const int r = (nw * AL + q) * 8 + (lane >> 3);
                const int k = step * BK + ((lane & 7) ^ rows_key(r)) * 8;
                const void* src = reinterpret_cast<const uint8_t*>(p.A) + a_off[q] + (size_t)step * (BK * 2);
                dma16(k < p.K ? src : (const void*)zeros16, dst + q * 1024);
            }
        }
    };
    auto load_w = [&](int pair) {
        const uint32_t dst = w_ring + (uint32_t)((pair % WS) * F::W_BYTES);
        const uint32_t g = (uint32_t)min(pair, npairs - 1);
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int q = 0; q < 2; q++) {
                if (WHOLE) {
                    dma16(wblk[b] + g * 16, w_off[q], dst + b * 2048 + q * 1024);
                } else {  // units past the row's end re-read its last one (against activations and scales that are zero)
                    const int r = 16 * q + (lane >> 2);
                    const uint32_t unit = g * 4 + ((lane & 3) ^ ((r >> 1) & 3));
                    dma16(wblk[b], ((uint32_t)(r * p.C) + min(unit, (uint32_t)p.C - 1)) * 16, dst + b * 2048 + q * 1024);
                }
            }
    };
    // Scales and zeros travel for 8 pairs at a time (a zeros dword covers that many): asked for pair by pair they are 64
    // lanes on 64 cache lines each.  A row's 8 scales may start on either half of a dword: 5 dwords, always.
    auto load_zs = [&](int oct) {
        const uint32_t dst = w_ring + (uint32_t)(WS * F::W_BYTES + (oct & 1) * F::ZS_BYTES);
        int l = lane;
        asm volatile("" : "+v"(l));  // (or its addresses would be kept in registers across the K loop)
#pragma unroll
        for (int i = 0; i < 6; i++) {
            if (i < 5) {
                const int idx = i * 64 + l, r = idx / 5;
                const size_t first = (size_t)row_of(r) * p.sh;
                const size_t d = min(((first + min(oct * 8, p.sh - 1)) >> 1) + idx % 5, (first + p.sh - 1) >> 1);
                dma4(reinterpret_cast<const uint32_t*>(mat_of(mat_row(r), p.s)) + d, dst + i * 256);
            } else {
                dma4(mat_of(mat_row(l), p.z) + (size_t)row_of(l) * p.pzh + min(oct, p.pzh - 1), dst + i * 256);
            }
        }
    };
    Group gc[2];
    u32x4 wq[2];
    const int s_odd[2] = {((cg.row0 + lrow) * p.sh) & 1, ((cg.row1 + lrow) * p.sh) & 1};  // (8 groups further on it is the same)
    auto read_w = [&](int step) {  // the lane's packed dwords of a step and, at the start of a pair, its group's constants
        const int pair = step >> 1;
        if ((step & 1) == 0) {
            const uint32_t* zs = reinterpret_cast<const uint32_t*>(lds_bytes + w_ring + WS * F::W_BYTES + ((pair >> 3) & 1) * F::ZS_BYTES);
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const int o = s_odd[b] + (pair & 7);
                const uint32_t sw = zs[(b * 32 + lrow) * 5 + (o >> 1)], zw = zs[320 + b * 32 + lrow];
                gc[b] = group_consts((zw >> (4 * (pair & 7))) & 0xFu, (uint16_t)(sw >> (16 * (o & 1))));
            }
        }
        const uint8_t* ws = lds_bytes + w_ring + (pair % WS) * F::W_BYTES + lrow * 64;
        const int unit = (step & 1) * 2 + lhalf;
        if (!WHOLE && step * BK + lhalf * 32 >= p.K) {  // past K: zero scales (a weight that is not finite is not undone by a zero activation)
            const h16x2 none = {(h16_t)0.0f, (h16_t)0.0f};
            gc[0].s2 = gc[1].s2 = none;
        }
#pragma unroll
        for (int b = 0; b < 2; b++) wq[b] = *reinterpret_cast<const u32x4*>(ws + b * 2048 + ((unit ^ ((lrow >> 1) & 3)) << 4));
    };
    // K mapping of the four fragments of a step: fragment j multiplies K chunk j (lanes 0-31) and chunk 4 + j (lanes
    // 32-63), i.e. dword j of each lane's 16 bytes against the matching 8 activations.
    struct Frag {
        h16x8 a[MT], b[2];
    };
    auto fetch = [&](Frag& f, int step, int j) {
        const uint16_t* at = reinterpret_cast<const uint16_t*>(lds_bytes + a_ring + (step % AS) * F::A_BYTES);
#pragma unroll
        for (int i = 0; i < MT; i++) f.a[i] = *reinterpret_cast<const h16x8*>(&at[i * 32 * BK + lrow * BK + (((j + 4 * lhalf) ^ rows_key(lrow)) << 3)]);
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const u32x4 dq = dequant8(wq[b][j], gc[b], magic);
            f.b[b] = __builtin_bit_cast(h16x8, APERM ? dq : unpermute8(dq));
        }
    };
    auto multiply = [&](const Frag& f) {
#pragma unroll
        for (int i = 0; i < MT; i++) {
            acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[i], f.b[0], acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[i], f.b[1], acc[i][1], 0, 0, 0);
        }
    };
    // The end of a step: what the next one needs is in LDS, `newer` later requests may still be on their way, and this wave's
    // LDS reads are done (the next requests overwrite what they read).
    auto step_end = [&](auto newer) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(newer)::value) : "memory");
        if (SHARED) __syncthreads();
    };
    // needed next: activation tile step + 1, requested AS - 2 steps ago; tile step + 2 and weight pair + 1
    constexpr std::integral_constant<int, AS == 3 ? AL + WL : WL> newer_even{};
    constexpr std::integral_constant<int, AS == 3 ? (WS == 3 ? AL + WL : AL) : 0> newer_odd{};

    const int s0 = p_begin * 2;
    load_zs(p_begin >> 3);
    load_w(p_begin);
    if (WS == 3) load_w(p_begin + 1);
    load_a(s0);
    if (AS == 3) load_a(s0 + 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // Fragments are read and dequantised one ahead of the products that use them, across steps too: the last products of a
    // step run behind its barrier, under the first reads of the next.
    Frag f[2];
    read_w(s0);
    fetch(f[0], s0, 0);
    for (int t = 0; t < trips; t++) {
        const int pair = p_begin + t, step = 2 * pair;
        if (SHARED && KW > 1 && pair >= p_end) {  // (this slice is a pair shorter than its neighbours)
            step_end(newer_even);
            step_end(newer_odd);
            continue;
        }
        if (t == 0 || (pair & 7) == 0) load_zs((pair >> 3) + 1);
        load_a(step + AS - 1);
        load_w(pair + WS - 1);
#pragma unroll
        for (int j = 0; j < 3; j++) {
            fetch(f[(j + 1) & 1], step, j + 1);
            multiply(f[j & 1]);
        }
        read_w(step + 1);
        step_end(newer_even);
        load_a(step + AS);
        fetch(f[0], step + 1, 0);
        multiply(f[1]);
#pragma unroll
        for (int j = 0; j < 3; j++) {
            fetch(f[(j + 1) & 1], step + 1, j + 1);
            multiply(f[j & 1]);
        }
        if (WS == 3) read_w(step + 2);
        step_end(newer_odd);
        if (WS == 2) read_w(step + 2);
        fetch(f[0], step + 2, 0);
        multiply(f[1]);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // no direct-to-LDS load is still on its way
    __syncthreads();

    // ---- epilogue: the accumulators pass through the idle rings as fp32 [wave][RB * 32 rows][64 columns]; an item is 8
    // columns of a row in both blocks, the K slices of which the item's lane adds up in slice order.
    constexpr int REG = F::RB * 32 * 64;  // floats per wave
    constexpr int ITEMS = F::ITEMS, PER = F::PER;  // items per column wave, shared by its KW slices
    float* tile_f = reinterpret_cast<float*>(lds_bytes);
    auto put = [&](int round) {
        float* mine = tile_f + wave * REG + (lane >> 5) * 256 + (lane & 31);
#pragma unroll
        for (int i = 0; i < F::RB; i++)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int j = 0; j < 16; j++) mine[(i * 32 + (j >> 2) * 8 + (j & 3)) * 64 + b * 32] = acc[round * F::RB + i][b][j];
    };
    auto get = [&](int item, float (&v)[2][8]) {  // the sum over the workgroup's K slices
#pragma unroll
        for (int k = 0; k < KW; k++) {
            const float* src = tile_f + (k * NW + nw) * REG + (item >> 2) * 64 + (item & 3) * 8;
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const f32x4 t = *reinterpret_cast<const f32x4*>(src + b * 32 + h * 4);
#pragma unroll
                    for (int e = 0; e < 4; e++) v[b][h * 4 + e] = k == 0 ? t[e] : v[b][h * 4 + e] + t[e];
                }
        }
    };
    auto pack8 = [](const float (&v)[8]) {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (uint32_t)float_to_half_bits(v[2 * e]) | ((uint32_t)float_to_half_bits(v[2 * e + 1]) << 16);
        return o;
    };
    uint16_t* const obase = (cg.mat0 == 0 ? p.out[0] : (cg.mat0 == 1 ? p.out[1] : p.out[2])) +
                            (size_t)(cg.mat0 == 0 ? p.out_off[0] : (cg.mat0 == 1 ? p.out_off[1] : p.out_off[2]));
    const size_t ld = (size_t)(cg.mat0 == 0 ? p.ldo[0] : (cg.mat0 == 1 ? p.ldo[1] : p.ldo[2]));
    auto finish = [&](int m, int chunk, float (&v)[2][8]) {
        if (m >= p.M) return;
        uint16_t* o0 = obase + (size_t)m * ld + cg.row0 + chunk * 8;
        uint16_t* o1 = obase + (size_t)m * ld + cg.row1 + chunk * 8;
        if (p.epi == EPI_FFN) {
            float r[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float g = v[0][e];
                const float s = g * (1.0f / (1.0f + expf(-g)));
                r[e] = s * v[1][e];
            }
            const u32x4 h = pack8(r);
            *reinterpret_cast<u32x4*>(o0) = p.out_perm ? permute8(h) : h;
            return;
        }
        if (p.epi == EPI_QKV && p.rope && cg.mat0 < 2) {
            // values are rounded to fp16 first and rotated in fp32, as the separate kernel does on the stored q and k
            // (gpu_kernels.h:351-361); (cos, sin) of 8 consecutive pairs are 64 contiguous bytes of the table
            const int pair0 = (cg.row0 & (p.head_size - 1)) + chunk * 8;
            const f32x4* cs = reinterpret_cast<const f32x4*>(p.rope + (size_t)(p.rope_pos0 + m) * (p.head_size >> 1) + pair0);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float a = half_bits_to_float(float_to_half_bits(v[0][e])), b = half_bits_to_float(float_to_half_bits(v[1][e]));
                rope_rotate(a, b, cs[e >> 1][(e & 1) * 2], cs[e >> 1][(e & 1) * 2 + 1], v[0][e], v[1][e]);
            }
        }
        if (p.epi == EPI_RESID) {
            const u32x4 x0 = *reinterpret_cast<const u32x4*>(o0), x1 = *reinterpret_cast<const u32x4*>(o1);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                v[0][e] += half_bits_to_float((uint16_t)(x0[e >> 1] >> (16 * (e & 1))));
                v[1][e] += half_bits_to_float((uint16_t)(x1[e >> 1] >> (16 * (e & 1))));
            }
        }
        *reinterpret_cast<u32x4*>(o0) = pack8(v[0]);
        *reinterpret_cast<u32x4*>(o1) = pack8(v[1]);
    };
    // Split K: each workgroup writes its fp32 sums through to memory and counts itself in; the last one adds all of them in
    // slice order, so that the result does not depend on who that is.
    const size_t tile_id = (size_t)tile * p.mtiles + m_index;
    float* tile_part = p.part + tile_id * p.ksplit * F::PART_FLOATS + tid;
#pragma unroll
    for (int round = 0; round < F::ROUNDS; round++) {
        if (round > 0) __syncthreads();
        put(round);
        __syncthreads();
#pragma unroll
        for (int it = 0; it < PER; it++) {
            const int item = (it * KW + kw) * 64 + lane;
            if (item < ITEMS) {
                float v[2][8];
                get(item, v);
                if (p.epi == EPI_PART) {
                    const int m = m0 + round * F::RB * 32 + (item >> 2);
                    float* dst = p.part + ((size_t)ks * p.M + m) * p.N[0] + (item & 3) * 8;
                    if (m < p.M) {
#pragma unroll
                        for (int b = 0; b < 2; b++)
#pragma unroll
                            for (int h = 0; h < 2; h++)
                                *reinterpret_cast<f32x4*>(dst + (b ? cg.row1 : cg.row0) + h * 4) =
                                    f32x4{v[b][h * 4], v[b][h * 4 + 1], v[b][h * 4 + 2], v[b][h * 4 + 3]};
                    }
                } else if (p.ksplit == 1) {
                    finish(m0 + round * F::RB * 32 + (item >> 2), item & 3, v);
                } else {
                    float* dst = tile_part + (size_t)ks * F::PART_FLOATS + (round * PER + it) * 16 * NT;
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        __hip_atomic_store(dst + e * NT, v[e >> 3][e & 7], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
    }
    if (p.ksplit == 1 || p.epi == EPI_PART) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    unsigned int* arrival = reinterpret_cast<unsigned int*>(lds_bytes);
    if (tid == 0) *arrival = __hip_atomic_fetch_add(&p.part_counter[tile_id], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*arrival != (unsigned int)p.ksplit - 1) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (tid == 0) p.part_counter[tile_id] = 0;  // ready for the next launch
#pragma unroll
    for (int round = 0; round < F::ROUNDS; round++)
#pragma unroll
        for (int it = 0; it < PER; it++) {
            const int item = (it * KW + kw) * 64 + lane;
            if (item < ITEMS) {
                const float* src = tile_part + (round * PER + it) * 16 * NT;
                float v[2][8];
#pragma unroll
                for (int e = 0; e < 16; e++) v[e >> 3][e & 7] = src[e * NT];
                for (int k = 1; k < p.ksplit; k++)
#pragma unroll
                    for (int e = 0; e < 16; e++) v[e >> 3][e & 7] += src[(size_t)k * F::PART_FLOATS + e * NT];
                finish(m0 + round * F::RB * 32 + (item >> 2), item & 3, v);
            }
        }
}

}  // namespace pf

// ---------------------------------------------------------------- which form a product takes
namespace {

template <class F>
int launch_form(awq_ctx* ctx, pf::GemmParams& p, int groups, int ksplit, bool a_perm, const char* what) {
    p.mtiles = div_up(p.M, F::BMR);
    p.ntiles = groups / F::NW;
    p.ksplit = ksplit;
    const dim3 grid(8 * div_up(p.mtiles * ksplit * p.ntiles, 8)), block(F::WAVES * 64);
    if (a_perm)
        hipLaunchKernelGGL((pf::gemm_rows_kernel<F, true, true>), grid, block, F::LDS, ctx->stream, p);
    else if ((p.K & 127) == 0)
        hipLaunchKernelGGL((pf::gemm_rows_kernel<F, false, true>), grid, block, F::LDS, ctx->stream, p);
    else
        hipLaunchKernelGGL((pf::gemm_rows_kernel<F, false, false>), grid, block, F::LDS, ctx->stream, p);
    return awq_check_launch(what);
}

template <class F>
hipError_t raise_lds() {
    const void* kernels[3] = {(const void*)pf::gemm_rows_kernel<F, true, true>, (const void*)pf::gemm_rows_kernel<F, false, true>,
                              (const void*)pf::gemm_rows_kernel<F, false, false>};
    for (const void* k : kernels) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, F::LDS);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Measured over K 2048 .. 28672, N 2560 .. 57344 and 16 .. 2000 rows with weights from memory: us per K step of 64 with
// single workgroups on few compute units, on all of them, and with two on each (where the LDS holds two).  The estimate
// made of them was within 15 % of the time of 145 of 148 products besides those it was fitted to (1 .. 2048 rows; up to 18 %
// low).  Forms closer together than that are a toss-up: between one and two workgroups on a compute unit the unsplit
// 64 x 128 form is put up to 15 % too low, and at 600 to 1000 rows of long K is taken where the 128 x 128 kernel is 2 to 8 %
// faster (879 x 11008 x 4096: 116 us, 107); step times that correct it lose as much where that kernel stalls (859 x 10592 x
// 4352: 126 us, 159).
struct Form {
    int rows, nw, kw, per_cu;
    awq_step_us step;
    size_t part_floats;
    int (*launch)(awq_ctx*, pf::GemmParams&, int, int, bool, const char*);
    hipError_t (*raise)();
};
template <int MT, int NW, int KW, int AS, int WS>
constexpr Form form(awq_step_us step) {
    using F = pf::RowsForm<MT, NW, KW, AS, WS>;
    return Form{F::BMR, NW, KW, F::PER_CU > 1 ? 2 : 1, step, (size_t)F::PART_FLOATS, launch_form<F>, raise_lds<F>};
}
const Form kForms[] = {
    form<1, 1, 4, 2, 2>({0.56f, 0.62f, 0.97f}),  // 32 x 64, four K slices
    form<2, 1, 4, 3, 3>({0.68f, 0.80f, 0.80f}),  // 64 x 64, four K slices
    form<2, 2, 2, 2, 2>({0.69f, 0.85f, 1.25f}),  // 64 x 128, two K slices
    form<2, 4, 1, 3, 2>({0.60f, 0.72f, 1.15f}),  // 64 x 256
    form<3, 4, 1, 3, 2>({0.68f, 0.85f, 1.50f}),  // 96 x 256
    form<4, 4, 1, 2, 2>({0.72f, 1.02f, 1.90f}),  // 128 x 256
};
constexpr int kMaxSplit = 4;

}  // namespace

// Expected time of `wgs` workgroups of `steps` K steps each.
float awq_gemm_us(int cus, int per_cu, long long wgs, int steps, const awq_step_us& t) {
    const long long slots = (long long)per_cu * cus, full = wgs / slots, rest = wgs % slots;
    const float f = (float)rest / cus;
    float per_step = full * t.twice;
    if (rest > 0) per_step += f <= 1.0f ? t.alone + (t.once - t.alone) * f : t.once + (t.twice - t.once) * (0.6f + 0.4f * (f - 1.0f));
    return 2.5f + 2.0f * (full + (rest > 0)) + steps * per_step;
}

int awq_gemm_rows_setup() {
    for (const Form& f : kForms) {
        const hipError_t e = f.raise();
        if (e != hipSuccess) {
            awq_set_error("hipFuncSetAttribute(gemm_rows) failed: %s", hipGetErrorString(e));
            return AWQ_ERR_HIP;
        }
    }
    return AWQ_OK;
}

awq_rows_plan awq_plan_gemm_rows(int cus, int M, int K, int groups, bool may_split, bool parts) {
    awq_rows_plan best{-1, 1, 1e30f};
    const int npairs = div_up(K, 128);
    for (int i = 0; i < (int)(sizeof(kForms) / sizeof(kForms[0])); i++) {
        const Form& f = kForms[i];
        if (groups % f.nw) continue;
        const long long tiles = (long long)(groups / f.nw) * div_up(M, f.rows);
        for (int s = 1; s <= (may_split ? kMaxSplit : 1); s++) {
            const long long wgs = tiles * s;
            // a split is for matrices that leave compute units idle, and has to fit the workspace
            const size_t part = s == 1 ? 0 : (parts ? (size_t)s * M * groups * 64 : wgs * f.part_floats) * sizeof(float);
            if (s > 1 && (tiles >= cus || (!parts && tiles > kPartTiles) || part > kPartBytes || npairs < 2 * f.kw * s)) break;
            // partial tiles that meet in the launch cost it 2 us and 0.65 per MB; sums left to the next launch cost the two
            // of them 0.5 us and 0.2 to 0.3 per MB (512 x 4096, four parts: its norm 5.1 -> 9.1 us)
            const float extra = s == 1 ? 0.0f : (parts ? 0.5f + 0.3e-6f * part : 2.0f + 0.65e-6f * part);
            const float us = awq_gemm_us(cus, f.per_cu, wgs, 2 * div_up(npairs, f.kw * s), f.step) + extra;
            if (us < best.us) best = awq_rows_plan{i, s, us};
        }
    }
    return best;
}

int awq_launch_gemm_rows(awq_ctx* ctx, pf::GemmParams& p, int groups, int form, int ksplit, bool a_perm, const char* what) {
    return kForms[form].launch(ctx, p, groups, ksplit, a_perm, what);
}

void awq_rows_form(int form, int* tile) {
    tile[0] = kForms[form].rows;
    tile[1] = kForms[form].nw * 64;
    tile[2] = kForms[form].kw;
}
