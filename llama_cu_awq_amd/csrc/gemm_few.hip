#include "common.hpp"
#include "gemm_tile.hpp"

typedef float f32x2 __attribute__((ext_vector_type(2)));

namespace pf {

template <int MT_, int NU_>
struct FewForm {
    static constexpr int MT = MT_, NU = NU_;  // 32-row tiles; units of a workgroup
    static constexpr int WAVES = 8;
    static constexpr int SLOTS = 2;                      // quantisation groups of packed weights in a wave's ring
    static constexpr int AD = MT <= 2 ? 8 : (MT * NU < 8 ? 4 : 2);  // activation fragments in flight (8 a group): what the registers hold
    static constexpr int W_BYTES = NU * 2048;            // a group of the workgroup's rows
    static constexpr int ROW = 36, TILE = 32 * ROW;      // floats of a sum's row and tile in LDS (rows padded: no bank conflicts)
    // units and tiles whose sums pass through LDS at a time
    static constexpr int RU = MT % 2 == 1 && NU % 2 == 0 ? 2 : 1, RT = MT % 2 == 0 ? 2 : 1, ROUNDS = (NU / RU) * (MT / RT);
    static constexpr int MEET = WAVES * RU * RT * TILE * 4;
    static constexpr int RING = WAVES * SLOTS * W_BYTES;
    static constexpr int LDS = RING > (ROUNDS > 1 ? 2 : 1) * MEET ? RING : (ROUNDS > 1 ? 2 : 1) * MEET;
};

// C[m][n] = sum_k A[m][k] * half((q[n][k] - z) * s) of up to 128 rows: prefill.hip's product, rounding points and epilogues.  A
// workgroup of 8 waves owns NU units of 32 weight rows; its waves (and ksplit workgroups) share K, a contiguous run of
// quantisation groups each, and their sums meet in LDS.
//  * No wave reads what another one loaded, so there is no barrier before the sums meet and each wave waits for its own requests
//    alone.  A comes in fragment order (the kernels before write it so) straight into registers, 1 KB an instruction, a whole
//    group ahead; in rows of a matrix the 64 lanes of an operand would lie on 64 cache lines.
//  * Packed weights go through LDS, the group after the one in hand, because a load straight into operand order has consecutive
//    lanes on different rows: 64 cycles an instruction instead of 16.
//  * 32x32x16 products, weights as the first operand: between two of them another wave's dequantisation finds room.  (In 16x16x32
//    products the two hardly overlap: 3 of them and 13 vector instructions take 81 ns a wave, 2 of 32x32x16 and the same 69.)
// What bounds it (7B gate/up, 37 rows, 22 us = 44 000 clocks, by counters): with two waves a SIMD its matrix core is busy 12 300
// clocks and its vector instructions take 15 000, of which 10 000 are the 13 that dequantise a packed dword; the two overlap in part.
// Waves wait a quarter of their life for memory or LDS: about 4 us until the first activations and weights are there, 3 us until the
// sums have met.  More waves of fewer registers, column groups that share A through L1, or weights left in cache change nothing.
// Measured, us, the row forms -> this one: 7B shape, 37 rows QKV 17.9 -> 15.6, O 9.5 -> 8.5, gate/up 30.3 -> 21.5, down 16.5 ->
// 14.5; 64 rows gate/up 30.2 -> 22.4.  96 rows, from memory, QKV 26.9 -> 20.0, O 12.3 -> 10.2, gate/up 41.9 -> 33.2, 13824 columns of 5120 35.9 -> 24.5;
// 128 rows QKV 27.8 -> 23.0, 13824 of 5120 36.3 -> 28.0, but gate/up 42.2 -> 44.2: two rounds of workgroups, since three units a workgroup
// would need more registers than there are.
// KIND: EPI_QKV, EPI_FFN (out in fragment order), or EPI_STORE for the single-matrix forms (p.epi says which).
template <class F, int KIND>
__global__ __launch_bounds__(F::WAVES * 64, 2) void gemm_few_kernel(const GemmParams p) {
    constexpr int MT = F::MT, NU = F::NU, W = F::WAVES, SLOTS = F::SLOTS, AD = F::AD;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_bytes[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int first = (int)blockIdx.x * NU, ks = (int)blockIdx.z;

    // A unit is 32 weight rows, two runs of 16 whose results meet in the epilogue: consecutive rows (single matrices, V), the gate
    // and up rows of the same indices (FFN), or the two halves of rotation pairs (Q and K with RoPE).
    struct Unit {
        int mat, row0, row1;
    };
    auto unit_of = [&](int u) {
        if (KIND == EPI_FFN) return Unit{0, u * 16, u * 16};
        int mat = 0;
        if (KIND == EPI_QKV) {
            const int t0 = p.N[0] >> 5, t1 = p.N[1] >> 5;
            if (u >= t0 + t1) {
                mat = 2;
                u -= t0 + t1;
            } else if (u >= t0) {
                mat = 1;
                u -= t0;
            }
            if (p.rope && mat < 2) {
                const int shift = __builtin_ctz(p.head_size) - 5;  // (heads of 64, 128, 256)
                const int row = (u >> shift) * p.head_size + (u & ((1 << shift) - 1)) * 16;
                return Unit{mat, row, row + (p.head_size >> 1)};
            }
        }
        return Unit{mat, u * 32, u * 32 + 16};
    };
    // This wave's quantisation groups: the first `extra` slices have one more.
    const int slice = ks * W + wave;
    const int k_begin = slice * p.few_per + min(slice, p.few_extra);
    const int nk = p.few_per + (slice < p.few_extra ? 1 : 0), k_end = k_begin + nk;
    const int k_last = p.sh - 1;

    // Packed weights travel global -> LDS, 16 rows (one run) an instruction, 4 lanes x 16 bytes a row; 16-byte piece c of row r lies
    // at c ^ ((r >> 1) & 3) (free of bank conflicts).  Scales and zeros of four groups come into registers, row r's in lanes
    // 2 r and 2 r + 1: two scales each, and the zeros dwords of the first and of the last group.
    const int lrow = lane >> 2, quarter = lane & 3;
    const uint32_t rb = (uint32_t)p.C * 16;
    const uint32_t w_lane = (uint32_t)lrow * rb + ((quarter ^ ((lrow >> 1) & 3)) << 4);
    const uint32_t z_lane = (uint32_t)((lane >> 1) & 15) * (p.pzh * 4), s_lane = (uint32_t)((lane >> 1) & 15) * (p.sh * 2);
    const uint8_t *wu[NU][2], *zu[NU][2], *su[NU][2];
#pragma unroll
    for (int u = 0; u < NU; u++) {
        const Unit un = unit_of(min(first + u, p.ntiles - 1));
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int mat = KIND == EPI_FFN ? b : un.mat, row = b ? un.row1 : un.row0;
            wu[u][b] = reinterpret_cast<const uint8_t*>(mat == 0 ? p.w[0] : (mat == 1 ? p.w[1] : p.w[2])) + (size_t)row * rb;
            zu[u][b] = reinterpret_cast<const uint8_t*>(mat == 0 ? p.z[0] : (mat == 1 ? p.z[1] : p.z[2])) + (size_t)row * (p.pzh * 4);
            su[u][b] = reinterpret_cast<const uint8_t*>(mat == 0 ? p.s[0] : (mat == 1 ? p.s[1] : p.s[2])) + (size_t)row * (p.sh * 2);
        }
    }
    typedef __attribute__((address_space(3))) void lptr;
    const uint32_t ring = (uint32_t)wave * (SLOTS * F::W_BYTES);
    // Loads are unconditional (one that sits in a branch is waited for with everything before it); those past the slice's end all
    // read one line that is there already.
    auto load_w = [&](int k, int slot) {
        const uint32_t in = (uint32_t)((k - k_end) >> 31), at = (uint32_t)k * 64 & in, off = w_lane & in;
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int b = 0; b < 2; b++)
                dma16(wu[u][b] + at, off, ring + slot * F::W_BYTES + u * 2048 + b * 1024);
    };
    // rows past M are computed, never stored: their lanes read the last row's line
    const uint32_t a_lane = (uint32_t)lane * 16, a_last = (uint32_t)((lane & 32) + min(lane & 31, p.M - 1 - (MT - 1) * 32)) * 16;
    const uint8_t* const abase = reinterpret_cast<const uint8_t*>(p.A);
    h16x8 a[AD][MT];
    auto load_a = [&](int f, int k) {
        k += f >> 3;
        const uint32_t in = (uint32_t)((k - k_end) >> 31);
        const uint8_t* src = abase + ((uint32_t)((k * 8 + (f & 7)) * p.a_tiles) * 1024u & in);
#pragma unroll
        for (int i = 0; i < MT; i++) a[f % AD][i] = *reinterpret_cast<const h16x8*>(src + ((i == MT - 1 ? a_last : a_lane) & in) + i * 1024);
    };
    uint32_t cs[NU], cz[NU];
    auto load_c = [&](int k) {
        const uint32_t ks0 = (uint32_t)min(k + 2 * (lane & 1), k_last - 1), kz = (uint32_t)min(k + 3 * (lane & 1), k_last) >> 3;
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const uint8_t *s = lane < 32 ? su[u][0] : su[u][1], *z = lane < 32 ? zu[u][0] : zu[u][1];
            __builtin_memcpy(&cs[u], s + s_lane + ks0 * 2, 4);
            cz[u] = *reinterpret_cast<const uint32_t*>(z + z_lane + kz * 4);
        }
    };
    // what the matrix instruction takes: row l % 32 of the unit, half l / 32
    const int r32 = lane & 31, half = lane >> 5;
    const uint32_t piece0 = (uint32_t)(uintptr_t)(lptr*)(lds_bytes + ring) + (uint32_t)(r32 * 64 + ((half ^ ((r32 >> 1) & 3)) << 4));
    u32x4 cur[NU][2];
    auto read_w = [&](int slot) {
        const uint32_t a0 = piece0 + slot * F::W_BYTES, a1 = a0 ^ 32u;
        static_assert(NU <= 3, "");
        if constexpr (NU == 1)
            asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)" : "=&v"(cur[0][0]), "=&v"(cur[0][1]) : "v"(a0), "v"(a1) : "memory");
        else if constexpr (NU == 2)
            asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %4 offset:2048\n\tds_read_b128 %3, %5 offset:2048\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(cur[0][0]), "=&v"(cur[0][1]), "=&v"(cur[1][0]), "=&v"(cur[1][1]) : "v"(a0), "v"(a1) : "memory");
        else
            asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %7\n\tds_read_b128 %2, %6 offset:2048\n\tds_read_b128 %3, %7 offset:2048\n\t"
                         "ds_read_b128 %4, %6 offset:4096\n\tds_read_b128 %5, %7 offset:4096\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(cur[0][0]), "=&v"(cur[0][1]), "=&v"(cur[1][0]), "=&v"(cur[1][1]), "=&v"(cur[NU - 1][0]), "=&v"(cur[NU - 1][1]) : "v"(a0), "v"(a1) : "memory");
    };
    Group gc[NU];
    auto constants = [&](int t, int k) {
        const int s_shift = 16 * (k - min(k - (t & 1), k_last - 1));  // (the last pair is that of the row's last two scales)
        const int s_from = (r32 * 2 + ((t >> 1) & 1)) * 4, z_from = (r32 * 2 + ((k >> 3) != ((k - (t & 3)) >> 3))) * 4;
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const uint32_t sc = (uint32_t)__builtin_amdgcn_ds_bpermute(s_from, (int)cs[u]), zr = (uint32_t)__builtin_amdgcn_ds_bpermute(z_from, (int)cz[u]);
            gc[u] = group_consts((zr >> (4 * (k & 7))) & 0xFu, (uint16_t)(sc >> s_shift));
        }
    };

    // Requests stay where they are written, in this order: the wait for the weights below counts them, and the compiler would move
    // them to where their results are used.
    auto pin = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    uint32_t magic = 0x64006400u;
    asm("" : "+v"(magic));
    load_c(k_begin);
    load_w(k_begin, 0);
#pragma unroll
    for (int f = 0; f < AD; f++) {
        load_a(f, k_begin);
        pin();
    }
    f32x16 acc[NU][MT];
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 16; j++) acc[u][i][j] = 0.0f;
    for (int t = 0; t < nk; t++) {
        const int k = k_begin + t;
        load_w(k + 1, (t + 1) & 1);
        constants(t, k);
        if ((t & 3) == 3) load_c(k + 1);
        // the group's weights are in LDS: behind their request came the activations of a group and the next one's weights
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NU + AD * MT) : "memory");
        read_w(t & 1);
        h16x8 b[2];
        b[0] = __builtin_bit_cast(h16x8, dequant8(cur[0][0][0], gc[0], magic));
#pragma unroll
        for (int s = 0; s < 8 * NU; s++) {  // a step: fragment s / NU of unit s % NU; the next one's weights are made under its products
            const int f = s / NU, u = s % NU, fn = (s + 1) / NU, un = (s + 1) % NU;
            if (s + 1 < 8 * NU) b[(s + 1) & 1] = __builtin_bit_cast(h16x8, dequant8(cur[un][fn >> 2][fn & 3], gc[un], magic));
#pragma unroll
            for (int i = 0; i < MT; i++) acc[u][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[s & 1], a[f % AD][i], acc[u][i], 0, 0, 0);
            if (u == NU - 1) {
                load_a(f + AD, k);
                pin();
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // no direct-to-LDS load is still on its way
    __syncthreads();

    // ---- epilogue: the waves' sums pass through LDS, [wave][unit][tile][row][32 columns], and are added in K order.  A lane takes
    // four columns of both runs: consecutive ones, or (FFN) those whose results are neighbours in the order a packed dword has.
    constexpr int TR = MT / F::RT;  // rounds of a unit
    float* lds = reinterpret_cast<float*>(lds_bytes);
    auto put = [&](int round) {
        float* mine = lds + (round & 1) * (F::MEET / 4) + wave * F::RU * F::RT * F::TILE + r32 * F::ROW + half * 4;
#pragma unroll
        for (int u = 0; u < F::RU; u++)
#pragma unroll
            for (int i = 0; i < F::RT; i++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const f32x16& v = acc[round / TR * F::RU + u][round % TR * F::RT + i];
                    *reinterpret_cast<f32x4*>(mine + (u * F::RT + i) * F::TILE + q * 8) = f32x4{v[q * 4], v[q * 4 + 1], v[q * 4 + 2], v[q * 4 + 3]};
                }
    };
    auto pack4 = [](const float (&v)[4]) {
        return u32x2{(uint32_t)float_to_half_bits(v[0]) | ((uint32_t)float_to_half_bits(v[1]) << 16), (uint32_t)float_to_half_bits(v[2]) | ((uint32_t)float_to_half_bits(v[3]) << 16)};
    };
    auto finish = [&](const Unit& un, int q, int m, float (&v)[2][4]) {
        if (KIND == EPI_FFN) {  // columns 2 h, 4 + 2 h, 1 + 2 h, 5 + 2 h of an octet
            float r[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float gt = v[0][e];
                const float s = gt * (1.0f / (1.0f + expf(-gt)));
                r[e] = s * v[1][e];
            }
            *reinterpret_cast<u32x2*>(p.out[0] + fragment_offset(m, un.row0 + (q >> 1) * 8, p.out_tiles) + (q & 1) * 4) = pack4(r);
            return;
        }
        const int c0 = un.row0 + q * 4, c1 = un.row1 + q * 4;
        if (KIND == EPI_STORE && p.epi == EPI_PART) {
            float* dst = p.part + ((size_t)ks * p.M + m) * p.N[0];
            *reinterpret_cast<f32x4*>(dst + c0) = f32x4{v[0][0], v[0][1], v[0][2], v[0][3]};
            *reinterpret_cast<f32x4*>(dst + c1) = f32x4{v[1][0], v[1][1], v[1][2], v[1][3]};
            return;
        }
        const int mat = un.mat;
        uint16_t* const o = (mat == 0 ? p.out[0] : (mat == 1 ? p.out[1] : p.out[2])) +
                            (size_t)(mat == 0 ? p.out_off[0] : (mat == 1 ? p.out_off[1] : p.out_off[2])) +
                            (size_t)m * (size_t)(mat == 0 ? p.ldo[0] : (mat == 1 ? p.ldo[1] : p.ldo[2]));
        if (KIND == EPI_QKV && p.rope && mat < 2) {
            // rounded to fp16 first and rotated in fp32, as the separate kernel does on the stored q and k (gpu_kernels.h:351-361)
            const f32x4* cs4 = reinterpret_cast<const f32x4*>(p.rope + (size_t)(p.rope_pos0 + m) * (p.head_size >> 1) + (c0 & (p.head_size - 1)));
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x = half_bits_to_float(float_to_half_bits(v[0][e])), y = half_bits_to_float(float_to_half_bits(v[1][e]));
                rope_rotate(x, y, cs4[e >> 1][(e & 1) * 2], cs4[e >> 1][(e & 1) * 2 + 1], v[0][e], v[1][e]);
            }
        }
        if (KIND == EPI_STORE && p.epi == EPI_RESID) {
            const u32x2 x0 = *reinterpret_cast<const u32x2*>(o + c0), x1 = *reinterpret_cast<const u32x2*>(o + c1);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[0][e] += half_bits_to_float((uint16_t)(x0[e >> 1] >> (16 * (e & 1))));
                v[1][e] += half_bits_to_float((uint16_t)(x1[e >> 1] >> (16 * (e & 1))));
            }
        }
        *reinterpret_cast<u32x2*>(o + c0) = pack4(v[0]);
        *reinterpret_cast<u32x2*>(o + c1) = pack4(v[1]);
    };
    put(0);
#pragma unroll
    for (int round = 0; round < F::ROUNDS; round++) {
        __syncthreads();
        if (round + 1 < F::ROUNDS) put(round + 1);
        if (tid < F::RU * F::RT * 128) {
            const int q = tid & 3, r = (tid >> 2) % (F::RT * 32), u = tid / (F::RT * 128);
            const float* src = lds + (round & 1) * (F::MEET / 4) + (u * F::RT + (r >> 5)) * F::TILE + (r & 31) * F::ROW;
            float v[2][4];
#pragma unroll
            for (int k = 0; k < W; k++) {
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    const float* at = src + k * F::RU * F::RT * F::TILE + b * 16;
                    f32x4 t;
                    if (KIND == EPI_FFN) {
                        const f32x2 lo = *reinterpret_cast<const f32x2*>(at + (q >> 1) * 8 + (q & 1) * 2), hi = *reinterpret_cast<const f32x2*>(at + (q >> 1) * 8 + (q & 1) * 2 + 4);
                        t = f32x4{lo[0], hi[0], lo[1], hi[1]};
                    } else {
                        t = *reinterpret_cast<const f32x4*>(at + q * 4);
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++) v[b][e] = k == 0 ? t[e] : v[b][e] + t[e];
                }
            }
            const int unit = first + round / TR * F::RU + u, m = round % TR * F::RT * 32 + r;
            if (unit < p.ntiles && m < p.M) finish(unit_of(unit), q, m, v);
        }
    }
}

}  // namespace pf

// ---------------------------------------------------------------- which form a product takes
namespace {

// us: what a round of workgroups (one on every compute unit) takes, its part that does not scale with K and that of a
// quantisation group of each wave's
struct FewFormInfo {
    int units;
    float fixed, group;
};
// Measured over 128 .. 504 workgroups, 1 .. 8 groups a wave, weights from memory; 2.5 us besides for the launch itself.
constexpr int kFewForms = 3;
const FewFormInfo kFew[4][kFewForms] = {  // by 32-row tiles (four by three units: more registers than there are)
    {{1, 0.9f, 1.6f}, {2, 1.2f, 2.7f}, {3, 1.6f, 4.0f}},
    {{1, 1.6f, 2.2f}, {2, 2.4f, 3.4f}, {3, 3.3f, 4.7f}},
    {{1, 1.3f, 3.0f}, {2, 1.9f, 4.0f}, {3, 3.8f, 5.8f}},
    {{1, 1.2f, 3.5f}, {2, 2.2f, 4.6f}, {0, 0.0f, 0.0f}},
};
constexpr int kFewMaxSplit = 4;

template <int MT, int NU>
void few_launch(awq_ctx* ctx, const pf::GemmParams& p) {
    using F = pf::FewForm<MT, NU>;
    const dim3 grid(div_up(p.ntiles, NU), 1, p.ksplit), block(F::WAVES * 64);
    if (p.epi == pf::EPI_QKV)
        hipLaunchKernelGGL((pf::gemm_few_kernel<F, pf::EPI_QKV>), grid, block, F::LDS, ctx->stream, p);
    else if (p.epi == pf::EPI_FFN)
        hipLaunchKernelGGL((pf::gemm_few_kernel<F, pf::EPI_FFN>), grid, block, F::LDS, ctx->stream, p);
    else
        hipLaunchKernelGGL((pf::gemm_few_kernel<F, pf::EPI_STORE>), grid, block, F::LDS, ctx->stream, p);
}

template <int MT, int NU>
hipError_t few_raise() {
    using F = pf::FewForm<MT, NU>;
    const void* kernels[3] = {(const void*)pf::gemm_few_kernel<F, pf::EPI_QKV>, (const void*)pf::gemm_few_kernel<F, pf::EPI_FFN>,
                              (const void*)pf::gemm_few_kernel<F, pf::EPI_STORE>};
    for (const void* k : kernels) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, F::LDS);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

int awq_gemm_few_setup() {
    hipError_t (*const raise[])() = {few_raise<1, 1>, few_raise<1, 2>, few_raise<1, 3>, few_raise<2, 1>,
                                    few_raise<2, 2>, few_raise<2, 3>, few_raise<3, 1>, few_raise<3, 2>, few_raise<3, 3>, few_raise<4, 1>, few_raise<4, 2>};
    for (auto f : raise) {
        const hipError_t e = f();
        if (e != hipSuccess) {
            awq_set_error("hipFuncSetAttribute(gemm_few) failed: %s", hipGetErrorString(e));
            return AWQ_ERR_HIP;
        }
    }
    return AWQ_OK;
}

awq_few_plan awq_plan_gemm_few(int cus, int M, int K, int N, bool may_split) {
    awq_few_plan best{0, 1, 1e30f};
    if (M > kFewRows || K < 256 || (K & 127) || (N & 31)) return best;
    const int groups = K / 128, units = N / 32;
    for (int i = 0; i < kFewForms; i++) {
        const FewFormInfo& f = kFew[div_up(M, 32) - 1][i];
        if (!f.units) break;
        for (int s = 1; s <= (may_split ? kFewMaxSplit : 1); s++) {
            const size_t part = s == 1 ? 0 : (size_t)s * M * N * sizeof(float);
            if (s > 1 && (part > kPartBytes || groups < 8 * s)) break;
            const int wgs = div_up(units, f.units) * s, rounds = div_up(wgs, cus);
            const float fill = (float)wgs / ((float)rounds * cus);  // a chip that is not full has its bandwidth for fewer
            const float us = 2.5f + rounds * (f.fixed + div_up(groups, 8 * s) * f.group * (0.8f + 0.2f * fill)) + (s == 1 ? 0.0f : 0.5f + 0.3e-6f * part);
            if (us < best.us) best = awq_few_plan{f.units, s, us};
        }
    }
    return best;
}

int awq_launch_gemm_few(awq_ctx* ctx, pf::GemmParams& p, int N, const awq_few_plan& plan, const char* what) {
    p.ntiles = N / 32;
    p.ksplit = plan.ksplit;
    p.a_tiles = div_up(p.M, 32);
    p.out_tiles = p.a_tiles;
    p.few_per = p.sh / (8 * plan.ksplit);
    p.few_extra = p.sh % (8 * plan.ksplit);
    switch (p.a_tiles * 4 + plan.units) {
        case 5: few_launch<1, 1>(ctx, p); break;
        case 6: few_launch<1, 2>(ctx, p); break;
        case 7: few_launch<1, 3>(ctx, p); break;
        case 9: few_launch<2, 1>(ctx, p); break;
        case 10: few_launch<2, 2>(ctx, p); break;
        case 11: few_launch<2, 3>(ctx, p); break;
        case 13: few_launch<3, 1>(ctx, p); break;
        case 14: few_launch<3, 2>(ctx, p); break;
        case 15: few_launch<3, 3>(ctx, p); break;
        case 17: few_launch<4, 1>(ctx, p); break;
        case 18: few_launch<4, 2>(ctx, p); break;
        default: awq_set_error("%s: no few-row form of %d units", what, plan.units); return AWQ_ERR_ARG;
    }
    return awq_check_launch(what);
}
