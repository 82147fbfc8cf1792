// Device-side building blocks of the int4-weight GEMMs over many activation rows (prefill.hip, gemm_rows.hip):
// the argument block, the bit-exact dequantisation of a packed dword, direct global -> LDS loads.
#pragma once

#include "common.hpp"

typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace pf {

constexpr int BM = 128;  // tokens per tile
constexpr int BN = 128;  // weight rows per tile
constexpr int BK = 64;   // K per step: 128 bytes of fp16 per LDS tile row

// EPI_PART: fp32 sums of each part of K, [part][row][column], for whoever reads the result to add up
enum Epi { EPI_STORE = 0, EPI_RESID = 1, EPI_QKV = 2, EPI_FFN = 3, EPI_PART = 4 };

struct GemmParams {
    const uint16_t* A;  // [M][lda] fp16 activations
    int lda, M, K;
    const uint32_t* w[3];
    const uint32_t* z[3];
    const uint16_t* s[3];
    int N[3];  // rows of each matrix
    int C, pzh, sh;
    int epi;
    int mtiles, ntiles;
    int ksplit;                  // workgroups that share a tile, each taking a part of K
    float* part;                 // ksplit > 1: fp32 partial tiles [tile][ksplit][rows x columns]
    unsigned int* part_counter;  // ksplit > 1: arrivals per tile, zero between launches
    // QKV: RoPE of the q and k tiles in the epilogue (prefill.hip: 128-wide heads, one per tile), (cos, sin) from the table
    // [position][pair]; row m of the GEMM is position rope_pos0 + m.  Null: no rotation.
    const float2* rope;
    int head_size;
    int rope_pos0;
    // FFN form: write the output with every 8 columns in the order (0,4,1,5,2,6,3,7), the order a permuted-A GEMM reads
    int out_perm;
    // few-row form: 32-row tiles of A, which is in fragment order, and of the FFN form's output (0: rows, as out_perm says)
    int a_tiles, out_tiles;
    int few_per, few_extra;  // its K slices: quantisation groups of each, and how many of them have one more
    uint16_t* out[3];
    long long ldo[3];       // output row stride in elements
    long long out_off[3];   // element offset of output row 0 (KV cache: loff + pos0 * kv_dim)
};

// (h0,h1)(h2,h3)(h4,h5)(h6,h7) -> (h0,h4)(h1,h5)(h2,h6)(h3,h7): the order in which one packed dword unpacks
__device__ __forceinline__ u32x4 permute8(const u32x4 v) {
    u32x4 o;
    o[0] = __builtin_amdgcn_perm(v[2], v[0], 0x05040100u);
    o[1] = __builtin_amdgcn_perm(v[2], v[0], 0x07060302u);
    o[2] = __builtin_amdgcn_perm(v[3], v[1], 0x05040100u);
    o[3] = __builtin_amdgcn_perm(v[3], v[1], 0x07060302u);
    return o;
}

// Fragment order: activations as the few-row form's 32x32x16 products take them, the 64 lanes of an operand 1 KB in a row:
// [column / 128][fragment][row / 32][half][row % 32][8 columns], where fragment f holds eighth f % 4 of quarters 2 (f / 4) and
// 2 (f / 4) + 1 of the 128 columns (a lane's dwords of packed weights).  `tiles`: 32-row tiles of the block.
__device__ __forceinline__ size_t fragment_offset(int row, int col, int tiles) {
    const int f = ((col >> 6) & 1) * 4 + ((col >> 3) & 3);
    return ((((size_t)(col >> 7) * 8 + f) * tiles + (row >> 5)) * 64 + ((col >> 5) & 1) * 32 + (row & 31)) * 8 + (col & 7);
}

// The constants of one quantisation group of a weight row.
struct Group {
    h16x2 zlo, zhi, s2;  // -(1024 + z), -(64 + z), scale
};
__device__ __forceinline__ Group group_consts(uint32_t z, uint16_t scale_bits) {
    const uint32_t zz = z | (z << 16), ss = (uint32_t)scale_bits | ((uint32_t)scale_bits << 16);
    return Group{as_h2(0xE400E400u | zz), as_h2(0xD400D400u | (zz << 4)), as_h2(ss)};
}

// 8 nibbles of one dword -> 8 dequantised fp16 weights in the order (w0,w4)(w1,w5)(w2,w6)(w3,w7).
// magic = 0x64006400 held in a vector register: v_and_or_b32 takes no literal, and with the constant in a register
// the mask-and-merge of a nibble pair is one instruction.
__device__ __forceinline__ u32x4 dequant8(uint32_t d, const Group& g, uint32_t magic) {
    const h16x2 sixteenth = {(h16_t)0.0625f, (h16_t)0.0625f};
    const uint32_t d8 = d >> 8;
    const h16x2 t0 = as_h2((d & 0x000F000Fu) | magic) + g.zlo;                                      // exact q - z
    const h16x2 t1 = __builtin_elementwise_fma(as_h2((d & 0x00F000F0u) | magic), sixteenth, g.zhi);  // exact
    const h16x2 t2 = as_h2((d8 & 0x000F000Fu) | magic) + g.zlo;
    const h16x2 t3 = __builtin_elementwise_fma(as_h2((d8 & 0x00F000F0u) | magic), sixteenth, g.zhi);
    return u32x4{as_u32(t0 * g.s2), as_u32(t1 * g.s2), as_u32(t2 * g.s2), as_u32(t3 * g.s2)};  // one rounding each
}

// The activation tile in LDS is [rows][64 halves] with the 16-byte chunk index XOR-ed with a key of the row, so
// that a wave's fragment reads (32 consecutive rows, one chunk) spread over all banks without padding.
__device__ __forceinline__ int lds_key(int row) { return (row ^ (row >> 3)) & 7; }
__device__ __forceinline__ int lds_off(int row, int chunk) { return row * BK + ((chunk ^ lds_key(row)) << 3); }

// what a 16-byte load of activations past K reads instead
static __device__ const __align__(16) uint32_t zeros16[4] = {0u, 0u, 0u, 0u};

// Direct global -> LDS loads: lane L's 16 (4) bytes land at lds_byte_off + 16 (4) * L.  Issued as inline assembly,
// so the compiler's wait-count bookkeeping does not see them; the kernel counts and waits for them itself.
__device__ __forceinline__ void dma16(const void* gptr, uint32_t lds_byte_off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_byte_off), "v"(gptr) : "memory");
}
// Same with the address as a wave-uniform base plus a 32-bit byte offset per lane (no 64-bit vector arithmetic).
__device__ __forceinline__ void dma16(const void* sbase, uint32_t voff, uint32_t lds_byte_off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_byte_off), "v"(voff), "s"(sbase) : "memory");
}
// A pointer that is the same in all lanes, in scalar registers whatever the compiler can prove of it.
template <typename T>
__device__ __forceinline__ const T* uniform_ptr(const T* ptr) {
    const uint64_t v = reinterpret_cast<uint64_t>(ptr);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const T*>(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ void dma4(const void* gptr, uint32_t lds_byte_off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds_byte_off), "v"(gptr) : "memory");
}

// inverse of permute8: (h0,h4)(h1,h5)(h2,h6)(h3,h7) -> (h0,h1)(h2,h3)(h4,h5)(h6,h7)
__device__ __forceinline__ u32x4 unpermute8(const u32x4 v) {
    u32x4 o;
    o[0] = __builtin_amdgcn_perm(v[1], v[0], 0x05040100u);
    o[1] = __builtin_amdgcn_perm(v[3], v[2], 0x05040100u);
    o[2] = __builtin_amdgcn_perm(v[1], v[0], 0x07060302u);
    o[3] = __builtin_amdgcn_perm(v[3], v[2], 0x07060302u);
    return o;
}

}  // namespace pf

// Split-K workspace, of a context or of the device: fp32 partial tiles, then an arrival counter per tile.
constexpr int kPartTiles = 256;
constexpr size_t kPartBytes = (size_t)kPartTiles * 2 * pf::BM * pf::BN * sizeof(float);  // 32 MiB

// gemm_rows.hip
struct awq_rows_plan {
    int form, ksplit;
    float us;  // what the launch is expected to take
};
struct awq_step_us {
    float alone, once, twice;  // us per K step: few workgroups; one on every compute unit; two on every compute unit
};
float awq_gemm_us(int cus, int per_cu, long long wgs, int steps, const awq_step_us& t);
int awq_gemm_rows_setup();  // once per device, with that device current
// parts: the K parts of a split stay apart (EPI_PART)
awq_rows_plan awq_plan_gemm_rows(int cus, int M, int K, int groups, bool may_split, bool parts = false);
int awq_launch_gemm_rows(awq_ctx* ctx, pf::GemmParams& p, int groups, int form, int ksplit, bool a_perm, const char* what);
void awq_rows_form(int form, int* tile);  // rows, columns, K slices inside a workgroup

// gemm_few.hip
constexpr int kFewRows = 128;  // the most it takes
struct awq_few_plan {
    int units, ksplit;  // 32-row units of weights a workgroup; workgroups that share them, each with a part of K
    float us;           // what the launch is expected to take
};
int awq_gemm_few_setup();  // once per device, with that device current
awq_few_plan awq_plan_gemm_few(int cus, int M, int K, int N, bool may_split);
int awq_launch_gemm_few(awq_ctx* ctx, pf::GemmParams& p, int N, const awq_few_plan& plan, const char* what);
