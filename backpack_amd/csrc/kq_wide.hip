// kq_wide.hip — fp32 activations of many tokens against k-quant weights on the matrix cores: up to 64 tokens share
// every weight byte (decode steps of many sequences, short fp32 batches, mixture layers of a prompt).
//
// What bounds it.  The 16-token tile kernel (kq_mtile.hip) walks the weights once per 16 tokens and scales every
// product of 32 elements on the vector units, once per token: its vector work grows with the tokens and the matrix
// cores wait.  Here a weight is turned into (quant * sub-block scale) once for all tokens of the workgroup — an
// integer of at most 63 * 31 (Q4_K, Q5_K), exact in fp16 — so a superblock's 256 elements accumulate in one chain of
// matrix instructions and the vector units see one fused multiply-add per output and superblock.
//
// Activations.  A pass of its own (wide_x_kernel, with the call's prologue folded in) splits fp32 X once per call,
// where the tile kernel did so in every workgroup: per (token, superblock) a power of two puts the largest magnitude
// just below 2^15, x * s = hi + lo with both fp16 (22 bits), in operand order, 1 KB; beside it the eight sub-block
// sums (hi and lo fp16, the factor of the Q4_K / Q5_K minima, one matrix instruction per superblock) and 1 / s.
//
// Q6_K.  scale * (q - 32) has up to 13 bits: it is Wh = fp16(product) and the exact rest Wl = fma(scale, q - 32, -Wh),
// and the product takes three instructions, hi * Wh + lo * Wh + hi * Wl; the dropped lo * Wl is below 2^-22 of x * W.
//
// Operand order.  v_mfma_f32_16x16x32_f16 gives lane l eight of the 32 k of row l % 16, and any order of k will do as
// long as both operands use it.  Lane group kq = l / 16 takes 64 consecutive weights' bytes of the superblock (Q4_K,
// Q5_K: 32 bytes, sub-blocks 2kq and 2kq+1; Q6_K: 16 positions of a half, all four 32-element runs), so a lane reads
// its bytes in 16-byte loads and needs two (four) scales per superblock.  Step j of eight multiplies
//   Q4_K, Q5_K  elements 64 kq + 32 (j & 1) + 8 (j >> 1) ..+7        (low nibbles, then high ones)
//   Q6_K        elements 128 (kq >> 1) + 32 (j >> 1) + 16 (kq & 1) + 8 (j & 1) ..+7
// each group of eight in the order 0 2 1 3 4 6 5 7 (what masking dwords leaves).
//
// Work split.  Eight waves of two 16-row tiles each; the X of a superblock (TT tiles of 16 tokens, 16 KB each) is
// staged in LDS, shared by the waves.  K is cut over blockIdx.z when rows give too few workgroups; a second launch
// adds the partial tiles in split order.
//
// The walk.  X (halves of a superblock, a ring of three) and W (each wave its own rows) go from memory to LDS without
// registers, requested a superblock ahead and spread over its eight steps; a step's LDS reads and its expansion of weights
// stand between the matrix instructions of the step before (sched_group_barrier), and the two meetings per superblock lie
// ahead of a step whose operands are already in registers.  What that replaced: every lane fetched its 16-byte pieces
// of W and X itself (52 cache accesses per load instruction, 20 now) and the compiler read operands right ahead of their
// use.  What is left at 32 tokens and more: vector and matrix instructions on split operands (issue of both, and waits for 0.3 of the waves'
// cycles), at a core clock of 1.8 .. 2.0 GHz of 2.43 while all CUs are in these kernels, in a launch alone as behind a thousand others
// (s_memtime against s_memrealtime of each workgroup).  A walk with W a step earlier in registers gained 1 %, fewer vector
// instructions more (v_perm for the Q6_K fields: 31 -> 24 per eight weights, 5 to 7 % of its launches).  At 16 tokens and fewer it is the
// memory: 144 and 210 B pieces of rows reach 83 to 92 % of a contiguous read.  With one tile of 16 tokens a step is too short for the
// fixed order (`schedule`).
//
// A workgroup may walk several groups of 256 rows against the same tokens as one sequence of superblocks (groups_per_wg): its
// start (records, addresses, the first loads' way: 8 us of 25 .. 40) is paid once and a group's stores go under the next
// group's walk.
//
// Mixture layers (records of pairs of one expert): consecutive workgroups go to the same XCD, so a record's row groups
// and an expert's records meet their X and W in that L2 (128 experts x 8 slots, 2048 / 768, 2048 tokens: 750 -> 703 us).
// us with the router, now / with the walk before / on the 16-token tiles: 2048 tokens 547 / 739 / 1264, 256 tokens
// 158 / 191 / 267, 24 tokens 117 / 128 / 153.
#include "kq_format.h"
#include "kq_gemm_plan.h"
#include "kq_group.h"
#include "kq_kernels.h"
#include "kq_wave.h"
#include <cmath>

namespace kq {

typedef _Float16 w_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 w_half2 __attribute__((ext_vector_type(2)));
typedef float w_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t w_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t w_u32x2 __attribute__((ext_vector_type(2)));

constexpr int WIDE_WAVES = 8;
constexpr int WIDE_MAX_GROUPS = 8;   // of rows, that a workgroup walks for a record
constexpr uint32_t WIDE_XA = 1024, WIDE_XV = 32, WIDE_XI = 4;   // bytes per (token, superblock)

WideX wide_x_layout(void* xa, void* rest, uint32_t rows, uint32_t n_blocks)
{
    const size_t n = (size_t)rows * n_blocks;
    WideX x;
    x.xa = (uint8_t*)xa;
    x.xv = rest ? (uint8_t*)rest : (uint8_t*)xa + n * WIDE_XA;
    x.xi = (float*)(x.xv + n * WIDE_XV);
    return x;
}
size_t wide_x_bytes(uint32_t rows, uint32_t n_blocks) { return (size_t)rows * n_blocks * (WIDE_XA + WIDE_XV + WIDE_XI); }
size_t wide_x_rest_bytes(uint32_t rows, uint32_t n_blocks) { return (size_t)rows * n_blocks * (WIDE_XV + WIDE_XI); }

// ------------------------------------------------------------------------------------------------------------------
// silu (2) or gelu_tanh (3)
__device__ __forceinline__ float wide_act(int act, float g)
{
    return act == 2 ? g / (expf(-g) + 1.0f) : 0.5f * g * (1.0f + tanhf(0.7978845608f * (g + 0.044715f * g * g * g)));
}

// Eight elements of superblock `cell` (a token's), run `sub` of its 32, split and put in operand order by the half wave that has them.
__device__ __forceinline__ void wide_split(const float (&v)[8], uint32_t sub, size_t cell, int q6, uint8_t* xa, uint8_t* xv, float* xi)
{
    uint32_t amax = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = max(amax, __builtin_bit_cast(uint32_t, v[i]) & 0x7FFFFFFFu);
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) amax = max(amax, (uint32_t)__shfl_xor((int)amax, o, 32));
    uint32_t e = amax >> 23;
    e = e < 15u ? 15u : (e > 253u ? 253u : e);
    const float s = __builtin_bit_cast(float, (268u - e) << 23);     // 2^(141-e): amax * s in [2^14, 2^15)
    if (sub == 0) xi[cell] = __builtin_bit_cast(float, (e - 14u) << 23);
    _Float16 h[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float a = v[i] * s;
        h[i] = (_Float16)a;
        l[i] = (_Float16)(a - (float)h[i]);
    }
    // the step and lane group that take this run of eight
    const uint32_t j = q6 ? 2u * ((sub >> 2) & 3u) + (sub & 1u) : 2u * (sub & 3u) + ((sub >> 2) & 1u);
    const uint32_t kq = q6 ? 2u * (sub >> 4) + ((sub >> 1) & 1u) : sub >> 3;
    uint8_t* dst = xa + cell * WIDE_XA + j * 64u + kq * 16u;
    *(w_half8*)dst = w_half8{h[0], h[2], h[1], h[3], h[4], h[6], h[5], h[7]};
    *(w_half8*)(dst + 512) = w_half8{l[0], l[2], l[1], l[3], l[4], l[6], l[5], l[7]};
    if (!q6) {
        float t = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        t += group_partner<1>(t);
        t += group_partner<2>(t);
        if ((sub & 3u) == 0) {
            const float a = t * (s * 0.03125f);   // 32 elements of at most 2^15 fit an fp16
            const _Float16 th = (_Float16)a;
            _Float16* o = (_Float16*)(xv + cell * WIDE_XV) + (sub >> 2);
            o[0] = th;
            o[8] = (_Float16)(a - (float)th);
        }
    }
}

// One workgroup: 16 superblocks of a row at a time, 32 threads each, 8 consecutive elements per thread.  pro as in
// MatmulArgs (the stand-alone prologue kernels' formulas).  The norm needs the whole row first, so its workgroup
// walks the row; the others spread it over blockIdx.y.  xa may be X itself: a superblock is read and written by the
// same half wave, and its exponent needs every element of it before the first store.
__global__ __launch_bounds__(512) void wide_x_kernel(const float* X, const float* norm_w, float eps, uint32_t n_blocks,
                                                     int pro, int q6, uint8_t* xa, uint8_t* xv, float* xi)
{
    __shared__ float part[8];
    const uint32_t tok = blockIdx.x, sub = threadIdx.x & 31u, at = threadIdx.x >> 5;
    const uint32_t K = n_blocks * KQ_QK;
    const float* row = X + (size_t)tok * (pro >= 2 ? 2u * (size_t)K : (size_t)K);
    float rstd = 1.0f;
    if (pro == 1) {
        float ss = 0.0f;
        for (uint32_t k = threadIdx.x * 4u; k < K; k += 2048u) {
            const float4 v = *(const float4*)(row + k);
            ss = fmaf(v.x, v.x, ss); ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss);
        }
        ss = wave_total(ss);
        if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = ss;
        __syncthreads();
        ss = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
        rstd = 1.0f / sqrtf(ss / (float)K + eps);
    }
    for (uint32_t b = blockIdx.y * 16u + at; b < n_blocks; b += 16u * gridDim.y) {
        const uint32_t k = b * KQ_QK + sub * 8u;
        float v[8];
        *(float4*)v = *(const float4*)(row + k);
        *(float4*)(v + 4) = *(const float4*)(row + k + 4);
        if (pro == 1) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = v[i] * rstd * norm_w[k + i];
        } else if (pro >= 2) {
            float u[8];
            *(float4*)u = *(const float4*)(row + K + k);
            *(float4*)(u + 4) = *(const float4*)(row + K + k + 4);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float g = v[i];
                v[i] = wide_act(pro, g) * u[i];
            }
        }
        wide_split(v, sub, (size_t)tok * n_blocks + b, q6, xa, xv, xi);
    }
}

hipError_t launch_wide_x(int type, const float* X, int pro, const float* norm_w, float eps, uint32_t rows,
                         uint32_t n_blocks, const WideX& x, hipStream_t s)
{
    hipLaunchKernelGGL(wide_x_kernel, dim3(rows, pro == 1 ? 1u : (n_blocks + 15u) / 16u), dim3(512), 0, s, X, norm_w, eps,
                       n_blocks, pro, type == KQ_TYPE_Q6_K ? 1 : 0, x.xa, x.xv, x.xi);
    return hipGetLastError();
}

// A mixture layer's start in one launch: the first workgroup buckets the pairs, the others split X, a half wave per superblock.  The two
// need nothing from each other, and as launches of their own they cost 2.7 us more: 128 experts x 8, 2048 / 768, with the router, 24 /
// 256 / 2048 tokens 116.5 / 159.8 / 534.5 -> 113.9 / 156.9 / 529.5, 8 experts x 2, 1024 / 512, 8 tokens 29.9 -> 27.8.
template <int KEEP, bool MORE>
__global__ __launch_bounds__(1024) void wide_prepare_kernel(const uint32_t* __restrict__ expert_idx, uint32_t n_pairs, uint32_t n_experts,
                                                            uint32_t cap, uint32_t* __restrict__ records, uint32_t* __restrict__ n_records,
                                                            const float* X, uint64_t cells, int q6, uint8_t* xa, uint8_t* xv, float* xi)
{
    extern __shared__ uint32_t sm[];
    if (blockIdx.x == 0) {
        group_pairs<KEEP, MORE>(expert_idx, n_pairs, n_experts, cap, records, n_records, sm);
        return;
    }
    const uint32_t sub = threadIdx.x & 31u;
    for (uint64_t cell = (uint64_t)(blockIdx.x - 1u) * 32u + (threadIdx.x >> 5); cell < cells; cell += (uint64_t)(gridDim.x - 1u) * 32u) {
        const float* x = X + (size_t)cell * KQ_QK + sub * 8u;
        float v[8];
        *(float4*)v = *(const float4*)x;
        *(float4*)(v + 4) = *(const float4*)(x + 4);
        wide_split(v, sub, (size_t)cell, q6, xa, xv, xi);
    }
}

hipError_t launch_wide_prepare(const uint32_t* expert_idx, uint32_t n_pairs, uint32_t n_experts, uint32_t cap, uint32_t* records,
                               uint32_t* n_records, int type, const float* X, uint32_t rows, uint32_t n_blocks, const WideX& x, hipStream_t s)
{
    if (n_experts > 8192u) return hipErrorInvalidValue;   // three LDS arrays of n_experts words, eight experts per thread
    const uint64_t cells = (uint64_t)rows * n_blocks, wgs = (cells + 31u) / 32u;
    const dim3 grid(1u + (uint32_t)(wgs < 65536u ? wgs : 65536u));
    const int q6 = type == KQ_TYPE_Q6_K ? 1 : 0;
    const auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(1024), 3 * n_experts * sizeof(uint32_t), s, expert_idx, n_pairs, n_experts, cap, records,
                           n_records, X, cells, q6, x.xa, x.xv, x.xi);
    };
    if (n_pairs <= 4096u) go(wide_prepare_kernel<4, false>);
    else go(wide_prepare_kernel<16, true>);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------------------------
struct WideParams {
    WideX x;
    const uint8_t* W;
    const uint8_t* W2;       // act != 0: where the second tile's row 0 is (gate rows in W, up rows in W2)
    const float* bias;       // [N] (act: [2N], the up half N on); nullptr for none
    const float* residual;
    float* Y;
    uint32_t M, N;           // rows of x; outputs
    uint32_t n_blocks, row_stride_bytes, y_offset, ldy;
    uint32_t n_splits, blocks_per_split;
    float* partial;          // [split][token group][row group][token][256 columns]
    uint32_t row_groups, per_wg;        // groups of 256 rows (act: 128 gate and their up rows); how many a workgroup walks (dense)
    int act;                 // 0, or 2 / 3: Y = silu / gelu_tanh (W x) * (W2 x)
    // grouped (records != nullptr): workgroups walk records {expert, count, pair ids ...}; W and W2 advance by N rows per expert, a
    // pair's X row is itself (x_per_slot) or pair / k_slots, its Y row the pair.  How many groups of rows a workgroup walks is chosen
    // here, when the number of records is known (a round more than the choice counted on costs as much as all of them: 129
    // records of which 128 were expected, three groups each, 334 us instead of 206; chosen here 201 and 203): wgs_of[c - 1] workgroups to a record at c
    // groups, `walk` us per group, `start` beside them.  Records of 16 pairs: one group, always.  Over 2069 such layers that was
    // 2 % ahead of the choice, which was the better one by 3 % on 2 % of them, and the choice itself takes 0.8 us at a workgroup's
    // start (3 tokens, 4 experts x 2, 256 / 512: 23.4 us for the layer with it, 22.5 without).
    const uint32_t* records;
    const uint32_t* n_records;
    uint32_t record_words, k_slots;
    uint32_t wgs_of[WIDE_MAX_GROUPS];
    float per_cu, walk, start;
    int x_per_slot;
};

// A row tile's bytes of one superblock, as this lane holds them.
template <int TYPE> struct WideW;
template <> struct WideW<KQ_TYPE_Q4_K> {
    w_u32x4 hdr, q[2];
    __device__ __forceinline__ void load_lds(const uint8_t* blk, const uint8_t*, uint32_t kq)
    {
        hdr = *(const w_u32x4*)blk;
        q[0] = *(const w_u32x4*)(blk + 16 + 32 * kq);
        q[1] = *(const w_u32x4*)(blk + 32 + 32 * kq);
    }
    __device__ __forceinline__ void arrived() const { asm volatile("" ::"v"(hdr), "v"(q[0]), "v"(q[1]) : "memory"); }
};
template <> struct WideW<KQ_TYPE_Q5_K> {
    w_u32x4 hdr, q[2], f[2];
    __device__ __forceinline__ void load_lds(const uint8_t* blk, const uint8_t*, uint32_t kq)
    {
        hdr = *(const w_u32x4*)blk;
        f[0] = *(const w_u32x4*)(blk + 16);
        f[1] = *(const w_u32x4*)(blk + 32);
        q[0] = *(const w_u32x4*)(blk + 48 + 32 * kq);
        q[1] = *(const w_u32x4*)(blk + 64 + 32 * kq);
    }
    __device__ __forceinline__ void arrived() const { asm volatile("" ::"v"(hdr), "v"(f[0]), "v"(f[1]), "v"(q[0]), "v"(q[1]) : "memory"); }
};
template <> struct WideW<KQ_TYPE_Q6_K> {
    w_u32x4 ql[2], qh;
    w_u32x2 sc;
    uint16_t d;
    // the block's 208 bytes ahead of d on a 16-byte boundary, d in the upper half of a word of its own
    __device__ __forceinline__ void load_lds(const uint8_t* blk, const uint8_t* dw, uint32_t kq)
    {
        const uint32_t h = kq >> 1, lh = kq & 1u;
        ql[0] = *(const w_u32x4*)(blk + 64 * h + 16 * lh);
        ql[1] = *(const w_u32x4*)(blk + 64 * h + 32 + 16 * lh);
        qh = *(const w_u32x4*)(blk + 128 + 32 * h + 16 * lh);
        sc = *(const w_u32x2*)(blk + 192 + 8 * h);
        d = (uint16_t)(*(const uint32_t*)dw >> 16);
    }
    __device__ __forceinline__ void arrived() const { asm volatile("" ::"v"(ql[0]), "v"(ql[1]), "v"(qh), "v"(sc), "v"((uint32_t)d) : "memory"); }
};

__device__ __forceinline__ uint32_t w_mul2(uint32_t a, w_half2 s)
{
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(w_half2, a) * s);
}

// Memory -> LDS without registers: lane l's 16 (4) bytes land at m0 + 16 l (4 l).  Inline asm, because the compiler
// would wait for such a load ahead of every LDS read that it cannot tell apart from its target; the waits are the
// kernel's own (wide_meet).  No register is written, so none can be reused while a load is in flight.  The compiler does not
// see into these statements, so the wait states between a vector instruction that writes a scalar register (a spill read
// back, a readfirstlane) and a load that uses it (5), and ahead of a load that uses m0 (1), stand in them.
// SKIP: not at all where go is 0 (the branch lies inside the statement, so the steps of the walk stay one basic block).
#define WIDE_SKIP "s_cmp_eq_u32 %2, 0\n\ts_mov_b32 m0, %0\n\ts_cbranch_scc1 .Lwide_skip%=\n\t"
template <bool SKIP> __device__ __forceinline__ void lds_dma16(uint32_t lds, const uint8_t* src, int go)
{
    if constexpr (SKIP) asm volatile(WIDE_SKIP "global_load_lds_dwordx4 %1, off\n.Lwide_skip%=:" ::"s"(lds), "v"(src), "s"(go) : "scc", "memory");
    else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory");
}
template <bool SKIP> __device__ __forceinline__ void lds_dma16(uint32_t lds, const uint8_t* base, uint32_t off, int go)
{
    if constexpr (SKIP)
        asm volatile(WIDE_SKIP "s_nop 1\n\tglobal_load_lds_dwordx4 %1, %3\n.Lwide_skip%=:" ::"s"(lds), "v"(off), "s"(go), "s"(base) : "scc", "memory");
    else asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
// ... with the lanes of `lanes` only (none: it moves nothing).  Called with every lane active.
template <bool SKIP> __device__ __forceinline__ void lds_dma16(uint32_t lds, const uint8_t* base, uint32_t off, uint64_t lanes, int go)
{
    if constexpr (SKIP)
        asm volatile(WIDE_SKIP "s_mov_b64 exec, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\ts_mov_b64 exec, -1\n.Lwide_skip%=:" ::"s"(lds), "v"(off), "s"(go), "s"(base), "s"(lanes) : "scc", "memory");
    else asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\ts_nop 2\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1" ::"s"(lds), "v"(off), "s"(base), "s"(lanes) : "memory");
}
template <bool SKIP> __device__ __forceinline__ void lds_dma4(uint32_t lds, const uint8_t* base, uint32_t off, uint64_t lanes, int go)
{
    if constexpr (SKIP)
        asm volatile(WIDE_SKIP "s_mov_b64 exec, %4\n\ts_nop 0\n\tglobal_load_lds_dword %1, %3\n\ts_mov_b64 exec, -1\n.Lwide_skip%=:" ::"s"(lds), "v"(off), "s"(go), "s"(base), "s"(lanes) : "scc", "memory");
    else asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\ts_nop 2\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b64 exec, -1" ::"s"(lds), "v"(off), "s"(base), "s"(lanes) : "memory");
}
template <bool SKIP> __device__ __forceinline__ void lds_dma4(uint32_t lds, const void* src, int go)
{
    static_assert(SKIP, "");
    asm volatile(WIDE_SKIP "global_load_lds_dword %1, off\n.Lwide_skip%=:" ::"s"(lds), "v"(src), "s"(go) : "scc", "memory");
}
#undef WIDE_SKIP
// (an int: all lanes or none)
__device__ __forceinline__ void lds_dma16_or_none(uint32_t lds, const uint8_t* src, int lanes)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_lo, %2\n\ts_mov_b32 exec_hi, %2\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b64 exec, -1" ::"s"(lds), "v"(src), "s"(lanes) : "memory");
}
__device__ __forceinline__ void lds_dma4_or_none(uint32_t lds, const void* src, int lanes)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_lo, %2\n\ts_mov_b32 exec_hi, %2\n\tglobal_load_lds_dword %1, off\n\ts_mov_b64 exec, -1" ::"s"(lds), "v"(src), "s"(lanes) : "memory");
}
// ... from 64-bit addresses
__device__ __forceinline__ void lds_dma16_lanes(uint32_t lds, const uint8_t* src, uint64_t lanes)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %2\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b64 exec, -1" ::"s"(lds), "v"(src), "s"(lanes) : "memory");
}
__device__ __forceinline__ void lds_dma4_lanes(uint32_t lds, const uint8_t* src, uint64_t lanes)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %2\n\tglobal_load_lds_dword %1, off\n\ts_mov_b64 exec, -1" ::"s"(lds), "v"(src), "s"(lanes) : "memory");
}
// At most N of this wave's loads are still in flight, its LDS reads have returned, and so have the other waves'.
template <int N>
__device__ __forceinline__ void wide_meet() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }

// None of this wave's loads is still in flight, if go is 0.  (wide_meet's counts take all of the walk's loads to have been sent;
// the branch lies inside the statement.)
__device__ __forceinline__ void wide_drain_unless(int go)
{
    asm volatile("s_cmp_lg_u32 %0, 0\n\ts_cbranch_scc1 .Lwide_go%=\n\ts_waitcnt vmcnt(0)\n.Lwide_go%=:" ::"s"(go) : "scc", "memory");
}

// The kernel's LDS, in bytes.  X: a ring of three halves of a superblock, [token][hi, lo][16 pieces of 16 bytes], a piece's
// place exchanged by its token (^ token % 16) so that the 16 tokens that a wave reads a piece of lie in different banks.
// W: per wave its two row tiles' blocks as they are in memory (9, 11 or 13 units of 16 bytes per row: odd, so 16 rows start
// in different banks), Q6_K's d behind them.  S: two buffers of the sums and the scales of X.
template <int TYPE, int TT> struct WideLds {
    static constexpr bool Q6 = TYPE == KQ_TYPE_Q6_K;
    static constexpr uint32_t UNITS = TYPE == KQ_TYPE_Q4_K ? 9u : TYPE == KQ_TYPE_Q5_K ? 11u : 13u;   // per row and superblock
    static constexpr uint32_t W_INSTR = (16u * UNITS + 63u) / 64u, W_LAST = 16u * UNITS - 64u * (W_INSTR - 1u);   // per tile
    static constexpr uint32_t W_TILE = 256u * UNITS, W_WAVE = 2u * W_TILE + (Q6 ? 128u : 0u);
    static constexpr uint32_t X_HALF = TT * 8192u, V_BUF = Q6 ? 0u : (TT > 2 ? 2048u : 1024u), I_BUF = 256u;
    static constexpr uint32_t W_AT = 3u * X_HALF, V_AT = W_AT + 8u * W_WAVE, I_AT = V_AT + 2u * V_BUF, R_AT = I_AT + 2u * I_BUF, BYTES = R_AT + TT * 1024u;
    static constexpr int N_W = 2 * (int)W_INSTR + (Q6 ? 2 : 0);   // a wave's loads for its weights of a superblock
};

// A workgroup's walk: its groups of rows from group0 on against up to TT tiles of 16 tokens, t0 .. t0 + count - 1 or a record's
// `count` pairs.
template <int TYPE, int TT>
__device__ __forceinline__ void wide_walk(const WideParams& p, uint8_t* lds, uint32_t bx, uint32_t per_wg, const uint32_t* rec,
                                          uint32_t t0, uint32_t count, const uint8_t* W, const uint8_t* W2)
{
    using L = WideLds<TYPE, TT>;
    constexpr bool Q6 = TYPE == KQ_TYPE_Q6_K, Q5 = TYPE == KQ_TYPE_Q5_K;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, kq = lane >> 4, r16 = lane & 15u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    constexpr uint32_t BB = TYPE == KQ_TYPE_Q4_K ? KQ_Q4K_BYTES : TYPE == KQ_TYPE_Q5_K ? KQ_Q5K_BYTES : KQ_Q6K_BYTES;
    const uint32_t b0 = blockIdx.z * p.blocks_per_split, b1 = min(b0 + p.blocks_per_split, p.n_blocks);
    // The slots' rows of Y and X, a copy per wave (no meeting).  A record's go straight into LDS, all its words (those beyond the
    // count have no meaning: no wait for the count); the first weights are requested behind them and are under way while the
    // rows are turned into addresses.  Slots beyond the count repeat the last slot's X: their outputs are dropped.
    uint32_t* const out_rows = (uint32_t*)(lds + L::R_AT + wave * (TT * 128u));
    uint32_t* const x_rows = out_rows + TT * 16u;
    const uint32_t last = min(count, TT * 16u) - 1u;
    if (rec) lds_dma4<false>(lds0 + L::R_AT + wave * (TT * 128u), (const uint8_t*)rec, lane * 4u, TT == 4 ? ~0ull : (1ull << (TT * 16u % 64u)) - 1ull, -1);

    // W: the wave's two tiles of 16 rows, unit after unit.  The last rows of a matrix that does not fill its tiles are read from
    // N - 16 on (what a tile has of an earlier one is not stored), so a lane's offsets are the same for every tile.
    const uint32_t rows = min(p.N, 16u);
    uint32_t woff[L::W_INSTR];
#pragma unroll
    for (uint32_t i = 0; i < L::W_INSTR; ++i) {
        const uint32_t n = i * 64u + lane, row = n / L::UNITS, u = n % L::UNITS;
        woff[i] = min(row, rows - 1u) * p.row_stride_bytes + u * 16u;
    }
    const uint32_t doff = min(r16, rows - 1u) * p.row_stride_bytes + 206u;   // (d in the upper half; ends with the block)
    auto tile_row = [&](uint32_t group, int r) { return (group * WIDE_WAVES + wave) * (p.act ? 16u : 32u) + (p.act ? 0u : 16u * r); };
    const uint8_t* wbase[2];
    auto set_w = [&](uint32_t group, uint32_t sb) {   // (no branch: the steps of the walk stay one basic block)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint64_t at = (uint64_t)((r && p.act ? W2 : W) + (size_t)min(tile_row(group, r), p.N - rows) * p.row_stride_bytes + (size_t)((b0 + sb) * BB));
            // (scalar registers: the compiler would keep the choice of a superblock in vector registers)
            wbase[r] = (const uint8_t*)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)at));
        }
    };
    const uint32_t group0 = bx * per_wg, n_groups = min(per_wg, p.row_groups - group0);
    set_w(group0, 0);
    const uint32_t w_lds = lds0 + L::W_AT + wave * L::W_WAVE;
    // piece k of a superblock's weights: whole loads first, then each tile's last lanes (and d)
    constexpr bool SKIP = TT == 1 && Q6;
    auto request_w = [&](int k, int go) {
        constexpr int WHOLE = 2 * ((int)L::W_INSTR - 1);
        if (k < WHOLE) {
            const uint32_t r = (uint32_t)k & 1u, i = (uint32_t)k >> 1;
            lds_dma16<SKIP>(w_lds + r * L::W_TILE + i * 1024u, wbase[r], woff[i], go);
        } else if (k < WHOLE + 2) {
            const uint32_t r = (uint32_t)k & 1u;
            lds_dma16<SKIP>(w_lds + r * L::W_TILE + (L::W_INSTR - 1u) * 1024u, wbase[r], woff[L::W_INSTR - 1u], (1ull << L::W_LAST) - 1ull, go);
        } else {
            const uint32_t r = (uint32_t)k & 1u;
            lds_dma4<SKIP>(w_lds + 2u * L::W_TILE + r * 64u, wbase[r], doff, 0xFFFFull, go);
        }
    };
    // The walk: n_groups groups of rows against the same tokens, n_sb superblocks each, as one sequence of `all` superblocks:
    // W and X of the next group are under way while a group's outputs leave.  Half h of it is superblock h / 2.  Requested
    // ahead: X by two halves, W by one superblock (into the place it was read from), S half a superblock less.  Past the
    // end the last is requested again, and waited for at the end — or, for Q6_K at 16 tokens (SKIP), nothing is.  Elsewhere the test
    // for it costs more than the loads (means as at `schedule` below, us, without / with it: Q4_K 1.0 / 1.7 and -1.4 / -1.4, Q5_K
    // -0.5 / 0.5 and -3.7 / -3.3, Q6_K -8.7 / -9.1 on the dense calls; 28672 x 4096 at 48 tokens 37.0 and 38.1 us).
    constexpr int WAS = (TT + L::N_W + 3) / 4, XBS = (TT + 3) / 4;   // requests per step
    const uint32_t n_sb = b1 - b0, all = n_groups * n_sb;
    auto wrap = [&](uint32_t sb) { return sb + 1u == n_sb ? 0u : sb + 1u; };
    uint32_t w_group = group0;   // the group whose W is requested
    auto next_w = [&](uint32_t at, uint32_t sb) {   // from superblock `at`, number sb of its group, to the one behind it
        const uint32_t go = SKIP || at + 1u < all ? 1u : 0u, to = wrap(sb);
        w_group += to == 0u ? go : 0u;
        set_w(w_group, go ? to : sb);
    };
    // the way of X from the second half of superblock `at`, number sb of its group; of S from the superblock
    auto x_step = [&](uint32_t at, uint32_t sb) -> int { return !SKIP && at + 1u >= all ? -256 : wrap(sb) ? 768 : -(int)(sb * WIDE_XA) - 256; };
    auto s_step = [&](uint32_t at, uint32_t sb) -> int { return !SKIP && at + 1u >= all ? 0 : wrap(sb) ? 1 : -(int)sb; };
    // is superblock `at` there (a scalar register, as below)
    auto there = [&](uint32_t at) -> int {
        int go = -1;
        if constexpr (SKIP) {
            const int in = at < all ? -1 : 0;
            asm("s_nop 1\n\tv_readfirstlane_b32 %0, %1" : "=s"(go) : "v"(in));
        }
        return go;
    };
#pragma unroll
    for (int k = 0; k < L::N_W; ++k) request_w(k, -1);
    next_w(0, 0);

    if (rec) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L::N_W) : "memory");   // the record's words
        const uint32_t pair = out_rows[min(lane, last)];
        if (lane < TT * 16u) x_rows[lane] = p.x_per_slot ? pair : pair / p.k_slots;
    } else if (lane < TT * 16u) {
        out_rows[lane] = x_rows[lane] = t0 + min(lane, last);
    }
    // X: load i of the wave takes half a superblock of two tokens
    const uint8_t* xp[TT];
#pragma unroll
    for (int i = 0; i < TT; ++i) {
        const uint32_t tok = 2u * (wave * TT + i) + (lane >> 5);
        xp[i] = p.x.xa + ((size_t)x_rows[tok] * p.n_blocks + b0) * WIDE_XA + ((lane >> 4) & 1u) * 512u + ((lane ^ tok) & 15u) * 16u;
    }
    // its sums (waves 0, 1) and scales (the last wave)
    const uint32_t vn = (wave & 1u) * 64u + lane;
    const uint8_t* vp = p.x.xv + ((size_t)x_rows[min((vn >> 5) * 16u + (vn & 15u), TT * 16u - 1u)] * p.n_blocks + b0) * WIDE_XV + ((vn >> 4) & 1u) * 16u;
    const float* ip = p.x.xi + (size_t)x_rows[min(lane, TT * 16u - 1u)] * p.n_blocks + b0;
    int s_lanes = wave < (TT > 2 ? 2u : 1u) ? -1 : 0, i_lanes = wave == WIDE_WAVES - 1u ? -1 : 0;   // all or none
    // (a scalar register each: the compiler would keep such a choice in a vector register)
    asm("s_nop 1\n\tv_readfirstlane_b32 %0, %1" : "=s"(s_lanes) : "v"(s_lanes));
    asm("s_nop 1\n\tv_readfirstlane_b32 %0, %1" : "=s"(i_lanes) : "v"(i_lanes));
    auto request_x = [&](uint32_t ring, int i, int step, int go) {   // piece i, which moves on by `step` bytes
        lds_dma16<SKIP>(lds0 + ring * L::X_HALF + (wave * TT + i) * 1024u, xp[i], go);
        xp[i] += step;
    };
    auto request_s = [&](uint32_t buf, int step, int go) {   // step: superblocks
        if constexpr (SKIP) {
            lds_dma4<true>(lds0 + L::I_AT + buf * L::I_BUF, (const void*)ip, i_lanes & go);
        } else {
            if constexpr (!Q6) lds_dma16_or_none(lds0 + L::V_AT + buf * L::V_BUF + (wave & 1u) * 1024u, vp, s_lanes);
            lds_dma4_or_none(lds0 + L::I_AT + buf * L::I_BUF, (const void*)ip, i_lanes);
        }
        vp += step * (int)WIDE_XV;
        ip += step;
    };

    // operands of X for step j: four places of the exchanged pieces
    uint32_t a_lane[4];
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) a_lane[jj] = r16 * 512u + (((4u * jj + kq) ^ r16) & 15u) * 16u;
    w_half8 A[2][2][TT];   // [step % 2][hi, lo][tile]
    auto read_a = [&](uint32_t ring, int j) {
        const uint8_t* x = lds + ring * L::X_HALF + a_lane[j & 3];
#pragma unroll
        for (int hl = 0; hl < 2; ++hl)
#pragma unroll
            for (int t = 0; t < TT; ++t) A[j & 1][hl][t] = *(const w_half8*)(x + t * 8192 + hl * 256);
    };

    WideW<TYPE> w[2];
    auto read_w = [&]() {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint8_t* row = lds + L::W_AT + wave * L::W_WAVE + r * L::W_TILE + r16 * (L::UNITS * 16u);
            w[r].load_lds(row, lds + L::W_AT + wave * L::W_WAVE + 2u * L::W_TILE + r * 64u + r16 * 4u, kq);
        }
    };
    // what a superblock needs of its headers: per-lane scales as pairs, minima operands, super-scales
    w_half2 sc[2][Q6 ? 4 : 2];
    w_u32x4 bmn[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
    float d24[2] = {0.0f, 0.0f}, m24[2] = {0.0f, 0.0f};
    auto headers = [&]() {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if constexpr (Q6) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const uint32_t word = t < 2 ? w[r].sc.x : w[r].sc.y;
                    const int v = (int)(int8_t)(word >> (16 * (t & 1) + 8 * (kq & 1u)));
                    const _Float16 h = (_Float16)(float)v;
                    sc[r][t] = w_half2{h, h};
                }
            } else {
                const w_u32x4 h = w[r].hdr;
                const uint32_t scA = h.y & 0x3F3F3F3Fu;
                const uint32_t scB = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
                const uint32_t s2 = (kq < 2u ? scA : scB) >> (16u * (kq & 1u));
                const _Float16 a = (_Float16)(float)(s2 & 255u), c = (_Float16)((float)((s2 >> 8) & 255u) * 0.0625f);
                sc[r][0] = w_half2{a, a};
                sc[r][1] = w_half2{c, c};   // (high nibbles sit four bits up)
            }
        }
    };
    auto headers2 = [&]() {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if constexpr (Q6) {
                d24[r] = half_bits_to_float(w[r].d);
            } else {
                const w_u32x4 h = w[r].hdr;
                const uint32_t mnA = h.z & 0x3F3F3F3Fu, mnB = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
                // the eight minima as fp16 subnormals mn * 2^-24, against the hi sums (kq 0) and the lo sums (kq 1)
                const uint32_t keep = kq < 2u ? 0xFFFFFFFFu : 0u;
                bmn[r] = w_u32x4{__builtin_amdgcn_perm(0u, mnA, 0x0c010c00u) & keep, __builtin_amdgcn_perm(0u, mnA, 0x0c030c02u) & keep,
                                 __builtin_amdgcn_perm(0u, mnB, 0x0c010c00u) & keep, __builtin_amdgcn_perm(0u, mnB, 0x0c030c02u) & keep};
                d24[r] = half_bits_to_float(h.x & 0xFFFFu) * 16777216.0f;
                m24[r] = half_bits_to_float(h.x >> 16) * (16777216.0f * 32.0f);
            }
        }
    };
    w_half8 Bh[2][2], Bl[2][2];   // [step % 2][tile]
    // Q6_K: two of a word's bytes become 1024 + q in one byte permute against this constant, the shift that joins ql and qh is
    // the one that takes the field to its place: 24 vector instructions per eight weights where masks and ors took 31:
    // 128256 x 4096 at 48 / 16 tokens 181.7 / 128.7 -> 174.7 / 123.3 us, 65536 x 4096 at 32 67.8 -> 64.4.
    uint32_t magic = 0x64646464u;
    asm("" : "+v"(magic));   // (in a vector register: v_perm_b32 takes one scalar)
    auto expand = [&](int j) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            w_u32x4 o;
            if constexpr (Q6) {
                const int t = j >> 1, u = j & 1;
                const uint32_t l0 = w[r].ql[t & 1][2 * u], l1 = w[r].ql[t & 1][2 * u + 1];
                const uint32_t h0 = w[r].qh[2 * u], h1 = w[r].qh[2 * u + 1];
                const uint32_t c0 = ((l0 >> (4 * (t >> 1))) & 0x0F0F0F0Fu) | ((t < 2 ? h0 << (4 - 2 * t) : h0 >> (2 * t - 4)) & 0x30303030u);
                const uint32_t c1 = ((l1 >> (4 * (t >> 1))) & 0x0F0F0F0Fu) | ((t < 2 ? h1 << (4 - 2 * t) : h1 >> (2 * t - 4)) & 0x30303030u);
                w_u32x4 lo;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t oi = __builtin_amdgcn_perm(magic, i < 2 ? c0 : c1, i & 1 ? 0x04030401u : 0x04020400u);   // 1024 + q
                    const w_half2 q = __builtin_bit_cast(w_half2, oi) - w_half2{(_Float16)1056.0f, (_Float16)1056.0f};
                    const w_half2 hi = q * sc[r][t];
                    o[i] = __builtin_bit_cast(uint32_t, hi);
                    lo[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q, sc[r][t], -hi));
                }
                Bl[j & 1][r] = __builtin_bit_cast(w_half8, lo);
            } else {
                const int i = j >> 1;
                const uint32_t d0 = w[r].q[i >> 1][2 * (i & 1)], d1 = w[r].q[i >> 1][2 * (i & 1) + 1];
                const uint32_t e0 = d0 >> 8, e1 = d1 >> 8;
                const uint32_t m = (j & 1) ? 0x00F000F0u : 0x000F000Fu;
                o = w_u32x4{d0 & m, e0 & m, d1 & m, e1 & m};
                if constexpr (Q5) {
                    // bit 2kq (2kq + 1) of a byte of fifth bits: bit 4 beside a low nibble, bit 8 beside a high one
                    const uint32_t g0 = w[r].f[i >> 1][2 * (i & 1)] >> (2u * kq), g1 = w[r].f[i >> 1][2 * (i & 1) + 1] >> (2u * kq);
                    if (j & 1) {
                        o.x |= (g0 << 7) & 0x01000100u; o.y |= (g0 >> 1) & 0x01000100u;
                        o.z |= (g1 << 7) & 0x01000100u; o.w |= (g1 >> 1) & 0x01000100u;
                    } else {
                        o.x |= (g0 << 4) & 0x00100010u; o.y |= (g0 >> 4) & 0x00100010u;
                        o.z |= (g1 << 4) & 0x00100010u; o.w |= (g1 >> 4) & 0x00100010u;
                    }
                }
#pragma unroll
                for (int n = 0; n < 4; ++n) o[n] = w_mul2(o[n], sc[r][j & 1]);
            }
            Bh[j & 1][r] = __builtin_bit_cast(w_half8, o);
        }
    };
    w_f32x4 D[2][TT], tot[2][TT];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int t = 0; t < TT; ++t) { D[r][t] = w_f32x4{0, 0, 0, 0}; tot[r][t] = w_f32x4{0, 0, 0, 0}; }
    auto multiply = [&](int j) {
        const int s = j & 1;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < 2; ++r)
                D[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[s][0][t], Bh[s][r], j == 0 ? w_f32x4{0, 0, 0, 0} : D[r][t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < 2; ++r) D[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[s][1][t], Bh[s][r], D[r][t], 0, 0, 0);
        if constexpr (Q6) {
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int r = 0; r < 2; ++r) D[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[s][0][t], Bl[s][r], D[r][t], 0, 0, 0);
        }
    };

    auto add_up = [&](uint32_t sbuf) {   // a finished superblock's products, scaled
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const w_f32x4 inv = *(const w_f32x4*)(lds + L::I_AT + sbuf * L::I_BUF + (16 * t + 4u * kq) * 4u);
            if constexpr (Q6) {
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int i = 0; i < 4; ++i) tot[r][t][i] = fmaf(inv[i] * d24[r], D[r][t][i], tot[r][t][i]);
            } else {
                const w_half8 av = *(const w_half8*)(lds + L::V_AT + sbuf * L::V_BUF + t * 512 + (lane & 31u) * 16u);
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    w_f32x4 V = {0, 0, 0, 0};
                    V = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(w_half8, bmn[r]), V, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) tot[r][t][i] += inv[i] * fmaf(d24[r], D[r][t][i], -(m24[r] * V[i]));
                }
            }
        }
    };

    // A step's matrix instructions with the next step's LDS reads and vector work between them
    auto schedule = [&]() {
        // One tile: four matrix instructions a step are too few to hide the next step's LDS reads, so in the fixed order every step
        // waits for its operands; there the compiler's own order is better (Q5_K: within a step).  Mean difference to the walk
        // through registers that came before, us, in the fixed order / the compiler's, over layers of 1.25 .. 4 pairs per expert and
        // over dense calls of 9 .. 16 tokens on 61441 rows and more: Q4_K 1.0 / 0.4 and -1.4 / -1.9, Q5_K -0.5 / -0.7 and -3.7 / -4.0
        // (1.5 slower where steps may mix).
        if constexpr (TT == 1 && !Q6) {
            if constexpr (Q5) __builtin_amdgcn_sched_barrier(0);
            return;
        }
        constexpr int NM = (Q6 ? 6 : 4) * TT, NV = Q6 ? 4 : Q5 ? 4 : 2;
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (i < 2 * TT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    request_s(0, s_step(0, 0), -1);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < TT; ++i) request_x(h, i, h == 0 ? 256 : x_step(0, 0), -1);
    wide_meet<TT>();
    read_w();
    w[0].arrived(); w[1].arrived();
    int go = there(1);   // is there a superblock behind the one under way
#pragma unroll
    for (int k = 0; k < WAS; ++k) request_w(k, go);
    headers();
    read_a(0, 0);
    expand(0);

    // The group's outputs, from the accumulators: 64 bytes of a token's row per tile (128 for both; an activation's in one).
    auto store = [&](uint32_t group) {
        uint32_t n[2];
        bool mine[2];
        float bias[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint32_t from = tile_row(group, r);
            n[r] = min(min(from, p.N - rows) + r16, p.N - 1u);
            mine[r] = n[r] >= from && r16 < rows;
            bias[r] = p.bias ? p.bias[n[r] + (p.act && r ? p.N : 0u)] : 0.0f;
        }
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            __builtin_amdgcn_sched_barrier(0);   // (a tile's addresses at a time: registers)
            const w_u32x4 row = *(const w_u32x4*)(out_rows + 16 * t + 4u * kq);
            if (p.act) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float y = wide_act(p.act, tot[0][t][i] + bias[0]) * (tot[1][t][i] + bias[1]);
                    if (16u * t + 4u * kq + i < count && mine[0]) p.Y[(size_t)row[i] * p.ldy + p.y_offset + n[0]] = y;
                }
            } else {
                float y[2][4];
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[r][i] = tot[r][t][i] + bias[r];
                if (p.residual) {
                    // (slots beyond the count, rows beyond the last: a value that is not stored.)  All of a tile's requested, then
                    // added: each waited for by itself took 50 us where this takes 36 (Q5_K 23877 x 768, 150 tokens).
                    float q[2][4];
#pragma unroll
                    for (int r = 0; r < 2; ++r)
#pragma unroll
                        for (int i = 0; i < 4; ++i) q[r][i] = p.residual[(size_t)row[i] * p.ldy + p.y_offset + n[r]];
#pragma unroll
                    for (int r = 0; r < 2; ++r)
#pragma unroll
                        for (int i = 0; i < 4; ++i) y[r][i] += q[r][i];
                }
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (16u * t + 4u * kq + i < count && mine[r]) p.Y[(size_t)row[i] * p.ldy + p.y_offset + n[r]] = y[r][i];
            }
        }
    };

    // The requests are spread over the steps: all of them behind the meetings, they found the memory path's queue full and
    // the waves stood in front of it (6900 of a superblock's 19000 cycles).
    uint32_t ring = 0;   // where the superblock's first half lies
    uint32_t sb = 0, group = group0;
    for (uint32_t at = 0; at < all; ++at) {
        const uint32_t ring1 = ring + 1u == 3u ? 0u : ring + 1u, ring2 = 3u - ring - ring1;
        const uint32_t sb1 = wrap(sb);   // number of the superblock behind this one in its group
        const int go2 = there(at + 2u);
        add_up(at == 0u ? 0u : (at - 1u) & 1u);   // of the superblock before (a group's last is done: nothing)
        headers2();
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (j == 3) {
                // every wave has read the first half; the second has arrived
                if constexpr (SKIP) wide_drain_unless(go);
                wide_meet<TT + L::N_W>();
                request_s((at + 1u) & 1u, s_step(at + 1u, sb1), go);
                read_a(ring1, 4);
                expand(4);
            } else if (j == 7) {
                wide_meet<TT>();
                read_w();
                read_a(ring2, 0);
                w[0].arrived(); w[1].arrived();
#pragma unroll
                for (int k = 0; k < WAS; ++k) request_w(k, go2);
                headers();
                expand(0);
            } else {
                read_a(j < 3 ? ring : ring1, j + 1);
                expand(j + 1);
                if (j < 3) {
#pragma unroll
                    for (int k = (j + 1) * WAS; k < (j + 2) * WAS && k < TT + L::N_W; ++k) {
                        if (k < L::N_W) request_w(k, go);
                        else request_x(ring2, k - L::N_W, 256, go);
                    }
                }
            }
            if (j >= 3 && j < 7) {
#pragma unroll
                for (int i = (j - 3) * XBS; i < (j - 2) * XBS && i < TT; ++i) request_x(ring, i, x_step(at + 1u, sb1), go);
            }
            multiply(j);
            if (j == 0) __builtin_amdgcn_sched_barrier(0);   // (with the scaling of the superblock before: the compiler's own order)
            else schedule();
            if (j == 2) next_w(at + 1u, sb1);
        }
        if (sb1 == 0u && p.n_splits == 1u) {   // the group's last
            __builtin_amdgcn_sched_barrier(0);
            add_up(at & 1u);
            store(group++);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                d24[r] = m24[r] = 0.0f;
                bmn[r] = w_u32x4{0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < TT; ++t) D[r][t] = tot[r][t] = w_f32x4{0, 0, 0, 0};
            }
        }
        sb = sb1;
        ring = ring2;
        go = go2;
    }
    // no load may land in LDS that is no longer this workgroup's (SKIP: none is under way since the last superblock's first meeting)
    if constexpr (!SKIP) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (p.n_splits == 1u) return;
    // A share of K (dense calls, one group): wide_sum_kernel adds the shares' tiles.  They change hands through LDS and leave in
    // whole rows (from the accumulators, in 64-byte pieces, a 28672 x 4096 call of 48 tokens took 1.5 us more).
    add_up((all - 1u) & 1u);
    __syncthreads();
    constexpr uint32_t OP = 260;   // floats between tokens: the four lane groups write to different banks
    static_assert(TT * 16 * OP * 4 <= L::R_AT, "the output tile fits");
    float* ot = (float*)lds;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint32_t from = tile_row(group0, r), col = wave * 32u + 16u * r + min(from, p.N - rows) + r16 - from;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (col >= wave * 32u + 16u * r && col < wave * 32u + 16u * r + 16u) ot[(16u * t + 4u * kq + i) * OP + col] = tot[r][t][i];
    }
    __syncthreads();
    float* tile = p.partial + (((size_t)blockIdx.z * gridDim.y + blockIdx.y) * p.row_groups + group0) * (TT * 16u * 256u);
    for (uint32_t n = tid; n < TT * 1024u; n += 512u)
        *(float4*)(tile + 4u * n) = *(const float4*)(ot + (n >> 6) * OP + 4u * (n & 63u));
}

template <int TYPE, int TT>
__global__ __launch_bounds__(512, TT == 1 ? 4 : 2) void wide_kernel(const WideParams p)
{
    __shared__ __align__(16) uint8_t lds[WideLds<TYPE, TT>::BYTES];
    const uint32_t t0 = blockIdx.y * (TT * 16u);
    wide_walk<TYPE, TT>(p, lds, blockIdx.x, p.per_wg, nullptr, t0, min(p.M - t0, TT * 16u), p.W, p.W2);
}

// Records of up to TT * 16 pairs: a workgroup walks the tiles that its record fills, each number of tiles with a walk of its own
// (a branch per tile inside one would cut its steps into pieces).  An expert's last record is half empty in the mean: with all tiles
// walked 128 experts x 8, 2048 / 768, took 555.8 / 194.1 / 154.2 us at 2048 / 512 / 256 tokens (64 / 48 / 32 pairs per record), now
// 538.9 / 183.3 / 147.3.  Records of 48 and 64 pairs walk two tiles where one is filled: a walk for it, too, gave 0.3 % more.
template <int TYPE, int TT>
__global__ __launch_bounds__(512, TT == 1 ? 4 : 2) void wide_records_kernel(const WideParams p)
{
    __shared__ __align__(16) uint8_t lds[WideLds<TYPE, TT>::BYTES];
    const uint32_t records = *p.n_records, bx = blockIdx.x + gridDim.x * blockIdx.y;
    uint32_t per_wg = p.per_wg, wgs = p.wgs_of[0];
    if constexpr (TT > 1) {   // (of 16 pairs: one group each)
        float best = 3e38f;
#pragma unroll
        for (int c = 1; c <= WIDE_MAX_GROUPS; ++c) {
            const float n = fmaxf(ceilf(((float)(p.wgs_of[c - 1] * records) - 0.5f) * p.per_cu), 1.0f);
            const float us = n * ((float)c * p.walk + p.start);
            if (us < best) { best = us; per_wg = (uint32_t)c; wgs = p.wgs_of[c - 1]; }
        }
        per_wg = (uint32_t)__builtin_amdgcn_readfirstlane((int)per_wg);
        wgs = (uint32_t)__builtin_amdgcn_readfirstlane((int)wgs);
    }
    const uint32_t all = records * wgs, share = (all + 7u) >> 3, at = (bx & 7u) * share + (bx >> 3);
    if ((bx >> 3) >= share || at >= all) return;   // whole workgroup
    const uint32_t record = (uint32_t)__builtin_amdgcn_readfirstlane((int)(at / wgs)), group = at - record * wgs;
    const uint32_t* rec = p.records + (size_t)record * p.record_words;
    const uint32_t expert = (uint32_t)__builtin_amdgcn_readfirstlane((int)rec[0]), count = (uint32_t)__builtin_amdgcn_readfirstlane((int)rec[1]);
    const size_t skip = (size_t)expert * p.N * p.row_stride_bytes;
    const uint8_t *W = p.W + skip, *W2 = p.W2 + skip;
    rec += 2;
    if constexpr (TT > 2)
        if (count <= 32u) return wide_walk<TYPE, 2>(p, lds, group, per_wg, rec, 0, count, W, W2);
    if constexpr (TT > 3)
        if (count <= 48u) return wide_walk<TYPE, 3>(p, lds, group, per_wg, rec, 0, count, W, W2);
    if constexpr (TT == 2)
        if (count <= 16u) return wide_walk<TYPE, 1>(p, lds, group, per_wg, rec, 0, count, W, W2);
    wide_walk<TYPE, TT>(p, lds, group, per_wg, rec, 0, count, W, W2);
}

// Adds the splits' partial tiles in split order, with the call's epilogue.  Workgroup (x, y): 256 columns of four
// tokens.  A launch of its own: added by the last workgroup of a tile to arrive, the splits were read one round
// trip after the other by that one workgroup (19 us of a 64-token call with eight splits).
__global__ __launch_bounds__(256) void wide_sum_kernel(const WideParams p, uint32_t tokens, uint32_t groups)
{
    const uint32_t slot = blockIdx.y * 4u + (threadIdx.x >> 6);          // token over all groups of `tokens`
    const uint32_t c = (threadIdx.x & 63u) * 4u;
    if (slot >= p.M) return;
    const uint32_t group = slot / tokens;
    const float* src = p.partial + (((size_t)group * gridDim.x + blockIdx.x) * tokens + slot % tokens) * 256u + c;
    const size_t zs = (size_t)groups * gridDim.x * tokens * 256u;
    float4 a = {0, 0, 0, 0};
#pragma unroll 8
    for (uint32_t z = 0; z < p.n_splits; ++z) {
        const float4 v = *(const float4*)(src + z * zs);
        a.x += v.x; a.y += v.y; a.z += v.z; a.w += v.w;
    }
    const size_t at = (size_t)slot * p.ldy + p.y_offset;
    float y[4] = {a.x, a.y, a.z, a.w};
    if (p.act) {
        // 16 gate columns, then their 16 up columns: the up quad sits four lanes on
        const uint32_t n = blockIdx.x * 128u + (c >> 5) * 16u + (c & 15u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float u = __shfl_down(y[i], 4, 64);
            if ((c & 16u) || n + i >= p.N) continue;
            float g = y[i];
            if (p.bias) { g += p.bias[n + i]; u += p.bias[p.N + n + i]; }
            p.Y[at + n + i] = wide_act(p.act, g) * u;
        }
        return;
    }
    const uint32_t n = blockIdx.x * 256u + c;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (n + i >= p.N) continue;
        float v = y[i];
        if (p.bias) v += p.bias[n + i];
        if (p.residual) v += p.residual[at + n + i];
        p.Y[at + n + i] = v;
    }
}

template <int TYPE>
static void launch_wide_type(const WideParams& p, uint32_t tt, dim3 grid, hipStream_t s)
{
    const auto go = [&](auto dense, auto grouped) {
        if (p.records) hipLaunchKernelGGL(grouped, grid, dim3(512), 0, s, p);
        else hipLaunchKernelGGL(dense, grid, dim3(512), 0, s, p);
    };
    if (tt == 1u) go(wide_kernel<TYPE, 1>, wide_records_kernel<TYPE, 1>);
    else if (tt == 2u) go(wide_kernel<TYPE, 2>, wide_records_kernel<TYPE, 2>);
    else if (tt == 3u) go(wide_kernel<TYPE, 3>, wide_records_kernel<TYPE, 3>);
    else go(wide_kernel<TYPE, 4>, wide_records_kernel<TYPE, 4>);
}

static hipError_t launch_wide_any(int type, const WideParams& p, uint32_t tt, dim3 grid, hipStream_t s)
{
    if (type == KQ_TYPE_Q4_K) launch_wide_type<KQ_TYPE_Q4_K>(p, tt, grid, s);
    else if (type == KQ_TYPE_Q5_K) launch_wide_type<KQ_TYPE_Q5_K>(p, tt, grid, s);
    else launch_wide_type<KQ_TYPE_Q6_K>(p, tt, grid, s);
    return hipGetLastError();
}

bool wide_supported(const MatmulArgs& a)
{
    // X in 16-byte loads; Q4_K and Q5_K blocks too (their 144 and 176 bytes keep a 16-byte aligned row aligned)
    if (((uintptr_t)a.X | (uintptr_t)a.norm_w) & 15u) return false;
    if (a.n_blocks * KQ_QK != a.K || a.N == 0) return false;
    if ((uint64_t)16u * a.row_stride_bytes > 0xFFFFFFFFull) return false;   // a tile's rows lie at 32-bit offsets
    if (a.type == KQ_TYPE_Q6_K) return !((uintptr_t)a.W & 1u) && !((uintptr_t)a.W2 & 1u);
    return !(((uintptr_t)a.W | (uintptr_t)a.W2) & 15u) && !(a.row_stride_bytes & 15u);
}

// Groups of rows that a workgroup walks one after the other are chosen by a launch's price in us: the busiest CU's workgroups,
// at `walk` per group and `start` beside them, [0] for one alone on its CU, [1] for two that share it.  At 16 tokens two
// workgroups do: a step of one takes half the two's, and its start goes under the other's walk; alone on it — all of one round,
// the odd one of several — a workgroup is a sixth slower than that (too few bytes under way).  Of 3730 dense calls of 9 to
// 16 tokens on 61441 to 262144 rows this choice is 0.3 % behind the best of one to four groups (priced without the odd one
// apart 0.9 %, by up to 16 %: Q5_K 160000 x 256 at 10 tokens 16.1 us against 14.5 with three groups; 13.9 with the compiler's order).
// Measured, us, with one group / with those chosen: 128 experts x 8, 2048 / 768, gate and up, then down: 256 tokens (3, 4) 77 / 73
// and 80 / 68, 2048 tokens (2, 2) 295 / 285 and 255 / 233.
struct WideWalk { double walk[2], start[2]; };
static WideWalk wide_walk(int type, uint32_t tt, uint32_t blocks)
{
    const bool q5 = type == KQ_TYPE_Q5_K, q6 = type == KQ_TYPE_Q6_K;
    if (tt == 1u) return {{blocks * (q6 ? 3.6 : q5 ? 2.5 : 2.1), blocks * (q6 ? 3.4 : q5 ? 2.1 : 1.75)}, {6.0, 3.0}};
    const double step = q6 ? 2.4 + 0.9 * tt : 0.8 + 0.8 * tt;
    return {{blocks * step, blocks * step}, {9.0, 9.0}};
}

static uint32_t groups_per_wg(uint32_t row_groups, uint32_t others, int type, uint32_t tt, uint32_t blocks, uint32_t cus, double* price)
{
    const WideWalk w = wide_walk(type, tt, blocks);
    uint32_t best = 1;
    double best_us = 1e30;
    for (uint32_t c = 1; c <= row_groups && c <= 64u; ++c) {
        const uint64_t n = ((uint64_t)((row_groups + c - 1u) / c) * others + cus - 1u) / cus;
        const double us = (double)(n / 2u * 2u) * (c * w.walk[1] + w.start[1]) + (double)(n % 2u) * (c * w.walk[0] + w.start[0]);
        if (us < best_us) { best_us = us; best = c; }
    }
    if (price) *price = best_us;
    return best;
}

// K is cut where the rows alone leave CUs idle (one workgroup per CU).  Prices in us, measured: a superblock of a
// workgroup's walk 0.8 + 0.7 per tile of tokens (Q6_K 3 + 0.9), the launch that adds the splits 5, and its
// traffic, written and read once, at 4 TB/s.  (Of the walk before this one; the choice is still within 4 % of the best of
// eight forced ones on 80 calls, 20 to 128 tokens, Q4_K and Q6_K.)  splits: at most so many, 0 = the cheapest.
static uint32_t wide_cut(int type, uint32_t tt, uint32_t row_groups, uint32_t token_groups, uint32_t n_blocks, const SplitScratch& sc, int splits)
{
    const double step_us = type == KQ_TYPE_Q6_K ? 3.0 + 0.9 * tt : 0.8 + 0.7 * tt;
    const size_t tile_floats = (size_t)token_groups * tt * 16u * row_groups * (WIDE_WAVES * 32u);
    uint32_t z = 1;
    double best = 1e30;
    for (uint32_t c = 1; c <= n_blocks && c <= 16u; ++c) {
        if (c > 1u && c * tile_floats > sc.capacity_floats) break;
        const uint32_t rounds = (row_groups * token_groups * c + sc.cus - 1u) / sc.cus;
        const double t = (double)rounds * ((n_blocks + c - 1u) / c) * step_us + (c > 1u ? 5.0 + 2e-6 * c * tile_floats : 0.0);
        if (splits ? (uint32_t)splits >= c : t < best) { best = t; z = c; }
    }
    return z;
}

double wide_price_16(int type, uint32_t N, uint32_t n_blocks, uint32_t cus)
{
    double us;
    groups_per_wg((N + 255u) / 256u, 1, type, 1, n_blocks, cus, &us);
    return us + 4.0;   // (the split of X in front)
}

double wide_price_5_to_16(const MatmulArgs& a, const SplitScratch& sc)
{
    const uint32_t outs = a.epi ? a.N / 2u : a.N, per_wg = a.epi ? WIDE_WAVES * 16u : WIDE_WAVES * 32u, gx = (outs + per_wg - 1u) / per_wg;
    const uint32_t cut = wide_cut(a.type, 1, gx, 1, a.n_blocks, sc, 0), per = (a.n_blocks + cut - 1u) / cut, z = (a.n_blocks + per - 1u) / per;
    double walk;
    if (z > 1u) {
        const WideWalk w = wide_walk(a.type, 1, per);
        const uint32_t n = (gx * z + sc.cus - 1u) / sc.cus;
        walk = (double)(n / 2u * 2u) * (w.walk[1] + w.start[1]) + (double)(n % 2u) * (w.walk[0] + w.start[0]);
    } else {
        groups_per_wg(gx, 1, a.type, 1, a.n_blocks, sc.cus, &walk);
    }
    // The launches' sum, walk, the one that adds the splits and its floats, 10^6 outputs, a norm (a workgroup walks its row first) and a
    // superblock of it: fitted to 128000 timed calls of 5 to 16 tokens (32 to 64000 rows, plain, with a norm, a residual, an epilogue), 4 to 5 % rms
    const double c[3][7] = {{1.364, 0.727, 3.638, 2.948, 2.733, 0.211, 0.07}, {1.165, 0.803, 3.669, 3.173, 3.368, 0.339, 0.063}, {0.953, 0.772, 4.486, 2.371, 3.407, 0.404, 0.057}};
    const double* k = c[a.type == KQ_TYPE_Q4_K ? 0 : a.type == KQ_TYPE_Q5_K ? 1 : 2];
    return k[0] + k[1] * walk + (z > 1u ? k[2] + k[3] * 1e-6 * z * 16.0 * gx * 256.0 : 0.0) + k[4] * 1e-6 * (double)a.M * outs +
           (a.pro == 1 ? k[5] + k[6] * a.n_blocks : 0.0);
}

hipError_t launch_wide(const MatmulArgs& a, const SplitScratch& sc, void* x_scratch, size_t x_bytes, int splits, hipStream_t s)
{
    const uint32_t outs = a.epi ? a.N / 2u : a.N;
    const size_t per_row = wide_x_bytes(1, a.n_blocks);
    size_t step = x_bytes / per_row;
    if (step < a.M) step = step / 64u * 64u;
    if (step == 0) return hipErrorInvalidValue;
    const uint32_t x_row = a.pro >= 2 ? 2u * a.K : a.K;
    for (uint32_t m0 = 0; m0 < a.M; m0 += (uint32_t)step) {
        const uint32_t M = a.M - m0 < step ? a.M - m0 : (uint32_t)step;
        WideParams p{};
        p.x = wide_x_layout(x_scratch, nullptr, M, a.n_blocks);
        if (hipError_t e = launch_wide_x(a.type, (const float*)a.X + (size_t)m0 * x_row, a.pro, a.norm_w, a.eps, M, a.n_blocks, p.x, s);
            e != hipSuccess) return e;
        p.W = a.W; p.W2 = a.W + (size_t)outs * a.row_stride_bytes;
        p.bias = a.bias;
        p.residual = a.residual ? a.residual + (size_t)m0 * a.ldy : nullptr;
        p.Y = a.Y + (size_t)m0 * a.ldy;
        p.M = M; p.N = outs; p.n_blocks = a.n_blocks; p.row_stride_bytes = a.row_stride_bytes;
        p.y_offset = a.y_offset; p.ldy = a.ldy; p.act = a.epi;
        const uint32_t gy = (M + 63u) / 64u, tiles = (M + 15u) / 16u, tt = (tiles + gy - 1u) / gy;
        const uint32_t gy2 = (tiles + tt - 1u) / tt;
        const uint32_t per_wg = a.epi ? WIDE_WAVES * 16u : WIDE_WAVES * 32u, gx = (outs + per_wg - 1u) / per_wg;
        const uint32_t z = wide_cut(a.type, tt, gx, gy2, a.n_blocks, sc, splits);
        p.blocks_per_split = (a.n_blocks + z - 1u) / z;
        p.n_splits = (a.n_blocks + p.blocks_per_split - 1u) / p.blocks_per_split;
        p.partial = sc.partial;
        p.row_groups = gx;
        p.per_wg = p.n_splits > 1u ? 1u : groups_per_wg(gx, gy2, a.type, tt, a.n_blocks, sc.cus, nullptr);
        if (hipError_t e = launch_wide_any(a.type, p, tt, dim3((gx + p.per_wg - 1u) / p.per_wg, gy2, p.n_splits), s); e != hipSuccess) return e;
        if (p.n_splits > 1u) {
            hipLaunchKernelGGL(wide_sum_kernel, dim3(gx, (M + 3u) / 4u), dim3(256), 0, s, p, tt * 16u, gy2);
            if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

hipError_t launch_wide_grouped(const MatmulArgs& a, const WideX& x, const uint32_t* records, const uint32_t* n_records,
                               uint32_t bound, uint32_t cap, hipStream_t s)
{
    WideParams p{};
    p.x = x;
    p.W = a.W; p.W2 = a.W2 ? a.W2 : a.W;
    p.Y = a.Y;
    p.M = a.M; p.N = a.N; p.n_blocks = a.n_blocks; p.row_stride_bytes = a.row_stride_bytes; p.ldy = a.ldy;
    p.n_splits = 1; p.blocks_per_split = a.n_blocks; p.per_wg = 1;
    p.act = a.W2 ? 2 : 0;
    p.records = records; p.n_records = n_records; p.record_words = 2u + cap; p.k_slots = a.k_slots; p.x_per_slot = a.x_per_slot;
    const uint32_t per_wg = a.W2 ? WIDE_WAVES * 16u : WIDE_WAVES * 32u;
    p.row_groups = (a.N + per_wg - 1u) / per_wg;
    const uint32_t tt = cap / 16u;
    const WideWalk w = wide_walk(a.type, tt, a.n_blocks);
    p.per_cu = 1.0f / (float)device_cu_count();
    p.walk = (float)w.walk[0]; p.start = (float)w.start[0];
    for (uint32_t c = 1; c <= WIDE_MAX_GROUPS; ++c) p.wgs_of[c - 1u] = (p.row_groups + c - 1u) / c;
    // (a dimension of the grid holds fewer than 2^32 threads; its first one a multiple of the XCDs)
    const uint64_t wgs = ((uint64_t)p.row_groups * bound + 7u) / 8u * 8u, most = a.grid_x ? a.grid_x : 1u << 22;
    const uint64_t gx = wgs < most ? wgs : most, gy = (wgs + gx - 1u) / gx;
    if (gy > 65535u) return hipErrorInvalidValue;
    return launch_wide_any(a.type, p, tt, dim3((uint32_t)gx, (uint32_t)gy), s);
}

// ------------------------------------------------------------------------------------------------------------------
// bf16 rows of a short prompt (one launch serves up to 128 tokens per workgroup, K cut over workgroups).
//
// The GEMM's tiles of 128 and 256 tokens walk K in steps of 64 with one barrier each and mostly find one workgroup per
// CU here: 1.4 us per step and CU, whatever the tokens.  This kernel walks whole superblocks as wide_walk does: X (halves of a
// superblock, a ring of three) and W go from memory to LDS without registers, a step's LDS reads and the expansion of its weights
// stand between the matrix instructions of the step before.  A wave turns its 32 rows' weights into bf16 in registers (the GEMM's
// formula and its one rounding, so both compute the same products; the quants enter v_fma_mix_f32 as fp16 subnormals where their
// bits lie) and meets every token with them: no weight passes through LDS as bf16.  Accumulation is in fp32 over the workgroup's
// whole range of K.  Against X and W read through registers ahead of a superblock, and the operands right ahead of their use: 28672 x 4096
// Q4_K at 100 tokens 51.7 -> 41.9 us, 4096 x 14336 Q6_K 37.8 -> 32.5, 28672 x 4096 at 32 tokens 28.9 -> 24.5, a layer with the launches
// between its products at 100 tokens 158 -> 141.
typedef __bf16 w_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 w_bf16x2 __attribute__((ext_vector_type(2)));
typedef float w_f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t w_pack_bf16(float lo, float hi)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((w_f32x2{lo, hi}), w_bf16x2));
}

// Its LDS.  X: a ring of three halves of a superblock, [token][16 pieces of 16 bytes], a piece's place exchanged by its token
// (^ token % 16).  W: as in WideLds.
template <int TYPE, int TT> struct ShortLds {
    using L = WideLds<TYPE, 1>;
    static constexpr uint32_t X_HALF = TT * 4096u, W_AT = 3u * X_HALF, END = W_AT + 8u * L::W_WAVE, O_BYTES = TT * 16u * 260u * 4u;
    static constexpr uint32_t BYTES = END > O_BYTES ? END : O_BYTES;
    static constexpr int N_X = (TT + 1) / 2;   // a wave's loads for half a superblock of X
};

template <int TYPE, int TT>
__global__ __launch_bounds__(512, 2) void short_kernel(const WideParams p)
{
    using L = WideLds<TYPE, 1>;
    using S = ShortLds<TYPE, TT>;
    constexpr bool Q6 = TYPE == KQ_TYPE_Q6_K, Q5 = TYPE == KQ_TYPE_Q5_K;
    constexpr uint32_t OP = 260;   // floats between tokens of the output tile, as in wide_kernel
    __shared__ __align__(16) uint8_t lds[S::BYTES];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, kq = lane >> 4, r16 = lane & 15u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    const uint32_t t0 = blockIdx.y * (TT * 16u), count = min(p.M - t0, TT * 16u);
    constexpr uint32_t BB = TYPE == KQ_TYPE_Q4_K ? KQ_Q4K_BYTES : TYPE == KQ_TYPE_Q5_K ? KQ_Q5K_BYTES : KQ_Q6K_BYTES;
    const uint32_t b0 = blockIdx.z * p.blocks_per_split, all = min(b0 + p.blocks_per_split, p.n_blocks) - b0;

    // W: lane offsets (64 bits: any row stride) from the wave's two tiles' bases.  A matrix's last tile is read from its last 16
    // rows on, what it has of an earlier one is not stored.
    const uint32_t rows = min(p.N, 16u);
    uint64_t woff[L::W_INSTR];
#pragma unroll
    for (uint32_t i = 0; i < L::W_INSTR; ++i) {
        const uint32_t n = i * 64u + lane, row = n / L::UNITS, u = n % L::UNITS;
        woff[i] = (uint64_t)min(row, rows - 1u) * p.row_stride_bytes + u * 16u;
    }
    const uint64_t doff = (uint64_t)min(r16, rows - 1u) * p.row_stride_bytes + 206u;
    const uint32_t from0 = (blockIdx.x * WIDE_WAVES + wave) * 32u;
    const uint8_t* wsrc[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) wsrc[r] = p.W + (size_t)min(from0 + 16u * r, p.N - rows) * p.row_stride_bytes + (size_t)b0 * BB;
    const uint32_t w_lds = lds0 + S::W_AT + wave * L::W_WAVE;
    auto request_w = [&](int k) {   // piece k of a superblock's weights: whole loads, then each tile's last lanes (and d)
        constexpr int WHOLE = 2 * ((int)L::W_INSTR - 1);
        const int r = k & 1, i = k >> 1;
        if (k < WHOLE) lds_dma16<false>(w_lds + r * L::W_TILE + i * 1024u, wsrc[r] + woff[i], -1);
        else if (k < WHOLE + 2) lds_dma16_lanes(w_lds + r * L::W_TILE + (L::W_INSTR - 1u) * 1024u, wsrc[r] + woff[L::W_INSTR - 1u], (1ull << L::W_LAST) - 1ull);
        else lds_dma4_lanes(w_lds + 2u * L::W_TILE + r * 64u, wsrc[r] + doff, 0xFFFFull);
    };
    // X: load i of the wave takes half a superblock of four tokens (beyond the count the last again: outputs that are dropped).  The
    // halves are chosen so that a half's pieces lie together: Q4_K, Q5_K the low nibbles' elements, then the high ones' (64 bytes of each
    // 128), Q6_K elements 0 .. 63 of each 128, then 64 .. 127.
    const uint8_t* xp[S::N_X];
#pragma unroll
    for (int i = 0; i < S::N_X; ++i) {
        const uint32_t n = i * WIDE_WAVES + wave, tok = 4u * n + (lane >> 4), piece = (lane ^ tok) & 15u, jj = piece >> 2, g = piece & 3u;
        const uint32_t c = Q6 ? 16u * (g >> 1) + 4u * (jj >> 1) + 2u * (g & 1u) + (jj & 1u) : 8u * g + jj;
        xp[i] = p.x.xa + ((size_t)(t0 + min(tok, count - 1u)) * p.n_blocks + b0) * 512u + c * 16u;
    }
    int x_last = (S::N_X - 1) * WIDE_WAVES + wave < TT * 4u ? -1 : 0;   // is the last of these there: all lanes or none
    asm("s_nop 1\n\tv_readfirstlane_b32 %0, %1" : "=s"(x_last) : "v"(x_last));
    constexpr int HALF = Q6 ? 128 : 64;   // bytes from a piece to the second half's
    auto request_x = [&](uint32_t ring, int i, int step) {
        const uint32_t to = lds0 + ring * S::X_HALF + (i * WIDE_WAVES + wave) * 1024u;
        if (TT % 2 && i == S::N_X - 1) lds_dma16_or_none(to, xp[i], x_last);
        else lds_dma16<false>(to, xp[i], -1);
        xp[i] += step;
    };

    uint32_t a_lane[4];   // operands of X for step j: four places of the exchanged pieces
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) a_lane[jj] = r16 * 256u + (((4u * jj + kq) ^ r16) & 15u) * 16u;
    w_bf16x8 A[2][TT];
    auto read_a = [&](uint32_t ring, int j) {
        const uint8_t* x = lds + ring * S::X_HALF + a_lane[j & 3];
#pragma unroll
        for (int t = 0; t < TT; ++t) A[j & 1][t] = *(const w_bf16x8*)(x + t * 4096);
    };
    WideW<TYPE> w[2];
    auto read_w = [&]() {
#pragma unroll
        for (int r = 0; r < 2; ++r)
            w[r].load_lds(lds + S::W_AT + wave * L::W_WAVE + r * L::W_TILE + r16 * (L::UNITS * 16u),
                          lds + S::W_AT + wave * L::W_WAVE + 2u * L::W_TILE + r * 64u + r16 * 4u, kq);
    };
    // a weight is q * sa + sb, q read as an fp16 subnormal where its bits lie (q * 2^-24; Q4_K's high nibbles q * 2^-20: the scale
    // carries the power of two, which is exact, so the sum rounds the same value)
    float sa[2][Q6 ? 4 : 2], sb[2][Q6 ? 4 : 2];
    auto headers = [&]() {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if constexpr (Q6) {
                const float d = half_bits_to_float(w[r].d);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const uint32_t word = t < 2 ? w[r].sc.x : w[r].sc.y;
                    const float s = d * (float)(int)(int8_t)(word >> (16 * (t & 1) + 8 * (kq & 1u)));
                    sa[r][t] = s * 16777216.0f;
                    sb[r][t] = -32.0f * s;   // exact: the sum rounds once, as s * (q - 32) does
                }
            } else {
                const w_u32x4 h = w[r].hdr;
                const float d = half_bits_to_float(h.x & 0xFFFFu), dmin = half_bits_to_float(h.x >> 16);
                // (arithmetic, no choice between the two: the compiler would branch)
                const uint32_t sc = ((kq < 2u ? h.y : h.w) & 0x0F0F0F0Fu) | ((h.y >> (kq & 2u)) & 0x30303030u);
                const uint32_t mn = (((kq < 2u ? h.z : h.w) >> (2u * (kq & 2u))) & 0x0F0F0F0Fu) | ((h.z >> (kq & 2u)) & 0x30303030u);
                const uint32_t s2 = sc >> (16u * (kq & 1u)), m2 = mn >> (16u * (kq & 1u));
                sa[r][0] = d * (float)(s2 & 255u) * 16777216.0f;
                sa[r][1] = d * (float)((s2 >> 8) & 255u) * 1048576.0f;
                sb[r][0] = -(dmin * (float)(m2 & 255u));
                sb[r][1] = -(dmin * (float)((m2 >> 8) & 255u));
            }
        }
    };
    w_bf16x8 B[2][2];   // [step % 2][tile]
    auto expand = [&](int j) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            w_u32x4 o;
            const int n = Q6 ? j >> 1 : j >> 2;   // which scale
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                w_half2 a, b;   // elements 0 and 2, 1 and 3
                if constexpr (Q6) {
                    const int t = j >> 1, u = j & 1;
                    const uint32_t l = w[r].ql[t & 1][2 * u + i], h = w[r].qh[2 * u + i];
                    const uint32_t c = ((l >> (4 * (t >> 1))) & 0x0F0F0F0Fu) | ((t < 2 ? h << (4 - 2 * t) : h >> (2 * t - 4)) & 0x30303030u);
                    a = __builtin_bit_cast(w_half2, __builtin_amdgcn_perm(0u, c, 0x0c020c00u));
                    b = __builtin_bit_cast(w_half2, __builtin_amdgcn_perm(0u, c, 0x0c030c01u));
                } else {
                    const int i8 = j & 3;
                    const uint32_t d = w[r].q[i8 >> 1][2 * (i8 & 1) + i], m = n ? 0x00F000F0u : 0x000F000Fu;
                    uint32_t e = d & m, f = (d >> 8) & m;
                    if constexpr (Q5) {
                        // bit 2kq + n of a byte of fifth bits: bit 4 beside a low nibble, bit 8 beside a high one
                        const uint32_t g = w[r].f[i8 >> 1][2 * (i8 & 1) + i] >> (2u * kq);
                        e |= n ? (g << 7) & 0x01000100u : (g << 4) & 0x00100010u;
                        f |= n ? (g >> 1) & 0x01000100u : (g >> 4) & 0x00100010u;
                    }
                    a = __builtin_bit_cast(w_half2, e);
                    b = __builtin_bit_cast(w_half2, f);
                }
                const _Float16 a0 = a.x, a1 = a.y, c0 = b.x, c1 = b.y;
                o[2 * i] = w_pack_bf16(fmaf((float)a0, sa[r][n], sb[r][n]), fmaf((float)c0, sa[r][n], sb[r][n]));
                o[2 * i + 1] = w_pack_bf16(fmaf((float)a1, sa[r][n], sb[r][n]), fmaf((float)c1, sa[r][n], sb[r][n]));
            }
            B[j & 1][r] = __builtin_bit_cast(w_bf16x8, o);
        }
    };
    w_f32x4 acc[2][TT];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[r][t] = w_f32x4{0, 0, 0, 0};
    auto multiply = [&](int j) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < 2; ++r) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[j & 1][t], B[j & 1][r], acc[r][t], 0, 0, 0);
    };
    auto schedule = [&]() {
        constexpr int NV = ((Q6 ? 50 : Q5 ? 54 : 38) + 2 * TT - 1) / (2 * TT);
#pragma unroll
        for (int i = 0; i < 2 * TT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (i < TT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // The walk, as wide_walk's: W a superblock ahead, X two halves; past the end the last is requested again.
    constexpr int N_X = S::N_X, N_W = L::N_W, WAS = (N_X + N_W + 3) / 4, XBS = (N_X + 3) / 4;
    auto next_w = [&](uint32_t at) {
        const uint32_t step = at + 1u < all ? BB : 0u;
        wsrc[0] += step;
        wsrc[1] += step;
    };
    auto x_step = [&](uint32_t at) -> int { return at + 1u >= all ? -HALF : 512 - HALF; };
#pragma unroll
    for (int k = 0; k < N_W; ++k) request_w(k);
    next_w(0);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < N_X; ++i) request_x(h, i, h == 0 ? HALF : x_step(0));
    wide_meet<N_X>();
    read_w();
    w[0].arrived(); w[1].arrived();
#pragma unroll
    for (int k = 0; k < WAS; ++k) request_w(k);
    headers();
    read_a(0, 0);
    expand(0);
    uint32_t ring = 0;   // where the superblock's first half lies
    for (uint32_t at = 0; at < all; ++at) {
        const uint32_t ring1 = ring + 1u == 3u ? 0u : ring + 1u, ring2 = 3u - ring - ring1;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (j == 3) {
                // every wave has read the first half; the second has arrived
                wide_meet<N_X + N_W>();
                read_a(ring1, 4);
                expand(4);
            } else if (j == 7) {
                wide_meet<N_X>();
                read_w();
                read_a(ring2, 0);
                w[0].arrived(); w[1].arrived();
#pragma unroll
                for (int k = 0; k < WAS; ++k) request_w(k);
                headers();
                expand(0);
            } else {
                read_a(j < 3 ? ring : ring1, j + 1);
                expand(j + 1);
                if (j < 3) {
#pragma unroll
                    for (int k = (j + 1) * WAS; k < (j + 2) * WAS && k < N_X + N_W; ++k) {
                        if (k < N_W) request_w(k);
                        else request_x(ring2, k - N_W, HALF);
                    }
                }
            }
            if (j >= 3 && j < 7) {
#pragma unroll
                for (int i = (j - 3) * XBS; i < (j - 2) * XBS && i < N_X; ++i) request_x(ring, i, x_step(at + 1u));
            }
            multiply(j);
            schedule();
            if (j == 2) next_w(at + 1u);
        }
        ring = ring2;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load may land in the output tile
    __syncthreads();

    // outputs through LDS, as in wide_kernel
    float* ot = (float*)lds;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint32_t from = from0 + 16u * r, first = wave * 32u + 16u * r, col = first + min(from, p.N - rows) + r16 - from;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (col >= first && col < first + 16u) ot[(16 * t + 4u * kq + i) * OP + col] = acc[r][t][i];
    }
    __syncthreads();
    if (p.n_splits > 1) {   // wide_sum_kernel adds the splits' tiles
        float* tile = p.partial + (((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * (TT * 16u * 256u);
        for (uint32_t n = tid; n < TT * 1024u; n += 512u)
            *(float4*)(tile + 4u * n) = *(const float4*)(ot + (n >> 6) * OP + 4u * (n & 63u));
        return;
    }
    const uint32_t col = tid & 255u, n = blockIdx.x * 256u + col;
    if (n >= p.N) return;
    const float bv = p.bias ? p.bias[n] : 0.0f;
#pragma unroll 4
    for (uint32_t slot = tid >> 8; slot < count; slot += 2u) p.Y[(size_t)(t0 + slot) * p.ldy + n] = ot[slot * OP + col] + bv;
}

template <int TYPE>
static void launch_short_type(const WideParams& p, uint32_t tt, dim3 grid, hipStream_t s)
{
    switch (tt) {
    case 1: case 2: hipLaunchKernelGGL((short_kernel<TYPE, 2>), grid, dim3(512), 0, s, p); break;
    case 3: hipLaunchKernelGGL((short_kernel<TYPE, 3>), grid, dim3(512), 0, s, p); break;
    case 4: hipLaunchKernelGGL((short_kernel<TYPE, 4>), grid, dim3(512), 0, s, p); break;
    case 5: hipLaunchKernelGGL((short_kernel<TYPE, 5>), grid, dim3(512), 0, s, p); break;
    case 6: hipLaunchKernelGGL((short_kernel<TYPE, 6>), grid, dim3(512), 0, s, p); break;
    case 7: hipLaunchKernelGGL((short_kernel<TYPE, 7>), grid, dim3(512), 0, s, p); break;
    default: hipLaunchKernelGGL((short_kernel<TYPE, 8>), grid, dim3(512), 0, s, p); break;
    }
}

// How a call of M bf16 tokens is cut, its price in us and what the GEMM takes.  A superblock of a workgroup's walk costs
// 1.1 + 0.27 per tile of tokens (Q5_K 1.7 + 0.25, Q6_K 2.15 + 0.24), a round over the CUs 2.7 + 0.15 per tile and 2.5 behind the
// first, the launch that adds the splits 3.5 and 1.4 per 10^6 floats, 10^6 outputs 0.9: fitted to 31400 timed calls of 17 to 512
// tokens to 6 % rms.  Over these calls the choice is 0.5 % slower than the faster of the two kernels in the mean and more than 5 %
// slower on 1107; with the prices of the walk through registers that came before it was 6 % and 6145.  The GEMM has to be 5 %
// dearer: close calls stay where they were.  us at 100 / 128 / 256 tokens, with the walk before / this one / the GEMM: Q4_K
// 28672x4096 51.7 / 41.9 / 62.6, 57.5 / 46.6 / 60.0, 88.8 / 63.9 / 63.6; Q6_K 4096x14336 37.8 / 32.5 / 57.9, 40.4 / 35.2 / 58.3,
// 56.4 / 46.1 / 59.5.
ShortPlan plan_short(int type, uint32_t M, uint32_t N, uint32_t K, size_t capacity_floats, uint32_t cus)
{
    ShortPlan best{0, 0, 0, 0, 1e30, 0.0};
    const uint32_t n_blocks = K / KQ_QK, tiles = (M + 15u) / 16u, gy0 = (tiles + 7u) / 8u;
    uint32_t tt = (tiles + gy0 - 1u) / gy0;
    if (tt < 2u) tt = 2u;
    const uint32_t gy = (tiles + tt - 1u) / tt, gx = (N + 255u) / 256u;
    const double step_us = type == KQ_TYPE_Q4_K ? 1.1 + 0.27 * tt : type == KQ_TYPE_Q5_K ? 1.7 + 0.25 * tt : 2.15 + 0.24 * tt;
    const size_t tile_floats = (size_t)gy * tt * 16u * gx * 256u;
    const double out = 1e-6 * (double)M * N;
    for (uint32_t c = 1; c <= n_blocks && c <= 16u; ++c) {
        const uint32_t per = (n_blocks + c - 1u) / c, z = (n_blocks + per - 1u) / per;
        if (z > 1u && z * tile_floats > capacity_floats) break;
        const double rounds = (double)(((uint64_t)gx * gy * z + cus - 1u) / cus);
        const double us = 1.6 + 2.5 * (rounds - 1.0) + rounds * (per * step_us + 2.7 + 0.15 * tt) +
                          (z > 1u ? 3.5 + 1.4e-6 * (double)z * (double)tile_floats + 0.9 * out : 0.95 * out);
        if (us < best.us) best = ShortPlan{tt, gy, z, per, us, 0.0};
    }
    best.gemm_us = 0.95 * gemm_price_us(type, M, N, K, cus);
    return best;
}

hipError_t launch_short(const MatmulArgs& a, const ShortPlan& plan, const SplitScratch& sc, hipStream_t s)
{
    WideParams p{};
    p.x.xa = (uint8_t*)const_cast<void*>((const void*)a.X);
    p.W = a.W; p.bias = a.bias; p.Y = a.Y;
    p.M = a.M; p.N = a.N; p.n_blocks = a.n_blocks; p.row_stride_bytes = a.row_stride_bytes; p.ldy = a.ldy;
    p.blocks_per_split = plan.blocks_per_split;
    p.n_splits = plan.splits;
    p.partial = sc.partial;
    const dim3 grid((a.N + 255u) / 256u, plan.groups, plan.splits);
    if (a.type == KQ_TYPE_Q4_K) launch_short_type<KQ_TYPE_Q4_K>(p, plan.tiles, grid, s);
    else if (a.type == KQ_TYPE_Q5_K) launch_short_type<KQ_TYPE_Q5_K>(p, plan.tiles, grid, s);
    else launch_short_type<KQ_TYPE_Q6_K>(p, plan.tiles, grid, s);
    if (hipError_t e = hipGetLastError(); e != hipSuccess || plan.splits <= 1u) return e;
    hipLaunchKernelGGL(wide_sum_kernel, dim3(grid.x, (a.M + 3u) / 4u), dim3(256), 0, s, p, plan.tiles * 16u, plan.groups);
    return hipGetLastError();
}

}  // namespace kq
