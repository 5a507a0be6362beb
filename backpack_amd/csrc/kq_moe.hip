// kq_moe.hip — MoE expert path: on-GPU grouping of (token, slot) pairs by expert,
// the activation between gate/up and down, and the weighted combine.
//
// The reference dispatches one matvec per slot against offsets[slot] =
// expert * rowsPerExpert (compute_offsets.wgsl) and, for T > 1, one per token
// and slot with no reuse of an expert's weights between tokens.  Here the
// T*k pairs are bucketed by expert into tiles of up to CAP pairs; a tile is one
// grid.z slice of the row kernel, so an expert's rows are streamed once per
// tile and shared by its pairs.  Nothing returns to the host: tile count and
// contents stay in device memory and surplus grid slices exit at once.
#include <cmath>
#include "kq_format.h"
#include "kq_group.h"
#include "kq_kernels.h"

namespace kq {

template <int KEEP, bool MORE>
__global__ __launch_bounds__(1024) void moe_group_kernel(const uint32_t* __restrict__ expert_idx, uint32_t n_pairs,
                                                         uint32_t n_experts, uint32_t cap, uint32_t* __restrict__ tiles,
                                                         uint32_t* __restrict__ n_tiles)
{
    extern __shared__ uint32_t sm[];
    group_pairs<KEEP, MORE>(expert_idx, n_pairs, n_experts, cap, tiles, n_tiles, sm);
}

// act[p, i] = silu(gate[p, i]) * up[p, i] with silu(g) = g / (exp(-g) + 1)
__global__ __launch_bounds__(256) void moe_silu_mul_kernel(const float* __restrict__ gate, const float* __restrict__ up,
                                                           float* __restrict__ act, size_t n)
{
    const size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const float g = gate[i];
    act[i] = g / (expf(-g) + 1.0f) * up[i];
}

// out[t, h] = sum over slots, in slot order, of wt[t, s] * down[(t*k + s), h].  A pair that the grouping dropped (its id is
// no expert's) has no row of its own in down, which holds whatever the scratch memory did: it adds nothing.
__global__ __launch_bounds__(256) void moe_combine_kernel(const float* __restrict__ down, const float* __restrict__ wt,
                                                          const uint32_t* __restrict__ expert_idx, uint32_t n_experts,
                                                          float* __restrict__ out, uint32_t k, uint32_t hidden)
{
    const uint32_t t = blockIdx.y;
    const uint32_t h = blockIdx.x * 256u + threadIdx.x;
    if (h >= hidden) return;
    float a = -0.0f;   // (the sum's neutral element)
    for (uint32_t s = 0; s < k; ++s) {
        const float v = wt[(size_t)t * k + s] * down[((size_t)t * k + s) * hidden + h];
        const bool kept = expert_idx[(size_t)t * k + s] < n_experts;
        a = kept ? a + v : a;
    }
    out[(size_t)t * hidden + h] = a;
}

// The same in pieces of four outputs (hidden a multiple of four, pointers on 16 bytes), eight slots' rows in flight: 2048 x 8
// rows of 2048 (151 MB) 38 -> 23 us.
__global__ __launch_bounds__(64) void moe_combine4_kernel(const float* __restrict__ down, const float* __restrict__ wt,
                                                           const uint32_t* __restrict__ expert_idx, uint32_t n_experts,
                                                           float* __restrict__ out, uint32_t k, uint32_t hidden)
{
    const uint32_t t = blockIdx.y, h = 4u * (blockIdx.x * 64u + threadIdx.x);
    if (h >= hidden) return;
    const float* row = down + (size_t)t * k * hidden + h;
    float a[4] = {-0.0f, -0.0f, -0.0f, -0.0f};   // (the sum's neutral element)
    for (uint32_t s0 = 0; s0 < k; s0 += 8u) {
        float4 d[8];
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) d[i] = *(const float4*)(row + (size_t)min(s0 + i, k - 1u) * hidden);
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) {
            if (s0 + i >= k) break;
            const float w = wt[(size_t)t * k + s0 + i];
            const bool kept = expert_idx[(size_t)t * k + s0 + i] < n_experts;
            const float v[4] = {w * d[i].x, w * d[i].y, w * d[i].z, w * d[i].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) a[e] = kept ? a[e] + v[e] : a[e];
        }
    }
    *(float4*)(out + (size_t)t * hidden + h) = float4{a[0], a[1], a[2], a[3]};
}

int moe_sets_for(uint32_t n_pairs, uint32_t n_experts)
{
    const uint32_t per = (n_pairs + n_experts - 1u) / n_experts;
    return per <= 1u ? 1 : per <= 4u ? 2 : 4;
}

uint32_t moe_tiles_bound(uint32_t n_pairs, uint32_t n_experts, int sets)
{
    const uint32_t cap = 2u * (uint32_t)sets;
    const uint32_t a = n_pairs / cap + n_experts;   // every expert can add one partial tile
    return a < n_pairs ? a : n_pairs;
}

// Records that n_pairs pairs spread evenly (independently) over n_experts experts are expected to make at cap
// pairs per record: n_experts * E[ceil(n / cap)] for n ~ Poisson(n_pairs / n_experts).  Host arithmetic for launch
// shapes only; the device counts the real ones.
double moe_expected_records(uint32_t n_pairs, uint32_t n_experts, uint32_t cap)
{
    if (n_experts == 0u || cap == 0u) return 0.0;
    const double lambda = (double)n_pairs / (double)n_experts;
    if (lambda > 500.0) return (double)n_experts * (lambda / (double)cap + 0.5);
    double pmf = std::exp(-lambda), sum = 0.0;
    const uint32_t top = (uint32_t)(lambda + 12.0 * std::sqrt(lambda) + 24.0);
    for (uint32_t n = 1; n <= top; ++n) {
        pmf *= lambda / (double)n;
        sum += pmf * (double)((n + cap - 1u) / cap);
    }
    return (double)n_experts * sum;
}

size_t moe_tiles_words(uint32_t n_pairs, uint32_t n_experts, int sets)
{
    return (size_t)moe_tiles_bound(n_pairs, n_experts, sets) * (2u + 2u * (uint32_t)sets) + 1u;   // + n_tiles
}

hipError_t launch_moe_group(const uint32_t* expert_idx, uint32_t n_pairs, uint32_t n_experts, int sets, uint32_t* tiles,
                            uint32_t* n_tiles, hipStream_t s)
{
    if (n_experts > 8192u) return hipErrorInvalidValue;   // three LDS arrays of n_experts words, eight experts per thread
    if (n_pairs <= 4096u)
        hipLaunchKernelGGL((moe_group_kernel<4, false>), dim3(1), dim3(1024), 3 * n_experts * sizeof(uint32_t), s, expert_idx, n_pairs,
                           n_experts, 2u * (uint32_t)sets, tiles, n_tiles);
    else
        hipLaunchKernelGGL((moe_group_kernel<16, true>), dim3(1), dim3(1024), 3 * n_experts * sizeof(uint32_t), s, expert_idx, n_pairs,
                           n_experts, 2u * (uint32_t)sets, tiles, n_tiles);
    return hipGetLastError();
}

hipError_t launch_moe_silu_mul(const float* gate, const float* up, float* act, size_t n, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(moe_silu_mul_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, gate, up, act, n);
    return hipGetLastError();
}

hipError_t launch_moe_combine(const float* down, const float* wt, const uint32_t* expert_idx, uint32_t n_experts, float* out,
                              uint32_t T, uint32_t k, uint32_t hidden, hipStream_t s)
{
    for (uint32_t t0 = 0; t0 < T; t0 += 65535u) {
        const uint32_t tc = T - t0 < 65535u ? T - t0 : 65535u;
        if (hidden % 4u == 0 && !(((uintptr_t)down | (uintptr_t)out) & 15u)) {
            hipLaunchKernelGGL(moe_combine4_kernel, dim3((hidden / 4u + 63u) / 64u, tc), dim3(64), 0, s,
                               down + (size_t)t0 * k * hidden, wt + (size_t)t0 * k, expert_idx + (size_t)t0 * k, n_experts,
                               out + (size_t)t0 * hidden, k, hidden);
            continue;
        }
        hipLaunchKernelGGL(moe_combine_kernel, dim3((hidden + 255) / 256, tc), dim3(256), 0, s,
                           down + (size_t)t0 * k * hidden, wt + (size_t)t0 * k, expert_idx + (size_t)t0 * k, n_experts,
                           out + (size_t)t0 * hidden, k, hidden);
    }
    return hipGetLastError();
}

}  // namespace kq
