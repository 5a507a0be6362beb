// kq_group.h — (token, slot) pairs bucketed by expert into records, by one workgroup of 1024 threads.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace kq {

// One workgroup buckets all pairs.  tiles: records of (2 + cap) words
// {expert, count, pair ids...}; experts appear in ascending order, the pairs
// of an expert in arrival order (the per-pair results do not depend on it).
// One pass over the pairs: the LDS counter's old value is the pair's place inside its expert, and the
// first pairs of a thread stay in registers until the records' places are known; the first record of
// every expert comes from a scan over the workgroup (eight experts per thread, a wave scan, the waves'
// totals through LDS) instead of one thread walking all experts.
// KEEP: pairs per thread kept in registers; MORE: there may be others, which are read again, one dependent load after the other
// (16384 pairs took 17.5 us with 4 kept, 14 with all of them; up to 4096 pairs the short form is 0.7 us ahead).
// sm: three words per expert.
template <int KEEP, bool MORE>
__device__ __forceinline__ void group_pairs(const uint32_t* __restrict__ expert_idx, uint32_t n_pairs, uint32_t n_experts, uint32_t cap,
                                            uint32_t* __restrict__ tiles, uint32_t* __restrict__ n_tiles, uint32_t* sm)
{
    uint32_t* count = sm;                  // [n_experts]
    uint32_t* base = sm + n_experts;       // [n_experts] first tile of the expert
    uint32_t* fill = sm + 2 * n_experts;   // [n_experts] places taken by the kept pairs (where there are more)
    __shared__ uint32_t wave_total[16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    for (uint32_t e = tid; e < n_experts; e += 1024u) count[e] = 0;
    __syncthreads();
    uint32_t my_e[KEEP], my_pos[KEEP];
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const uint32_t p = tid + (uint32_t)i * 1024u;
        my_e[i] = 0xFFFFFFFFu;
        if ((uint32_t)i * 1024u >= n_pairs) continue;   // (uniform)
        if (p < n_pairs) my_e[i] = expert_idx[p];
    }
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        my_pos[i] = 0;
        if ((uint32_t)i * 1024u >= n_pairs) continue;   // (uniform)
        if (my_e[i] < n_experts) my_pos[i] = atomicAdd(&count[my_e[i]], 1u);   // out-of-range ids are dropped
    }
    __syncthreads();
    const bool more = MORE && n_pairs > KEEP * 1024u;   // (uniform)
    if (more) {
        // pairs beyond the kept ones: counted now, placed behind the kept ones by a second read below
        for (uint32_t e = tid; e < n_experts; e += 1024u) fill[e] = count[e];
        __syncthreads();
        for (uint32_t p = tid + KEEP * 1024u; p < n_pairs; p += 1024u) {
            const uint32_t e = expert_idx[p];
            if (e < n_experts) atomicAdd(&count[e], 1u);
        }
        __syncthreads();
    }
    // exclusive scan of the experts' record counts: thread t owns experts 8t .. 8t+7
    uint32_t nt[8], mine = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t e = tid * 8u + j;
        nt[j] = e < n_experts ? (count[e] + cap - 1u) / cap : 0u;
        mine += nt[j];
    }
    uint32_t incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t v = __shfl_up(incl, o, 64);
        if (lane >= (uint32_t)o) incl += v;
    }
    if (lane == 63u) wave_total[wave] = incl;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        const uint32_t v = wave_total[w];
        before += (uint32_t)w < wave ? v : 0u;
        all += v;
    }
    uint32_t run = before + incl - mine;
    const uint32_t stride = 2u + cap;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t e = tid * 8u + j;
        if (e < n_experts) {
            base[e] = run;
            for (uint32_t i = 0; i < nt[j]; ++i) {
                uint32_t* rec = tiles + (size_t)(run + i) * stride;
                rec[0] = e;
                rec[1] = min(cap, count[e] - i * cap);
            }
            run += nt[j];
        }
    }
    if (tid == 0) *n_tiles = all;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        if ((uint32_t)i * 1024u >= n_pairs) continue;   // (uniform)
        const uint32_t e = my_e[i];
        if (e < n_experts) tiles[(size_t)(base[e] + my_pos[i] / cap) * stride + 2u + my_pos[i] % cap] = tid + (uint32_t)i * 1024u;
    }
    if (more) {
        for (uint32_t p = tid + KEEP * 1024u; p < n_pairs; p += 1024u) {
            const uint32_t e = expert_idx[p];
            if (e >= n_experts) continue;
            const uint32_t pos = atomicAdd(&fill[e], 1u);
            tiles[(size_t)(base[e] + pos / cap) * stride + 2u + pos % cap] = p;
        }
    }
}

}  // namespace kq
