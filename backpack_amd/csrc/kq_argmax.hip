// kq_argmax.hip — the greedy-sampling tail behind the lm_head matvec: index of the largest logit per row.
//
// Replaces the two dispatches argmax + argmax_reduce (runtime/kernels/.../argmax.wgsl: per-workgroup
// scan of a chunk with `v > best` from best = -1e30, index 0; argmax_reduce.wgsl: the same over the
// partials; wired in runtime/model_runner.cpp:2441-2453) by one launch: up to ARGMAX_PARTS workgroups per
// row leave a partial each, the last of them to arrive (a ticket per row) reduces the partials and re-arms
// the ticket.  Among equal maxima the lowest index is returned (the reference's butterfly leaves that
// to the lane order); a row with nothing above -1e30 yields index 0.
#include <hip/hip_runtime.h>

#include "kq_kernels.h"
#include "kq_wave.h"

namespace kq {

// Best of a workgroup of 256 lanes; valid in thread 0.
__device__ __forceinline__ void argmax_block(float& v, uint32_t& i, float (&sv)[4], uint32_t (&si)[4])
{
    wave_best(v, i);
    if ((threadIdx.x & 63u) == 0) { sv[threadIdx.x >> 6] = v; si[threadIdx.x >> 6] = i; }
    __syncthreads();
    if (threadIdx.x == 0) {
        v = sv[0]; i = si[0];
#pragma unroll
        for (int w = 1; w < 4; ++w) best_of(v, i, sv[w], si[w]);
    }
}

__global__ __launch_bounds__(256) void argmax_rows_kernel(const float* logits, uint32_t N, uint32_t ld, int32_t* out_idx,
                                                          float* out_val, float* part_val, uint32_t* part_idx,
                                                          uint32_t* tickets)
{
    __shared__ float sv[4];
    __shared__ uint32_t si[4];
    __shared__ bool last;
    const uint32_t row = blockIdx.y, parts = gridDim.x;
    const float* x = logits + (size_t)row * ld;
    // (places beyond 32 bits where N is near 2^32: 64-bit ones, and a walk that counts from the part's start)
    const uint64_t chunk = (((uint64_t)N + parts - 1u) / parts + 3u) & ~3ull;
    const uint64_t at = blockIdx.x * chunk;
    const uint32_t begin = at < N ? (uint32_t)at : N, len = chunk < N - begin ? (uint32_t)chunk : N - begin;
    float v = -1e30f;
    uint32_t i = 0xFFFFFFFFu;   // "none yet": any real index is lower
    // four logits per lane and load (a row may start at any float), four loads in flight
    const uint32_t whole = len & ~3u;
    x += begin;
    for (uint32_t k0 = 4u * threadIdx.x; k0 < whole; k0 += 4096u) {
        float t[4][4];
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) __builtin_memcpy(t[u], x + min(k0 + 1024u * u, whole - 4u), 16);
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u)
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e)
                // ascending k per lane: the first of equals stays (a piece past the end is the last one again, seen by the lane
                // that owns it or lost to it: equal values, and best_of takes the lower index)
                if (t[u][e] > v) { v = t[u][e]; i = begin + min(k0 + 1024u * u, whole - 4u) + e; }
    }
    if (threadIdx.x < len - whole) {
        const float t = x[whole + threadIdx.x];
        if (t > v) { v = t; i = begin + whole + threadIdx.x; }
    }
    argmax_block(v, i, sv, si);
    if (threadIdx.x == 0) {
        const size_t cell = (size_t)row * parts + blockIdx.x;
        __hip_atomic_store(&part_val[cell], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&part_idx[cell], i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // Write-through stores acknowledged before the ticket, agent-scope loads by the last to arrive.  (An acquire / release
        // ticket wrote back and invalidated the XCD's L2 once per workgroup: 48 rows of 128256 logits 39 us.)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const uint32_t t = __hip_atomic_fetch_add(&tickets[row], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = t == parts - 1u;
    }
    __syncthreads();
    if (!last) return;
    asm volatile("" ::: "memory");
    v = -1e30f;
    i = 0xFFFFFFFFu;
    for (uint32_t q = threadIdx.x; q < parts; q += 256u) {
        const size_t cell = (size_t)row * parts + q;
        const float pv = __hip_atomic_load(&part_val[cell], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t pi = __hip_atomic_load(&part_idx[cell], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        best_of(v, i, pv, pi);
    }
    __syncthreads();   // sv / si are reused
    argmax_block(v, i, sv, si);
    if (threadIdx.x == 0) {
        out_idx[row] = i == 0xFFFFFFFFu ? 0 : (int32_t)i;
        if (out_val) out_val[row] = v;
        __hip_atomic_store(&tickets[row], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // re-armed for the next launch
    }
}

// Scratch of the entry point that allocates nothing (bpk_argmax_rows_static): partial values | partial
// indices | tickets, the layout of the allocated scratch of bpk_argmax_rows, 132 096 bytes that every GPU
// the library runs on holds until the process ends.  Zero when the code object is loaded; the last
// workgroup of a row to arrive puts the row's ticket back to zero, so every launch finds its tickets
// cleared.  In host code this name stands for the array only as a symbol: its device address, one per
// GPU, comes from hipGetSymbolAddress below and is what launches are given.
static __device__ __align__(256) __attribute__((used)) uint32_t scratch[ARGMAX_STATIC_WORDS];

hipError_t argmax_static_scratch(uint32_t** out)
{
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));   // of the current device
    if (e != hipSuccess) return e;
    *out = (uint32_t*)ptr;
    return hipSuccess;
}

// scratch: ARGMAX_MAX_ROWS * ARGMAX_PARTS floats, as many words, ARGMAX_MAX_ROWS tickets (zero between launches)
hipError_t launch_argmax_rows(const float* logits, uint32_t M, uint32_t N, uint32_t ld, int32_t* out_idx,
                              float* out_val, float* part_val, uint32_t* part_idx, uint32_t* tickets, hipStream_t s)
{
    const uint32_t at_most = 2u * device_cu_count();
    for (uint32_t m0 = 0; m0 < M; m0 += ARGMAX_MAX_ROWS) {
        const uint32_t rows = M - m0 < ARGMAX_MAX_ROWS ? M - m0 : ARGMAX_MAX_ROWS;
        // a part is worth at least a few thousand logits, and a launch at most two workgroups per CU: the partials and tickets
        // of more, past the non-coherent cache levels, cost more than their loads in flight give.  Calls in a row, without
        // this bound, with four per CU and with two: 48 rows of 128256 15.5, 11.0, 10.6 us (10.4 is the host's share),
        // 128 rows 27.8, 13.9, 13.5, 256 rows 39.0, 21.8, 22.3; 48 rows of 262144 32.5, 15.5, 12.7, 256 rows 81, 42, 40.
        uint32_t parts = (uint32_t)(((uint64_t)N + 4095u) / 4096u);
        parts = parts < ARGMAX_PARTS ? parts : ARGMAX_PARTS;
        parts = parts * rows <= at_most ? parts : at_most / rows;
        parts = parts < 1u ? 1u : parts;
        hipLaunchKernelGGL(argmax_rows_kernel, dim3(parts, rows), dim3(256), 0, s, logits + (size_t)m0 * ld, N, ld,
                           out_idx + m0, out_val ? out_val + m0 : nullptr, part_val, part_idx, tickets);
    }
    return hipGetLastError();
}

}  // namespace kq
