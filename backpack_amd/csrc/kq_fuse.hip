// kq_fuse.hip — the stand-alone forms of what the lanes-along-K decode kernels fold into their activation
// prologue and their stores: RMSNorm of a row, act(gate) * up, and the residual add.  They serve the
// shapes those kernels decline (more than two tokens, rows longer than their registers hold), so that
// the fused entry point computes the same function for every shape.
//
// Reference forms: norm/rms_norm.wgsl:15-20 and quant_kq/q4k_matmul_norm.wgsl:50-91 (y = x * rstd * w,
// rstd = 1/sqrt(mean(x^2) + eps)); fused/silu_mul_fused.wgsl:39-49; fused/gelu_mul_fused.wgsl:22-32; the
// add_inplace dispatch after down (runtime/model_runner.cpp:3775-3793).
#include <hip/hip_runtime.h>

#include "kq_kernels.h"
#include "kq_wave.h"

namespace kq {

// An output element as fp32, or as bf16 (round to nearest even: the activation rows of the prefill GEMM).
__device__ __forceinline__ void put_out(float* out, size_t at, float v) { out[at] = v; }
__device__ __forceinline__ void put_out(uint16_t* out, size_t at, float v)
{
    out[at] = __builtin_bit_cast(uint16_t, (__bf16)v);
}

// One workgroup of 256 lanes per row.
template <typename OUT>
__global__ __launch_bounds__(256) void rms_norm_rows_kernel(const float* X, const float* w, float eps, uint32_t K,
                                                            OUT* out)
{
    __shared__ float part[4];
    const float* x = X + (size_t)blockIdx.x * K;
    float ss = 0.0f;
    for (uint32_t k = threadIdx.x; k < K; k += 256u) ss = __builtin_fmaf(x[k], x[k], ss);
    ss = wave_total(ss);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float rstd = 1.0f / sqrtf(((part[0] + part[1]) + (part[2] + part[3])) / (float)K + eps);
    const size_t o = (size_t)blockIdx.x * K;
    for (uint32_t k = threadIdx.x; k < K; k += 256u) put_out(out, o + k, x[k] * rstd * w[k]);
}

// Rows in pieces of four (K a multiple of four, pointers on 16 bytes: what every k-quant row has; the scalar forms above and
// below serve the rest).  One pass over memory: a lane's pieces of X and w stay in registers across the row's sum.
__device__ __forceinline__ void put_four(float* out, size_t at, float4 v) { *(float4*)(out + at) = v; }
__device__ __forceinline__ void put_four(uint16_t* out, size_t at, float4 v)
{
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    *(bf16x4*)(out + at) = bf16x4{(__bf16)v.x, (__bf16)v.y, (__bf16)v.z, (__bf16)v.w};
}

// 1280 to 8192 elements, 512 lanes (fewer than 2^23 rows: a grid holds fewer than 2^32 threads).  2048 rows of 4096 17 -> 10 us, 100
// rows 10 -> 6 (bf16 out; one dependent pass less, and 16 bytes a load).  Shorter rows leave most lanes idle and stay on the scalar
// form: 8008 rows of 256 9.9 us here, 5.6 there, 2048 rows of 1024 4.2 and 4.0, of 1280 4.3 and 4.5.
template <typename OUT>
__global__ __launch_bounds__(512) void rms_norm_rows4_kernel(const float* X, const float* w, float eps, uint32_t K, OUT* out)
{
    __shared__ float part[8];
    const uint32_t k4 = K / 4u;
    const float4* x = (const float4*)(X + (size_t)blockIdx.x * K);
    float4 v[4], g[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
        const uint32_t k = threadIdx.x + 512u * i;
        v[i] = k < k4 ? x[k] : float4{0, 0, 0, 0};
        g[i] = k < k4 ? ((const float4*)w)[k] : float4{0, 0, 0, 0};
    }
    float ss = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
        ss = fmaf(v[i].x, v[i].x, ss); ss = fmaf(v[i].y, v[i].y, ss); ss = fmaf(v[i].z, v[i].z, ss); ss = fmaf(v[i].w, v[i].w, ss);
    }
    ss = wave_total(ss);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
    const float rstd = 1.0f / sqrtf(ss / (float)K + eps);
    const size_t o = (size_t)blockIdx.x * K;
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
        const uint32_t k = threadIdx.x + 512u * i;
        if (k < k4) put_four(out, o + 4u * k, float4{v[i].x * rstd * g[i].x, v[i].y * rstd * g[i].y, v[i].z * rstd * g[i].z, v[i].w * rstd * g[i].w});
    }
}

// out[m, k] = X[m, k] converted (blockIdx.y = row)
__global__ __launch_bounds__(256) void cast_rows_bf16_kernel(const float* X, uint32_t K, uint16_t* out)
{
    const uint32_t k = blockIdx.x * 256u + threadIdx.x;
    if (k >= K) return;
    const size_t at = (size_t)blockIdx.y * K + k;
    put_out(out, at, X[at]);
}

__global__ __launch_bounds__(256) void cast_rows4_bf16_kernel(const float* X, uint32_t n4, uint16_t* out)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n4) put_four(out, 4u * (size_t)i, ((const float4*)X)[i]);
}

template <bool GELU>
__device__ __forceinline__ float act_of(float gv)
{
    if (GELU) {
        const float inner = 0.7978845608f * (gv + 0.044715f * gv * gv * gv);
        return 0.5f * gv * (1.0f + tanhf(inner));
    }
    return gv / (expf(-gv) + 1.0f);
}

// GU rows are gate | up (2K floats); out rows are K floats.  P pieces of four per lane, all their loads in flight: with two, 2048 rows
// of 14336 (294 MB) 75 -> 55 us.
template <int P, bool GELU, typename OUT>
__global__ __launch_bounds__(256) void act_mul_rows4_kernel(const float* GU, uint32_t K, OUT* out)
{
    const float* row = GU + (size_t)blockIdx.y * 2u * K;
    float4 g[P], u[P];
    uint32_t k[P];
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)P; ++i) {
        k[i] = 4u * (blockIdx.x * (256u * P) + i * 256u + threadIdx.x);
        if (k[i] >= K) continue;
        g[i] = *(const float4*)(row + k[i]);
        u[i] = *(const float4*)(row + K + k[i]);
    }
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)P; ++i)
        if (k[i] < K)
            put_four(out, (size_t)blockIdx.y * K + k[i], float4{act_of<GELU>(g[i].x) * u[i].x, act_of<GELU>(g[i].y) * u[i].y,
                                                               act_of<GELU>(g[i].z) * u[i].z, act_of<GELU>(g[i].w) * u[i].w});
}

// GU rows are gate | up (2K floats); out rows are K floats.
template <bool GELU, typename OUT>
__global__ __launch_bounds__(256) void act_mul_rows_kernel(const float* GU, uint32_t K, OUT* out)
{
    const float* g = GU + (size_t)blockIdx.y * 2u * K;
    const uint32_t k = blockIdx.x * 256u + threadIdx.x;
    if (k >= K) return;
    const float gv = g[k], uv = g[K + k];   // (both requested ahead of tanhf's branches)
    put_out(out, (size_t)blockIdx.y * K + k, act_of<GELU>(gv) * uv);
}

// Y[m, y_offset + n] = T[m, n] + R[m, y_offset + n]   (R may be Y)
__global__ __launch_bounds__(256) void add_residual_kernel(const float* T, const float* R, float* Y, uint32_t N,
                                                           uint32_t ldy, uint32_t y_offset)
{
    const uint32_t n = blockIdx.x * 256u + threadIdx.x;
    if (n >= N) return;
    const size_t at = (size_t)blockIdx.y * ldy + y_offset + n;
    Y[at] = T[(size_t)blockIdx.y * N + n] + R[at];
}

template <typename OUT>
static hipError_t launch_prologue_rows_as(int pro, const float* X, const float* norm_w, float eps, uint32_t M, uint32_t K,
                                          OUT* out, hipStream_t s)
{
    const bool fours = K >= 4u && K % 4u == 0 && !(((uintptr_t)X | (uintptr_t)out | (pro == 1 ? (uintptr_t)norm_w : 0u)) & 15u);
    if (fours && pro != 1) {
        // Two pieces per lane from 2^22 outputs on, unless workgroups of 2048 outputs would leave more than a quarter of theirs beyond
        // the row; other calls need the workgroups more than the loads in flight.  us, scalar / two pieces / one: GELU 521 x 2560 3.4 /
        // 4.3 / 3.3, 1292 x 2560 6.5 / 8.0 / 5.0, SILU 2048 x 2560 10.0 / 10.4 / 8.7; with two SILU 2048 x 14336 66 / 43.
        const bool fits = (uint64_t)(K + 2047u) / 2048u * 2048u * 4u <= 5ull * K;
        const uint32_t P = fits && (uint64_t)M * K >= (1u << 22) ? 2u : 1u;
        const dim3 grid((K / 4u + 256u * P - 1u) / (256u * P), M);
        if (pro == 2 && P == 2u) hipLaunchKernelGGL((act_mul_rows4_kernel<2, false, OUT>), grid, dim3(256), 0, s, X, K, out);
        else if (pro == 2) hipLaunchKernelGGL((act_mul_rows4_kernel<1, false, OUT>), grid, dim3(256), 0, s, X, K, out);
        else if (P == 2u) hipLaunchKernelGGL((act_mul_rows4_kernel<2, true, OUT>), grid, dim3(256), 0, s, X, K, out);
        else hipLaunchKernelGGL((act_mul_rows4_kernel<1, true, OUT>), grid, dim3(256), 0, s, X, K, out);
    } else if (fours && K >= 1280u && K <= 8192u && M < (1u << 23)) hipLaunchKernelGGL(rms_norm_rows4_kernel<OUT>, dim3(M), dim3(512), 0, s, X, norm_w, eps, K, out);
    else if (pro == 1) hipLaunchKernelGGL(rms_norm_rows_kernel<OUT>, dim3(M), dim3(256), 0, s, X, norm_w, eps, K, out);
    else if (pro == 2) hipLaunchKernelGGL((act_mul_rows_kernel<false, OUT>), dim3((K + 255u) / 256u, M), dim3(256), 0, s, X, K, out);
    else hipLaunchKernelGGL((act_mul_rows_kernel<true, OUT>), dim3((K + 255u) / 256u, M), dim3(256), 0, s, X, K, out);
    return hipGetLastError();
}

hipError_t launch_prologue_rows(int pro, const float* X, const float* norm_w, float eps, uint32_t M, uint32_t K,
                                float* out, hipStream_t s)
{
    return launch_prologue_rows_as(pro, X, norm_w, eps, M, K, out, s);
}

// pro 0: the rows as they are
hipError_t launch_prologue_rows_bf16(int pro, const float* X, const float* norm_w, float eps, uint32_t M, uint32_t K,
                                     uint16_t* out, hipStream_t s)
{
    if (pro != 0) return launch_prologue_rows_as(pro, X, norm_w, eps, M, K, out, s);
    const uint64_t n = (uint64_t)M * K;
    if (n % 4u == 0 && n / 4u < 0xFFFFFF00ull && !(((uintptr_t)X | (uintptr_t)out) & 15u)) {
        hipLaunchKernelGGL(cast_rows4_bf16_kernel, dim3((uint32_t)((n / 4u + 255u) / 256u)), dim3(256), 0, s, X, (uint32_t)(n / 4u), out);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(cast_rows_bf16_kernel, dim3((K + 255u) / 256u, M), dim3(256), 0, s, X, K, out);
    return hipGetLastError();
}

hipError_t launch_add_residual(const float* T, const float* R, float* Y, uint32_t M, uint32_t N, uint32_t ldy,
                               uint32_t y_offset, hipStream_t s)
{
    hipLaunchKernelGGL(add_residual_kernel, dim3((N + 255u) / 256u, M), dim3(256), 0, s, T, R, Y, N, ldy, y_offset);
    return hipGetLastError();
}

}  // namespace kq
