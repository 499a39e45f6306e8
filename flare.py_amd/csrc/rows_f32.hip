// Row passes around the library's fp32 products of a token-wise MLP in training: activation slope and bias gradient of the backward,
// LayerNorm / RMSNorm each way (pdebench/models/flare.py:45-59, 204-215, lra/models/backends.py:625-672 run these as separate
// torch layers).  fp32 [T,C] rows, contiguous, C in {32, 64, 128, 256}.
//
// Every pass is bound by its bytes: one read of each input, one write of each output.  65,536 rows of 128 channels (33.5 MB an
// array), the torch kernels replaced / these:  gelu's backward, column sum and the residual's gradient sum 51 / 25 us;  the last
// two alone 35 / 12 us;  LayerNorm forward 65 / 13 us, backward (dx, dgamma, dbeta) 104 / 18 us.
//
// A thread owns four consecutive channels, the same for all its rows, so the sums over rows stay in its registers; a
// workgroup leaves one partial row, and the partial rows are added in a fixed order by one small launch.
#include <algorithm>

#include "rows_f32.hpp"

namespace flare {

namespace {

// the workgroup's sums over its rows -> one partial row: thread x % quads owns four channels
template <int N>
__device__ __forceinline__ void column_sums(f32x4 (&acc)[N], int quads, float* part)
{
    __shared__ f32x4 red[256];
    const int tid = threadIdx.x;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        if (k) __syncthreads();
        red[tid] = acc[k];
        __syncthreads();
        if (tid < quads) {
            f32x4 s = red[tid];
            for (int i = tid + quads; i < 256; i += quads) s += red[i];
            *reinterpret_cast<f32x4*>(part + ((size_t)k * quads + tid) * 4) = s;
        }
    }
}

// tanh-GELU as the separate torch layer rounds it, bit for bit (x + 0.044715 x^3 with one rounding, every other operation with its
// own): a chain's outputs do not depend on whether it comes here.  Compared over 2^24 values drawn from N(0, 4) and 2^24 bit patterns.
__device__ __forceinline__ float gelu_tanh(float x)
{
#pragma clang fp contract(off)
    const float inner = 0.79788456080286535588f * fmaf(0.044715f, (x * x) * x, x);
    return (0.5f * x) * (1.f + tanhf(inner));
}

// y = [res +] ([x +] act(t)): one pass instead of one per operation (65,536 rows of 128 channels: activation and sum 27 us as two, 15 us; a
// block's step 2.31 -> 2.12 ms)
template <int ACT>
__global__ __launch_bounds__(256) void rows_act_fwd_kernel(const f32x4* t, const f32x4* x, const f32x4* res, f32x4* y, int64_t n4)
{
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) {
        f32x4 v = t[i];
        const f32x4 a = x ? x[i] : v, r = res ? res[i] : v;
        if (ACT)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(v[e]);
        if (x) v = a + v;
        if (res) v = r + v;
        y[i] = v;
    }
}

// dt = ds act'(t) and the partial column sums of dt; ACT 0: the sums of ds alone, no dt.  copy (or null): receives ds, for the
// product that adds W^T dt to it in place (a copy of its own would read ds once more).
template <int ACT>
__global__ __launch_bounds__(256) void rows_act_bwd_kernel(const f32x4* ds, const f32x4* t, f32x4* dt, f32x4* copy, int64_t n4, int quads, float* part)
{
    f32x4 acc[1] = {{0.f, 0.f, 0.f, 0.f}};
    // 256 is a multiple of quads: a thread meets the same channels in every step
    const int64_t step = (int64_t)gridDim.x * 256;
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    auto one = [&](f32x4 v, f32x4 x, int64_t at) {
        if (copy) copy[at] = v;
        if (ACT != 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] *= act_slope<ACT>(x[r]);
            dt[at] = v;
        }
        acc[0] += v;
    };
    for (; i + step < n4; i += 2 * step) {
        const f32x4 v0 = ds[i], v1 = ds[i + step];
        f32x4 x0 = v0, x1 = v1;
        if (ACT != 0) { x0 = t[i]; x1 = t[i + step]; }
        one(v0, x0, i);
        one(v1, x1, i + step);
    }
    if (i < n4) one(ds[i], ACT != 0 ? t[i] : ds[i], i);
    column_sums<1>(acc, quads, part + (size_t)blockIdx.x * 4 * quads);
}

template <int Q> __device__ __forceinline__ float row_sum(float v)      // over the Q lanes that share a row
{
#pragma unroll
    for (int o = 1; o < Q; o <<= 1) v += __shfl_xor(v, o);
    return v;
}

// Q = C / 4 lanes per row
template <int Q>
__global__ __launch_bounds__(256) void rows_norm_kernel(RowsNormArgs a)
{
    constexpr int R = 256 / Q;
    const int q = threadIdx.x % Q, rl = threadIdx.x / Q;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f}, one = {1.f, 1.f, 1.f, 1.f};
    const f32x4 gm = a.gamma ? reinterpret_cast<const f32x4*>(a.gamma)[q] : one;
    const f32x4 bt = a.beta ? reinterpret_cast<const f32x4*>(a.beta)[q] : zero;
    for (int64_t r0 = (int64_t)blockIdx.x * R; r0 < a.T; r0 += (int64_t)gridDim.x * R) {
        const int64_t row = r0 + rl < a.T ? r0 + rl : a.T - 1;
        const f32x4 x = reinterpret_cast<const f32x4*>(a.x)[row * Q + q];
        const float mean = a.norm == 1 ? row_sum<Q>(x[0] + x[1] + x[2] + x[3]) * (1.f / (4 * Q)) : 0.f;
        const f32x4 d = x - mean;
        const float rstd = 1.f / sqrtf(row_sum<Q>(d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + d[3] * d[3]) * (1.f / (4 * Q)) + a.eps);
        if (r0 + rl < a.T) {
            reinterpret_cast<f32x4*>(a.y)[row * Q + q] = d * rstd * gm + bt;
            if (q == 0) *reinterpret_cast<float2*>(a.stats + 2 * row) = make_float2(mean, rstd);
        }
    }
}

// dx = [add +] rstd (g - mean(g) - xhat mean(g xhat)), g = dy gamma (no mean(g) for RMSNorm); partial sums of dy xhat and dy
template <int Q>
__global__ __launch_bounds__(256) void rows_norm_bwd_kernel(RowsNormArgs a)
{
    constexpr int R = 256 / Q;
    const int q = threadIdx.x % Q, rl = threadIdx.x / Q;
    const f32x4 one = {1.f, 1.f, 1.f, 1.f};
    const f32x4 gm = a.gamma ? reinterpret_cast<const f32x4*>(a.gamma)[q] : one;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    for (int64_t r0 = (int64_t)blockIdx.x * R; r0 < a.T; r0 += (int64_t)gridDim.x * R) {
        const bool live = r0 + rl < a.T;
        const int64_t row = live ? r0 + rl : a.T - 1;
        const f32x4 x = reinterpret_cast<const f32x4*>(a.x)[row * Q + q];
        const f32x4 dy = reinterpret_cast<const f32x4*>(a.dy)[row * Q + q];
        const float2 st = *reinterpret_cast<const float2*>(a.stats + 2 * row);
        const f32x4 xh = (x - st.x) * st.y, g = dy * gm, gx = g * xh;
        const float m1 = a.norm == 1 ? row_sum<Q>(g[0] + g[1] + g[2] + g[3]) * (1.f / (4 * Q)) : 0.f;
        const float m2 = row_sum<Q>(gx[0] + gx[1] + gx[2] + gx[3]) * (1.f / (4 * Q));
        if (live) {
            f32x4 dx = st.y * (g - m1 - xh * m2);
            if (a.add) dx += reinterpret_cast<const f32x4*>(a.add)[row * Q + q];
            reinterpret_cast<f32x4*>(a.y)[row * Q + q] = dx;
            acc[0] += dy * xh;
            acc[1] += dy;
        }
    }
    column_sums<2>(acc, Q, a.gb_part + (size_t)blockIdx.x * 8 * Q);
}

template <typename F> hipError_t with_quads(int C, F&& f)
{
    switch (C) {
        case 32:  f(std::integral_constant<int, 8>{}); break;
        case 64:  f(std::integral_constant<int, 16>{}); break;
        case 128: f(std::integral_constant<int, 32>{}); break;
        case 256: f(std::integral_constant<int, 64>{}); break;
        default:  return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

bool rows_f32_supported(int C) { return C == 32 || C == 64 || C == 128 || C == 256; }

// workgroups of the passes that leave partial rows: four per compute unit, at least eight steps of a thread each
int rows_f32_parts(int64_t T, int C)
{
    const int64_t steps = (T * (C / 4) + 256 * 8 - 1) / (256 * 8);
    return (int)std::max<int64_t>(1, std::min<int64_t>(steps, 4 * (int64_t)device_cus()));
}

hipError_t launch_rows_act_bwd(int act, const float* ds, const float* t, float* dt, float* copy, float* part, float* db, int64_t T, int C, hipStream_t st)
{
    const int parts = rows_f32_parts(T, C);
    hipError_t e = with_row_act(act, [&](auto ac) {
        hipLaunchKernelGGL(rows_act_bwd_kernel<decltype(ac)::value>, dim3((unsigned)parts), dim3(256), 0, st, (const f32x4*)ds,
                           (const f32x4*)t, (f32x4*)dt, (f32x4*)copy, T * C / 4, C / 4, part);
    });
    return e != hipSuccess || !db ? e : launch_sum_parts(part, db, C, parts, st);
}

hipError_t launch_rows_act_fwd(int act, const float* t, const float* x, const float* res, float* y, int64_t n, hipStream_t st)
{
    const unsigned grid = (unsigned)std::min<int64_t>((n / 4 + 255) / 256, 32 * (int64_t)device_cus());
    const auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, st, (const f32x4*)t, (const f32x4*)x, (const f32x4*)res, (f32x4*)y, n / 4);
    };
    if (act < 0) go(rows_act_fwd_kernel<0>);
    else go(rows_act_fwd_kernel<1>);
    return hipGetLastError();
}

hipError_t launch_rows_norm(const RowsNormArgs& a, hipStream_t st)
{
    const unsigned grid = (unsigned)std::min<int64_t>((a.T * (a.C / 4) + 255) / 256, 16 * (int64_t)device_cus());
    return with_quads(a.C, [&](auto qc) { hipLaunchKernelGGL(rows_norm_kernel<decltype(qc)::value>, dim3(grid), dim3(256), 0, st, a); });
}

hipError_t launch_rows_norm_bwd(const RowsNormArgs& a, hipStream_t st)
{
    const int parts = rows_f32_parts(a.T, a.C);
    hipError_t e = with_quads(a.C, [&](auto qc) {
        hipLaunchKernelGGL(rows_norm_bwd_kernel<decltype(qc)::value>, dim3((unsigned)parts), dim3(256), 0, st, a);
    });
    return e != hipSuccess || !a.gb ? e : launch_sum_parts(a.gb_part, a.gb, 2 * a.C, parts, st);
}

}  // namespace flare
