// The narrow ends of a model in training under autocast (the lift in_dim -> C with its activation and the last layer C -> out_dim of
// pdebench/models/flare.py:285-310, both dims at most 4): forward and backward each one pass over the rows.  16-bit compute type,
// C in {32, 64, 128}; operands and results are rounded to it where the separate torch layers round them (input, weights, bias, product
// with bias, activation, and in the backward the gradients of those), sums are kept in fp32.
//
// As torch layers the two ends were twenty launches of a step, among them a weight gradient [C, in_dim] that the library runs as one
// long product with nothing to parallelise (50 us at 4096 points).  Everything here is bound by latency, not by its rows: at 4096 points and 128
// channels, as nodes of a replayed step (3 us of each are the node's), the first layer takes 8.8 us forward and 19.5 us backward, the last one 4.0
// and 11.5 us; the backward is 64 workgroups of 64 tokens there, which walk them in turns, one trip to memory behind the other.
// The replayed step of 8 blocks at 4096 points: 128 channels 1608 -> 1518 us, 64 channels 1273 -> 1171 us; 4 blocks of 128 channels at
// 12,000 points 1600 -> 1459 us.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace flare {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T> __device__ __forceinline__ float rnd(float v) { return to_f32(from_f32<T>(v)); }
template <typename T> __device__ __forceinline__ f32x4 load_quad(const T* p)
{
    const uint2 r = *reinterpret_cast<const uint2*>(p);
    const T* e = reinterpret_cast<const T*>(&r);
    return f32x4{to_f32(e[0]), to_f32(e[1]), to_f32(e[2]), to_f32(e[3])};
}
template <typename T> __device__ __forceinline__ void store_quad(T* p, f32x4 v)
{
    const T e[4] = {from_f32<T>(v[0]), from_f32<T>(v[1]), from_f32<T>(v[2]), from_f32<T>(v[3])};
    *reinterpret_cast<uint2*>(p) = *reinterpret_cast<const uint2*>(e);
}
// element of rows in fp32, bf16 or f16
__device__ __forceinline__ float load_any(const void* p, int dt, int64_t i)
{
    return dt == 0 ? static_cast<const float*>(p)[i] : dt == 1 ? to_f32(static_cast<const bf16_t*>(p)[i]) : to_f32(static_cast<const f16_t*>(p)[i]);
}

// value and slope of tanh-GELU (kind 0) / SiLU (kind 1): both are x gate(a), gate = 1 / (1 + exp(-a))
__device__ __forceinline__ void act_fwd_slope(int kind, float x, float& value, float& slope)
{
    const float a = kind == 0 ? 1.5957691216057308f * x * fmaf(0.044715f * x, x, 1.f) : x;
    const float da = kind == 0 ? 1.5957691216057308f * fmaf(3.f * 0.044715f * x, x, 1.f) : 1.f;
    const float e = fminf(expf(-a), 3.0e38f), r = 1.f / (1.f + e);
    value = x * r;
    slope = r * fmaf(x * (e * r), da, 1.f);
}

// Every kernel: a thread owns four channels (quad q of C / 4), the S = 1024 / C threads of a quad share a workgroup's tokens.

// t = x W^T + b and, with an activation, y = act(t); act < 0: y alone
template <typename T>
__global__ __launch_bounds__(256) void narrow_in_kernel(NarrowArgs a)
{
    const int Q = a.C / 4, S = 256 / Q, q = threadIdx.x % Q, s = threadIdx.x / Q, K = a.K;
    float w[4][4], b[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        b[r] = a.b ? rnd<T>(a.b[4 * q + r]) : 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[r][j] = j < K ? rnd<T>(a.w[(4 * q + r) * K + j]) : 0.f;
    }
    for (int64_t t = (int64_t)blockIdx.x * S + s; t < a.T; t += (int64_t)gridDim.x * S) {
        f32x4 v = {b[0], b[1], b[2], b[3]};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float x = j < K ? rnd<T>(load_any(a.x, a.x_dtype, t * a.xs + j)) : 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = fmaf(x, w[r][j], v[r]);
        }
        T* y = static_cast<T*>(a.y) + t * a.C + 4 * q;
        if (a.act >= 0) {
            store_quad<T>(static_cast<T*>(a.t) + t * a.C + 4 * q, v);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float u, sl;
                act_fwd_slope(a.act, rnd<T>(v[r]), u, sl);
                v[r] = u;
            }
        }
        store_quad<T>(y, v);
    }
}

// sums over the S threads of a quad, in slot order; slot 0 gets them
template <int N> __device__ __forceinline__ void slot_sums(f32x4 (&v)[N], int Q)
{
    __shared__ f32x4 red[256];
    const int tid = threadIdx.x;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        if (k) __syncthreads();
        red[tid] = v[k];
        __syncthreads();
        if (tid < Q)
            for (int i = tid + Q; i < 256; i += Q) v[k] += red[i];
    }
}

// dt = dy act'(t); partial dW [C][K] and db [C] over the workgroup's tokens
template <typename T>
__global__ __launch_bounds__(256) void narrow_in_bwd_kernel(NarrowArgs a)
{
    const int Q = a.C / 4, S = 256 / Q, q = threadIdx.x % Q, s = threadIdx.x / Q, K = a.K;
    f32x4 acc[5] = {};                                              // K columns of dW for the four channels, then db
    const int64_t t0 = (int64_t)blockIdx.x * a.tokens_per_wg, t1 = t0 + a.tokens_per_wg < a.T ? t0 + a.tokens_per_wg : a.T;
    for (int64_t t = t0 + s; t < t1; t += S) {
        f32x4 g = load_quad<T>(static_cast<const T*>(a.dy) + t * a.C + 4 * q);
        if (a.act >= 0) {
            const f32x4 v = load_quad<T>(static_cast<const T*>(a.t) + t * a.C + 4 * q);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float u, sl;
                act_fwd_slope(a.act, v[r], u, sl);
                g[r] = rnd<T>(g[r] * sl);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < K) acc[j] += g * rnd<T>(load_any(a.x, a.x_dtype, t * a.xs + j));
        acc[4] += g;
    }
    slot_sums<5>(acc, Q);
    if (s == 0) {
        float* dw = a.dw_part + ((size_t)blockIdx.x * a.C + 4 * q) * K;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j < K) dw[r * K + j] = acc[j][r];
        *reinterpret_cast<f32x4*>(a.db_part + (size_t)blockIdx.x * a.C + 4 * q) = acc[4];
    }
}

// y = x W^T + b, K output columns: the C / 4 threads of a token meet by lane swaps
template <typename T>
__global__ __launch_bounds__(256) void narrow_out_kernel(NarrowArgs a)
{
    const int Q = a.C / 4, S = 256 / Q, q = threadIdx.x % Q, s = threadIdx.x / Q, K = a.K;
    f32x4 w[4] = {};
    for (int o = 0; o < 4; ++o)
        if (o < K)
#pragma unroll
            for (int r = 0; r < 4; ++r) w[o][r] = rnd<T>(a.w[o * a.C + 4 * q + r]);
    const int64_t step = (int64_t)gridDim.x * S;
    for (int64_t t0 = (int64_t)blockIdx.x * S; t0 < a.T; t0 += step) {
        const int64_t t = t0 + s < a.T ? t0 + s : a.T - 1;
        const f32x4 x = load_quad<T>(static_cast<const T*>(a.x) + t * a.C + 4 * q);
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            if (o >= K) break;
            float v = x[0] * w[o][0] + x[1] * w[o][1] + x[2] * w[o][2] + x[3] * w[o][3];
            for (int m = 1; m < Q; m <<= 1) v += __shfl_xor(v, m);
            if (q == 0 && t0 + s < a.T) {
                v = rnd<T>(v + (a.b ? rnd<T>(a.b[o]) : 0.f));
                const int64_t i = t * K + o;
                if (a.y_dtype == 0) static_cast<float*>(a.y)[i] = v;
                else if (a.y_dtype == 1) static_cast<bf16_t*>(a.y)[i] = from_f32<bf16_t>(v);
                else static_cast<f16_t*>(a.y)[i] = from_f32<f16_t>(v);
            }
        }
    }
}

// dx = dy W; partial dW [K][C] and db [4] over the workgroup's tokens
template <typename T>
__global__ __launch_bounds__(256) void narrow_out_bwd_kernel(NarrowArgs a)
{
    const int Q = a.C / 4, S = 256 / Q, q = threadIdx.x % Q, s = threadIdx.x / Q, K = a.K;
    f32x4 w[4] = {}, acc[5] = {};
    for (int o = 0; o < 4; ++o)
        if (o < K)
#pragma unroll
            for (int r = 0; r < 4; ++r) w[o][r] = rnd<T>(a.w[o * a.C + 4 * q + r]);
    const int64_t t0 = (int64_t)blockIdx.x * a.tokens_per_wg, t1 = t0 + a.tokens_per_wg < a.T ? t0 + a.tokens_per_wg : a.T;
    for (int64_t t = t0 + s; t < t1; t += S) {
        const f32x4 x = load_quad<T>(static_cast<const T*>(a.x) + t * a.C + 4 * q);
        f32x4 dx = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            const float g = o < K ? rnd<T>(load_any(a.dy, a.y_dtype, t * K + o)) : 0.f;
            dx += g * w[o];
            if (o < K) acc[o] += g * x;
            acc[4][o] += g;
        }
        if (a.dx) store_quad<T>(static_cast<T*>(a.dx) + t * a.C + 4 * q, dx);
    }
    slot_sums<5>(acc, Q);
    if (s == 0) {
#pragma unroll
        for (int o = 0; o < 4; ++o)
            if (o < K) *reinterpret_cast<f32x4*>(a.dw_part + ((size_t)blockIdx.x * K + o) * a.C + 4 * q) = acc[o];
        if (q == 0) *reinterpret_cast<f32x4*>(a.db_part + (size_t)blockIdx.x * 4) = acc[4];
    }
}

}  // namespace

// workgroups of the backward passes: 64 tokens each until they fill the device four times
static int64_t tokens_per_wg(int64_t T) { return std::max<int64_t>(64, ((T + 4 * (int64_t)device_cus() - 1) / (4 * (int64_t)device_cus()) + 63) / 64 * 64); }
int mlp_narrow_parts(int64_t T) { return (int)((T + tokens_per_wg(T) - 1) / tokens_per_wg(T)); }

hipError_t launch_mlp_narrow(const NarrowArgs& a0, bool out, bool bwd, int dtype, float* dw, float* db, hipStream_t st)
{
    NarrowArgs a = a0;
    a.tokens_per_wg = tokens_per_wg(a.T);
    const int S = 1024 / a.C;
    const unsigned grid = bwd ? (unsigned)mlp_narrow_parts(a.T) : (unsigned)std::min<int64_t>((a.T + S - 1) / S, 16 * (int64_t)device_cus());
    const auto go = [&](auto t) {
        using T = decltype(t);
        auto kern = out ? (bwd ? narrow_out_bwd_kernel<T> : narrow_out_kernel<T>) : (bwd ? narrow_in_bwd_kernel<T> : narrow_in_kernel<T>);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, st, a);
        return hipGetLastError();
    };
    const hipError_t e = dtype == 1 ? go(bf16_t{}) : go(f16_t{});
    if (e != hipSuccess || !bwd) return e;
    return launch_sum_two_parts(a.dw_part, dw, (int64_t)a.C * a.K, a.db_part, db, out ? 4 : a.C, (int)grid, st);
}

}  // namespace flare
