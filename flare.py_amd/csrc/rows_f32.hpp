// Shared pieces of the fp32 row kernels (rows_f32.hip, rows_layer_f32_mfma.hip).
#pragma once

#include <type_traits>

#include "common.hpp"

namespace flare {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// GELU's gate 0.5 (1 + tanh u) is 1 / (1 + exp(-2 u)), 2 u = 1.5957691 x (1 + 0.044715 x^2): no cancellation for negative x.
// gate = 1 / (1 + e), 1 - gate = e / (1 + e), e kept finite.
template <int ACT> __device__ __forceinline__ float act_slope(float x)
{
    const float a = ACT == 1 ? 1.5957691216057308f * x * fmaf(0.044715f * x, x, 1.f) : x;
    const float da = ACT == 1 ? 1.5957691216057308f * fmaf(3.f * 0.044715f * x, x, 1.f) : 1.f;
    const float e = fminf(expf(-a), 3.0e38f), r = 1.f / (1.f + e);
    return r * fmaf(x * (e * r), da, 1.f);
}

// act: -1 none, else FLARE_ACT_*
template <typename F> hipError_t with_row_act(int act, F&& f)
{
    switch (act) {
        case -1: f(std::integral_constant<int, 0>{}); break;
        case 0:  f(std::integral_constant<int, 1>{}); break;
        case 1:  f(std::integral_constant<int, 2>{}); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

}  // namespace flare
