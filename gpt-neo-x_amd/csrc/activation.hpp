// The activations of the MLP, element by element in fp32: tanh-GeLU and the functions of a gate.
#pragma once

#include "common.hpp"

namespace nhp {

// tanh-GeLU of the reference (megatron/model/activations.py:79-97) with x^2 shared and tanh
// eliminated. With u = 0.79788456 x (1 + 0.044715 x^2), e = exp(2u) and s = 1 / (1 + e):
//   tanh(u) = 1 - 2s, so  gelu(x) = 0.5 x (1 + tanh u) = x (1 - s)
//   and, with 1 - tanh^2 = 4 s (1 - s) and the reference's polynomial 0.79788456 + 0.1070322243 x^2,
//   gelu'(x) = 0.5 x (1 - tanh^2)(0.79788456 + 0.1070322243 x^2) + 0.5 (1 + tanh u)
//            = (1 - s) + (1 - s) x s (1.59576912 + 0.2140644486 x^2).
// Two transcendental instructions (exp2, rcp) and 7 / 11 other operations per element instead of
// 17 / 27 for the expressions written out in source order: the backward was bound by the vector
// ALU, not by memory. 1 - s carries the same absolute error (about 2^-24) as the `1 + tanh` of the
// source order; e = inf gives s = 0 and the limits gelu = x, gelu' = 1.
__device__ __forceinline__ float gelu_gate(float x, float x2)
{
    // exp2 argument 2 log2(e) u, the constants folded
    const float w = __builtin_fmaf(2.0f * kLog2e * 0.79788456f * 0.044715f, x2, 2.0f * kLog2e * 0.79788456f);
    const float e = exp2_raw(x * w);
    return __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ float gelu_fwd(float x)
{
    const float s = gelu_gate(x, x * x);
    return x * (1.0f - s);
}

__device__ __forceinline__ float gelu_grad(float x)
{
    const float x2 = x * x;
    const float s = gelu_gate(x, x2);
    const float poly = __builtin_fmaf(2.0f * 0.1070322243f, x2, 2.0f * 0.79788456f);
    // (1 - s) x and s poly are formed first: each factor that reaches 0 does so before it can meet an
    // overflowed partner, so the result is finite wherever x^2 is (the domain of the reference's expression)
    const float q = 1.0f - s;
    return __builtin_fmaf(q * x, s * poly, q);
}

enum GateAct {
    kActSwish = NHP_GATE_SWISH,
    kActGelu = NHP_GATE_GELU,
    kActRelu = NHP_GATE_RELU,
    kActSigmoid = NHP_GATE_SIGMOID,
    kActIdentity = NHP_GATE_IDENTITY
};

__device__ __forceinline__ float sigmoid_fast(float v)
{
    return __builtin_amdgcn_rcpf(1.0f + exp2_raw(-v * kLog2e));
}

// act(g) and d act / d g
template <int ACT>
__device__ __forceinline__ void gate_eval(float g, float& act, float& dact)
{
    if constexpr (ACT == kActSwish) {
        const float s = sigmoid_fast(g);
        act = g * s;
        dact = s * (1.0f + g * (1.0f - s));
    } else if constexpr (ACT == kActGelu) {
        const float cdf = 0.5f * (1.0f + erff(g * 0.70710678118654752f));
        const float pdf = 0.3989422804014327f * exp2_raw((-0.5f * kLog2e) * g * g);
        act = g * cdf;
        dact = cdf + g * pdf;
    } else if constexpr (ACT == kActRelu) {
        act = g > 0.0f ? g : 0.0f;
        dact = g > 0.0f ? 1.0f : 0.0f;
    } else if constexpr (ACT == kActSigmoid) {
        const float s = sigmoid_fast(g);
        act = s;
        dact = s * (1.0f - s);
    } else {
        act = g;
        dact = 1.0f;
    }
}

}  // namespace nhp
