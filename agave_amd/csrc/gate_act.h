// A gated feed-forward's activations in 32 bits.
#pragma once
#include "common.h"

__device__ __forceinline__ float gelu_tanh(float x) {
    const float c = 0.7978845608028654f;
    return 0.5f * x * (1.0f + tanhf(c * (x + 0.044715f * x * x * x)));
}

// The gate's activation, by number (the feed-forward part knows the names): 0 gelu, tanh form;
// 1 silu, x / (1 + exp(-x)); 2 gelu with the error function; 3 relu.  Another one is another case
// here.  A 32-bit product of a few rows ends in any of them (gemm.hip), the matrix-core products in the tanh form, silu and the clamped
// swish in a form of their own (gemm_mfma.hip).
#define AGAVE_GATE_ACTS 4
#define AGAVE_GATE_SWISH_CLAMPED 6     // a gated form with two numbers of its own, known to gate_form only
__device__ __forceinline__ float gate_act(float x, int act) {
    switch (act) {
        case 0: return gelu_tanh(x);
        case 1: return x / (1.0f + expf(-x));
        case 2: return 0.5f * x * (1.0f + erff(x * 0.7071067811865476f));
        default: return x > 0.f ? x : 0.f;
    }
}
// act(gate) * up
__device__ __forceinline__ float gate_form(float g, float u, int act, float p0, float p1) {
    if (act == AGAVE_GATE_SWISH_CLAMPED) {
        // g' = min(g, p0), u' = clamp(u, -p0, p0);  g' sigmoid(p1 g') (u' + 1)
        const float gc = fminf(g, p0), uc = fminf(fmaxf(u, -p0), p0);
        return gc / (1.0f + expf(-p1 * gc)) * (uc + 1.0f);
    }
    return gate_act(g, act) * u;
}
