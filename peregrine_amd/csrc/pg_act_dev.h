// The experts' activations in f32, for every kernel that multiplies act(gate) by up.
#pragma once
#include <hip/hip_runtime.h>
#include "pg_internal.h"

__device__ __forceinline__ float act_silu(float x) {
    const float sig = 1.0f / (1.0f + expf(-x));
    return x * sig;
}
__device__ __forceinline__ float act_gelu_tanh(float x) {
    const float c = sqrtf(2.0f / 3.14159265358979323846f);
    const float inner = c * (x + 0.044715f * x * x * x);
    return 0.5f * x * (1.0f + tanhf(inner));
}
__device__ __forceinline__ float pg_act(int act, float x) { return act == PG_ACT_GELU_TANH ? act_gelu_tanh(x) : act_silu(x); }
