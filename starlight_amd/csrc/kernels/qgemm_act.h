// The activation a q-GEMM's split kernel reads, shared by both splits.
#pragma once

#include "common.h"

namespace slhip {

// Four activation elements: a, or with a second input u (SwiGlu's down
// projection) silu(a) * u, the elementwise kernels' formula
// (elementwise.rs:10-12): (a * (1 / (1 + exp(-a)))) * u.
__device__ __forceinline__ float4 act4(const float4* row, const float4* urow, uint32_t i) {
    float4 v = row[i];
    if (urow != nullptr) {
        const float4 u = urow[i];
        v.x = (v.x * (1.0f / (1.0f + expf(-v.x)))) * u.x;
        v.y = (v.y * (1.0f / (1.0f + expf(-v.y)))) * u.y;
        v.z = (v.z * (1.0f / (1.0f + expf(-v.z)))) * u.z;
        v.w = (v.w * (1.0f / (1.0f + expf(-v.w)))) * u.w;
    }
    return v;
}

}  // namespace slhip
