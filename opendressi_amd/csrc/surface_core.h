// surface_core.h -- device helpers shared by the torch surface's kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace dressi {

// Orders a one-wave workgroup's LDS accesses.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The sum of gradient contributions as the reference's backward builder
// forms it (src/core/build_backward.cpp:36-57): groups of at most four, each
// summed left to right, level by level. Contributions come one at a time; a
// level holds the sum of its unfinished group.
struct ContribSum {
    static constexpr int kLevels = 10;  // 4^9 contributions
    float acc[kLevels];
    uint32_t count[kLevels];
    __device__ ContribSum() {
#pragma unroll
        for (int l = 0; l < kLevels; l++) {
            acc[l] = 0.f;
            count[l] = 0;
        }
    }
    __device__ __forceinline__ void push(float x) {
        bool go = true;
#pragma unroll
        for (int l = 0; l < kLevels; l++) {
            if (go) {
                acc[l] = count[l] ? acc[l] + x : x;
                count[l]++;
                go = count[l] == 4;
                if (go) {
                    x = acc[l];
                    count[l] = 0;
                }
            }
        }
    }
    __device__ __forceinline__ float sum() const {
        float carry = 0.f;
        bool have = false;
#pragma unroll
        for (int l = 0; l < kLevels; l++) {
            if (count[l]) {
                carry = have ? acc[l] + carry : acc[l];
                have = true;
            }
        }
        return carry;
    }
};

}  // namespace dressi
