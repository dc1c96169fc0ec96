// surface_core.h -- device helpers shared by the torch surface's kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace dressi {

// A lane's way through a box of an image in raster order, `stride` pixels a
// step (the lanes that share the box): an add and a carry in place of a
// division per pixel.
struct BoxWalk {
    uint32_t o;  // the pixel's index in the image
    uint32_t col, bw, step_col, step_o, wrap;
    __device__ __forceinline__ BoxWalk(uint32_t x0, uint32_t y0, uint32_t box_w, uint32_t img_w,
                                       uint32_t lane, uint32_t stride = 64)
        : bw(box_w) {
        const uint32_t row = lane / bw, rows = stride / bw;
        col = lane - row * bw;
        o = (y0 + row) * img_w + x0 + col;
        step_col = stride - rows * bw;
        step_o = rows * img_w + step_col;
        wrap = img_w - bw;
    }
    __device__ __forceinline__ void next() {
        col += step_col;
        o += step_o;
        if (col >= bw) {
            col -= bw;
            o += wrap;
        }
    }
};

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
