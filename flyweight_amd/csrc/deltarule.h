// What the kernels of the gated delta rule share.
#pragma once
#include "fw_common.h"

__device__ __forceinline__ float fw_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float fw_softplus(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

// A sum over the 16 lanes of a row of the wave (every lane gets it): neighbours, pairs, then the two
// mirrors, all inside the vector unit (no trip through the LDS crossbar). After each step the lanes
// that have met hold one value, so the mirrors may stand for the exchanges between quads and halves.
template <int CTRL>
__device__ __forceinline__ float delta_dpp(float x) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float delta_row_sum(float x) {
    x += delta_dpp<0xB1>(x);        // quad_perm [1, 0, 3, 2]
    x += delta_dpp<0x4E>(x);        // quad_perm [2, 3, 0, 1]
    x += delta_dpp<0x141>(x);       // row_half_mirror
    x += delta_dpp<0x140>(x);       // row_mirror
    return x;
}

// The short convolutions' memory moves on by a step's segments (several rows long).
// proj [rows][proj_stride] float32 or bfloat16 by `dtype`.
void fw_launch_conv_state(const void* proj, int dtype, int proj_stride, float* conv_state, const int32_t* seg_row0, const int32_t* seg_slot,
                          int channels, int taps_count, int segments, hipStream_t stream);
