// What the two GEMM kernels over GGUF weights share (qgemm.hip, qgemm_big.hip):
// the formats and what their weights are.
//
//   Every block format is  w = s_g * q + o_g  over groups g of 16 or 32
//   consecutive weights, q a small integer:
//     Q4_K  q in [0, 15],     s = d * sc_g, o = -dmin * m_g  (groups of 32)
//     Q6_K  q in [-32, 31],   s = d * sc_g, o = 0            (groups of 16)
//     Q8_0  q in [-128, 127], s = d,        o = 0            (groups of 32)
//   x goes into the MFMAs as f16 x_hi + x_lo.
#pragma once

#include "common.hpp"

namespace lmx {

enum GType { kGF16 = 1, kGQ8_0 = 8, kGQ4K = 12, kGQ6K = 14, kGBF16 = 30 };

// Sum over each aligned group of 8 lanes; every lane of the group gets it.
__device__ __forceinline__ float sum8(float x) {
    x += dpp<0xB1>(x);   // quad_perm [1,0,3,2]
    x += dpp<0x4E>(x);   // quad_perm [2,3,0,1]
    return x + dpp<0x141>(x);  // row_half_mirror: lane i with 7 - i of its 8
}

}  // namespace lmx
