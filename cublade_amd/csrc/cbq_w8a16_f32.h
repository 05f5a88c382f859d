// cbq_w8a16_f32.h - the fp32-activation W8A16 linear on the int8 matrix cores
// (cbq_w8a16_f32.hip), called by cbq_w8a16_linear.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cbq {
namespace f32lin {

// Whether the path takes a call (operands 16-byte aligned besides): no outlier
// columns, K % 64 == 0, 32-bit operand offsets, and M > 64 or a weight of at
// least 8 MB (below that the general kernel's single launch is as fast).
bool applies(int64_t M, int64_t N, int64_t K, int64_t n_out);

// Scratch bytes, 256-byte aligned.
int64_t ws_bytes(int64_t M, int64_t N, int64_t K);

int run(const float* x, const int8_t* wq, const float* scales, const float* bias, int64_t M,
        int64_t N, int64_t K, void* scratch, float* y, hipStream_t s, const char* what);

}  // namespace f32lin
}  // namespace cbq
