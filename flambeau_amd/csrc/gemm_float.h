// The 32-bit matrix product on the matrix cores (gemm_float.hip): the bits of gemm_plain_kernel, faster.
#pragma once
#include <hip/hip_runtime.h>

// Whether the kernels take the operands: rows in whole 16-byte pieces (K a multiple of 4, aligned pointers), and a K that is
// long enough for them to be the faster ones.
bool gemm_float_takes(const void* x, const void* w, const void* out, int M, int N, int K);
// out[M][N] = x[M][K] w[N][K]^T; the caller checks sizes and, after it, the launch.
void gemm_float_launch(const float* x, const float* w, float* out, int M, int N, int K, hipStream_t stream);
