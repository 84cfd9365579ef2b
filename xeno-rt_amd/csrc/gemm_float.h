// Float32 products of more than 16 rows of a on the matrix cores (gemm_float.hip).
#pragma once
#include <hip/hip_runtime.h>

// Whether such a product can take them: whole pieces of 16 bytes, and offsets inside a tile that 32 bits hold.
bool xrt_linear_float_accepts(const void* a, const void* w, int M, int K);
int xrt_linear_float(const float* a, const float* w, float* out, int M, int N, int K, int mode, int activation, hipStream_t s);
