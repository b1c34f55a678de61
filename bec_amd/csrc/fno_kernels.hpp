// Fused kernels of the surrogate network (fno_kernels.hip), used by fno.hip for
// the shapes they cover; other shapes run the general strided GEMM (gemm.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace bec {

// ranges of rows a weight gradient is split into (the GEMM's split, so that both
// give the same bits)
constexpr int WGRAD_SPLITS = 256;

// [dW (K x N); db (N)] = [X^T; 1^T] D over rows, for K, N <= 64 and rows a
// multiple of 32; out holds K N + N floats, part WGRAD_SPLITS times as many.
bool wgrad_covers(int K, int N, long rows);
hipError_t run_wgrad(const float *X, int K, const float *D, int N, long rows, float *part, float *out, hipStream_t s);

} // namespace bec
