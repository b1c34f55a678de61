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

// Offset of entry (m, k) of an M x K BF16 matrix stored as MFMA operands:
// [M / 16][K / 32][lane][8], lane (m % 16) + 16 ((k % 32) / 8)
constexpr long operand_at(long m, long k, long K)
{
    return ((m / 16 * (K / 32) + k / 32) * 64 + m % 16 + 16 * (k % 32 / 8)) * 8 + k % 8;
}

// out[p] = A in[p] for `planes` planes: A M x K in BF16 (operand_at), in[p] K x W, out[p] M x W; per > 0: K in chunks of `per` 32-value tiles, added in
// order.  W a power of two up to 64, M a multiple of 16, K of 32 up to 1024.
bool plane_dft_covers(int M, int K, int W);
hipError_t run_plane_dft(const unsigned short *A, const float *in, float *out, int M, int K, int W, int planes, int per,
                         hipStream_t s);

// out[b] = A in[b]: A M x K operands (operand_at, M rounded up to 16 with zeros),
// in[b] K x N, out[b] M x N; per as above.  M <= 64, K % 32 == 0, N % 64 == 0.
bool z_dft_covers(int M, int K, long N);
hipError_t run_z_dft(const unsigned short *A, const float *in, float *out, int M, int K, int N, int batch, int per,
                     hipStream_t s);

// What leaves a spectral layer, forward (back = 0): r = h W + bias + Fz^T s, and
// with g set gelu(r) there (r may then be null); backward (back = 1):
// r = h W^T + Fz^T s, times gelu'(u) when u is set.  h, r, g, u [batch][nz][P][W];
// s [batch][ms][P][W]; FzT nz x ms operands (ms rounded up to 32 with zeros).
// W 16, 32 or 64; nz % 32 == 0.
struct LayerOut {
    const unsigned short *FzT;
    const float *s, *h, *Wm, *bias, *u;
    float *r, *g;
    int ms, nz, P, W, batch, back;
};
bool layer_out_covers(int nz, int W);
hipError_t run_layer_out(const LayerOut &a, hipStream_t s);

// out[rows][W] = x[rows][K] P + bias.  K % 8 == 0 up to 32; W 16, 32 or 64; rows % 16 == 0.
bool lift_covers(int K, int W, long rows);
hipError_t run_lift(const float *x, int K, const float *P, const float *bias, int W, long rows, float *out, hipStream_t s);

// y[rows][co] = gelu(h Q1 + q1) Q2 + q2; with g1 set the hidden values before and
// after GELU go to g1 and a1 [rows][H].  W, H 16, 32 or 64; co <= 16; rows % 16 == 0.
bool project_covers(int W, int H, int co, long rows);
hipError_t run_project(const float *h, const float *Q1, const float *q1, const float *Q2, const float *q2, int W, int H,
                       int co, long rows, float *g1, float *a1, float *y, hipStream_t s);
// its gradient: dg1 = (dy Q2^T) gelu'(g1), dh = dg1 Q1^T
hipError_t run_project_back(const float *dy, const float *Q1, const float *Q2, const float *g1, int W, int H, int co,
                            long rows, float *dg1, float *dh, hipStream_t s);

// The channel mixing of the mz * mxy retained modes (layout [sample][mz][re, im]
// [mxy][W]): C = A R[mode] with the FP32 parameters R[mode][W][W][re, im], and its
// gradient dA = D conj(R)^T, dR = conj(A)^T-sums over the samples.  W 16, 32 or 64.
bool mode_covers(int W);
hipError_t run_mode_mix(const float *A, const float *R, float *C, int W, long mxy, long mz, int B, hipStream_t s);
hipError_t run_mode_back(const float *A, const float *D, const float *R, float *dA, float *dR, int W, long mxy, long mz,
                         int B, hipStream_t s);

} // namespace bec
