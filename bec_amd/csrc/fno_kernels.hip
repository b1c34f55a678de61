// Kernels of the surrogate network that the general strided GEMM served badly:
// each reads its activations once, straight into MFMA operands.
//
// All use gfx950's 16x16x32 BF16 MFMA with FP32 accumulation: lane l supplies
// row (A) or column (B) l % 16 at the eight K positions 8 (l / 16) + i; result
// D[4 (l / 16) + q][l % 16], q = 0..3.  Operands are FP32 in memory and rounded
// to BF16 (nearest even) on the way in, as the GEMM rounds them.
#include "fno_kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace bec {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8_t to_bf16x8(f32x8_t v) { return __builtin_convertvector(v, bf16x8_t); }

__device__ __forceinline__ f32x4_t mfma(bf16x8_t a, bf16x8_t b, f32x4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// 1, 2 or 4 blocks of 16: the instantiated sizes
template <class F> hipError_t with_blocks(int n, F &&f)
{
    if (n <= 16) return f(std::integral_constant<int, 1>{});
    if (n <= 32) return f(std::integral_constant<int, 2>{});
    return f(std::integral_constant<int, 4>{});
}

// Weight and bias gradients: memory-bound (X and D are read once, 134 MB for a
// batch of 16 at width 32).  Workgroup = one of the WGRAD_SPLITS ranges of rows,
// one wavefront per 16 x 16 block of the result; its operands need eight rows
// per lane at one column, loaded directly (16 lanes read 64 contiguous bytes of
// a row, the blocks of a row its whole lines), U tiles of 32 rows ahead of the
// products, so nothing passes through LDS.  The bias is one more product, by a
// row of ones.  The range's tiles are accumulated in order and the ranges are
// added in order (sum_partials), as the split-K GEMM does, so the gradients are
// the same bits: a training run amplifies any other rounding of them.  At
// 524288 x 32 x 32: 23.7 us (5.7 TB/s) and 5.2 us for the sum; as two GEMMs
// (weights, bias) it took 107 us each and 57 us for each sum.
template <int U>
__device__ __forceinline__ void load_tiles(const float *__restrict__ P, int width, int at, long t, f32x8_t (&v)[U])
{
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float *row = P + ((t + u) * 32 + k) * width;   // uniform
            v[u][k] = row[at];
        }
}

template <int MB, int NB>
__global__ __launch_bounds__(64 * MB * NB) void wgrad_kernel(const float *__restrict__ X, int M,
                                                             const float *__restrict__ D, int N, long tiles, int per,
                                                             float *__restrict__ part)
{
    constexpr int U = MB * NB > 8 ? 1 : 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = wave / NB, j = wave % NB;
    const int cm = i * 16 + (lane & 15), cn = j * 16 + (lane & 15), kq = (lane >> 4) * 8;
    // a block's columns beyond the matrix read its last one: what they give is not stored
    const int am = kq * M + min(cm, M - 1), an = kq * N + min(cn, N - 1);
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f}, accb = {0.f, 0.f, 0.f, 0.f};
    const float o = (lane & 15) == 0 ? 1.0f : 0.0f;
    const bf16x8_t ones = to_bf16x8((f32x8_t){o, o, o, o, o, o, o, o});
    const long t0 = (long)blockIdx.x * per, t1 = min(tiles, t0 + per);
    auto step = [&](f32x8_t a, f32x8_t b) {
        const bf16x8_t bb = to_bf16x8(b);
        acc = mfma(to_bf16x8(a), bb, acc);
        if (i == 0) accb = mfma(ones, bb, accb);   // uniform
    };
    long t = t0;
    f32x8_t a0[U], b0[U], a1[U], b1[U];
    if (t + U <= t1) {
        load_tiles<U>(X, M, am, t, a0);
        load_tiles<U>(D, N, an, t, b0);
        for (; t + 3 * U <= t1; t += 2 * U) {
            load_tiles<U>(X, M, am, t + U, a1);
            load_tiles<U>(D, N, an, t + U, b1);
#pragma unroll
            for (int u = 0; u < U; ++u) step(a0[u], b0[u]);
            load_tiles<U>(X, M, am, t + 2 * U, a0);
            load_tiles<U>(D, N, an, t + 2 * U, b0);
#pragma unroll
            for (int u = 0; u < U; ++u) step(a1[u], b1[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) step(a0[u], b0[u]);
        t += U;
    }
    for (; t < t1; ++t) {
        f32x8_t a[1], b[1];
        load_tiles<1>(X, M, am, t, a);
        load_tiles<1>(D, N, an, t, b);
        step(a[0], b[0]);
    }
    float *out = part + (long)blockIdx.x * ((long)M * N + N);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int m = i * 16 + 4 * (lane >> 4) + q;
        if (m < M && cn < N) out[(long)m * N + cn] = acc[q];
    }
    if (i == 0 && lane < 16 && cn < N) out[(long)M * N + cn] = accb[0];
}

// out[i] = the n partials added in order, 32 of them in flight per thread (one
// at a time took 57 us for 256 partials)
__global__ __launch_bounds__(64) void sum_partials(const float *__restrict__ part, int n, int total,
                                                   float *__restrict__ out)
{
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= total) return;
    float s = 0.f;
    for (int k = 0; k < n; k += 32) {   // n is a multiple of 32
        float v[32];
#pragma unroll
        for (int j = 0; j < 32; ++j) v[j] = part[(long)(k + j) * total + i];
#pragma unroll
        for (int j = 0; j < 32; ++j) s += v[j];
    }
    out[i] = s;
}

} // namespace

bool wgrad_covers(int K, int N, long rows) { return K <= 64 && N <= 64 && rows % 32 == 0; }

hipError_t run_wgrad(const float *X, int K, const float *D, int N, long rows, float *part, float *out, hipStream_t s)
{
    if (!wgrad_covers(K, N, rows)) return hipErrorInvalidValue;
    const long tiles = rows / 32;
    const int per = (int)((tiles + WGRAD_SPLITS - 1) / WGRAD_SPLITS);
    hipError_t e = with_blocks(K, [&](auto mb) {
        return with_blocks(N, [&](auto nb) {
            constexpr int MB = decltype(mb)::value, NB = decltype(nb)::value;
            hipLaunchKernelGGL((wgrad_kernel<MB, NB>), dim3(WGRAD_SPLITS), dim3(64 * MB * NB), 0, s, X, K, D, N, tiles,
                               per, part);
            return hipGetLastError();
        });
    });
    if (e != hipSuccess) return e;
    const int total = K * N + N;
    hipLaunchKernelGGL(sum_partials, dim3((total + 63) / 64), dim3(64), 0, s, part, WGRAD_SPLITS, total, out);
    return hipGetLastError();
}

} // namespace bec
