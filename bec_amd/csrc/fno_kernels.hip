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

// The 2D transforms of all retained kz planes: out[b] = A in[b] with the plane's
// DFT matrix A (M x K, BF16, stored as the wavefronts' operands: [M / 16][K / 32]
// [lane][8]) the same for every plane b.  A workgroup stages its plane's columns
// (K x W) once in LDS, as BF16 and K contiguous, and its four wavefronts take
// 16 MB rows of A each, straight from L2, 1 KB per load.  per > 0 splits K into chunks of `per` tiles that are added in order: the
// rounding of the split-K GEMM it stands for.
template <int NB, int MB, bool SPLIT>
__global__ __launch_bounds__(256) void plane_dft_kernel(const unsigned short *__restrict__ A,
                                                        const float *__restrict__ in, float *__restrict__ out, int M,
                                                        int K, int W, int per)
{
    extern __shared__ __align__(16) unsigned short Bs[];   // [NB * 16][K + 8], column w at row (w % NB) 16 + w / NB
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, ld = K + 8;
    const int m0 = (blockIdx.x * 4 + wave) * 16 * MB;
    const float *src = in + (long)blockIdx.y * K * W;
    // G tiles of A are in flight: the first group under the staging loads
    constexpr int G = 16 / MB;
    const int tiles = K / 32;
    const bool mine = m0 < M;   // M is a multiple of 16 MB
    const unsigned short *afrag = A + (long)((mine ? m0 : 0) / 16) * tiles * 512 + lane * 8;
    bf16x8_t a[G][MB], an[G][MB];
    auto fetch = [&](bf16x8_t (&v)[G][MB], int t0) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < MB; ++i) v[g][i] = *(const bf16x8_t *)(afrag + (i * tiles + min(t0 + g, tiles - 1)) * 512);
    };
    fetch(a, 0);
#pragma unroll 4
    for (int e = threadIdx.x; e < K / 8 * W; e += 256) {
        const int w = e & (W - 1), k8 = e / W;
        f32x8_t v;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = src[(k8 * 8 + i) * W + w];
        *(bf16x8_t *)&Bs[((w % NB) * 16 + w / NB) * ld + k8 * 8] = to_bf16x8(v);
    }
    __syncthreads();
    if (!mine) return;
    const unsigned short *brow = Bs + (lane & 15) * ld + (lane >> 4) * 8;
    f32x4_t acc[MB][NB], sum[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = sum[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    for (int t0 = 0; t0 < tiles; t0 += G) {
        if (t0 + G < tiles) fetch(an, t0 + G);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int t = t0 + g;
            if (t < tiles) {
                bf16x8_t b[NB];
#pragma unroll
                for (int j = 0; j < NB; ++j) b[j] = *(const bf16x8_t *)(brow + j * 16 * ld + t * 32);
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j) acc[i][j] = mfma(a[g][i], b[j], acc[i][j]);
                if (SPLIT && ((t + 1) % per == 0 || t + 1 == tiles)) {
#pragma unroll
                    for (int i = 0; i < MB; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j) {
                            sum[i][j] += acc[i][j];
                            acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                        }
                }
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < MB; ++i) a[g][i] = an[g][i];
    }
    float *dst = out + (long)blockIdx.y * M * W;
    const int w0 = (lane & 15) * NB;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float *row = dst + (long)(m0 + i * 16 + 4 * (lane >> 4) + q) * W + w0;
            float v[NB];
#pragma unroll
            for (int j = 0; j < NB; ++j) v[j] = SPLIT ? sum[i][j][q] : acc[i][j][q];
            if (NB == 4) *(float4 *)row = make_float4(v[0], v[1 % NB], v[2 % NB], v[3 % NB]);
            else if (NB == 2) *(float2 *)row = make_float2(v[0], v[1 % NB]);
            else if (w0 < W) row[0] = v[0];
        }
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

bool plane_dft_covers(int M, int K, int W)
{
    return M % 16 == 0 && K % 32 == 0 && W <= 64 && (W & (W - 1)) == 0 && K <= 1024;
}

hipError_t run_plane_dft(const unsigned short *A, const float *in, float *out, int M, int K, int W, int planes, int per,
                         hipStream_t s)
{
    if (!plane_dft_covers(M, K, W) || planes < 1 || planes > 65535) return hipErrorInvalidValue;
    // 64 rows of A per wavefront while that leaves two workgroups for every CU,
    // else 16: the planes of a single sample would fill a quarter of the chip
    const bool wide = M % 64 == 0 && (long)planes * (M / 64) >= 1024;
    return with_blocks(W, [&](auto nb) {
        constexpr int NB = decltype(nb)::value;
        const size_t lds = sizeof(unsigned short) * NB * 16 * (K + 8);
        auto go = [&](auto mb, auto split) {
            constexpr int MB = decltype(mb)::value;
            hipLaunchKernelGGL((plane_dft_kernel<NB, MB, decltype(split)::value>),
                               dim3((M + 64 * MB - 1) / (64 * MB), planes), dim3(256), lds, s, A, in, out, M, K, W, per);
            return hipGetLastError();
        };
        using M1 = std::integral_constant<int, 1>;
        using M4 = std::integral_constant<int, 4>;
        if (per > 0) return wide ? go(M4{}, std::true_type{}) : go(M1{}, std::true_type{});
        return wide ? go(M4{}, std::false_type{}) : go(M1{}, std::false_type{});
    });
}

} // namespace bec
