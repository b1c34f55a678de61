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
                                                        int K, int W, int per, int m_blocks)
{
    extern __shared__ __align__(16) unsigned short Bs[];   // [NB * 16][K + 8], column w at row (w % NB) 16 + w / NB
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, ld = K + 8;
    // the planes in the grid's x dimension, which alone holds more than 65535
    const int mb = blockIdx.x % m_blocks;
    const long plane = blockIdx.x / m_blocks;
    const int m0 = (mb * 4 + wave) * 16 * MB;
    const float *src = in + plane * K * W;
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
    float *dst = out + plane * M * W;
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

// Transform along z: out[b] = A in[b], A the M x K operand matrix (rows beyond M
// zero), in[b] K x N, out[b] M x N.  A wavefront owns 64 columns, four adjacent
// ones per lane (256-byte row segments), and reads them once.
template <int MB, bool SPLIT>
__global__ __launch_bounds__(256) void z_dft_kernel(const unsigned short *__restrict__ A, const float *__restrict__ in,
                                                    float *__restrict__ out, int M, int K, int N, int per)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kq = (lane >> 4) * 8, tiles = K / 32;
    const int n0 = (blockIdx.x * 4 + wave) * 64 + (lane & 15) * 4;
    if (n0 - (lane & 15) * 4 >= N) return;   // N is a multiple of 64
    const float *src = in + (long)blockIdx.y * K * N + (long)kq * N + n0;
    const unsigned short *afrag = A + lane * 8;
    f32x4_t acc[MB][4], sum[MB][4], v[8];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = sum[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = *(const f32x4_t *)(src + (long)k * N);
    for (int t = 0; t < tiles; ++t) {
        f32x4_t vn[8];
        bf16x8_t a[MB];
        if (t + 1 < tiles)
#pragma unroll
            for (int k = 0; k < 8; ++k) vn[k] = *(const f32x4_t *)(src + ((long)(t + 1) * 32 + k) * N);
#pragma unroll
        for (int i = 0; i < MB; ++i) a[i] = *(const bf16x8_t *)(afrag + (i * tiles + t) * 512);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bf16x8_t b =
                to_bf16x8((f32x8_t){v[0][j], v[1][j], v[2][j], v[3][j], v[4][j], v[5][j], v[6][j], v[7][j]});
#pragma unroll
            for (int i = 0; i < MB; ++i) acc[i][j] = mfma(a[i], b, acc[i][j]);
        }
        if (SPLIT && ((t + 1) % per == 0 || t + 1 == tiles)) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    sum[i][j] += acc[i][j];
                    acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
                }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = vn[k];
    }
    float *dst = out + (long)blockIdx.y * M * N + n0;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int m = i * 16 + 4 * (lane >> 4) + q;
            if (m >= M) continue;
            f32x4_t r;
#pragma unroll
            for (int j = 0; j < 4; ++j) r[j] = SPLIT ? sum[i][j][q] : acc[i][j][q];
            *(f32x4_t *)(dst + (long)m * N) = r;
        }
}

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

// gelu'(x) = Phi(x) + x phi(x)
__device__ __forceinline__ float gelu_slope(float x)
{
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

template <int V> struct VecF;
template <> struct VecF<1> { typedef float type __attribute__((ext_vector_type(1))); };
template <> struct VecF<2> { typedef float type __attribute__((ext_vector_type(2))); };
template <> struct VecF<4> { typedef float type __attribute__((ext_vector_type(4))); };

// What leaves a spectral layer: r = h W (+ b) + Fz^T s, one pass over h and s
// (the z modes of the layer's spectral part), both products in one wavefront's
// registers: 32 z values of one column (b, y, x).  BACK applies W^T and no bias.
// EPI: 0 stores r; 1 stores r and gelu(r); 2 stores gelu(r) alone; 3 stores
// r gelu'(u).  It stands for the transform, the per-cell GEMM that read its
// result again and a GELU kernel (46 + 64 + 28 us at batch 16).
template <int V, bool BACK, int EPI>
__global__ __launch_bounds__(256) void layer_out_kernel(const unsigned short *__restrict__ FzT,
                                                        const float *__restrict__ s, int ms,
                                                        const float *__restrict__ h, const float *__restrict__ Wm,
                                                        const float *__restrict__ bias, int nz, int P,
                                                        const float *__restrict__ u, float *__restrict__ r_out,
                                                        float *__restrict__ g_out)
{
    constexpr int W = 16 * V, WT = (W + 31) / 32, ZB = 2;
    using vec = typename VecF<V>::type;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, kq = (lane >> 4) * 8;
    const int p = blockIdx.x * 4 + wave, zb0 = blockIdx.y * ZB, w0 = c * V;
    if (p >= P) return;
    const long b = blockIdx.z;
    const int st = (ms + 31) / 32;
    // the layer input's rows first: the longest reads
    f32x8_t ha[ZB][WT];
#pragma unroll
    for (int i = 0; i < ZB; ++i)
#pragma unroll
        for (int t = 0; t < WT; ++t) {
            const float *row = h + ((b * nz + (zb0 + i) * 16 + c) * P + p) * W + t * 32 + kq;
            ha[i][t] = (f32x8_t){0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (W >= 32 || kq < W) {
                const f32x4_t lo = *(const f32x4_t *)row, hi = *(const f32x4_t *)(row + 4);
                ha[i][t] = (f32x8_t){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            }
        }
    f32x4_t az[ZB][V], aw[ZB][V];
#pragma unroll
    for (int i = 0; i < ZB; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) az[i][j] = aw[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t < st; ++t) {
        vec v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int m = t * 32 + kq + k;
            v[k] = *(const vec *)(s + ((b * ms + min(m, ms - 1)) * P + p) * W + w0);
            if (m >= ms) v[k] = (vec)(0.f);
        }
        bf16x8_t a[ZB];
#pragma unroll
        for (int i = 0; i < ZB; ++i) a[i] = *(const bf16x8_t *)(FzT + ((long)((zb0 + i) * st + t) * 64 + lane) * 8);
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const bf16x8_t bb =
                to_bf16x8((f32x8_t){v[0][j], v[1][j], v[2][j], v[3][j], v[4][j], v[5][j], v[6][j], v[7][j]});
#pragma unroll
            for (int i = 0; i < ZB; ++i) az[i][j] = mfma(a[i], bb, az[i][j]);
        }
    }
#pragma unroll
    for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int j = 0; j < V; ++j) {
            f32x8_t w;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int i = t * 32 + kq + k;
                w[k] = i < W ? (BACK ? Wm[(w0 + j) * W + i] : Wm[i * W + w0 + j]) : 0.f;
            }
            const bf16x8_t bb = to_bf16x8(w);
#pragma unroll
            for (int i = 0; i < ZB; ++i) aw[i][j] = mfma(to_bf16x8(ha[i][t]), bb, aw[i][j]);
        }
    vec bv = (vec)(0.f);
    if (!BACK) bv = *(const vec *)(bias + w0);
#pragma unroll
    for (int i = 0; i < ZB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const long at = ((b * nz + (zb0 + i) * 16 + 4 * (lane >> 4) + q) * P + p) * W + w0;
            vec r, g;
#pragma unroll
            for (int j = 0; j < V; ++j) {
                r[j] = aw[i][j][q] + az[i][j][q];
                if (!BACK) r[j] += bv[j];
            }
            if (EPI == 3) {
                const vec uv = *(const vec *)(u + at);
#pragma unroll
                for (int j = 0; j < V; ++j) r[j] *= gelu_slope(uv[j]);
            }
            if (EPI != 2) *(vec *)(r_out + at) = r;
            if (EPI == 1 || EPI == 2) {
#pragma unroll
                for (int j = 0; j < V; ++j) g[j] = gelu(r[j]);
                *(vec *)(g_out + at) = g;
            }
        }
}

// Eight consecutive K values of a row-major FP32 operand row as BF16; zeros from
// `width` on (a multiple of 8).
__device__ __forceinline__ bf16x8_t row_operand(const float *row, int k, int width)
{
    f32x8_t v = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (k < width) {
        const f32x4_t lo = *(const f32x4_t *)(row + k), hi = *(const f32x4_t *)(row + k + 4);
        v = (f32x8_t){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
    return to_bf16x8(v);
}

// The lift: out = x P + p, 16 rows at a time per wavefront, P in registers.
template <int V>
__global__ __launch_bounds__(256) void lift_kernel(const float *__restrict__ x, int K, const float *__restrict__ P,
                                                   const float *__restrict__ bias, long tiles, float *__restrict__ out)
{
    constexpr int W = 16 * V;
    using vec = typename VecF<V>::type;
    const int lane = threadIdx.x & 63, c = lane & 15, kq = (lane >> 4) * 8, w0 = c * V;
    bf16x8_t pb[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        f32x8_t w;
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = kq + k < K ? P[(kq + k) * W + w0 + j] : 0.f;
        pb[j] = to_bf16x8(w);
    }
    const vec bv = *(const vec *)(bias + w0);
    for (long t = (long)blockIdx.x * 4 + (threadIdx.x >> 6); t < tiles; t += (long)gridDim.x * 4) {
        const bf16x8_t a = row_operand(x + (t * 16 + c) * K, kq, K);
        f32x4_t acc[V];
#pragma unroll
        for (int j = 0; j < V; ++j) acc[j] = mfma(a, pb[j], (f32x4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            vec r;
#pragma unroll
            for (int j = 0; j < V; ++j) r[j] = acc[j][q] + bv[j];
            *(vec *)(out + (t * 16 + 4 * (lane >> 4) + q) * W + w0) = r;
        }
    }
}

// A 16-row tile of BF16 values between the result layout of one product (rows
// 4 (l / 16) + q, columns V c + j) and the operand layout of the next (row
// l % 16, eight consecutive columns), through this wavefront's LDS rows.
template <int V>
__device__ __forceinline__ void tile_put(unsigned short *T, int ld, int lane, int q, const float (&v)[V])
{
    typedef float fV __attribute__((ext_vector_type(V)));
    typedef __bf16 bV __attribute__((ext_vector_type(V)));
    fV f;
#pragma unroll
    for (int j = 0; j < V; ++j) f[j] = v[j];
    *(bV *)&T[(4 * (lane >> 4) + q) * ld + (lane & 15) * V] = __builtin_convertvector(f, bV);
}

__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The projection y = gelu(h Q1 + q1) Q2 + q2 in one pass over h; with KEEP the
// hidden values before and after GELU are stored for the backward pass.  As
// three launches the hidden values (134 MB at batch 16) were written, read,
// written and read again: 72 + 64 + 64 us.
template <int VW, int VH, bool KEEP>
__global__ __launch_bounds__(256) void project_kernel(const float *__restrict__ h, const float *__restrict__ Q1,
                                                      const float *__restrict__ q1, const float *__restrict__ Q2,
                                                      const float *__restrict__ q2, int co, long tiles,
                                                      float *__restrict__ g1, float *__restrict__ a1,
                                                      float *__restrict__ y)
{
    constexpr int W = 16 * VW, H = 16 * VH, WT = (W + 31) / 32, HT = (H + 31) / 32, LD = HT * 32 + 8;
    using vec = typename VecF<VH>::type;
    __shared__ __align__(16) unsigned short lds[4][16 * LD];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, kq = (lane >> 4) * 8, h0 = c * VH;
    unsigned short *T = lds[wave];
    for (int i = lane; i < 16 * LD; i += 64) T[i] = 0;   // columns beyond H stay zero
    bf16x8_t w1[WT][VH], w2[HT];
#pragma unroll
    for (int t = 0; t < WT; ++t)
#pragma unroll
        for (int j = 0; j < VH; ++j) {
            f32x8_t w;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int i = t * 32 + kq + k;
                w[k] = i < W ? Q1[i * H + h0 + j] : 0.f;
            }
            w1[t][j] = to_bf16x8(w);
        }
#pragma unroll
    for (int t = 0; t < HT; ++t) {
        f32x8_t w;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int i = t * 32 + kq + k;
            w[k] = i < H && c < co ? Q2[i * co + c] : 0.f;
        }
        w2[t] = to_bf16x8(w);
    }
    const vec b1 = *(const vec *)(q1 + h0);
    const float b2 = c < co ? q2[c] : 0.f;
    wave_fence();
    for (long t = (long)blockIdx.x * 4 + wave; t < tiles; t += (long)gridDim.x * 4) {
        f32x4_t acc[VH], yo = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < VH; ++j) acc[j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < WT; ++i) {
            const bf16x8_t a = row_operand(h + (t * 16 + c) * W, i * 32 + kq, W);
#pragma unroll
            for (int j = 0; j < VH; ++j) acc[j] = mfma(a, w1[i][j], acc[j]);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const long at = (t * 16 + 4 * (lane >> 4) + q) * H + h0;
            vec u, g;
            float v[VH];
#pragma unroll
            for (int j = 0; j < VH; ++j) {
                u[j] = acc[j][q] + b1[j];
                g[j] = v[j] = gelu(u[j]);
            }
            if (KEEP) {
                *(vec *)(g1 + at) = u;
                *(vec *)(a1 + at) = g;
            }
            tile_put<VH>(T, LD, lane, q, v);
        }
        wave_fence();
#pragma unroll
        for (int i = 0; i < HT; ++i) yo = mfma(*(const bf16x8_t *)&T[c * LD + i * 32 + kq], w2[i], yo);
        wave_fence();
        if (c < co)
#pragma unroll
            for (int q = 0; q < 4; ++q) y[(t * 16 + 4 * (lane >> 4) + q) * co + c] = yo[q] + b2;
    }
}

// Its gradient: dg1 = (dy Q2^T) gelu'(g1) (kept for the weight gradients) and
// dh = dg1 Q1^T, in one pass over g1.
template <int VW, int VH>
__global__ __launch_bounds__(256) void project_back_kernel(const float *__restrict__ dy, int co,
                                                           const float *__restrict__ Q1, const float *__restrict__ Q2,
                                                           const float *__restrict__ g1, long tiles,
                                                           float *__restrict__ dg1, float *__restrict__ dh)
{
    constexpr int W = 16 * VW, H = 16 * VH, HT = (H + 31) / 32, LD = HT * 32 + 8;
    using vec = typename VecF<VH>::type;
    using vew = typename VecF<VW>::type;
    __shared__ __align__(16) unsigned short lds[4][16 * LD];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, kq = (lane >> 4) * 8, h0 = c * VH;
    unsigned short *T = lds[wave];
    for (int i = lane; i < 16 * LD; i += 64) T[i] = 0;
    bf16x8_t w2[VH], w1[HT][VW];
#pragma unroll
    for (int j = 0; j < VH; ++j) {
        f32x8_t w;
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = kq + k < co ? Q2[(h0 + j) * co + kq + k] : 0.f;
        w2[j] = to_bf16x8(w);
    }
#pragma unroll
    for (int t = 0; t < HT; ++t)
#pragma unroll
        for (int j = 0; j < VW; ++j) w1[t][j] = row_operand(Q1 + (c * VW + j) * H, t * 32 + kq, H);
    wave_fence();
    for (long t = (long)blockIdx.x * 4 + wave; t < tiles; t += (long)gridDim.x * 4) {
        f32x8_t d;
#pragma unroll
        for (int k = 0; k < 8; ++k) d[k] = kq + k < co ? dy[(t * 16 + c) * co + kq + k] : 0.f;
        const bf16x8_t a = to_bf16x8(d);
        f32x4_t acc[VH], ao[VW];
#pragma unroll
        for (int j = 0; j < VH; ++j) acc[j] = mfma(a, w2[j], (f32x4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const long at = (t * 16 + 4 * (lane >> 4) + q) * H + h0;
            const vec u = *(const vec *)(g1 + at);
            vec g;
            float v[VH];
#pragma unroll
            for (int j = 0; j < VH; ++j) g[j] = v[j] = acc[j][q] * gelu_slope(u[j]);
            *(vec *)(dg1 + at) = g;
            tile_put<VH>(T, LD, lane, q, v);
        }
        wave_fence();
#pragma unroll
        for (int j = 0; j < VW; ++j) ao[j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < HT; ++i) {
            const bf16x8_t b = *(const bf16x8_t *)&T[c * LD + i * 32 + kq];
#pragma unroll
            for (int j = 0; j < VW; ++j) ao[j] = mfma(b, w1[i][j], ao[j]);
        }
        wave_fence();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            vew r;
#pragma unroll
            for (int j = 0; j < VW; ++j) r[j] = ao[j][q];
            *(vew *)(dh + (t * 16 + 4 * (lane >> 4) + q) * W + c * VW) = r;
        }
    }
}

// Where the values of mode t lie: the real channels of sample b at
// b * sample + t's offset, the imaginary ones `part` floats behind.
struct ModeAt {
    long base, part;
};
__device__ __forceinline__ ModeAt mode_at(long t, long mxy, int W)
{
    return {(t / mxy * 2 * mxy + t % mxy) * W, mxy * W};
}

// Eight samples from b0 on of V channels of one part, as V operands whose K is the sample.
template <int V>
__device__ __forceinline__ void sample_operands(const float *A, long sample, int b0, int B, bf16x8_t (&out)[V])
{
    using vec = typename VecF<V>::type;
    vec v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        vec z;
#pragma unroll
        for (int j = 0; j < V; ++j) z[j] = 0.f;
        v[k] = b0 + k < B ? *(const vec *)(A + (b0 + k) * sample) : z;
    }
#pragma unroll
    for (int j = 0; j < V; ++j)
        out[j] = to_bf16x8((f32x8_t){v[0][j], v[1][j], v[2][j], v[3][j], v[4][j], v[5][j], v[6][j], v[7][j]});
}

// The operand of a product over 2 W channels of sample b (K tile i of 32).
template <int V>
__device__ __forceinline__ bf16x8_t channel_operand(const float *A, long sample, const ModeAt &m, int b, int B, int k)
{
    f32x8_t v = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (b < B) {
        const float *r = A + b * sample + m.base + (k < 16 * V ? k : m.part + k - 16 * V);
        const f32x4_t lo = *(const f32x4_t *)r, hi = *(const f32x4_t *)(r + 4);
        v = (f32x8_t){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
    return to_bf16x8(v);
}

// C = A (re + i im) for the 2 W channels of 16 samples at a time, given the
// products' operands: re[i][j], im[i][j] of K tile i (of the W input channels;
// with W = 16 one tile holds both parts, already signed) and output column
// 16 V-wide block j.  `conj` the other sign of im (the adjoint).
template <int V, bool CONJ>
__device__ __forceinline__ void mix_samples(const float *A, float *C, long sample, const ModeAt &m, int B,
                                            const bf16x8_t (&re)[(V + 1) / 2][V], const bf16x8_t (&im)[(V + 1) / 2][V],
                                            const bf16x8_t (&nim)[(V + 1) / 2][V])
{
    using vec = typename VecF<V>::type;
    constexpr int T = V / 2;
    const int lane = threadIdx.x & 63, c = lane & 15, kq = (lane >> 4) * 8;
    for (int b0 = 0; b0 < B; b0 += 16) {
        f32x4_t acc[2][V];
#pragma unroll
        for (int j = 0; j < V; ++j) acc[0][j] = acc[1][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const bf16x8_t a = channel_operand<V>(A, sample, m, b0 + c, B, i * 32 + kq);
#pragma unroll
            for (int j = 0; j < V; ++j) {
                if (V == 1 || i < T) {
                    acc[0][j] = mfma(a, re[i][j], acc[0][j]);
                    acc[1][j] = mfma(a, V > 1 && CONJ ? nim[i][j] : im[i][j], acc[1][j]);
                } else {
                    acc[0][j] = mfma(a, CONJ ? im[i - T][j] : nim[i - T][j], acc[0][j]);
                    acc[1][j] = mfma(a, re[i - T][j], acc[1][j]);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int b = b0 + 4 * (lane >> 4) + q;
            if (b < B)
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    vec v;
#pragma unroll
                    for (int j = 0; j < V; ++j) v[j] = acc[r][j][q];
                    *(vec *)(C + b * sample + m.base + r * m.part + c * V) = v;
                }
        }
    }
}

// The channel mixing of every retained mode, C[b][t] = A[b][t] R[t] (complex):
// bound by memory (R is read once, 33 MB per layer at width 32 and 4096 modes).
// One wavefront per mode holds R[t] in registers as BF16 operands, read straight
// from the FP32 parameters in whole rows; as a GEMM over the expanded real
// matrices it took 31 us at batch 16 and the matrices another 16 us per change
// of the parameters.
template <int V>
__global__ __launch_bounds__(256) void mode_mix_kernel(const float *__restrict__ A, const float *__restrict__ R,
                                                       float *__restrict__ C, long mxy, long sample, int B, long modes)
{
    constexpr int W = 16 * V, I = (V + 1) / 2;
    typedef float vec2 __attribute__((ext_vector_type(2 * V)));
    const long t = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= modes) return;
    const int lane = threadIdx.x & 63, c = lane & 15, kq = (lane >> 4) * 8;
    const bool second = V == 1 && kq >= W;   // width 16: these lanes' K is the imaginary part
    const float *r = R + t * (2 * W * W) + c * 2 * V;
    bf16x8_t re[I][V], im[I][V], nim[I][V];
#pragma unroll
    for (int i = 0; i < I; ++i) {
        vec2 v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = *(const vec2 *)(r + (i * 32 + (kq & (V == 1 ? 15 : 31)) + k) * 2 * W);
#pragma unroll
        for (int j = 0; j < V; ++j) {
            f32x8_t x, y;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                x[k] = second ? -v[k][2 * j + 1] : v[k][2 * j];
                y[k] = second ? v[k][2 * j] : v[k][2 * j + 1];
            }
            re[i][j] = to_bf16x8(x);
            im[i][j] = to_bf16x8(y);
            nim[i][j] = to_bf16x8(-y);
        }
    }
    mix_samples<V, false>(A, C, sample, mode_at(t, mxy, W), B, re, im, nim);
}

// Its gradient, per mode: dA = dC conj(R)^T and dR = A^T-products of A and dC
// over the samples (re: AreDre + AimDim, im: AreDim - AimDre), in one pass over
// R, A and dC.  As two GEMMs and a fold of the four real products: 35 + 16 + 31 us.
template <int V>
__global__ __launch_bounds__(256) void mode_back_kernel(const float *__restrict__ A, const float *__restrict__ D,
                                                        const float *__restrict__ R, float *__restrict__ dA,
                                                        float *__restrict__ dR, long mxy, long sample, int B, long modes)
{
    constexpr int W = 16 * V, I = (V + 1) / 2, JS = V < 2 ? V : 2;
    const long t = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= modes) return;
    const int lane = threadIdx.x & 63, c = lane & 15, kq = (lane >> 4) * 8;
    const bool second = V == 1 && kq >= W;
    const ModeAt m = mode_at(t, mxy, W);
    {
        bf16x8_t re[I][V], im[I][V], nim[I][V];
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const float *r = R + t * (2 * W * W) + (c * V + j) * 2 * W + (i * 32 + (kq & (V == 1 ? 15 : 31))) * 2;
                f32x8_t x, y;
#pragma unroll
                for (int k = 0; k < 8; k += 2) {
                    const f32x4_t v = *(const f32x4_t *)(r + 2 * k);
                    x[k] = second ? v[1] : v[0];
                    y[k] = second ? v[0] : -v[1];
                    x[k + 1] = second ? v[3] : v[2];
                    y[k + 1] = second ? v[2] : -v[3];
                }
                re[i][j] = to_bf16x8(x);
                nim[i][j] = to_bf16x8(y);
                im[i][j] = V == 1 ? nim[i][j] : to_bf16x8(-y);
            }
        mix_samples<V, true>(D, dA, sample, m, B, re, im, nim);
    }
    for (int jb = 0; jb < V; jb += JS) {
        typedef float vecj __attribute__((ext_vector_type(2 * JS)));
        f32x4_t acc[4][V][JS];   // re re, im im, re im, im re
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int i = 0; i < V; ++i)
#pragma unroll
                for (int j = 0; j < JS; ++j) acc[p][i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        for (int b0 = 0; b0 < B; b0 += 32) {
            bf16x8_t ar[V], ai[V], dr[JS], di[JS];
            const float *a = A + m.base + c * V, *d = D + m.base + c * V + jb;
            sample_operands<V>(a, sample, b0 + kq, B, ar);
            sample_operands<V>(a + m.part, sample, b0 + kq, B, ai);
            sample_operands<JS>(d, sample, b0 + kq, B, dr);
            sample_operands<JS>(d + m.part, sample, b0 + kq, B, di);
#pragma unroll
            for (int i = 0; i < V; ++i)
#pragma unroll
                for (int j = 0; j < JS; ++j) {
                    acc[0][i][j] = mfma(ar[i], dr[j], acc[0][i][j]);
                    acc[1][i][j] = mfma(ai[i], di[j], acc[1][i][j]);
                    acc[2][i][j] = mfma(ar[i], di[j], acc[2][i][j]);
                    acc[3][i][j] = mfma(ai[i], dr[j], acc[3][i][j]);
                }
        }
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                vecj v;
#pragma unroll
                for (int j = 0; j < JS; ++j) {
                    v[2 * j] = acc[0][i][j][q] + acc[1][i][j][q];
                    v[2 * j + 1] = acc[2][i][j][q] - acc[3][i][j][q];
                }
                *(vecj *)(dR + t * (2 * W * W) + ((4 * (lane >> 4) + q) * V + i) * 2 * W + (c * V + jb) * 2) = v;
            }
    }
}

// The mixing for a single sample at width 32 (a product would use one row of
// 16): one wavefront per mode, lane l owns the outputs 4 (l % 8) + i and the
// inputs l / 8 + 8 j, so one load covers whole rows of R; the partial sums are
// combined over the lanes in a fixed butterfly order.  Operands rounded to BF16
// as the products round them, products exact in FP32.
__global__ __launch_bounds__(256) void mode_row_kernel(const float *__restrict__ A, const float *__restrict__ R,
                                                       float *__restrict__ C, long mxy, long modes)
{
    const long t = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= modes) return;
    const int lane = threadIdx.x & 63, o = 4 * (lane & 7), kp = lane >> 3;
    const ModeAt m = mode_at(t, mxy, 32);
    f32x8_t w[4], acc[2] = {};   // acc: re outputs, im outputs (4 each used)
    float xr[4], xi[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float *r = R + t * 2048 + (kp + 8 * j) * 64 + 2 * o;
        const f32x4_t lo = *(const f32x4_t *)r, hi = *(const f32x4_t *)(r + 4);
        w[j] = __builtin_convertvector(to_bf16x8((f32x8_t){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}), f32x8_t);
        xr[j] = A[m.base + kp + 8 * j];
        xi[j] = A[m.base + m.part + kp + 8 * j];
    }
    const f32x8_t x = __builtin_convertvector(
        to_bf16x8((f32x8_t){xr[0], xr[1], xr[2], xr[3], xi[0], xi[1], xi[2], xi[3]}), f32x8_t);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[0][i] = fmaf(x[j], w[j][2 * i], acc[0][i]);
            acc[1][i] = fmaf(x[j], w[j][2 * i + 1], acc[1][i]);
        }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[0][i] = fmaf(x[4 + j], -w[j][2 * i + 1], acc[0][i]);
            acc[1][i] = fmaf(x[4 + j], w[j][2 * i], acc[1][i]);
        }
#pragma unroll
    for (int off = 8; off < 64; off <<= 1)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[0][i] += __shfl_xor(acc[0][i], off);
            acc[1][i] += __shfl_xor(acc[1][i], off);
        }
    if (kp < 2) {
        const f32x8_t v = acc[kp ? 1 : 0];
        *(f32x4_t *)(C + m.base + kp * m.part + o) = (f32x4_t){v[0], v[1], v[2], v[3]};
    }
}

// workgroups of a kernel whose wavefronts walk `tiles` tiles: eight per CU
int row_grid(long tiles) { return (int)std::min<long>(2048, (tiles + 3) / 4); }

bool vec_width(int n) { return n == 16 || n == 32 || n == 64; }

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
    if (!plane_dft_covers(M, K, W) || planes < 1) return hipErrorInvalidValue;
    // 64 rows of A per wavefront while that leaves two workgroups for every CU,
    // else 16: the planes of a single sample would fill a quarter of the chip
    const bool wide = M % 64 == 0 && (long)planes * (M / 64) >= 1024;
    return with_blocks(W, [&](auto nb) {
        constexpr int NB = decltype(nb)::value;
        const size_t lds = sizeof(unsigned short) * NB * 16 * (K + 8);
        auto go = [&](auto mb, auto split) {
            constexpr int MB = decltype(mb)::value;
            const int m_blocks = (M + 64 * MB - 1) / (64 * MB);
            const long wgs = (long)m_blocks * planes;
            if (wgs > 0xffffffffL / 256) return hipErrorInvalidValue;   // threads of a launch
            hipLaunchKernelGGL((plane_dft_kernel<NB, MB, decltype(split)::value>), dim3((unsigned)wgs), dim3(256), lds, s, A,
                               in, out, M, K, W, per, m_blocks);
            return hipGetLastError();
        };
        using M1 = std::integral_constant<int, 1>;
        using M4 = std::integral_constant<int, 4>;
        if (per > 0) return wide ? go(M4{}, std::true_type{}) : go(M1{}, std::true_type{});
        return wide ? go(M4{}, std::false_type{}) : go(M1{}, std::false_type{});
    });
}

bool z_dft_covers(int M, int K, long N) { return M <= 64 && K % 32 == 0 && N % 64 == 0; }

hipError_t run_z_dft(const unsigned short *A, const float *in, float *out, int M, int K, int N, int batch, int per,
                     hipStream_t s)
{
    if (!z_dft_covers(M, K, N) || batch < 1 || batch > 65535) return hipErrorInvalidValue;
    return with_blocks(M, [&](auto mb) {
        constexpr int MB = decltype(mb)::value;
        const dim3 grid((N / 64 + 3) / 4, batch);
        if (per > 0) hipLaunchKernelGGL((z_dft_kernel<MB, true>), grid, dim3(256), 0, s, A, in, out, M, K, N, per);
        else hipLaunchKernelGGL((z_dft_kernel<MB, false>), grid, dim3(256), 0, s, A, in, out, M, K, N, per);
        return hipGetLastError();
    });
}

bool layer_out_covers(int nz, int W) { return nz % 32 == 0 && (W == 16 || W == 32 || W == 64); }

hipError_t run_layer_out(const LayerOut &a, hipStream_t s)
{
    if (!layer_out_covers(a.nz, a.W) || a.batch < 1 || a.batch > 65535) return hipErrorInvalidValue;
    const dim3 grid((a.P + 3) / 4, a.nz / 32, a.batch);
    return with_blocks(a.W, [&](auto v) {
        constexpr int V = decltype(v)::value;
        auto go = [&](auto back, auto epi) {
            hipLaunchKernelGGL((layer_out_kernel<V, decltype(back)::value, decltype(epi)::value>), grid, dim3(256), 0, s,
                               a.FzT, a.s, a.ms, a.h, a.Wm, a.bias, a.nz, a.P, a.u, a.r, a.g);
            return hipGetLastError();
        };
        using E0 = std::integral_constant<int, 0>;
        if (a.back) return a.u ? go(std::true_type{}, std::integral_constant<int, 3>{}) : go(std::true_type{}, E0{});
        if (!a.g) return go(std::false_type{}, E0{});
        return a.r ? go(std::false_type{}, std::integral_constant<int, 1>{})
                   : go(std::false_type{}, std::integral_constant<int, 2>{});
    });
}

bool lift_covers(int K, int W, long rows) { return K % 8 == 0 && K <= 32 && vec_width(W) && rows % 16 == 0; }

hipError_t run_lift(const float *x, int K, const float *P, const float *bias, int W, long rows, float *out, hipStream_t s)
{
    if (!lift_covers(K, W, rows)) return hipErrorInvalidValue;
    return with_blocks(W, [&](auto v) {
        hipLaunchKernelGGL(lift_kernel<decltype(v)::value>, dim3(row_grid(rows / 16)), dim3(256), 0, s, x, K, P, bias,
                           rows / 16, out);
        return hipGetLastError();
    });
}

bool project_covers(int W, int H, int co, long rows)
{
    return vec_width(W) && vec_width(H) && co <= 16 && rows % 16 == 0;
}

hipError_t run_project(const float *h, const float *Q1, const float *q1, const float *Q2, const float *q2, int W, int H,
                       int co, long rows, float *g1, float *a1, float *y, hipStream_t s)
{
    if (!project_covers(W, H, co, rows)) return hipErrorInvalidValue;
    return with_blocks(W, [&](auto vw) {
        return with_blocks(H, [&](auto vh) {
            constexpr int VW = decltype(vw)::value, VH = decltype(vh)::value;
            const dim3 grid(row_grid(rows / 16));
            if (g1)
                hipLaunchKernelGGL((project_kernel<VW, VH, true>), grid, dim3(256), 0, s, h, Q1, q1, Q2, q2, co, rows / 16,
                                   g1, a1, y);
            else
                hipLaunchKernelGGL((project_kernel<VW, VH, false>), grid, dim3(256), 0, s, h, Q1, q1, Q2, q2, co,
                                   rows / 16, g1, a1, y);
            return hipGetLastError();
        });
    });
}

hipError_t run_project_back(const float *dy, const float *Q1, const float *Q2, const float *g1, int W, int H, int co,
                            long rows, float *dg1, float *dh, hipStream_t s)
{
    if (!project_covers(W, H, co, rows)) return hipErrorInvalidValue;
    return with_blocks(W, [&](auto vw) {
        return with_blocks(H, [&](auto vh) {
            hipLaunchKernelGGL((project_back_kernel<decltype(vw)::value, decltype(vh)::value>), dim3(row_grid(rows / 16)),
                               dim3(256), 0, s, dy, co, Q1, Q2, g1, rows / 16, dg1, dh);
            return hipGetLastError();
        });
    });
}

bool mode_covers(int W) { return vec_width(W); }

hipError_t run_mode_mix(const float *A, const float *R, float *C, int W, long mxy, long mz, int B, hipStream_t s)
{
    if (!mode_covers(W)) return hipErrorInvalidValue;
    const long modes = mz * mxy, sample = 2 * modes * W;
    const dim3 grid((unsigned)((modes + 3) / 4));
    if (B == 1 && W == 32) {
        hipLaunchKernelGGL(mode_row_kernel, grid, dim3(256), 0, s, A, R, C, mxy, modes);
        return hipGetLastError();
    }
    return with_blocks(W, [&](auto v) {
        hipLaunchKernelGGL(mode_mix_kernel<decltype(v)::value>, grid, dim3(256), 0, s, A, R, C, mxy, sample, B, modes);
        return hipGetLastError();
    });
}

hipError_t run_mode_back(const float *A, const float *D, const float *R, float *dA, float *dR, int W, long mxy, long mz,
                         int B, hipStream_t s)
{
    if (!mode_covers(W)) return hipErrorInvalidValue;
    const long modes = mz * mxy, sample = 2 * modes * W;
    return with_blocks(W, [&](auto v) {
        hipLaunchKernelGGL(mode_back_kernel<decltype(v)::value>, dim3((unsigned)((modes + 3) / 4)), dim3(256), 0, s, A, D,
                           R, dA, dR, mxy, sample, B, modes);
        return hipGetLastError();
    });
}

} // namespace bec
