// Density projections: the ensemble sums of the vacuum-subtracted densities after
// halfPiRotate(alpha) (wigner_kernel.cu:283-286,344-360), projected onto the xy
// and zy planes and the z axis (wigner.cu:279-303,388-410).  FP64 sums in a
// fixed order.
//
// A wavefront owns 64/N planes at fixed z and a few trajectories.  A lane ends
// with a whole row (fixed z and y) in registers, so its zy value needs no
// exchange, and the planes of a workgroup (four wavefronts) are added before
// they leave it; the second kernel adds the partial planes and rows.  One
// wavefront per z that walked every trajectory left the chip idle: 32
// wavefronts at 128 x 16 x 16, 183 us for 64 trajectories and 36 us for one
// thread per output value; split over the trajectories, 2048 wavefronts.
#include <algorithm>

#include "launch.hpp"

namespace bec {

namespace {

constexpr int WAVES = 4;   // wavefronts of a workgroup, each with 64/N planes

// planes of a workgroup and the trajectory splits of a launch: as many splits
// as trajectories while the partial sums stay below 4 MiB (what the fixed
// workspace of bec_projections_static holds beside the results)
int planes_per_wg(const DevGroup &g) { return WAVES * (64 / g.nx); }

long split_doubles(const DevGroup &g)
{
    return 2L * g.nx * g.ny * (g.nz / planes_per_wg(g)) + 2L * g.ny * g.nz;
}

int splits(const DevGroup &g)
{
    const int most = (int)std::max(1L, std::min((long)g.ntraj, (4L << 20) / 8 / split_doubles(g)));
    const int chunk = (g.ntraj + most - 1) / most;
    return (g.ntraj + chunk - 1) / chunk;
}

long result_doubles(const DevGroup &g) { return 2 * ((long)g.nx * g.ny + (long)g.ny * g.nz + g.nz); }

// LDS exchange within one wavefront: its own operations complete in order
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <typename T, int N>
__global__ void __launch_bounds__(64 * WAVES) plane_sums_kernel(const cpx<T> *__restrict__ a,
                                                                const cpx<T> *__restrict__ b, int nz, int ntraj,
                                                                int chunk, double ca, double sa, double vac,
                                                                double *__restrict__ xy_part,
                                                                double *__restrict__ zy_part)
{
    constexpr int PPW = 64 / N, TILE = PPW * N * (N + 1);
    constexpr int BYTES_T = WAVES * TILE * (int)sizeof(cpx<T>), BYTES_S = WAVES * 2 * N * N * 8;
    __shared__ __align__(16) char lds[BYTES_T > BYTES_S ? BYTES_T : BYTES_S];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, pl = lane / N, t = lane % N;
    const int z = (blockIdx.x * WAVES + wave) * PPW + pl;
    cpx<T> *tile = (cpx<T> *)lds + wave * TILE + pl * N * (N + 1);
    const double r = 0.70710678118654752440;
    double acc[2][N];
#pragma unroll
    for (int x = 0; x < N; ++x) acc[0][x] = acc[1][x] = 0.0;
    const int t0 = blockIdx.y * chunk, t1 = min(ntraj, t0 + chunk);
    for (int traj = t0; traj < t1; ++traj) {
        const long base = ((long)traj * nz + z) * (N * N);
        cpx<T> v[2][N];
#pragma unroll
        for (int y = 0; y < N; ++y) {
            v[0][y] = a[base + y * N + t];
            v[1][y] = b[base + y * N + t];
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            dft<T, N, -1>(v[c]);
#pragma unroll
            for (int y = 0; y < N; ++y) tile[y * (N + 1) + t] = v[c][y];
            wave_fence();
#pragma unroll
            for (int x = 0; x < N; ++x) v[c][x] = tile[t * (N + 1) + x];
            wave_fence();
            dft<T, N, -1>(v[c]);
        }
#pragma unroll
        for (int x = 0; x < N; ++x) {
            const double ar = v[0][x].x, ai = v[0][x].y, br = v[1][x].x, bi = v[1][x].y;
            // a' = (a + b (sin - i cos))/sqrt2, b' = (a (-sin - i cos) + b)/sqrt2
            const double anr = (ar + br * sa + bi * ca) * r, ani = (ai + bi * sa - br * ca) * r;
            const double bnr = (-ar * sa + ai * ca + br) * r, bni = (-ai * sa - ar * ca + bi) * r;
            acc[0][x] += anr * anr + ani * ani - vac;
            acc[1][x] += bnr * bnr + bni * bni - vac;
        }
    }
    // the row's sum over x: the zy value of (t, z)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        double s = 0.0;
#pragma unroll
        for (int x = 0; x < N; ++x) s += acc[c][x];
        zy_part[(((long)blockIdx.y * 2 + c) * N + t) * nz + z] = s;
    }
    // the sum of the wavefront's planes, then of the workgroup's
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int x = 0; x < N; ++x) {
            double v = acc[c][x], w = v;
            if (N == 16) {
                swap16(v, w);
                v += w;
                w = v;
            }
            swap32(v, w);
            acc[c][x] = v + w;
        }
    __syncthreads();   // every wavefront is done with its tile
    double *sum = (double *)lds;
    if (pl == 0)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int x = 0; x < N; ++x) sum[((wave * 2 + c) * N + t) * N + x] = acc[c][x];
    __syncthreads();
    double *out = xy_part + ((long)blockIdx.y * gridDim.x + blockIdx.x) * (2 * N * N);
    for (int i = threadIdx.x; i < 2 * N * N; i += 64 * WAVES) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) s += sum[w * 2 * N * N + i];
        out[i] = s;
    }
}

// out = {xy[2][ny][nx], zy[2][ny][nz], axial[2][nz]}: 16 values per workgroup,
// each by 16 threads that take every sixteenth term, combined in order.
__global__ void __launch_bounds__(256) projection_reduce_kernel(const double *__restrict__ xy_part,
                                                                const double *__restrict__ zy_part, int nxy, int ny,
                                                                int nz, int splits, int z_blocks,
                                                                double *__restrict__ out)
{
    __shared__ double part[16][17];
    const int n_xy = 2 * nxy, n_zy = 2 * ny * nz, lo = threadIdx.x & 15, sl = threadIdx.x >> 4;
    const int o = blockIdx.x * 16 + lo;   // the sections are multiples of 16
    double s = 0.0;
    if (o < n_xy) {
#pragma unroll 4
        for (int i = sl; i < splits * z_blocks; i += 16) s += xy_part[(long)i * n_xy + o];
    } else if (o < n_xy + n_zy) {
#pragma unroll 4
        for (int i = sl; i < splits; i += 16) s += zy_part[(long)i * n_zy + o - n_xy];
    } else {
        const int q = o - n_xy - n_zy, c = q / nz, z = q - c * nz;
#pragma unroll 4
        for (int i = sl; i < splits * ny; i += 16) {
            const int sp = i / ny, y = i - sp * ny;
            s += zy_part[(long)sp * n_zy + (long)(c * ny + y) * nz + z];
        }
    }
    part[sl][lo] = s;
    __syncthreads();
    if (sl == 0) {
        double v = 0.0;
#pragma unroll
        for (int i = 0; i < 16; ++i) v += part[i][lo];
        out[o] = v;
    }
}

} // namespace

long projection_doubles(const DevGroup &g) { return result_doubles(g) + splits(g) * split_doubles(g); }
long projection_results(const DevGroup &g) { return result_doubles(g); }

hipError_t run_projections(const DevGroup &g, double alpha, double vac, double *buf, hipStream_t s)
{
    const double ca = cos(alpha), sa = sin(alpha);
    const int sp = splits(g), chunk = (g.ntraj + sp - 1) / sp, zb = g.nz / planes_per_wg(g);
    double *xy_part = buf + result_doubles(g), *zy_part = xy_part + 2L * g.nx * g.ny * zb * sp;
    hipError_t e = dispatch(g, [&](auto Tt, auto Nt, auto) -> hipError_t {
        using T = typename decltype(Tt)::type;
        constexpr int N = decltype(Nt)::value;
        if (g.nz % (WAVES * (64 / N))) return hipErrorInvalidValue;
        hipLaunchKernelGGL((plane_sums_kernel<T, N>), dim3(zb, sp), dim3(64 * WAVES), 0, s, (const cpx<T> *)g.a,
                           (const cpx<T> *)g.b, g.nz, g.ntraj, chunk, ca, sa, vac, xy_part, zy_part);
        return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(projection_reduce_kernel, dim3((unsigned)(result_doubles(g) / 16)), dim3(256), 0, s, xy_part,
                       zy_part, g.nx * g.ny, g.ny, g.nz, sp, zb, buf);
    return hipGetLastError();
}

} // namespace bec
