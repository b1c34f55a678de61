// The 1D two-component program (programs/bec_wigner_2d.cpp/wigner_1d.cpp) on
// the GPU: calculate_steady_state (wigner_1d.cpp:166-243) and main_loop
// (wigner_1d.cpp:245-445), FP64.
//
// A trajectory is one workgroup (one wavefront up to 63 cells).  The program's
// lattice has an odd, generally prime, number n = 2 h + 1 of cells (41), so the
// transforms are direct DFTs, folded about the middle: with
// S_j = x_j + x_{n-j} and D_j = x_j - x_{n-j} (S_0 = x_0),
//   X_k     = sum_{j<=h} S_j cos(2 pi j k / n) +- i sum_{j<=h} D_j sin(2 pi j k / n),
//   X_{n-k} = the same with the other sign,
// so a thread that owns cells k and n - k of one component forms both outputs
// with 4 multiply-adds per j, a quarter of the plain sum's.  It stages its own
// S_k and D_k into LDS; the j loop reads them as broadcasts.  Up to h = 31 the
// thread keeps its cosines and sines in registers; longer lattices step
// the index (j k) mod n into a table in LDS.  The components meet through their
// densities (nonlinear step) and at the pulses, exchanged through LDS.  The
// samples' five sums are reduced together, halving the values a lane carries
// while the lanes combine, and the square root and division of a sample wait
// until the run is over, when the lanes do them in parallel.
//
// Conventions of the program (and of the oracle's restatement): the k-space
// factor is -k^2 with k = dk j for 2j <= nv else dk (j - nv), dk = pi/zmax;
// x -> k is the +i transform over nv cells, k -> x the unnormalised -i
// transform; the trap term is mu - z^2/4 with z = -zmax + dz j.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include "backend1d.hpp"
#include "fastmath.hpp"
#include "fft_reg.hpp"
#include "philox.hpp"

namespace bec {

namespace {

constexpr int MAXNV = W1D_MAX_NV;

__device__ __forceinline__ double2 cm(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
// a (b + lo), lo below the rounding of b
__device__ __forceinline__ double2 cm_ext(double2 a, double2 b, double2 lo)
{
    return make_double2(fma(a.x, b.x, fma(-a.y, b.y, fma(a.x, lo.x, -(a.y * lo.y)))),
                        fma(a.x, b.y, fma(a.y, b.x, fma(a.x, lo.y, a.y * lo.x))));
}
__device__ __forceinline__ double2 cs(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ __forceinline__ double nrm(double2 a) { return a.x * a.x + a.y * a.y; }

__device__ __forceinline__ double kval(int j, int n, double dk) { return (2 * j > n) ? dk * (j - n) : dk * j; }

// the phase factors e^{i x}, e^{i y} (both at once: two independent chains)
__device__ __forceinline__ void phases(double x, double y, double2 &u, double2 &v)
{
    if (fmax(fabs(x), fabs(y)) < DSINCOS_MAX) {
        fast_sincos_f64(x, &u.y, &u.x);
        fast_sincos_f64(y, &v.y, &v.x);
    } else {
        sincos(x, &u.y, &u.x);
        sincos(y, &v.y, &v.x);
    }
}

// A thread's share of a line of n = 2 h + 1 values of NC components: the pair
// (k, n - k) of component c (k = 0 alone), for the first NC (h + 1) threads.
struct Line {
    int n, h, hs, k, c;   // hs: stride between the components' LDS rows (odd: their broadcasts meet no bank twice)
    bool on, two;         // has a pair; has a second cell
    double2 *S, *D;       // [NC][hs]
    const double2 *tw;    // (cos, sin)(2 pi m / n), m < n
};

// LDS row of S or D: h + 1 values and zeros up to a (non-zero) multiple of eight, an odd length
__host__ __device__ constexpr int row_len(int n) { return (n < 2 ? 8 : (n / 2 + 7) & ~7) + 1; }

// LDS: the factor table, then S and D (one row of each per component).
template <int NC> __device__ __forceinline__ Line make_line(int n, double2 *lds)
{
    Line l;
    l.n = n;
    l.h = n >> 1;
    l.hs = row_len(n);
    l.c = NC > 1 && (int)threadIdx.x > l.h ? 1 : 0;
    l.k = (int)threadIdx.x - l.c * (l.h + 1);
    l.on = l.k <= l.h;
    l.two = l.on && l.k > 0;
    l.tw = lds;
    l.S = lds + n;
    l.D = l.S + NC * l.hs;
    for (int m = threadIdx.x; m < n; m += blockDim.x) {
        double s, c;
        unit_root(m, n, &c, &s);
        lds[m] = make_double2(c, s);
    }
    for (int m = threadIdx.x; m < 2 * NC * l.hs; m += blockDim.x) l.S[m] = make_double2(0.0, 0.0);
    if (!l.on) l.k = 0;
    __syncthreads();
    return l;
}

// The cosines and sines of a thread's output pair, read once and held in
// registers for lines of h <= H (H = 0: read from the table every time).
template <int H> struct Factors {
    double c[H + 1], s[H + 1];
    __device__ __forceinline__ void load(const Line &l)
    {
        if constexpr (H > 0) {
            int idx = 0;
#pragma unroll
            for (int j = 1; j <= H; ++j) {
                idx += l.k;
                idx -= idx >= l.n ? l.n : 0;
                const double2 w = l.tw[idx];
                c[j] = w.x;
                s[j] = w.y;
            }
        }
    }
};

// (x_k, x_{n-k}) <- sum_j x_j exp(SIGN 2 pi i j k / n) of the thread's pair
template <int SIGN, int H>
__device__ __forceinline__ void dft_line(const Line &l, const Factors<H> &f, double2 &x, double2 &y)
{
    if (l.on) {
        l.S[l.c * l.hs + l.k] = l.two ? make_double2(x.x + y.x, x.y + y.y) : x;
        l.D[l.c * l.hs + l.k] = make_double2(x.x - y.x, x.y - y.y);
    }
    __syncthreads();
    const double2 *S = l.S + l.c * l.hs, *D = l.D + l.c * l.hs;
    double2 e = S[0], o = make_double2(0.0, 0.0);
    auto add = [&](double2 sj, double2 dj, double c, double s) {
        e.x = fma(sj.x, c, e.x);
        e.y = fma(sj.y, c, e.y);
        o.x = fma(dj.x, s, o.x);
        o.y = fma(dj.y, s, o.y);
    };
    if constexpr (H > 0) {
        // straight line over H terms (the rows end in zeros), so that the reads run ahead of the sums
#pragma unroll
        for (int j = 1; j <= H; ++j) add(S[j], D[j], f.c[j], f.s[j]);
    } else {
        int idx = 0;
#pragma unroll 8
        for (int j = 1; j <= l.h; ++j) {
            idx += l.k;
            idx -= idx >= l.n ? l.n : 0;
            const double2 w = l.tw[idx];
            add(S[j], D[j], w.x, w.y);
        }
    }
    if (SIGN > 0) {
        x = make_double2(e.x - o.y, e.y + o.x);
        y = make_double2(e.x + o.y, e.y - o.x);
    } else {
        x = make_double2(e.x + o.y, e.y - o.x);
        y = make_double2(e.x - o.y, e.y + o.x);
    }
    __syncthreads();   // the staging rows may be overwritten
}

// Sums of K <= 8 values over the workgroup, in a fixed order; thread t returns
// sum t / 8 (in every wave).
template <int K> __device__ __forceinline__ double block_sums(const double (&v)[K], double *scratch)
{
    const double t = wave_sums<K>(v);
    const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
    if (waves == 1) return t;
    if ((lane & 7) == 0) scratch[threadIdx.x >> 3] = t;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < waves; ++w) s += scratch[w * 8 + (lane >> 3)];
    __syncthreads();
    return s;
}

// the sum of one value, in every thread
__device__ __forceinline__ double block_sum(double x, double *scratch)
{
    const double t = wave_sum(x);
    const int waves = blockDim.x >> 6;
    if (waves == 1) return t;
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = t;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < waves; ++w) s += scratch[w];
    __syncthreads();
    return s;
}

// calculate_steady_state (wigner_1d.cpp:166-243): uniform n0 start, ntG - 1
// imaginary-time steps with the itmax midpoint iteration, the N series after
// each pass; then the residual of the x-space result.  One workgroup.
template <int H>
__global__ __launch_bounds__(H ? 64 : 256) void w1d_ground_state_kernel(W1dParams p, int n, double2 *gs_out, double *ntot,
                                                               double *rep_out)
{
    extern __shared__ double2 lds[];
    __shared__ double scratch[32];
    const Line l = make_line<1>(n, lds);
    Factors<H> f;
    f.load(l);
    const double dk = M_PI / p.zmax, inv = 1.0 / n;
    const double kv = kval(l.k, n, dk), k2 = kv * kv, propG = exp(-k2 * p.dt / 2.0);   // the same for n - k
    const double z0 = -p.zmax + p.dz * l.k, z1 = -p.zmax + p.dz * (n - l.k);
    const double pG0 = p.mu - z0 * z0 / 4.0, pG1 = p.mu - z1 * z1 / 4.0;
    double2 a = make_double2(l.on ? p.n0 : 0.0, 0.0), b = make_double2(l.two ? p.n0 : 0.0, 0.0);
    auto to_k = [&](double2 &u, double2 &v) {
        dft_line<+1, H>(l, f, u, v);
        u = cs(u, inv);
        v = l.two ? cs(v, inv) : make_double2(0.0, 0.0);
    };
    auto to_x = [&](double2 &u, double2 &v) {
        dft_line<-1, H>(l, f, u, v);
        if (!l.two) v = make_double2(0.0, 0.0);
    };
    auto step = [&](double2 a1, double pG) {
        double2 v = a1;
        double da = 0.0;
        for (int i = 0; i < p.itmax; ++i) {
            da = exp(p.dt / 2.0 * (pG - p.g11 * nrm(v)));
            v = cs(a1, da);
        }
        return cs(v, da);
    };
    to_k(a, b);
    double N0 = 0.0;
    for (int it = 0; it < p.ntG; ++it) {
        if (it > 0) {
            a = cs(a, propG);
            b = cs(b, propG);
            to_x(a, b);
            a = step(a, pG0);
            b = step(b, pG1);
            to_k(a, b);
            a = cs(a, propG);
            b = cs(b, propG);
        }
        N0 = block_sum(l.on ? nrm(a) + nrm(b) : 0.0, scratch) * p.dz * n;
        if (ntot && threadIdx.x == 0) ntot[it] = N0;
    }
    to_x(a, b);
    if (l.on) gs_out[l.k] = a;
    if (l.two) gs_out[n - l.k] = b;
    // residual of (-d^2/dz^2 + z^2/4 + g11 |psi|^2) psi = mu psi
    double2 h0 = a, h1 = b;
    to_k(h0, h1);
    h0 = cs(h0, k2);
    h1 = cs(h1, k2);
    to_x(h0, h1);
    const double v0 = (p.mu - pG0) + p.g11 * nrm(a), v1 = (p.mu - pG1) + p.g11 * nrm(b);
    h0 = make_double2(h0.x + v0 * a.x, h0.y + v0 * a.y);
    h1 = make_double2(h1.x + v1 * b.x, h1.y + v1 * b.y);
    const double num = block_sum(l.on ? a.x * h0.x + a.y * h0.y + (l.two ? b.x * h1.x + b.y * h1.y : 0.0) : 0.0, scratch);
    const double den = block_sum(l.on ? nrm(a) + (l.two ? nrm(b) : 0.0) : 0.0, scratch);
    const double mu = num / den;
    const double r0 = nrm(make_double2(h0.x - mu * a.x, h0.y - mu * a.y));
    const double r1 = nrm(make_double2(h1.x - mu * b.x, h1.y - mu * b.y));
    const double rr = block_sum(l.on ? r0 + (l.two ? r1 : 0.0) : 0.0, scratch);
    if (threadIdx.x == 0) {
        rep_out[0] = N0;
        rep_out[1] = sqrt(rr / den) / fabs(mu);
        rep_out[2] = mu;
    }
}

// main_loop (wigner_1d.cpp:245-445) for one trajectory per workgroup.  meas:
// [traj][ntW][5]; {N1, N2, visibility} of every sample in the first three on
// return (the run stores the five sums they are made of); avn: [traj][nv]
// x-space density minus the vacuum term after the last step.
template <int H>
__global__ __launch_bounds__(H ? 64 : 512) void w1d_ensemble_kernel(W1dParams p, int n, const double2 *gs, double *meas,
                                                           double *avn, uint32_t k0, uint32_t k1, int first)
{
    extern __shared__ double2 lds[];
    __shared__ double scratch[64];
    const int traj = first + blockIdx.x;
    const Line l = make_line<2>(n, lds);
    Factors<H> f;
    f.load(l);
    const double dk = M_PI / p.zmax, nd = p.noise_dev / 0.5, inv = 1.0 / n;
    const double kv = kval(l.k, n, dk);   // k^2 is the same for n - k
    double sn, co;
    sincos(kv * kv * p.dt / 2.0, &sn, &co);
    const double2 kw = make_double2(co, sn);   // exp(+i k^2 dt/2)
    const double2 kwn = cs(kw, inv);
    // What kwn leaves of kw / (n |kw|^2): the roundings of the product, of 1 / n and of
    // kw's modulus, which every step applies again to the same mode.  With it and the
    // factors of unit_root the norm drifts by at most 4e-17 a step at 21 to 511 cells
    // (3.2e-16 without both, at 21), for 1% of the time of 20 trajectories of 41 cells.
    const double c2 = co * co, s2 = sn * sn;   // |kw|^2 - 1, exactly but for the last sum
    const double mod = (fmax(c2, s2) - 1.0) + fmin(c2, s2) + (fma(co, co, -c2) + fma(sn, sn, -s2));
    const double inv_lo = fma(-inv, (double)n, 1.0) * inv;
    const double2 kwl = make_double2(fma(co, inv, -kwn.x) + co * inv_lo - kwn.x * mod,
                                     fma(sn, inv, -kwn.y) + sn * inv_lo - kwn.y * mod);
    const double z0 = -p.zmax + p.dz * l.k, z1 = -p.zmax + p.dz * (n - l.k);
    const double base0 = p.mu - z0 * z0 / 4.0, base1 = p.mu - z1 * z1 / 4.0;
    const double gown = l.c ? p.g22 : p.g11, det = l.c ? -0.5 * p.E : 0.5 * p.E;
    // initial state: ground state + noise in x-space (:281-290), then to k-space
    auto start = [&](int cell) {
        double e[4];
        noise4((uint32_t)cell, (uint32_t)traj, 0u, k0, k1, e);
        if (l.c) return make_double2(p.Vb * nd * e[2], p.Vb * nd * e[3]);
        const double2 g = gs[cell];
        return make_double2(g.x + p.Va * nd * e[0], g.y + p.Va * nd * e[1]);
    };
    const double2 zero = make_double2(0.0, 0.0);
    double2 x = l.on ? start(l.k) : zero, y = l.two ? start(n - l.k) : zero;
    dft_line<+1, H>(l, f, x, y);
    x = cs(x, inv);
    y = l.two ? cs(y, inv) : zero;
    // the other component's pair, through the staging rows
    auto other = [&](double2 u, double2 v, double2 &ou, double2 &ov) {
        if (l.on) {
            l.S[l.c * l.hs + l.k] = u;
            l.D[l.c * l.hs + l.k] = v;
        }
        __syncthreads();
        ou = l.S[(1 - l.c) * l.hs + l.k];
        ov = l.D[(1 - l.c) * l.hs + l.k];
        __syncthreads();
    };
    const double r2 = sqrt(2.0), V = (p.Va + p.Vb) / 2.0;
    double *const mt = meas + (long)traj * p.ntW * 5;
    for (int nn = -p.ntW; nn < p.ntW; ++nn) {
        if (nn > -p.ntW) {
            if (nn == 0) {   // pi/2 pulse (:308-318): (a - i b)/sqrt 2, (b - i a)/sqrt 2
                double2 u, v;
                other(x, y, u, v);
                x = make_double2((x.x + u.y) / r2, (x.y - u.x) / r2);
                y = make_double2((y.x + v.y) / r2, (y.y - v.x) / r2);
            }
            x = cm(x, kw);
            y = cm(y, kw);
            dft_line<-1, H>(l, f, x, y);
            // single-shot nonlinear step (:331-337)
            const double n0 = nrm(x), n1 = nrm(y);
            double2 on, unused;
            other(make_double2(n0, n1), zero, on, unused);
            double2 e0, e1;
            phases(-p.dt * (-gown * n0 - p.g12 * on.x + base0 + det), -p.dt * (-gown * n1 - p.g12 * on.y + base1 + det),
                   e0, e1);
            x = cm(x, e0);
            y = l.two ? cm(y, e1) : zero;
            dft_line<+1, H>(l, f, x, y);
            x = cm_ext(x, kwn, kwl);
            y = l.two ? cm_ext(y, kwn, kwl) : zero;
        }
        if (nn >= 0) {   // second pulse U^+ and measurement in k-space (:358-391)
            double2 u, v;
            other(x, y, u, v);
            double s[5] = {0, 0, 0, 0, 0};
            if (l.on) {
                // (own + i other)/sqrt 2 is the rotated component of both lines
                const double2 q0 = make_double2(x.x - u.y, x.y + u.x), q1 = make_double2(y.x - v.y, y.y + v.x);
                const double rot = 0.5 * (nrm(q0) + nrm(q1));
                s[0] = l.c ? 0.0 : rot;
                s[1] = l.c ? rot : 0.0;
                if (!l.c) {
                    s[2] = x.x * u.x + x.y * u.y + y.x * v.x + y.y * v.y;
                    s[3] = x.x * u.y - x.y * u.x + y.x * v.y - y.y * v.x;
                }
                s[4] = nrm(x) + nrm(y);
            }
            const double t = block_sums<5>(s, scratch);
            if (threadIdx.x < 40 && (threadIdx.x & 7) == 0) mt[(long)nn * 5 + (threadIdx.x >> 3)] = t;
        }
    }
    // mean density after the last step (:396-400), of component a
    dft_line<-1, H>(l, f, x, y);
    if (l.c == 0) {
        if (l.on) avn[(long)traj * n + l.k] = nrm(x) - 0.5 * V / p.dz;
        if (l.two) avn[(long)traj * n + n - l.k] = nrm(y) - 0.5 * V / p.dz;
    }
    __syncthreads();   // the sums are written
    for (int t = threadIdx.x; t < p.ntW; t += blockDim.x) {
        double *m = mt + (long)t * 5;
        const double q[5] = {m[0], m[1], m[2], m[3], m[4]};
        m[0] = n * (q[0] * p.dz - 0.5 * V);
        m[1] = n * (q[1] * p.dz - 0.5 * V);
        m[2] = 2.0 * sqrt(q[2] * q[2] + q[3] * q[3]) / q[4];
    }
}

// Sums over trajectories in trajectory order (the order the program
// accumulates them in): thread t < ntW sums sample t, the next nv threads the
// cells of avn.
__global__ __launch_bounds__(256) void w1d_reduce_kernel(int ne, int ntW, int n, const double *meas, const double *avn,
                                                         double *sums, double *avn_sum)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < ntW) {
        double s[5] = {0, 0, 0, 0, 0};
        for (int j = 0; j < ne; ++j) {
            const double *q = meas + ((long)j * ntW + t) * 5;
            s[0] += q[0];
            s[1] += q[1];
            s[2] += q[0] * q[0];
            s[3] += q[1] * q[1];
            s[4] += q[2];
        }
        for (int i = 0; i < 5; ++i) sums[(long)i * ntW + t] = s[i];
    } else if (t < ntW + n) {
        const int c = t - ntW;
        double s = 0.0;
        for (int j = 0; j < ne; ++j) s += avn[(long)j * n + c];
        avn_sum[c] = s;
    }
}

// the factor table, then the rows S and D of every component
size_t lds_bytes(int n, int nc) { return sizeof(double2) * (n + 2 * (size_t)nc * row_len(n)); }

// threads of a workgroup: one per pair and component, whole wavefronts
int threads_for(int n, int nc) { return (nc * (n / 2 + 1) + 63) / 64 * 64; }

} // namespace

// Lines of h <= 31 run in one wavefront (both components) with their DFT
// factors in registers, 32 of them per 8 terms; longer ones read the table.
template <class Fn> static hipError_t with_terms(int n, Fn &&f)
{
    const int h = n / 2;
    if (n > MAXNV) return hipErrorInvalidValue;
    if (h <= 8) return f(std::integral_constant<int, 8>{});
    if (h <= 16) return f(std::integral_constant<int, 16>{});
    if (h <= 24) return f(std::integral_constant<int, 24>{});
    if (h <= 31) return f(std::integral_constant<int, 32>{});
    return f(std::integral_constant<int, 0>{});
}

hipError_t run_w1d_ground_state(const W1dParams &p, int n, double2 *gs_out, double *ntot, double *rep_out,
                                hipStream_t s)
{
    return with_terms(n, [&](auto Ht) {
        constexpr int H = decltype(Ht)::value;
        hipLaunchKernelGGL(w1d_ground_state_kernel<H>, dim3(1), dim3(threads_for(n, 1)), lds_bytes(n, 1), s, p, n, gs_out,
                           ntot, rep_out);
        return hipGetLastError();
    });
}

hipError_t run_w1d_ensemble(const W1dParams &p, int n, const double2 *gs, double *meas, double *avn, hipStream_t s)
{
    const uint32_t k0 = (uint32_t)p.seed, k1 = (uint32_t)(p.seed >> 32);
    return with_terms(n, [&](auto Ht) {
        constexpr int H = decltype(Ht)::value;
        // a launch holds less than 2^32 threads: 8.4 million trajectories of 511 cells
        const int threads = threads_for(n, 2), most = (int)(0xffffffffL / threads);
        hipError_t e = hipSuccess;
        for (int first = 0; first < p.ne && e == hipSuccess; first += most) {
            hipLaunchKernelGGL(w1d_ensemble_kernel<H>, dim3((unsigned)std::min(most, p.ne - first)), dim3(threads),
                               lds_bytes(n, 2), s, p, n, gs, meas, avn, k0, k1, first);
            e = hipGetLastError();
        }
        return e;
    });
}

hipError_t run_w1d_reduce(const W1dParams &p, int n, const double *meas, const double *avn, double *sums,
                          double *avn_sum, hipStream_t s)
{
    const int threads = p.ntW + n;
    hipLaunchKernelGGL(w1d_reduce_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, p.ne, p.ntW, n,
                       meas, avn, sums, avn_sum);
    return hipGetLastError();
}

} // namespace bec
