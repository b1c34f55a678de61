// The 2D two-component program (programs/bec_wigner_2d.cpp/wigner.cpp) on the
// GPU: calculate_steady_state (wigner.cpp:196-275) and main_loop
// (wigner.cpp:278-477), FP64.
//
// At these lattices (up to 64 x 64) a whole trajectory fits one workgroup's
// LDS: both components, 64 x 65 complex doubles each (rows padded by one
// element against bank conflicts), 133 KB of the 160 KB.  Each workgroup runs
// its trajectory's entire evolution -- noise, pulses, every split step and the
// measurements; HBM sees only the ground state read at the start and the
// measurements written.  The ground state runs the same way in one workgroup.
//
// The 2D transforms are in place, radix 8 or 4 in registers: a line of n
// points takes one stage (n = 4, 8) or two (n = 16, 32, 64), each thread
// holding one butterfly of each component, and one LDS round trip per stage.
// k-space stays in the digit-reversed order that the in-place stages leave it
// in (freq_of); everything done there is pointwise or a sum.  The pointwise
// steps work on the butterfly registers between two stages, so they cost no
// LDS pass: a split step of a 64 x 64 lattice is six LDS passes (two stages of
// rows and two of columns each way, the first and the last shared with the
// x-space and the k-space factor) where one radix-2 stage per pass took about
// thirty-three.  512 threads: one radix-8 butterfly each at 64 x 64, 256
// registers a thread, so both components, the trap and the kinetic factors
// stay in registers.
//
// Bound: FP64 issue and the LDS latency of two wavefronts per SIMD.  A step of
// 32 trajectories at 64 x 64 takes 15.2 us (82 us with the radix-2 passes), an
// imaginary-time step of the ground state 8.7 us.
//
// Conventions of the program (and of the oracle's restatement): the k-space
// kinetic factor is -k^2 with k = dk i for 2i <= n else dk (i - n),
// dk = pi/xmax, dx = 2 xmax/(n - 1); x -> k is the +i transform over n cells,
// k -> x the unnormalised -i transform; the trap term is mu - r^2/4.
#include <hip/hip_runtime.h>
#include <math.h>

#include "backend2d.hpp"
#include "fastmath.hpp"
#include "fft_reg.hpp"
#include "philox.hpp"

namespace bec {

namespace {

constexpr int THREADS = 512;
constexpr int SCRATCH = THREADS / 64 * 8;   // block_sum: up to 8 sums per wavefront
constexpr int MAXN = 64;
constexpr int LDMAX = MAXN + 1;

// One axis: n points, first radix r1 and second r2 (1: single stage); element
// stride es and line stride ls in LDS; `lines` lines.
struct Axis {
    int n, lg, r1, r2, es, ls, lines, lglines;
};

struct Geo {
    Axis x, y;
    int ld, n;
    double dx, dy, dkx, dky, xmax, ymax;
};

constexpr int first_radix(int lg) { return lg == 2 || lg == 4 ? 4 : 8; }
constexpr int second_radix(int lg) { return lg < 4 ? 1 : lg == 6 ? 8 : 4; }

__device__ __forceinline__ double2 cm(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ __forceinline__ double2 cs(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ __forceinline__ double nrm(double2 a) { return a.x * a.x + a.y * a.y; }

__device__ __forceinline__ double kval(int i, int n, double dk) { return (2 * i > n) ? dk * (i - n) : dk * i; }

// the frequency index held at position p of an axis
__device__ __forceinline__ int freq_of(const Axis &a, int p)
{
    const int sub = a.n / a.r1;
    return p / sub + a.r1 * (p % sub);
}

// the phase factors e^{i x}, e^{i y} of the two components
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

// A thread's butterfly of one stage: `on` when it has one, LDS offset of its
// first element, the stride of the others and the twiddle step j (n / L).
// Consecutive threads take consecutive lines: their addresses differ by the
// padded row (rows) or one element (columns), free of bank conflicts.
struct Fly {
    int off, step, tw;
    bool on;
};

// The thread index as a value the compiler does not see through: what depends on
// it (LDS offsets, coordinates) is computed where it is used instead of being
// held in registers over the whole step, where it would spill.
__device__ __forceinline__ int tid()
{
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

__device__ __forceinline__ Fly fly(const Axis &a, int radix, bool second)
{
    const int t = tid(), line = t & (a.lines - 1), q = t >> a.lglines;
    const int sub = a.n / a.r1;
    Fly f;
    f.on = q < a.n / radix;
    f.off = line * a.ls + (second ? q * radix : q) * a.es;
    f.step = second ? a.es : sub * a.es;
    f.tw = second ? 0 : q;
    return f;
}

// v[k] *= exp(SIGN 2 pi i j k / n): the twiddles of a first stage (tw = exp(-2 pi i k / n))
template <int R, int SIGN> __device__ __forceinline__ void twiddle(double2 (&v)[R], const Fly &f, const double2 *tw)
{
#pragma unroll
    for (int k = 1; k < R; ++k) {
        double2 w = tw[f.tw * k];
        if (SIGN > 0) w.y = -w.y;
        v[k] = cm(v[k], w);
    }
}

template <int R> __device__ __forceinline__ void get(double2 (&v)[R], const Fly &f, const double2 *buf)
{
#pragma unroll
    for (int m = 0; m < R; ++m) v[m] = buf[f.off + f.step * m];
}

template <int R> __device__ __forceinline__ void put(const double2 (&v)[R], const Fly &f, double2 *buf)
{
#pragma unroll
    for (int m = 0; m < R; ++m) buf[f.off + f.step * m] = v[m];
}

// x -> k (SIGN = +1): butterfly, then twiddles; k -> x (SIGN = -1): the reverse
template <int R, int SIGN>
__device__ __forceinline__ void butterfly(double2 (&v)[R], const Fly &f, bool tw, const double2 *table)
{
    if (SIGN < 0 && tw) twiddle<R, SIGN>(v, f, table);
    dft<double, R, SIGN>(v);
    if (SIGN > 0 && tw) twiddle<R, SIGN>(v, f, table);
}

// One buffer after the other (a scheduling barrier keeps them apart): the
// registers hold one butterfly at a time.
template <int R, int SIGN, int NB>
__device__ __forceinline__ void stage_r(const Axis &a, bool second, double2 *const (&buf)[NB], const double2 *tw)
{
    const Fly f = fly(a, R, second);
    if (f.on)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            double2 v[R];
            get<R>(v, f, buf[b]);
            butterfly<R, SIGN>(v, f, !second && a.r2 > 1, tw);
            put<R>(v, f, buf[b]);
            __builtin_amdgcn_sched_barrier(0);
        }
    __syncthreads();
}

template <int SIGN, int NB>
__device__ __forceinline__ void stage(const Axis &a, bool second, double2 *const (&buf)[NB], const double2 *tw)
{
    if ((second ? a.r2 : a.r1) == 8) stage_r<8, SIGN, NB>(a, second, buf, tw);
    else stage_r<4, SIGN, NB>(a, second, buf, tw);
}

// The stages between the first (rows) and the last (columns) one.
template <int NB>
__device__ __forceinline__ void mid_fwd(const Geo &g, double2 *const (&buf)[NB], const double2 *twx, const double2 *twy)
{
    if (g.x.r2 > 1) stage<+1, NB>(g.x, true, buf, twx);
    if (g.y.r2 > 1) stage<+1, NB>(g.y, false, buf, twy);
}

template <int NB>
__device__ __forceinline__ void mid_inv(const Geo &g, double2 *const (&buf)[NB], const double2 *twx, const double2 *twy)
{
    if (g.y.r2 > 1) stage<-1, NB>(g.y, false, buf, twy);
    if (g.x.r2 > 1) stage<-1, NB>(g.x, true, buf, twx);
}

// The transforms between a thread's x-space registers (its butterfly of the
// first row stage, radix RF) and its k-space registers (its butterfly of the
// last column stage, radix RL); unnormalised.
template <int RF, int RL, int NB> struct Fft {
    const Geo &g;
    double2 *const (&buf)[NB];
    const double2 *twx, *twy;
    __device__ __forceinline__ Fft(const Geo &g_, double2 *const (&b_)[NB], const double2 *twx_, const double2 *twy_)
        : g(g_), buf(b_), twx(twx_), twy(twy_)
    {
    }
    __device__ __forceinline__ Fly first() const { return fly(g.x, RF, false); }
    __device__ __forceinline__ Fly last() const { return fly(g.y, RL, g.y.r2 > 1); }
    // whether the thread has x-space values, k-space values
    __device__ __forceinline__ bool has_x() const { return (int)threadIdx.x < g.n / RF; }
    __device__ __forceinline__ bool has_k() const { return (int)threadIdx.x < g.n / RL; }
    __device__ __forceinline__ void to_k(double2 (&x)[NB][RF], double2 (&k)[NB][RL])
    {
        if (has_x()) {
            const Fly f = first();
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                butterfly<RF, +1>(x[b], f, g.x.r2 > 1, twx);
                put<RF>(x[b], f, buf[b]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
        mid_fwd<NB>(g, buf, twx, twy);
        if (has_k()) {
            const Fly f = last();
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                get<RL>(k[b], f, buf[b]);
                butterfly<RL, +1>(k[b], f, false, twy);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            clear<RL>(k);
        }
    }
    __device__ __forceinline__ void to_x(double2 (&k)[NB][RL], double2 (&x)[NB][RF])
    {
        if (has_k()) {
            const Fly f = last();
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                butterfly<RL, -1>(k[b], f, false, twy);
                put<RL>(k[b], f, buf[b]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
        mid_inv<NB>(g, buf, twx, twy);
        if (has_x()) {
            const Fly f = first();
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                get<RF>(x[b], f, buf[b]);
                butterfly<RF, -1>(x[b], f, g.x.r2 > 1, twx);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            clear<RF>(x);
        }
    }
    // a thread without values: defined, so that old registers don't stay live over the transform
    template <int R> static __device__ __forceinline__ void clear(double2 (&v)[NB][R])
    {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int m = 0; m < R; ++m) v[b][m] = make_double2(0.0, 0.0);
    }
    // coordinates of the thread's m-th x-space cell; r^2 there
    __device__ __forceinline__ int cell(int m) const
    {
        const int t = tid(), y = t & (g.y.n - 1), x = (t >> g.y.lg) + (g.x.n / RF) * m;
        return (y << g.x.lg) + x;
    }
    __device__ __forceinline__ double r2(int m) const
    {
        const int c = cell(m), x = c & (g.x.n - 1), y = c >> g.x.lg;
        const double xx = -g.xmax + g.dx * x, yy = -g.ymax + g.dy * y;
        return xx * xx + yy * yy;
    }
    // k^2 of the thread's m-th k-space value
    __device__ __forceinline__ double k2(int m) const
    {
        const int t = tid(), px = t & (g.x.n - 1), q = t >> g.x.lg;
        const int py = g.y.r2 > 1 ? q * RL + m : q + (g.y.n / RL) * m;
        const double kx = kval(freq_of(g.x, px), g.x.n, g.dkx), ky = kval(freq_of(g.y, py), g.y.n, g.dky);
        return kx * kx + ky * ky;
    }
};

// Sums of K doubles over the workgroup (within the waves, then LDS across
// them), in a fixed order; every thread receives the totals.
template <int K> __device__ __forceinline__ void block_sum(double (&v)[K], double *scratch)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const double t = K == 1 ? wave_sum(v[0]) : wave_sums<K>(v);
    if ((lane & 7) == 0 && lane / 8 < K) scratch[wave * K + lane / 8] = t;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < THREADS / 64; ++w) s += scratch[w * K + k];
        v[k] = s;
    }
    __syncthreads();
}

__device__ void make_twiddles(const Geo &g, double2 *twx, double2 *twy)
{
    for (int k = threadIdx.x; k < g.x.n; k += THREADS) {
        double s, c;
        sincospi(-2.0 * k / g.x.n, &s, &c);
        twx[k] = make_double2(c, s);
    }
    for (int k = threadIdx.x; k < g.y.n; k += THREADS) {
        double s, c;
        sincospi(-2.0 * k / g.y.n, &s, &c);
        twy[k] = make_double2(c, s);
    }
    __syncthreads();
}

__device__ Axis make_axis(int n, int es, int ls, int lines)
{
    Axis a;
    a.n = n;
    a.lg = 31 - __clz(n);
    a.r1 = first_radix(a.lg);
    a.r2 = second_radix(a.lg);
    a.es = es;
    a.ls = ls;
    a.lines = lines;
    a.lglines = 31 - __clz(lines);
    return a;
}

__device__ Geo make_geo(const W2dParams &p)
{
    Geo g;
    g.ld = p.nvx + 1;
    g.x = make_axis(p.nvx, 1, g.ld, p.nvy);
    g.y = make_axis(p.nvy, g.ld, 1, p.nvx);
    g.n = p.nvx * p.nvy;
    g.xmax = p.xmax;
    g.ymax = p.ymax;
    g.dx = 2.0 * p.xmax / (p.nvx - 1);
    g.dy = 2.0 * p.ymax / (p.nvy - 1);
    g.dkx = M_PI / p.xmax;
    g.dky = M_PI / p.ymax;
    return g;
}

// H psi of the x-space state ps, H = -lap + r^2/4 + g11 |psi|^2, its Rayleigh
// quotient and <psi, psi>, and the residual ||H psi - mu psi|| / (|mu| ||psi||);
// h returns H psi - mu psi.
template <int RF, int RL>
__device__ __forceinline__ double residual(Fft<RF, RL, 1> &F, const W2dParams &p, const double2 (&ps)[1][RF],
                                           double2 (&h)[1][RF], double *scratch, double *mu_out)
{
    double2 x[1][RF], k[1][RL];
#pragma unroll
    for (int m = 0; m < RF; ++m) x[0][m] = ps[0][m];
    F.to_k(x, k);
    const double inv = 1.0 / F.g.n;
#pragma unroll
    for (int m = 0; m < RL; ++m) k[0][m] = cs(k[0][m], F.k2(m) * inv);
    F.to_x(k, h);
    double s2[2] = {0.0, 0.0};
    if (F.has_x())
#pragma unroll
        for (int m = 0; m < RF; ++m) {
            const double2 v = ps[0][m];
            const double pot = F.r2(m) / 4.0 + p.g11 * nrm(v);
            h[0][m] = make_double2(h[0][m].x + pot * v.x, h[0][m].y + pot * v.y);
            s2[0] += v.x * h[0][m].x + v.y * h[0][m].y;
            s2[1] += nrm(v);
        }
    block_sum<2>(s2, scratch);
    const double mu = s2[0] / s2[1];
    double s1[1] = {0.0};
    if (F.has_x())
#pragma unroll
        for (int m = 0; m < RF; ++m) {
            h[0][m] = make_double2(h[0][m].x - mu * ps[0][m].x, h[0][m].y - mu * ps[0][m].y);
            s1[0] += nrm(h[0][m]);
        }
    block_sum<1>(s1, scratch);
    if (mu_out) *mu_out = mu;
    return sqrt(s1[0] / s2[1]) / fabs(mu);
}

// The tail of both ground states: atoms, x-space state, final residual.
template <int RF, int RL>
__device__ __forceinline__ void finish(Fft<RF, RL, 1> &F, const W2dParams &p, double2 (&ps)[1][RF], double atoms,
                                       int iters, double2 *gs_out, double *rep_out, double *scratch)
{
    double2 h[1][RF];
    if (F.has_x())
#pragma unroll
        for (int m = 0; m < RF; ++m) gs_out[F.cell(m)] = ps[0][m];
    double mu = 0.0;
    const double r = residual<RF, RL>(F, p, ps, h, scratch, &mu);
    if (threadIdx.x == 0) {
        rep_out[0] = atoms * F.g.dx * F.g.dy;
        rep_out[1] = iters;
        rep_out[2] = r;
        rep_out[3] = mu;
    }
}

// calculate_steady_state (wigner.cpp:196-275): uniform n0 start, imaginary
// time with the itmax midpoint iteration; ntG - 1 steps (reference rule) or
// until the residual is below gs_tol.  One workgroup.
template <int RF, int RL>
__global__ __launch_bounds__(THREADS) void w2d_ground_state_kernel(W2dParams p, double2 *gs_out, double *rep_out)
{
    __shared__ double2 A[MAXN * LDMAX];
    __shared__ double2 twx[MAXN], twy[MAXN];
    __shared__ double scratch[SCRATCH];
    const Geo g = make_geo(p);
    make_twiddles(g, twx, twy);
    double2 *const buf[1] = {A};
    Fft<RF, RL, 1> F(g, buf, twx, twy);
    double2 x[1][RF], k[1][RL];
    double pG[RF], kin[RL];
    const double inv = 1.0 / g.n;
#pragma unroll
    for (int m = 0; m < RF; ++m) {
        pG[m] = p.mu - F.r2(m) / 4.0;
        x[0][m] = make_double2(p.n0, 0.0);
    }
#pragma unroll
    for (int m = 0; m < RL; ++m) kin[m] = exp(-F.k2(m) * p.dtG / 2.0);
    F.to_k(x, k);
#pragma unroll
    for (int m = 0; m < RL; ++m) k[0][m] = cs(k[0][m], inv);
    const int total = p.gs_rule == 0 ? p.ntG - 1 : p.gs_max_iter;
    int iters = 0;
    for (int it = 0; it < total; ++it) {
#pragma unroll
        for (int m = 0; m < RL; ++m) k[0][m] = cs(k[0][m], kin[m]);
        F.to_x(k, x);
#pragma unroll
        for (int m = 0; m < RF; ++m) {
            const double2 a1 = x[0][m];
            double2 a = a1;
            double da = 0.0;
            for (int i = 0; i < p.itmax; ++i) {
                da = exp(p.dtG / 2.0 * (pG[m] - p.g11 * nrm(a)));
                a = cs(a1, da);
            }
            x[0][m] = cs(a, da);
        }
        F.to_k(x, k);
#pragma unroll
        for (int m = 0; m < RL; ++m) k[0][m] = cs(k[0][m], kin[m] * inv);
        ++iters;
        if (p.gs_rule == 1) {   // residual of the x-space iterate; the k-space one stays in registers
            double2 kk[1][RL], h[1][RF];
#pragma unroll
            for (int m = 0; m < RL; ++m) kk[0][m] = k[0][m];
            F.to_x(kk, x);
            if (residual<RF, RL>(F, p, x, h, scratch, nullptr) < p.gs_tol) break;   // uniform across the workgroup
        }
    }
    double s1[1] = {0.0};
    if (F.has_k())
#pragma unroll
        for (int m = 0; m < RL; ++m) s1[0] += nrm(k[0][m]);
    block_sum<1>(s1, scratch);
    F.to_x(k, x);
    finish<RF, RL>(F, p, x, s1[0] * g.n, iters, gs_out, rep_out, scratch);
}

// Ground state of n_atoms atoms (gs_rule 2; the program's own loop fixes mu):
// the preconditioned imaginary-time gradient flow
//   psi <- psi - tau P (H - mu) psi + beta (psi - psi_prev),  P = 1/(alpha + k^2),
// renormalised to dx dy sum |psi|^2 = n_atoms after every update, from the
// Thomas-Fermi profile sqrt(max(mu - r^2/4, 0) / g11), alpha = mu, until the
// residual ||H psi - mu psi|| / (|mu| ||psi||) is below gs_tol.  One
// workgroup; the iterate, the previous one and H psi are in registers.
template <int RF, int RL>
__global__ __launch_bounds__(THREADS) void w2d_flow_gs_kernel(W2dParams p, double2 *gs_out, double *rep_out)
{
    __shared__ double2 A[MAXN * LDMAX];
    __shared__ double2 twx[MAXN], twy[MAXN];
    __shared__ double scratch[SCRATCH];
    const Geo g = make_geo(p);
    make_twiddles(g, twx, twy);
    double2 *const buf[1] = {A};
    Fft<RF, RL, 1> F(g, buf, twx, twy);
    double2 x[1][RF], pv[RF], r[1][RF], k[1][RL];
    const double alpha = p.mu > 0 ? p.mu : 1.0, inv = 1.0 / g.n;
    double s0[2] = {0.0, 0.0};
#pragma unroll
    for (int m = 0; m < RF; ++m) {
        double v = p.mu - F.r2(m) / 4.0;
        v = v > 0 ? sqrt(v / p.g11) : 0.0;
        x[0][m] = make_double2(v, 0.0);
        if (F.has_x()) {
            s0[0] += v * v;
            s0[1] += v > 0 ? 1.0 : 0.0;
        }
    }
    block_sum<2>(s0, scratch);
    if (s0[1] == 0.0) {   // no Thomas-Fermi cloud on the lattice: uniform start
#pragma unroll
        for (int m = 0; m < RF; ++m) x[0][m] = make_double2(1.0, 0.0);
        s0[0] = g.n;
    }
    double sc = sqrt(p.n_atoms / (s0[0] * g.dx * g.dy));
#pragma unroll
    for (int m = 0; m < RF; ++m) pv[m] = x[0][m] = cs(x[0][m], sc);
    int iters = 0;
    for (;;) {
        const double res = residual<RF, RL>(F, p, x, r, scratch, nullptr);   // r = (H - mu) psi
        if (!(res == res) || res < p.gs_tol || iters >= p.gs_max_iter) break;   // uniform across the workgroup
        F.to_k(r, k);
#pragma unroll
        for (int m = 0; m < RL; ++m) k[0][m] = cs(k[0][m], inv / (alpha + F.k2(m)));
        F.to_x(k, r);
        double s4[1] = {0.0};
#pragma unroll
        for (int m = 0; m < RF; ++m) {
            const double2 cur = x[0][m], prev = pv[m], d = r[0][m];
            x[0][m] = make_double2(cur.x - p.gs_tau * d.x + p.gs_beta * (cur.x - prev.x),
                                   cur.y - p.gs_tau * d.y + p.gs_beta * (cur.y - prev.y));
            pv[m] = cur;
            if (F.has_x()) s4[0] += nrm(x[0][m]);
        }
        block_sum<1>(s4, scratch);
        sc = sqrt(p.n_atoms / (s4[0] * g.dx * g.dy));
#pragma unroll
        for (int m = 0; m < RF; ++m) x[0][m] = cs(x[0][m], sc);
        ++iters;
    }
    double s1[1] = {0.0};
    if (F.has_x())
#pragma unroll
        for (int m = 0; m < RF; ++m) s1[0] += nrm(x[0][m]);
    block_sum<1>(s1, scratch);
    finish<RF, RL>(F, p, x, s1[0], iters, gs_out, rep_out, scratch);
}

// main_loop (wigner.cpp:278-477) for one trajectory per workgroup.  meas:
// [traj][n_meas][3] = {N1, N2, visibility}; avn: [traj][cells] x-space
// density minus the vacuum term after the last step (may be null).
template <int RF, int RL>
__global__ __launch_bounds__(THREADS) void w2d_ensemble_kernel(W2dParams p, const double2 *gs, double *meas,
                                                               double *avn, uint32_t k0, uint32_t k1)
{
    __shared__ double2 A[MAXN * LDMAX], Bf[MAXN * LDMAX];
    __shared__ double2 twx[MAXN], twy[MAXN];
    __shared__ double scratch[SCRATCH];
    const Geo g = make_geo(p);
    const int traj = blockIdx.x;
    make_twiddles(g, twx, twy);
    double2 *const buf[2] = {A, Bf};
    Fft<RF, RL, 2> F(g, buf, twx, twy);
    double2 x[2][RF], k[2][RL], kw[RL];
    // initial state: ground state + noise (wigner.cpp:315-324); the program's
    // deviation 1/sqrt(dx dy) on top of the 0.5 of the normal deviates
    const double nd = p.noise_dev / 0.5, inv = 1.0 / g.n;
#pragma unroll
    for (int m = 0; m < RF; ++m) {
        x[0][m] = x[1][m] = make_double2(0.0, 0.0);
        if (F.has_x()) {
            const int c = F.cell(m);
            double z[4];
            noise4((uint32_t)c, (uint32_t)traj, 0u, k0, k1, z);
            x[0][m] = make_double2(gs[c].x + p.Va * nd * z[0], gs[c].y + p.Va * nd * z[1]);
            x[1][m] = make_double2(p.Vb * nd * z[2], p.Vb * nd * z[3]);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // kinetic factors exp(+i k^2 dtW/2) of the thread's values
#pragma unroll
    for (int m = 0; m < RL; ++m) {
        double s, co;
        sincos(F.k2(m) * p.dtW / 2.0, &s, &co);
        kw[m] = make_double2(co, s);
        __builtin_amdgcn_sched_barrier(0);
    }
    F.to_k(x, k);
#pragma unroll
    for (int m = 0; m < RL; ++m) {
        k[0][m] = cs(k[0][m], inv);
        k[1][m] = cs(k[1][m], inv);
    }
    const double r2 = sqrt(2.0), V = (p.Va + p.Vb) / 2.0;
    for (int nn = -p.ntW; nn < p.n_meas; ++nn) {
        if (nn > -p.ntW) {
            if (nn == 0)   // first pi/2 pulse (wigner.cpp:341-353)
#pragma unroll
                for (int m = 0; m < RL; ++m) {
                    const double2 a = k[0][m], b = k[1][m];
                    k[1][m] = make_double2((b.x + a.y) / r2, (b.y - a.x) / r2);   // (b - i a)/sqrt 2
                    k[0][m] = make_double2((a.x + b.y) / r2, (a.y - b.x) / r2);   // (a - i b)/sqrt 2
                }
#pragma unroll
            for (int m = 0; m < RL; ++m) {
                k[0][m] = cm(k[0][m], kw[m]);
                k[1][m] = cm(k[1][m], kw[m]);
            }
            F.to_x(k, x);
            if (F.has_x())
#pragma unroll
                for (int m = 0; m < RF; ++m) {
                    const double2 a = x[0][m], b = x[1][m];
                    const double na = nrm(a), nb = nrm(b), base = p.mu - F.r2(m) / 4.0;
                    const double dA = -p.g11 * na - p.g12 * nb + base + 0.5 * p.E;
                    const double dB = -p.g22 * nb - p.g12 * na + base - 0.5 * p.E;
                    double2 ea, eb;
                    phases(-p.dtW * dA, -p.dtW * dB, ea, eb);
                    x[0][m] = cm(a, ea);
                    x[1][m] = cm(b, eb);
                    __builtin_amdgcn_sched_barrier(0);   // one cell after the other: fewer registers
                }
            F.to_k(x, k);
#pragma unroll
            for (int m = 0; m < RL; ++m) {
                const double2 w = cs(kw[m], inv);   // 1/n is a power of two
                k[0][m] = cm(k[0][m], w);
                k[1][m] = cm(k[1][m], w);
            }
        }
        if (nn >= 0) {   // second pulse U^+ and measurement (wigner.cpp:393-425)
            double s[6] = {0, 0, 0, 0, 0, 0};
            if (F.has_k())
#pragma unroll
                for (int m = 0; m < RL; ++m) {
                    const double2 a = k[0][m], b = k[1][m];
                    // |(a + i b)/sqrt 2|^2, |(b + i a)/sqrt 2|^2
                    s[0] += 0.5 * nrm(make_double2(a.x - b.y, a.y + b.x));
                    s[1] += 0.5 * nrm(make_double2(b.x - a.y, b.y + a.x));
                    s[2] += a.x * b.x + a.y * b.y;
                    s[3] += a.x * b.y - a.y * b.x;
                    s[4] += nrm(a);
                    s[5] += nrm(b);
                }
            block_sum<6>(s, scratch);
            if (threadIdx.x == 0) {
                double *m = meas + ((long)traj * p.n_meas + nn) * 3;
                m[0] = g.n * (s[0] * g.dx * g.dy - 0.5 * V);
                m[1] = g.n * (s[1] * g.dx * g.dy - 0.5 * V);
                m[2] = 2.0 * sqrt(s[2] * s[2] + s[3] * s[3]) / (s[4] + s[5]);
            }
        }
    }
    if (avn) {
        F.to_x(k, x);
        if (F.has_x())
#pragma unroll
            for (int m = 0; m < RF; ++m)
                avn[(long)traj * g.n + F.cell(m)] = nrm(x[0][m]) - 0.5 * V / g.dx / g.dy;
    }
}

// Sums over trajectories in trajectory order, the products rounded on their own
// (no contraction), as the program accumulates them: thread t < n_meas sums
// sample t, the next threads the cells of avn.
__global__ __launch_bounds__(256) void w2d_reduce_kernel(int ne, int nm, int cells, const double *meas,
                                                         const double *avn, double *sums, double *avn_sum)
{
#pragma clang fp contract(off)
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < nm) {
        double s[5] = {0, 0, 0, 0, 0};
        for (int j = 0; j < ne; ++j) {
            const double *q = meas + ((long)j * nm + t) * 3;
            s[0] += q[0];
            s[1] += q[1];
            s[2] += q[0] * q[0];
            s[3] += q[1] * q[1];
            s[4] += q[2];
        }
        for (int i = 0; i < 5; ++i) sums[(long)i * nm + t] = s[i];
    } else if (avn && t < nm + cells) {
        double s = 0.0;
#pragma unroll 8
        for (int j = 0; j < ne; ++j) s += avn[(long)j * cells + t - nm];
        avn_sum[t - nm] = s;
    }
}

// the radices of the first row stage and of the last column stage
template <class Fn> hipError_t with_radices(const W2dParams &p, Fn &&f)
{
    const int lx = 31 - __builtin_clz(p.nvx), ly = 31 - __builtin_clz(p.nvy);
    const bool f8 = first_radix(lx) == 8, l8 = (second_radix(ly) > 1 ? second_radix(ly) : first_radix(ly)) == 8;
    using R4 = std::integral_constant<int, 4>;
    using R8 = std::integral_constant<int, 8>;
    if (f8 && l8) f(R8{}, R8{});
    else if (f8) f(R8{}, R4{});
    else if (l8) f(R4{}, R8{});
    else f(R4{}, R4{});
    return hipGetLastError();
}

} // namespace

hipError_t run_w2d_ground_state(const W2dParams &p, double2 *gs_out, double *rep_out, hipStream_t s)
{
    return with_radices(p, [&](auto rf, auto rl) {
        constexpr int RF = decltype(rf)::value, RL = decltype(rl)::value;
        if (p.gs_rule == 2)
            hipLaunchKernelGGL((w2d_flow_gs_kernel<RF, RL>), dim3(1), dim3(THREADS), 0, s, p, gs_out, rep_out);
        else
            hipLaunchKernelGGL((w2d_ground_state_kernel<RF, RL>), dim3(1), dim3(THREADS), 0, s, p, gs_out, rep_out);
    });
}

hipError_t run_w2d_ensemble(const W2dParams &p, const double2 *gs, double *meas, double *avn, hipStream_t s)
{
    const uint32_t k0 = (uint32_t)p.seed, k1 = (uint32_t)(p.seed >> 32);
    return with_radices(p, [&](auto rf, auto rl) {
        constexpr int RF = decltype(rf)::value, RL = decltype(rl)::value;
        hipLaunchKernelGGL((w2d_ensemble_kernel<RF, RL>), dim3((unsigned)p.ne), dim3(THREADS), 0, s, p, gs, meas, avn,
                           k0, k1);
    });
}

hipError_t run_w2d_reduce(const W2dParams &p, const double *meas, const double *avn, double *sums, double *avn_sum,
                          hipStream_t s)
{
    const int cells = p.nvx * p.nvy, threads = p.n_meas + (avn ? cells : 0);
    hipLaunchKernelGGL(w2d_reduce_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, p.ne, p.n_meas,
                       cells, meas, avn, sums, avn_sum);
    return hipGetLastError();
}

} // namespace bec
