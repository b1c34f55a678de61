// C ABI of the 1D program on the GPU (bec_1d_cells, bec_run_1d): validation,
// device buffers, the three launches (kernels1d.hip) and the final statistics
// of programs/bec_wigner_2d.cpp/wigner_1d.cpp:405-413 on the host.
#include <hip/hip_runtime.h>
#include <math.h>

#include <cmath>

#include <vector>

#include "backend1d.hpp"
#include "host_common.hpp"

namespace {

// the largest samples x trajectories product whose per-trajectory samples
// (40 B each) are staged on the device
constexpr long long W1D_MAX_SAMPLES = 1LL << 26;

int cells_1d(const bec_1d_params &p)
{
    if (!(p.zmax > 0) || !(p.dz > 0) || !std::isfinite(p.zmax) || !(p.zmax / p.dz < 1e6)) return -BEC_ERR_INVALID;
    const int nv = 1 + 2 * (int)(p.zmax / p.dz);
    if (nv > bec::W1D_MAX_NV) return -BEC_ERR_SHAPE;
    return nv;
}

int validate_1d(const bec_1d_params &p, int *nv)
{
    const int n = cells_1d(p);
    if (n < 0) return -n;
    if (!(p.dt > 0) || p.ntG < 1 || p.itmax < 0 || p.ntW < 1 || p.ne < 1) return BEC_ERR_INVALID;
    if ((long long)p.ne * p.ntW > W1D_MAX_SAMPLES || p.ne > 0x7fffffff / 2) return BEC_ERR_SHAPE;
    *nv = n;
    return BEC_OK;
}

// The device memory of one call: the results first (one copy back), then the
// per-trajectory values they are reduced from.
struct Slab {
    void *p = nullptr;
    ~Slab() { bec::dev_free(p); }
};

} // namespace

extern "C" int bec_1d_cells(const bec_1d_params *p)
{
    if (!p) return -BEC_ERR_INVALID;
    return cells_1d(*p);
}

extern "C" int bec_run_1d(const bec_1d_params *pp, double *m, double *var, double *vis, double *gs_x, double *avn,
                          double *ntot, bec_1d_report *rep)
{
    if (!pp || !m || !var) return BEC_ERR_INVALID;
    const bec_1d_params p = *pp;
    int n = 0;
    int st = validate_1d(p, &n);
    if (st != BEC_OK) return st;
    const int nt = p.ntW, ne = p.ne;
    hipStream_t s = nullptr;
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return BEC_ERR_HIP;
    struct StreamGuard {
        hipStream_t s;
        ~StreamGuard() { (void)hipStreamDestroy(s); }
    } guard{s};
    // doubles: ground state, report, sums over trajectories, N series | samples and densities per trajectory
    const size_t o_rep = 2 * (size_t)n, o_sums = o_rep + 3, o_avn = o_sums + 5 * (size_t)nt, o_ntot = o_avn + n;
    const size_t n_res = o_ntot + p.ntG, o_meas = n_res, o_av = o_meas + 5 * (size_t)ne * nt;
    Slab slab;
    BEC_HIP(bec::dev_alloc(&slab.p, sizeof(double) * (o_av + (size_t)ne * n)));
    double *d = (double *)slab.p;
    double2 *d_gs = (double2 *)d;
    hipEvent_t e0, e1;
    BEC_HIP(hipEventCreate(&e0));
    BEC_HIP(hipEventCreate(&e1));
    struct EventGuard {
        hipEvent_t a, b;
        ~EventGuard()
        {
            (void)hipEventDestroy(a);
            (void)hipEventDestroy(b);
        }
    } eg{e0, e1};
    BEC_HIP(hipEventRecord(e0, s));
    BEC_HIP(bec::run_w1d_ground_state(p, n, d_gs, d + o_ntot, d + o_rep, s));
    BEC_HIP(bec::run_w1d_ensemble(p, n, d_gs, d + o_meas, d + o_av, s));
    BEC_HIP(bec::run_w1d_reduce(p, n, d + o_meas, d + o_av, d + o_sums, d + o_avn, s));
    BEC_HIP(hipEventRecord(e1, s));
    std::vector<double> res(n_res);
    BEC_HIP(hipMemcpyAsync(res.data(), d, sizeof(double) * n_res, hipMemcpyDeviceToHost, s));
    BEC_HIP(hipStreamSynchronize(s));
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, e0, e1);

    const double *h_rep = &res[o_rep], *h_sums = &res[o_sums], *h_avn = &res[o_avn], *h_ntot = &res[o_ntot];
    // wigner_1d.cpp:405-413 as written: means, then sqrt((<N^2> - <N>^2) / (ne - 1))
    for (int i = 0; i < 2 * nt; ++i) {
        m[i] = h_sums[i] / ne;
        const double v = h_sums[2 * (size_t)nt + i] / ne - m[i] * m[i];
        var[i] = sqrt(v / (ne - 1));
    }
    if (vis)
        for (int i = 0; i < nt; ++i) vis[i] = h_sums[4 * (size_t)nt + i] / ne;
    if (avn)
        for (int c = 0; c < n; ++c) avn[c] = h_avn[c] / ne;
    if (ntot)
        for (int i = 0; i < p.ntG; ++i) ntot[i] = h_ntot[i];
    if (gs_x)
        for (int i = 0; i < 2 * n; ++i) gs_x[i] = res[i];
    if (rep) {
        rep->N0 = h_rep[0];
        rep->nv = n;
        rep->gs_residual = h_rep[1];
        rep->gs_mu = h_rep[2];
        rep->elapsed_ms = ms;
    }
    return BEC_OK;
}
