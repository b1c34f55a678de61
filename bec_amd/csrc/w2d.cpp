// C ABI of the 2D program on the GPU (bec_run_2d): validation, device buffers,
// the two launches (kernels2d.hip) and the ensemble statistics of
// programs/bec_wigner_2d.cpp/wigner.cpp:431-443 on the host.
#include <hip/hip_runtime.h>
#include <math.h>

#include <vector>

#include "backend2d.hpp"
#include "host_common.hpp"

namespace {

bool pow2_in(int v, int lo, int hi) { return v >= lo && v <= hi && (v & (v - 1)) == 0; }

int validate_2d(const bec_2d_params &p)
{
    if (!pow2_in(p.nvx, 4, bec::W2D_MAX_N) || !pow2_in(p.nvy, 4, bec::W2D_MAX_N)) return BEC_ERR_SHAPE;
    if (!(p.xmax > 0) || !(p.ymax > 0) || p.ne < 1 || p.n_meas < 1 || p.ntW < 0 || p.itmax < 0) return BEC_ERR_INVALID;
    if (!(p.dtG > 0) || !(p.dtW > 0)) return BEC_ERR_INVALID;
    if (p.gs_rule < 0 || p.gs_rule > 2) return BEC_ERR_INVALID;
    if (p.gs_rule == 0 && p.ntG < 1) return BEC_ERR_INVALID;
    if (p.gs_rule >= 1 && (p.gs_max_iter < 1 || !(p.gs_tol > 0))) return BEC_ERR_INVALID;
    if (p.gs_rule == 2 && (!(p.n_atoms > 0) || !(p.gs_tau > 0) || !(p.gs_beta >= 0) || !(p.g11 > 0)))
        return BEC_ERR_INVALID;
    if (p.ne > 65535) return BEC_ERR_SHAPE;
    return BEC_OK;
}

// The device memory of one call: the results first (one copy back), then the
// per-trajectory values they are reduced from.
struct Slab {
    void *p = nullptr;
    ~Slab() { bec::dev_free(p); }
};

} // namespace

extern "C" int bec_run_2d(const bec_2d_params *pp, double *m, double *var, double *vis, double *gs_x, double *avn,
                          bec_2d_report *rep)
{
    if (!pp || !m || !var) return BEC_ERR_INVALID;
    const bec_2d_params p = *pp;
    int st = validate_2d(p);
    if (st != BEC_OK) return st;
    const long cells = (long)p.nvx * p.nvy;
    hipStream_t s = nullptr;
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return BEC_ERR_HIP;
    struct StreamGuard {
        hipStream_t s;
        ~StreamGuard() { (void)hipStreamDestroy(s); }
    } guard{s};
    const int nm = p.n_meas, ne = p.ne;
    // doubles: ground state, report, sums over trajectories | samples and densities per trajectory
    const size_t o_rep = 2 * (size_t)cells, o_sums = o_rep + 4, o_avn = o_sums + 5 * (size_t)nm;
    const size_t n_res = o_avn + (avn ? cells : 0), o_meas = n_res, o_av = o_meas + 3 * (size_t)ne * nm;
    Slab slab;
    BEC_HIP(bec::dev_alloc(&slab.p, sizeof(double) * (o_av + (avn ? (size_t)ne * cells : 0))));
    double *d = (double *)slab.p, *d_av = avn ? d + o_av : nullptr;
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
    BEC_HIP(bec::run_w2d_ground_state(p, d_gs, d + o_rep, s));
    BEC_HIP(bec::run_w2d_ensemble(p, d_gs, d + o_meas, d_av, s));
    BEC_HIP(bec::run_w2d_reduce(p, d + o_meas, d_av, d + o_sums, d + o_avn, s));
    BEC_HIP(hipEventRecord(e1, s));
    std::vector<double> res(n_res);
    BEC_HIP(hipMemcpyAsync(res.data(), d, sizeof(double) * n_res, hipMemcpyDeviceToHost, s));
    BEC_HIP(hipStreamSynchronize(s));
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, e0, e1);

    const double *h_rep = &res[o_rep], *h_sums = &res[o_sums];
    // ensemble statistics (wigner.cpp:431-443): means, then sqrt(|<N^2> - <N>^2| / (ne - 1))
    for (int i = 0; i < 2 * nm; ++i) {
        m[i] = h_sums[i] / ne;
        const double v = h_sums[2 * (size_t)nm + i] / ne - m[i] * m[i];
        var[i] = ne > 1 ? sqrt(fabs(v) / (ne - 1)) : 0.0;
    }
    if (vis)
        for (int i = 0; i < nm; ++i) vis[i] = h_sums[4 * (size_t)nm + i] / ne;
    if (avn)
        for (long c = 0; c < cells; ++c) avn[c] = res[o_avn + c] / ne;
    if (gs_x)
        for (long i = 0; i < 2 * cells; ++i) gs_x[i] = res[i];
    if (rep) {
        rep->N0 = h_rep[0];
        rep->gs_iterations = (int)h_rep[1];
        rep->gs_residual = h_rep[2];
        rep->gs_mu = h_rep[3];
        rep->elapsed_ms = ms;
    }
    return BEC_OK;
}
