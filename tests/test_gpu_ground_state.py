"""GPU: calculateSteadyState (wigner.cu:84-175) and the residual-targeted solver."""
import numpy as np
import pytest

from tests.helpers import config1_model, gpu_calc, oracle_calc, rel_l2

pytestmark = pytest.mark.gpu


def test_split_step_reference_rule_matches_oracle(bec, oracle):
    m = config1_model(oracle, ne=1)
    c, oc = gpu_calc(bec, **m), oracle_calc(oracle, **m)
    ref, orep = oracle.ground_state(oc, rule=oracle.RULE_REFERENCE, tol=1e-6)
    with bec.Solver(c, precision=0) as s:
        psi, rep, st = s.calculate_steady_state(method=bec.GS_SPLIT_STEP, rule=bec.GS_RULE_REFERENCE,
                                                tol=1e-6, precision=bec.FP64)
    assert st == 0 and rep["converged"]
    assert rep["iterations"] == orep.iterations
    assert rel_l2(psi, ref) < 1e-10
    assert abs(rep["E_ref"] - orep.E_ref) < 1e-9 * abs(orep.E_ref)
    assert abs(rep["mu_ref"] - orep.mu_ref) < 1e-9 * abs(orep.mu_ref)
    assert abs(rep["E"] - orep.E) < 1e-9 * abs(orep.E)
    assert abs(rep["mu"] - orep.mu) < 1e-9 * abs(orep.mu)
    assert abs(rep["residual"] - orep.residual) < 1e-6 * orep.residual


def test_gradient_flow_reaches_residual(bec, oracle):
    m = config1_model(oracle, ne=1)
    c, oc = gpu_calc(bec, **m), oracle_calc(oracle, **m)
    with bec.Solver(c, precision=0) as s:
        psi, rep, st = s.calculate_steady_state(method=bec.GS_GRADIENT, rule=bec.GS_RULE_RESIDUAL, tol=1e-6,
                                                precision=bec.FP64, max_iter=2000)
    assert st == 0 and rep["converged"], rep
    assert rep["residual"] < 1e-6
    r, mu = oracle.residual(oc, psi)     # independent FP64 check of the returned state
    assert r < 1.05e-6
    assert abs(mu - rep["mu"]) < 1e-9 * abs(mu)
    E, mu2, N = oracle.energy_mu(oc, psi)
    assert abs(N - 30000) < 1e-6 * 30000
    assert abs(E - rep["E"]) < 1e-9 * abs(E)


def test_batched_ground_states_match_single(bec, oracle):
    base = config1_model(oracle, ne=1)
    params = [gpu_calc(bec, **dict(base, N=n, fz=fz)) for n, fz in [(20000, 11.96), (45000, 9.0), (8000, 15.0)]]
    out, reps, st = bec.ground_states_batched(params, method=bec.GS_GRADIENT, rule=bec.GS_RULE_RESIDUAL,
                                              tol=1e-6, precision=bec.FP64, max_iter=3000)
    assert st == 0
    for i, p in enumerate(params):
        oc = oracle.derive(oracle.model(**dict(base, N=[20000, 45000, 8000][i], fz=[11.96, 9.0, 15.0][i])))
        r, _ = oracle.residual(oc, out[i])
        assert r < 1.05e-6, (i, r)
        assert reps[i]["converged"]


SETS = [(20000, 11.96), (95000, 6.0), (8000, 19.0), (30000, 8.0), (60000, 14.0), (12000, 10.0), (5000, 20.0), (45000, 9.0)]


def _sets(bec, oracle, nz, n, sets):
    models = [config1_model(oracle, ne=1, nvx=n, nvy=n, nvz=nz, N=N, fz=fz) for N, fz in SETS[:sets]]
    return [gpu_calc(bec, **m) for m in models], [oracle_calc(oracle, **m) for m in models]


@pytest.mark.parametrize("nz,n,sets,tol", [(128, 16, 3, 1e-5), (256, 16, 3, 1e-4), (64, 32, 3, 1e-5), (128, 16, 8, 1e-4),
                                           (64, 16, 8, 1e-5)])
def test_batched_split_step_matches_oracle_set_by_set(bec, oracle, nz, n, sets, tol):
    """Sets of one solve stop at different iterations (2 to 312, in different blocks between two polls), in odd
    and XCD-placed counts; each one's iterations, state and energies are those of its own solve, at the bars
    of the single solve above."""
    params, oc = _sets(bec, oracle, nz, n, sets)
    out, reps, st = bec.ground_states_batched(params, tol=tol, precision=bec.FP64)
    assert st == 0
    ref = [oracle.ground_state(c, rule=oracle.RULE_REFERENCE, tol=tol) for c in oc]
    assert [r["iterations"] for r in reps] == [r.iterations for _, r in ref]
    assert len({r.iterations // 16 for _, r in ref}) > 1
    for psi, rep, (x, orep) in zip(out, reps, ref):
        assert rel_l2(psi, x) < 1e-10
        for key in ("E_ref", "mu_ref", "E", "mu"):
            assert abs(rep[key] - getattr(orep, key)) < 1e-9 * abs(getattr(orep, key)), key


@pytest.mark.parametrize("nz,n", [(128, 16), (64, 32)])
def test_split_step_residual_rule_every_third_iteration(bec, oracle, nz, n):
    """The residual test between fused iterations: its workspace is neither the state the next iteration
    starts from nor the one it returns."""
    params, oc = _sets(bec, oracle, nz, n, 3)
    out, reps, st = bec.ground_states_batched(params, rule=bec.GS_RULE_RESIDUAL, tol=3e-2, check_every=3, precision=bec.FP64)
    assert st == 0
    for psi, rep, c in zip(out, reps, oc):
        x, orep = oracle.ground_state(c, rule=oracle.RULE_RESIDUAL, tol=3e-2, check_every=3)
        assert rep["iterations"] == orep.iterations
        assert rel_l2(psi, x) < 1e-10
        assert abs(rep["residual"] - orep.residual) < 1e-6 * orep.residual


def test_fp32_split_step_follows_the_fp64_one(bec, oracle):
    """40 iterations of eight sets in FP32: about a dozen roundings of 6e-8 a cell and iteration, which the
    contracting steps don't amplify: 40 x sqrt(12) x 6e-8 = 8e-6 at most, were they all to add up."""
    params, _ = _sets(bec, oracle, 128, 16, 8)
    got = [bec.ground_states_batched(params, tol=1e-30, max_iter=40, precision=p) for p in (bec.FP32, bec.FP64)]
    assert all(r["iterations"] == 40 for _, reps, _ in got for r in reps)
    assert rel_l2(got[0][0], got[1][0], axis=(1, 2, 3)).max() < 8e-6
