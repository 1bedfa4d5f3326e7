"""HIP FV Poisson (potential app pressure solve) vs the oracle, whose
iteration counts and solutions are bit-identical to the reference build."""
import numpy as np
import pytest

from _cases import POTENTIAL_CASES
from nebulasem_amd import FVPoisson
from test_oracle import potential_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", POTENTIAL_CASES, ids=[c["name"] for c in POTENTIAL_CASES])
def test_fv_reference_mode_matches_oracle(oracle, tmp_path, case):
    print(f"[gpu] fv {case['name']}", flush=True)
    mesh, U, p, kp, vp = potential_inputs(tmp_path, case)
    om = oracle.OracleMesh(mesh)
    p_or = p.copy()
    st, it, r0, r = oracle.fv_poisson(om, kp, vp.reshape(-1), U.reshape(-1).copy(), p_or, 1e-10, 100000)
    n = mesh.info.nbcs
    fv = FVPoisson(mesh, kp, vp)
    assert fv.structured
    # dyadic spacings (8^3, 16^3) give bitwise-equal couplings per direction;
    # 12x8x6 over the unit cube rounds its face geometry differently per face
    assert fv.uniform == (case["ndiv"] in ((8, 8, 8), (16, 16, 16)))
    kU = np.zeros(len(mesh.boundaries), dtype=np.int32)
    fv.set_rhs_divergence(U[:n], kU, np.zeros((len(kU), 3)))
    x, res, rc = fv.solve(p[:n], mode=0, tol=1e-10)
    print(f"  iters gpu {res.iterations} oracle {it}; res {res.res_ref:.3e} vs {r:.3e}; "
          f"true {res.res_true:.2e}", flush=True)
    assert abs(res.iterations - it) <= 1
    err = np.linalg.norm(x - p_or[:n]) / np.linalg.norm(p_or[:n])
    assert err <= 1e-9, err
    # velocity correction U -= gradf(p): bit-identical to the oracle on the
    # same p (the oracle's matches the reference's output bit for bit)
    u_or = U.reshape(-1).copy()
    oracle.fv_correct_velocity(om, kp, vp.reshape(-1), p_or.copy(), u_or)
    u_gpu = fv.correct_velocity(p_or[:n], U[:n])
    assert np.array_equal(u_gpu.reshape(-1), u_or[:3 * n])
    # and on the device's own solution, within its 1e-9
    u_own = fv.correct_velocity(x, U[:n])
    du = np.linalg.norm(u_own.reshape(-1) - u_or[:3 * n]) / np.linalg.norm(u_or[:3 * n])
    print(f"  corrected U: bit-exact on the oracle's p; {du:.1e} on the device's own p", flush=True)
    assert du <= 1e-8
    fv.close()


def test_fv_modes_reach_true_residual(oracle, tmp_path):
    case = dict(name="pot_24", ndiv=(24, 20, 16), seed=11)
    mesh, U, p, kp, vp = potential_inputs(tmp_path, case)
    n = mesh.info.nbcs
    fv = FVPoisson(mesh, kp, vp)
    fv.set_rhs_divergence(U[:n], np.zeros(len(mesh.boundaries), dtype=np.int32),
                          np.zeros((len(mesh.boundaries), 3)))
    x1, r1, _ = fv.solve(mode=1, tol=1e-10)
    x2, r2, _ = fv.solve(mode=2, tol=1e-10)
    b = fv.rhs()
    for x, r in ((x1, r1), (x2, r2)):
        true = np.linalg.norm(b - fv.apply(x)) / np.linalg.norm(b)
        print(f"  mode iters {r.iterations} outer {r.outer_iterations} true {true:.2e}", flush=True)
        assert true <= 1e-10 * 1.01
    assert np.linalg.norm(x1 - x2) / np.linalg.norm(x1) < 1e-8
    fv.close()


def test_fv_march_with_partial_passes_reaches_true_residual(tmp_path):
    """256 x 256 cells per x-plane make the structured SpMV march 8 chunks of
    5 planes along x (40 planes): each chunk takes one full pass of 4 planes
    and one pass of a single plane.  The true residual is formed by the
    separate row-per-thread apply kernel, so a plane the march skips or
    repeats shows there."""
    print("[gpu] fv march 40x256x256", flush=True)
    case = dict(name="pot_march", ndiv=(40, 256, 256), seed=17)
    mesh, U, p, kp, vp = potential_inputs(tmp_path, case)
    n = mesh.info.nbcs
    fv = FVPoisson(mesh, kp, vp)
    assert fv.structured
    fv.set_rhs_divergence(U[:n], np.zeros(len(mesh.boundaries), dtype=np.int32),
                          np.zeros((len(mesh.boundaries), 3)))
    b = fv.rhs()
    for mode in (1, 2):
        x, r, rc = fv.solve(mode=mode, tol=1e-10)
        true = np.linalg.norm(b - fv.apply(x)) / np.linalg.norm(b)
        print(f"  mode {mode} iters {r.iterations} true {true:.2e} uniform {fv.uniform}", flush=True)
        assert rc == 0
        assert true <= 1e-10 * 1.01
    fv.close()


def test_fv_nonuniform_coefficient_keeps_stored_couplings(oracle, tmp_path):
    """A variable coefficient mu (as piso's rmu) makes the couplings differ,
    so the SpMV reads them; the solution still matches a dense solve of the
    same operator (applied through the device)."""
    case = dict(name="pot_mu", ndiv=(10, 8, 6), seed=13)
    mesh, U, p, kp, vp = potential_inputs(tmp_path, case)
    n = mesh.info.nbcs
    rng = np.random.default_rng(5)
    mu = rng.uniform(0.5, 2.0, size=mesh.info.ncells)
    fv = FVPoisson(mesh, kp, vp, mu=mu)
    assert fv.structured and not fv.uniform
    fv.set_rhs_divergence(U[:n], np.zeros(len(mesh.boundaries), dtype=np.int32),
                          np.zeros((len(mesh.boundaries), 3)))
    x, res, _ = fv.solve(mode=1, tol=1e-12)
    A = np.stack([fv.apply(e) for e in np.eye(n)], axis=1)
    xd = np.linalg.solve(A, fv.rhs())
    err = np.linalg.norm(x - xd) / np.linalg.norm(xd)
    print(f"  variable-mu PCG vs dense solve: {err:.1e} ({res.iterations} it)", flush=True)
    assert err <= 1e-9
    assert np.allclose(A, A.T, rtol=0, atol=1e-12 * np.abs(A).max())
    fv.close()


def test_fv_iteration_limit_reports_not_converged(tmp_path):
    """max_it reached before the tolerance: NSEM_ENOTCONVERGED with the
    iterate and its residuals returned."""
    mesh, U, p, kp, vp = potential_inputs(tmp_path, POTENTIAL_CASES[1])
    n = mesh.info.nbcs
    fv = FVPoisson(mesh, kp, vp)
    fv.set_rhs_divergence(U[:n], np.zeros(len(mesh.boundaries), dtype=np.int32),
                          np.zeros((len(mesh.boundaries), 3)))
    for mode in (0, 1, 2):
        x, res, rc = fv.solve(mode=mode, tol=1e-10, max_it=3, raise_on_error=False)
        print(f"  mode {mode}: rc {rc} iters {res.iterations} res {res.res_ref:.2e} true {res.res_true:.2e}",
              flush=True)
        assert rc == 7
        assert res.iterations <= 3 * max(res.outer_iterations, 1)
        assert np.all(np.isfinite(x)) and res.res_true > 1e-10
    fv.close()


def test_fv_indefinite_operator_reports_breakdown(tmp_path):
    """A negative coefficient (mu = -1) makes lap(p, mu) negative definite,
    so p.Ap < 0 at the first iteration: NSEM_EBREAKDOWN, not a NaN iterate."""
    mesh, U, p, kp, vp = potential_inputs(tmp_path, POTENTIAL_CASES[0])
    n = mesh.info.nbcs
    mu = -np.ones(mesh.info.ncells)
    fv = FVPoisson(mesh, kp, vp, mu=mu)
    fv.set_rhs_divergence(U[:n], np.zeros(len(mesh.boundaries), dtype=np.int32),
                          np.zeros((len(mesh.boundaries), 3)))
    x, res, rc = fv.solve(mode=0, tol=1e-10, max_it=100, raise_on_error=False)
    print(f"  rc {rc} breakdown {res.breakdown} iters {res.iterations}", flush=True)
    assert rc == 6 and res.breakdown == 1
    fv.close()


@pytest.mark.parametrize("ndiv,mu", [((1, 1, 600), False), ((16, 16, 16), True), ((17, 16, 16), True), ((3, 5, 700), True),
                                     ((67, 61, 59), False), ((67, 61, 59), True), ((96, 88, 80), True),
                                     ((128, 128, 128), False)])
def test_fv_on_chip_cg(tmp_path, ndiv, mu):
    """The conjugate gradient held on the chip: one work-group and several,
    boxes cut by the grid's end, one-cell-thick and long grids, held and
    re-read couplings, and the largest system it takes.  The true residual is
    formed by the row-per-thread apply kernel; a cell, face or halo that the
    on-chip kernel misses shows there.  The criterion uses the recursive
    residual, which drifts from the true one by some 1e-15 an iteration of
    |A||x|/|b|: 1e-2 of the tolerance at most on these sizes."""
    print(f"[gpu] fv on chip {ndiv} mu {mu}", flush=True)
    mesh, U, p, kp, vp = potential_inputs(tmp_path, dict(name="pot_chip", ndiv=ndiv, seed=23))
    n = mesh.info.nbcs
    m = np.random.default_rng(29).uniform(0.5, 2.0, size=mesh.info.ncells) if mu else None
    fv = FVPoisson(mesh, kp, vp, mu=m)
    fv.set_rhs_divergence(U[:n], np.zeros(len(mesh.boundaries), dtype=np.int32),
                          np.zeros((len(mesh.boundaries), 3)))
    b = fv.rhs()
    for mode in (1, 2):
        x, r, rc = fv.solve(mode=mode, tol=1e-9)
        y, r2, _ = fv.solve(mode=mode, tol=1e-9)
        true = np.linalg.norm(b - fv.apply(x)) / np.linalg.norm(b)
        print(f"  mode {mode} iters {r.iterations} true {true:.2e} uniform {fv.uniform}", flush=True)
        assert rc == 0 and true <= 1.01e-9
        assert np.array_equal(x, y) and r.iterations == r2.iterations
    fv.close()
