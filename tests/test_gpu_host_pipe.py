"""State transfers between the caller's arrays and the device: one chunk, one
thread's chunks and several threads' (the copies change form at 512 KiB and at
8 MiB), a last chunk that is cut, and non-finite results.  The values are
moved, so they come back bit for bit; the conserved form of a primitive state
is the same few FP64 operations on the device as here."""
import numpy as np
import pytest

from nebulasem_amd import DGEuler, Mesh, NsemError, euler_params

pytestmark = pytest.mark.gpu

CORNERS = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]


def make(ndiv):
    pts = np.array(CORNERS) * 1000.0
    faces = [(0, 1, 2, 3), (4, 5, 6, 7), (0, 1, 5, 4), (3, 2, 6, 7), (0, 3, 7, 4), (1, 2, 6, 5)]
    mesh = Mesh.box(pts, ndiv, patches=[("wall", [tuple(pts[i]) for i in f]) for f in faces], order=(3, 3, 3))
    return DGEuler(mesh, euler_params(1e-3), np.array([[0, 1, 0, 0]], dtype=np.int32), np.zeros((1, 6)))


@pytest.mark.parametrize("ndiv", [(1, 1, 1), (4, 4, 4), (8, 7, 5), (16, 15, 13), (24, 23, 19)])
def test_states_come_back_bit_for_bit(ndiv):
    print(f"[gpu] host pipe {ndiv}", flush=True)
    dg = make(ndiv)
    rng = np.random.default_rng(3)
    nb = dg.nb
    q = (rng.standard_normal(nb), rng.standard_normal(3 * nb), rng.standard_normal(nb))
    for _ in range(2):
        dg.set_conserved(*q)
        for a, b in zip(dg.get_conserved(), q):
            assert np.array_equal(a, b)
    _, rr = dg.background()
    rho, U, T, p = rr + 0.01 * q[0], q[1], q[2], rng.standard_normal(nb)
    dg.set_state(rho, U, T, p)
    for a, b in zip(dg.get_state(), (rho, U, T, p)):
        assert np.array_equal(a, b)
    rp, m, tp = dg.get_conserved()
    assert np.array_equal(rp, rho - rr)
    assert np.array_equal(m, np.repeat(rho, 3) * U)
    assert np.array_equal(tp, rho * (T + 300.0) - rr * 300.0)
    dg.close()


def test_non_finite_results_are_reported():
    print("[gpu] host pipe non-finite", flush=True)
    dg = make((4, 4, 4))
    nb = dg.nb
    z = np.zeros(nb)
    dg.set_conserved(z, np.zeros(3 * nb), z)
    lam = np.zeros((5, nb))
    lam[4, nb - 1] = np.inf
    with pytest.raises(NsemError) as e:
        dg.rk3_adjoint(1, lam)
    assert e.value.code == 5
    dg.set_conserved(z, np.zeros(3 * nb), z)
    bad = z.copy()
    bad[7] = np.nan
    dg.set_conserved(bad, np.zeros(3 * nb), z)
    with pytest.raises(NsemError) as e:
        dg.rk3_steps(1, 64)
    assert e.value.code == 5
    # the flag is taken with the error, and set anew by the next state only
    dg.set_conserved(z, np.zeros(3 * nb), z)
    dg.rk3_steps(1, 64)
    dg.close()
