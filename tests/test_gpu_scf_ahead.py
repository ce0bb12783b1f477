"""SCF iterations launched ahead of the host's convergence test: the iteration behind
the last one must leave nothing behind, at every end the loop can have."""
import numpy as np
import pytest

from electrostatic_amd import _lib, negf
from electrostatic_amd.workloads import gaussian_bumps

pytestmark = pytest.mark.gpu

SP = dict(Broyden_fraction=0.1, eps_r=3.9, R_ring_nm=0.665, R_image_nm=10.0)


def tubes_of(T, cells, eq_pts=(30, 30, 64), mu=(-1.0, -1.0)):
    return [negf.Tube(num_unitcells=cells, num_modes=1, contact_mu=mu, eq_integration_pts=eq_pts,
                      noneq_integration_pts=(100,), E_zPlus_imag=1e-5, E_valence_min=-10.0, E_pole_max=3.0)
            for _ in range(T)]


def same(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert np.array_equal(np.asarray(x), np.asarray(y))


@pytest.mark.parametrize("cells,mu,steps", [(1, (-1.0, -1.0), 200), (9, (-1.0, -1.1), 200), (68, (-1.0, -1.0), 200),
                                            (9, (-1.0, -1.0), 3)])
def test_single(cells, mu, steps):
    """Ends by convergence and (3 steps) by the step limit; the tube's potential and the
    next bias point start from the same state."""
    runs = []
    for ahead in (True, False):
        tube, = tubes_of(1, cells, mu=mu)
        scf = negf.Scf(tube, Broyden_max_norm=1e-6, Broyden_threshold_maxstep=steps, **SP)
        scf.set_external_potential(gaussian_bumps(tube.N, seed=3, amp=0.3))
        scf.use_graph(ahead)
        out = []
        for V in (0.3, 0.5):
            try:
                out += list(scf.bias_point(V))
            except _lib.NegfError as e:
                out.append(str(e))
            out.append(tube.solve(1)[0])
        runs.append(out)
        scf.close()
        tube.close()
    assert (steps == 3) == isinstance(runs[0][0], str)
    same(*runs)


@pytest.mark.parametrize("T,cells,eq_pts,steps", [(1, 5, (30, 30, 64), 200), (3, 13, (30, 30, 64), 200),
                                                  (2, 5, (400, 400, 400), 200), (3, 13, (30, 30, 64), 8)])
def test_batch(T, cells, eq_pts, steps):
    """Tubes that retire at different iterations; 1200 contour points (more than 16
    partial rows) keep the plan's own row sum; 8 steps end some or all by the limit."""
    runs = []
    for ahead in (True, False):
        tubes = tubes_of(T, cells, eq_pts)
        batch = negf.Batch(tubes)
        scf = negf.BatchScf(batch, Broyden_max_norm=1e-6, Broyden_threshold_maxstep=steps, **SP)
        N = tubes[0].N
        scf.set_external_potential(np.stack([gaussian_bumps(N, seed=t, amp=0.2) for t in range(T)]))
        scf.use_graph(ahead)
        out = []
        for k in range(2):
            scf.set_input_charge(np.zeros((T, N)))
            try:
                out += list(scf.run(np.linspace(0.0, 0.8, T)))
            except _lib.NegfError as e:
                out.append(str(e))
            out.append(scf.get_input_charge())
            out += [t.solve(1)[0] for t in tubes]
        runs.append(out)
        scf.close()
        batch.close()
        for t in tubes:
            t.close()
    assert (steps == 8) == isinstance(runs[0][0], str)
    same(*runs)


@pytest.mark.parametrize("T,cells", [(1, 1), (2, 16), (5, 33)])
def test_input_charge_round_trip(T, cells):
    tubes = tubes_of(T, cells)
    batch = negf.Batch(tubes)
    scf = negf.BatchScf(batch, Broyden_max_norm=1e-6, Broyden_threshold_maxstep=20, **SP)
    n = np.random.default_rng(T).normal(size=(T, tubes[0].N))
    for k in (1.0, -2.0):
        scf.set_input_charge(k * n)
        assert np.array_equal(scf.get_input_charge(), k * n)
    scf.close()
    batch.close()


@pytest.mark.parametrize("cells", [256, 257])
def test_batch_against_single(cells):
    """The last size of the small Broyden update and the first of the general one: both
    loops stop at a residual of 1e-8 e, so their potentials agree to 1e-6 V."""
    V = np.array([0.2, 0.6])
    tubes = tubes_of(2, cells)
    batch = negf.Batch(tubes)
    sp = dict(SP, Broyden_max_norm=1e-8, Broyden_threshold_maxstep=200)
    U_ext = np.stack([gaussian_bumps(tubes[0].N, seed=t, amp=0.2) for t in range(2)])
    scf = negf.BatchScf(batch, **sp)
    scf.set_external_potential(U_ext)
    scf.set_input_charge(np.zeros(U_ext.shape))
    U, Q, it, norms, _ = scf.run(V)
    scf.close()
    batch.close()
    for t in range(2):
        one = negf.Scf(tubes[t], **sp)
        one.set_external_potential(U_ext[t])
        U1, Q1 = one.bias_point(V[t])[:2]
        one.close()
        assert np.abs(U[t] - U1).max() < 1e-6 and np.abs(Q[t] - Q1).max() < 1e-6
