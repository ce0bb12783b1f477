"""A gate voltage or charge that is not a number ends a self-consistent run of many tubes with
the non-finite error, at the first iteration that meets it, and is never reported as
converged (a maximum norm formed with fmax reads 0 there)."""
import numpy as np
import pytest

from electrostatic_amd import _lib, negf
from electrostatic_amd.surrogate import Surrogate
from electrostatic_amd.workloads import gaussian_bumps

pytestmark = pytest.mark.gpu

ENAN = 5


class Setup:
    """T equal tubes, their batch and its SCF."""

    def __init__(self, T, cells, norm_type=0, max_norm=1e-6):
        self.tubes = [negf.Tube(num_unitcells=cells, num_modes=1, contact_mu=(-1.0, -1.0),
                                eq_integration_pts=(30, 30, 64), noneq_integration_pts=(100,), E_zPlus_imag=1e-5,
                                E_valence_min=-10.0, E_pole_max=3.0) for _ in range(T)]
        self.batch = negf.Batch(self.tubes)
        self.scf = negf.BatchScf(self.batch, Broyden_fraction=0.1, Broyden_max_norm=max_norm,
                                 Broyden_threshold_maxstep=200, Broyden_norm_type=norm_type, eps_r=3.9,
                                 R_ring_nm=0.665, R_image_nm=10.0)
        self.T, self.N = T, self.tubes[0].N
        self.U_ext = np.stack([gaussian_bumps(self.N, seed=t, amp=0.2) for t in range(T)])
        self.V = np.linspace(0.1, 0.8, T)
        self.scf.set_external_potential(self.U_ext)
        self.scf.set_input_charge(np.zeros((T, self.N)))

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.scf.close()
        self.batch.close()
        for t in self.tubes:
            t.close()


# 20 and 1028 sites: the Broyden update of at most 1024 sites and the general one
@pytest.mark.parametrize("cells", [5, 257])
@pytest.mark.parametrize("where", ["gate", "charge"])
@pytest.mark.parametrize("ahead", [True, False])
def test_nan_in_one_tube(dev, cells, where, ahead):
    T = 3
    with Setup(T, cells) as s:
        s.scf.use_graph(ahead)
        V, n = s.V.copy(), np.zeros((T, s.N))
        if where == "gate":
            V[1] = np.nan
        else:
            n[1, 3] = np.nan
        s.scf.set_input_charge(n)
        with pytest.raises(_lib.NegfError) as e:
            s.scf.run(V)
        assert e.value.code == ENAN and "tube 1 at iteration 1" in str(e.value)


@pytest.mark.parametrize("norm_type,max_norm", [(0, 1e-6), (1, 1e-3)])
def test_both_norms(dev, norm_type, max_norm):
    """The absolute and the relative norm see it; sound tubes converge with both."""
    with Setup(2, 5, norm_type, max_norm) as s:
        U, Q, it, norms, _ = s.scf.run(s.V)
        assert np.all(it > 1) and np.all(norms <= max_norm) and np.all(np.isfinite(Q))
        s.scf.set_input_charge(np.zeros((2, s.N)))
        with pytest.raises(_lib.NegfError) as e:
            s.scf.run(np.array([0.1, np.nan]))
        assert e.value.code == ENAN


@pytest.mark.parametrize("ahead", [True, False])
def test_preconditioned_run(dev, ahead):
    with Setup(2, 64) as s:
        sg = Surrogate(s.N, seed=1)
        s.scf.set_surrogate(sg)
        s.scf.use_graph(ahead)
        with pytest.raises(_lib.NegfError) as e:
            s.scf.run_surrogate(np.array([0.1, np.nan]), seed_iters=0, refresh_iter=0)
        assert e.value.code == ENAN
        sg.close()


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("max_iters", [0, 3])
def test_one_system_of_all_tubes(dev, graph, max_iters):
    with Setup(3, 13) as s:
        scf = negf.MultiScf(s.batch, Broyden_fraction=0.1, Broyden_max_norm=1e-6, Broyden_threshold_maxstep=200,
                            eps_r=3.9, R_ring_nm=0.665, R_image_nm=10.0)
        scf.use_graph(graph)
        with pytest.raises(_lib.NegfError) as e:
            scf.bias_point(np.array([0.1, np.nan, 0.2]), max_iters)
        assert e.value.code == ENAN and "iteration 1" in str(e.value)
        scf.close()


@pytest.mark.parametrize("ahead", [True, False])
@pytest.mark.parametrize("surrogate", [False, True])
def test_calls_after_an_error(dev, ahead, surrogate):
    """The iteration launched ahead of the error has ended when the call returns: solves
    on the same tubes and the next run give what they give on their own."""
    with Setup(3, 64) as s:
        s.scf.use_graph(ahead)
        sg = Surrogate(s.N, seed=1)
        s.scf.set_surrogate(sg)

        def run(V):
            s.scf.set_input_charge(np.zeros((3, s.N)))
            return s.scf.run_surrogate(V, seed_iters=0, refresh_iter=2) if surrogate else s.scf.run(V)

        want = run(s.V)
        for t, u in zip(s.tubes, s.U_ext):
            t.set_potential(u)
        alone = [t.solve(1)[0] for t in s.tubes]
        for _ in range(3):
            with pytest.raises(_lib.NegfError) as e:
                run(np.array([0.1, np.nan, 0.2]))
            assert e.value.code == ENAN
            for t, u, q in zip(s.tubes, s.U_ext, alone):
                t.set_potential(u)
                assert np.array_equal(t.solve(1)[0], q)
            for a, b in zip(run(s.V), want):
                assert np.array_equal(a, b)
        sg.close()
