"""A tube keeps the workspace of a DOS call for the next one only up to a bound."""
import numpy as np
import pytest
import torch

from electrostatic_amd import negf
from electrostatic_amd.workloads import gaussian_bumps

pytestmark = pytest.mark.gpu

MB = 1 << 20


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def make(cells, noneq=100, modes=2):
    t = negf.Tube(num_unitcells=cells, num_modes=modes, contact_mu=(-1.0, -1.1), eq_integration_pts=(30, 30, 64),
                  noneq_integration_pts=(noneq,), E_zPlus_imag=1e-5, E_valence_min=-10.0, E_pole_max=3.0)
    t.set_potential(gaussian_bumps(t.N, seed=1, amp=0.3))
    return t


def test_large_dos_and_current_give_their_memory_back(dev):
    """2 modes x 8192 energies x 20000 sites, and the current of 8000 energies: the
    segment matrices and states alone take over 400 MB.  At most the bound of 256
    MB and the chains with their results stay (16384 chains of 128 bytes: 2 MB)."""
    t = make(5000, noneq=8000)
    E = np.linspace(-2.0, 2.0, 8192)
    t.dos(E[:10])  # what any call keeps
    before = free()
    t.dos(E)
    assert before - free() < 272 * MB
    t.solve(1)
    after_solve = free()
    t.current()
    assert after_solve - free() < 272 * MB
    t.close()


def test_results_do_not_depend_on_what_is_kept(dev):
    """The workspace given back (large), kept (small) and kept from the other size."""
    E = np.linspace(-2.0, 2.0, 801) + 1e-5j
    got = []
    for big_first in (False, True):
        t = make(5000)
        if big_first:
            t.dos_complex(np.linspace(-2.0, 2.0, 1000) + 1e-5j, True)
        got.append([t.dos_complex(E[:n], True) for n in (801, 3, 801)])
        t.close()
    for a, b in zip(*got):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
