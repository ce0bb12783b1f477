"""LDOS of a tube, summed over its modes on the GPU, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_material import pair

pytestmark = pytest.mark.gpu


def check(tube, ot, U, nE):
    E = np.linspace(-1.5, 0.7, nE) + 1e-3j
    Uc = U[[0, -1]]
    tube.set_potential(U)
    got = tube.dos_complex(E, want_ldos=True)
    ref = O.dos_transmission(ot, U, Uc, E, 68, want_ldos=True)
    for g, r in zip(got, ref):
        assert np.abs(g - r).max() < 1e-9 * np.abs(r).max()


@pytest.mark.parametrize("modes", [1, 2, 5])
def test_sizes_and_repeats(modes):
    """4 sites x 1 energy (less than a block), 64 x 4 (exactly one) and 68 x 33; the
    same tube again with fewer and with more energies."""
    for cells, sizes in ((1, (1, 7, 2)), (16, (4,)), (17, (33, 5, 64))):
        tube, ot = pair(num_unitcells=cells, num_modes=modes)
        for k, nE in enumerate(sizes):
            U = 0.2 * np.sin(np.arange(tube.N) * (0.3 + k))
            check(tube, ot, U, nE)


def test_trace():
    """DOS = spin sum_n LDOS_n / atoms per unit cell (4 rings of 17)."""
    tube, _ = pair(num_unitcells=9, num_modes=3)
    E = np.linspace(-1.2, 0.9, 21) + 1e-4j
    U = 0.1 * np.cos(0.4 * np.arange(tube.N))
    tube.set_potential(U)
    dos, trans, ld = tube.dos_complex(E, want_ldos=True)
    assert np.abs(2.0 * ld.sum(axis=1) / 68 - dos).max() < 1e-12 * dos.max()
