"""GPU parity of the two-part block chain (coupling from the second part of a
block to the first part of the next only) against oracle/block_oracle.py, at
the part sizes, block counts and chunks where it can go wrong, and of chains
that keep the 32-wide path.

Im E = 0.05 eV keeps the condition of every block below about 1e3, so both
sides are within about 1e3 rounding errors (1e-13) of the exact diagonal;
tolerance 1e-11 relative.
"""
import numpy as np
import pytest

from electrostatic_amd import negf
from oracle import block_oracle as B

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def random_chain(m, h, nb, seed, dense=False):
    """Random symmetric H0 and a T from rows >= h to columns < h (or dense)."""
    rng = np.random.default_rng(seed)
    H0 = rng.normal(0.0, 0.5, (m, m))
    H0 = 0.5 * (H0 + H0.T)
    T = np.zeros((m, m))
    T[h:, :h] = rng.normal(0.0, 0.7, (m - h, h))
    if dense:
        T = rng.normal(0.0, 0.4, (m, m))
    return H0, T, rng.normal(0.0, 0.2, (nb, m))


def check(H0, T, v, Uc, E, scratch=None):
    nb, m = v.shape
    c = negf.BlockChain(nb, H0, T)
    c.set_potential(v, Uc)
    if scratch:
        c.set_scratch_limit(scratch)
    coef = np.exp(1j * np.arange(E.size))
    acc, dg, it = c.rgf(E, coef, want_diag=True)
    SLg, SRg, _ = c.self_energies(E)
    c.close()
    ref_acc = np.zeros((nb, m))
    for k, z in enumerate(E):
        SL, SR, its = B.lead_self_energies(z, H0, T, Uc)
        ref = B.dense_diag(z, H0, T, v, SL, SR)
        assert rel(dg[k], ref) < 1e-11, (k, rel(dg[k], ref))
        assert np.abs(SLg[k] - SL).max() < 1e-11 * max(1.0, np.abs(SL).max())
        assert np.abs(SRg[k] - SR).max() < 1e-11 * max(1.0, np.abs(SR).max())
        assert abs(it[k, 0] - its[0]) <= 1 and abs(it[k, 1] - its[1]) <= 1
        ref_acc += np.imag(coef[k] * ref)
    assert rel(acc, ref_acc) < 1e-10


E3 = np.array([0.3, -1.7, 0.011]) + 0.05j


@pytest.mark.parametrize("m,h", [(2, 1), (3, 1), (5, 4), (8, 4), (17, 1), (17, 16), (20, 9), (24, 12), (25, 13), (31, 16),
                                 (32, 16)])
@pytest.mark.parametrize("nb", [1, 2, 5])
def test_part_sizes(dev, m, h, nb):
    check(*random_chain(m, h, nb, seed=100 * m + nb), (0.1, -0.05), E3)


@pytest.mark.parametrize("scratch", [1, 2 * 7 * 2 * 256 * 16])
def test_energy_chunks(dev, scratch):
    # one energy per chunk; two energies per chunk and a remainder
    check(*random_chain(20, 10, 7, seed=3), (0.1, -0.05), E3, scratch)


@pytest.mark.parametrize("m,dense", [(1, False), (6, True), (32, True)])
def test_other_couplings_keep_the_wide_path(dev, m, dense):
    check(*random_chain(m, m, 3, seed=m, dense=True), (0.1, -0.05), E3)


def test_zero_coupling(dev):
    H0, T, v = random_chain(10, 5, 3, seed=5)
    check(H0, 0.0 * T, v, (0.1, -0.05), E3)


def test_singular_parts_take_the_pivoted_elimination(dev):
    """H_00 = H_11 = 0 with energies at the bare level: the first pivots of the
    leads' elimination are Im E, far below the couplings (limit 8).  The chain's own
    pivoted elimination is reached by test_gpu_block_pivot.py."""
    m, h, nb = 12, 6, 3
    rng = np.random.default_rng(7)
    H0 = np.zeros((m, m))
    H0[:h, h:] = rng.normal(0.0, 2.0, (h, m - h))
    H0[h:, :h] = H0[:h, h:].T
    T = np.zeros((m, m))
    T[h:, :h] = np.diag(np.full(h, 1e-3)) + 1.0 * np.eye(h, k=1)
    E = np.array([0.0 + 0.02j, 1e-3 + 0.02j])
    c = negf.BlockChain(nb, H0, T)
    v = np.zeros((nb, m))
    c.set_potential(v, (0.0, 0.0))
    _, dg, _ = c.rgf(E, want_diag=True)
    c.close()
    for k, z in enumerate(E):
        SL, SR, _ = B.lead_self_energies(z, H0, T, (0.0, 0.0))
        ref = B.dense_diag(z, H0, T, v, SL, SR)
        # couplings up to 6 over Im E = 0.02, squared: condition 1e5
        assert rel(dg[k], ref) < 1e-9, (k, rel(dg[k], ref))
