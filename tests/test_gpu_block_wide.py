"""The 32-wide block sweep and decimation, which every coupling takes that is not from
the second part of a block to the first of the next only: with g_b T kept and recomputed,
in one launch and in chunks of energies, against oracle/block_oracle.py.

Im E = 0.05 eV keeps the condition of every block below about 1e3: tolerance 1e-11.
"""
import numpy as np
import pytest

from electrostatic_amd import negf
from oracle import block_oracle as B
from tests.test_gpu_block_split import E3, check, random_chain

pytestmark = pytest.mark.gpu

G_BYTES = 2 * 32 * 32 * 8  # one complex g_b

E7 = np.concatenate([E3, np.array([0.9, -0.6, 2.2, -2.4]) + 0.05j])


@pytest.mark.parametrize("m", [1, 5, 20, 32])
@pytest.mark.parametrize("nb", [1, 2, 7])
@pytest.mark.parametrize("scratch", ["g and g T of all", "g of all", "g of two", "less than one"])
def test_dense_coupling(dev, m, nb, scratch):
    per = max(nb - 1, 1) * G_BYTES
    limit = {"g and g T of all": None, "g of all": E7.size * per, "g of two": 2 * per, "less than one": 1}[scratch]
    check(*random_chain(m, m, nb, seed=10 * m + nb, dense=True), (0.1, -0.05), E7, limit)


@pytest.mark.parametrize("m", [3, 20, 32])
@pytest.mark.parametrize("keep_x", [True, False])
def test_long_dense_chain(dev, m, keep_x):
    """Rounding errors must not grow along the chain."""
    nb = 40
    check(*random_chain(m, m, nb, seed=m, dense=True), (0.1, -0.05), E3,
          None if keep_x else E3.size * (nb - 1) * G_BYTES)


@pytest.mark.parametrize("m,h", [(5, 2), (20, 9), (32, 16)])
def test_long_split_chain(dev, m, h):
    check(*random_chain(m, h, 40, seed=m), (0.1, -0.05), E3)


def chunks(H0, T, v, coef, limits):
    out = []
    c = negf.BlockChain(len(v), H0, T)
    c.set_potential(v, (0.1, -0.05))
    for limit in limits:
        if limit:
            c.set_scratch_limit(limit)
        acc, dg, it = c.rgf(E7, coef, want_diag=True)
        out.append((acc, dg, it))
    c.close()
    for got in out[1:]:
        for a, b in zip(got, out[0]):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("m", [11, 32])
def test_wide_chunks_are_bit_identical(dev, m):
    """7 energies in one launch, in sweeps of 2, 2, 2, 1 (the last workgroup partly empty)
    and one by one; the energies are independent and the charge is summed in a fixed
    order."""
    nb = 9
    H0, T, v = random_chain(m, m, nb, seed=m, dense=True)
    per = (nb - 1) * G_BYTES
    chunks(H0, T, v, np.exp(1j * np.linspace(0.0, 1.0, 7)), (None, 7 * per, 2 * per, 1))


@pytest.mark.parametrize("m", [10, 16])
def test_split_chunks_are_bit_identical(dev, m):
    """The same of a ring chain, two wavefronts and 8 KiB a block and energy."""
    nb = 9
    H0, T = B.zigzag_blocks(m, 2.5)
    v = np.random.default_rng(m).normal(0.0, 0.05, (nb, 2 * m))
    per = nb * 2 * 256 * 16
    chunks(H0, T, v, np.exp(1j * np.linspace(0.0, 1.0, 7)), (None, 7 * per, 2 * per, 1))


def test_which_couplings_are_wide(dev):
    """One entry outside the second part x first part block sends the chain to the
    32-wide sweep, with the same result up to rounding where the entry is tiny."""
    H0, T, v = random_chain(12, 6, 4, seed=3)
    diag = []
    for extra in (0.0, 1e-14):
        T2 = T.copy()
        T2[0, 11] = extra
        c = negf.BlockChain(4, H0, T2)
        c.set_potential(v, (0.1, -0.05))
        diag.append(c.rgf(E7, want_diag=True)[1])
        c.close()
    assert not np.array_equal(*diag)
    assert np.abs(diag[0] - diag[1]).max() < 1e-11 * np.abs(diag[0]).max()
