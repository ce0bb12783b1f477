"""Rounding error of the lead self-energies of split chains, against Sancho-Rubio in 80-bit
floats: no larger than that of the same recursion in numpy (LAPACK inverses).

The doublings amplify every error by the same condition in both, so their errors differ
by the rounding of the elimination steps alone.  The mean of log10(error) over the
energies is compared; its scatter over 48 energies, each with a spread of about half a
decade between the two, is below 0.1: limit 0.3 (a factor of 2).
"""
import numpy as np
import pytest

from electrostatic_amd import negf
from oracle import block_oracle as B
from tests.test_gpu_block_split import random_chain

pytestmark = pytest.mark.gpu

L = np.clongdouble


def inverse(A):
    """Gauss-Jordan with partial pivoting of a stack of matrices."""
    n, e = A.shape[1], np.arange(len(A))
    A = np.concatenate([A, np.broadcast_to(np.eye(n, dtype=L), A.shape)], 2)
    for k in range(n):
        p = k + np.abs(A[:, k:, k]).argmax(1)
        row = A[e, p].copy()
        A[e, p] = A[:, k]
        A[:, k] = row / row[:, k][:, None]
        f = A[:, :, k].copy()
        f[:, k] = 0
        A -= f[:, :, None] * A[:, k][:, None, :]
    return A[:, :, n:]


def mm(a, b):
    return np.einsum("eij,ejk->eik", a, b)


def left_self_energy(E, H0, T, tol=1e-12):
    """T^T g T of every energy, g by Sancho-Rubio in 80 bits."""
    z = np.asarray(E, L)[:, None, None] * np.eye(len(H0), dtype=L)
    es = np.broadcast_to(H0.astype(L), z.shape).copy()
    eps, a = es.copy(), np.broadcast_to(T.T.astype(L), z.shape).copy()
    b = a.transpose(0, 2, 1).copy()
    on = np.arange(len(z))
    for _ in range(200):
        g = inverse(z[on] - eps[on])
        ga, gb = mm(g, a[on]), mm(g, b[on])
        agb, bga = mm(a[on], gb), mm(b[on], ga)
        es[on] += agb
        eps[on] += agb + bga
        a[on], b[on] = mm(a[on], ga), mm(b[on], gb)
        on = on[np.maximum(np.abs(a[on]).max((1, 2)), np.abs(b[on]).max((1, 2))) >= tol]
        if not len(on):
            break
    T = T.astype(L)
    return T.T @ inverse(z - es) @ T


@pytest.mark.parametrize("m,h,ring", [(32, 16, True), (20, 10, True), (20, 10, False), (18, 2, False)])
@pytest.mark.parametrize("eta", [1e-2, 1e-4])
def test_left_lead(dev, m, h, ring, eta):
    H0, T = B.zigzag_blocks(m // 2, 2.5) if ring else random_chain(m, h, 2, seed=m)[:2]
    E = np.random.default_rng(m).uniform(-3.0, 3.0, 48) + 1j * eta
    ref = left_self_energy(E, H0, T)
    c = negf.BlockChain(2, H0, T)
    c.set_potential(np.zeros((2, m)), (0.0, 0.0))
    got, _, _ = c.self_energies(E)
    c.close()
    numpy_ = np.stack([B.lead_self_energies(z, H0, T)[0] for z in E])

    def mean_log(x):
        e = np.abs(x - ref).max((1, 2)) / np.abs(ref).max((1, 2))
        return float(np.mean(np.log10(np.maximum(e.astype(float), 1e-17))))

    assert mean_log(got) < mean_log(numpy_) + 0.3, (mean_log(got), mean_log(numpy_))
