"""Two-part block chains whose parts need pivoting.  The symmetric sweep of a part
eliminates its orbitals in their order and hands the part to the pivoted elimination
where a multiplier of a later row exceeds 256.  The chains here are built so that a
chosen orbital's pivot is far below its couplings while the conditions stay moderate;
the multipliers that the kernel meets are replayed on the host (plain
Gaussian elimination of the same Schur complements) and asserted, so that each test
reaches the branch it is for.

Per part the kernel inverts one matrix (g from the lead on its own side) up to the
middle of the chain and two (g and G) beyond it, so there are four cases: the one, the
first, the second, or both.

Tolerance, given the kernel's own lead self-energies (compared with the oracle's to
1e-8 beside it): every inverse along the chain is within a few eps of its condition, so
the diagonal is within n eps kappa per part, kappa the largest condition among the
matrices that are inverted and the whole device's, n = 32 orbitals.
"""
import numpy as np
import pytest

from electrostatic_amd import negf
from oracle import block_oracle as B

pytestmark = pytest.mark.gpu

LIMIT = 256.0
# (orbitals per block, first part): parts of up to 4, 8, 12 and 16 columns, and uneven ones
SIZES = [(4, 2), (7, 3), (15, 7), (23, 12), (32, 16), (18, 2)]


def multiplier(A):
    """Largest |a_ik / a_kk| of an elimination in natural order."""
    A = A.astype(complex).copy()
    big = 0.0
    for k in range(len(A) - 1):
        f = A[k + 1:, k] / A[k, k]
        big = max(big, np.abs(f).max())
        A[k + 1:, k:] -= np.outer(f, A[k, k:])
    return big


def leads(E, H0, T):
    return B.lead_self_energies(E, H0, T, (0.0, 0.0))[:2]


class Parts:
    """The chain as 2 nb parts: on-site matrices, couplings and both self-energies."""

    def __init__(self, E, H0, T, h, v, SigL, SigR):
        nb, m = v.shape
        self.n = 2 * nb
        sl = [slice(0, h), slice(h, m)]
        E0 = [E * np.eye(s.stop - s.start) - H0[s, s] for s in sl]
        self.A = [E0[b % 2] - np.diag(v[b // 2, sl[b % 2]]) for b in range(2 * nb)]  # without self-energies
        C = [H0[sl[0], sl[1]], T[sl[1], sl[0]]]
        self.SL = [SigL[sl[0], sl[0]]]
        for b in range(2 * nb - 1):
            c = C[b % 2]
            self.SL.append(c.T @ np.linalg.inv(self.A[b] - self.SL[b]) @ c)
        self.SR = [SigR[sl[1], sl[1]]]
        for b in range(2 * nb - 1, 0, -1):
            c = C[(b - 1) % 2]
            self.SR.append(c @ np.linalg.inv(self.A[b] - self.SR[-1]) @ c.T)
        self.SR.reverse()

    def g(self, side, b):
        return self.A[b] - (self.SR if side else self.SL)[b]

    def G(self, b):
        return self.A[b] - self.SL[b] - self.SR[b]

    def counts(self):
        """Matrices over the limit: (single g, g of a pair only, G only, both)."""
        out = [0, 0, 0, 0]
        for side in range(2):
            for j in range(self.n):
                b = self.n - 1 - j if side else j
                big = multiplier(self.g(side, b)) > LIMIT
                if j < self.n // 2:
                    out[0] += big
                else:
                    Big = multiplier(self.G(b)) > LIMIT
                    out[1] += big and not Big
                    out[2] += Big and not big
                    out[3] += big and Big
        return out

    def condition(self):
        return max(np.linalg.cond(x) for b in range(self.n) for x in (self.g(0, b), self.g(1, b), self.G(b)))


def check(E, H0, T, h, v):
    nb, m = v.shape
    c = negf.BlockChain(nb, H0, T)
    c.set_potential(v, (0.0, 0.0))
    _, dg, _ = c.rgf(np.array([E]), want_diag=True)
    SL, SR, _ = c.self_energies(np.array([E]))
    c.close()
    SL, SR = SL[0], SR[0]
    for got, ref in zip((SL, SR), leads(E, H0, T)):
        assert np.abs(got - ref).max() < 1e-8 * np.abs(ref).max()
    H = np.zeros((nb * m, nb * m), complex)
    for b in range(nb):
        H[b * m:(b + 1) * m, b * m:(b + 1) * m] = H0 + np.diag(v[b])
        if b + 1 < nb:
            H[b * m:(b + 1) * m, (b + 1) * m:(b + 2) * m] = T
            H[(b + 1) * m:(b + 2) * m, b * m:(b + 1) * m] = T.T
    H[:m, :m] += SL
    H[-m:, -m:] += SR
    kappa = max(np.linalg.cond(E * np.eye(nb * m) - H), Parts(E, H0, T, h, v, SL, SR).condition())
    assert kappa < 1e6
    ref = B.dense_diag(E, H0, T, v, SL, SR)
    err = np.abs(dg[0] - ref).max() / np.abs(ref).max()
    assert err < 2 * nb * 32 * np.finfo(float).eps * kappa, (err, kappa)


def random_chain(m, h, nb, seed):
    rng = np.random.default_rng(seed)
    H0 = rng.normal(0.0, 0.5, (m, m))
    H0 = 0.5 * (H0 + H0.T)
    T = np.zeros((m, m))
    T[h:, :h] = rng.normal(0.0, 0.7, (m - h, h))
    return H0, T, rng.normal(0.0, 0.2, (nb, m))


def bare_chain(m, h, nb, E, parts):
    """The first orbital of each of the given parts (0, 1) lies at Re E and couples to
    the second one of its part only: its pivot is Im E in g and in G, its multiplier
    1 / Im E."""
    H0, T, v = random_chain(m, h, nb, seed=m)
    for o in ((0,), (h,), (0, h))[parts]:
        H0[o, :] = H0[:, o] = 0.0
        H0[o, o] = E.real
        H0[o, o + 1] = H0[o + 1, o] = 1.0
        T[o, :] = T[:, o] = 0.0
        v[:, o] = 0.0
    return H0, T, v


@pytest.mark.parametrize("m,h", SIZES)
@pytest.mark.parametrize("parts", [0, 1, 2])
@pytest.mark.parametrize("nb", [1, 2, 5])
def test_every_part(dev, m, h, parts, nb):
    E = 0.3 + 1e-3j
    H0, T, v = bare_chain(m, h, nb, E, parts)
    single, first, second, both = Parts(E, H0, T, h, v, *leads(E, H0, T)).counts()
    # all parts of the given kind, in each half of both sweeps
    assert single + both >= (4 * nb if parts == 2 else 2 * nb) and single > 0 and both > 0
    check(E, H0, T, h, v)


def tuned_chain(m, h, nb, E, beta, what):
    """A chain far outside its bands with the potential of one orbital (the first of
    part beta) tuned until its pivot is Im E in one matrix: G, or g from the left or
    right."""
    H0, T, v = random_chain(m, h, nb, seed=m + 1)
    p = Parts(E, H0, T, h, v, *leads(E, H0, T))
    a = {"G": p.G(beta), "left": p.g(0, beta), "right": p.g(1, beta)}[what][0, 0]
    v[beta // 2, h * (beta % 2)] += a.real
    return H0, T, v


@pytest.mark.parametrize("m,h", SIZES)
@pytest.mark.parametrize("beta", [0, 1, 4, 5, 8, 9])
@pytest.mark.parametrize("what", ["G", "left", "right"])
def test_one_matrix(dev, m, h, beta, what):
    nb, E = 5, 12.0 + 1e-4j
    H0, T, v = tuned_chain(m, h, nb, E, beta, what)
    counts = Parts(E, H0, T, h, v, *leads(E, H0, T)).counts()
    # a g beyond its sweep's middle is the first of a pair
    in_pair = beta >= nb if what == "left" else beta < nb
    want = [0, 0, 0, 0]
    want[2 if what == "G" else 1 if in_pair else 0] = 1
    assert counts == want
    check(E, H0, T, h, v)
