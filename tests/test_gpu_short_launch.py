"""Launches of few chain groups: short segments, transfer and scan fused from one
segment up, against the oracle and against the default segment length."""
import numpy as np
import pytest

from electrostatic_amd import _lib
from oracle import oracle as O
from tests.gpu_util import chain_params, dev_array, dev_zeros, ptr, smooth_potential, to_np
from tests.test_gpu_rgf import BETA17, GAMMA, energies, run_diag

pytestmark = pytest.mark.gpu


def rel_err(a, ref):
    return np.abs(a - ref).max() / np.abs(ref).max()


# 1, 2, 3, 16, 17 and 32 segments of 16, then of 32 and 48, then 64 sites, last ones
# partial; 2049 sites: the first length that keeps the default (17 segments of 128)
SIZES = [(2, 1), (16, 33), (17, 64), (40, 65), (256, 3), (257, 64), (500, 1), (512, 65), (513, 40), (1024, 64),
         (1030, 65), (2048, 64), (2049, 64), (2175, 64), (2176, 5),
         # above 32 chain groups: at most 16 segments, 32 chains per workgroup
         (40, 2048), (40, 2049), (600, 2112), (1024, 2305), (2048, 2049), (2049, 2049),
         # 128 chain groups and one more
         (40, 8192), (40, 8193), (300, 8192), (300, 8193)]


@pytest.mark.parametrize("N,nE", SIZES)
def test_against_oracle(N, nE):
    U = smooth_potential(N, seed=N)
    E = energies(nE - nE // 2, nE // 2, seed=N)
    rng = np.random.default_rng(N)
    coef = rng.normal(size=nE) + 1j * rng.normal(size=nE)
    Uc = (U[0], U[-1])
    ref, _ = O.accumulate_diagG(U, BETA17, GAMMA, Uc, BETA17, GAMMA, E, coef)
    acc, _ = run_diag(U, BETA17, GAMMA, Uc, E, coef, want_G=False)
    acc2, G = run_diag(U, BETA17, GAMMA, Uc, E, coef, want_G=True)
    G128 = run_diag(U, BETA17, GAMMA, Uc, E, coef, want_G=True, segment_length=128)[1]
    assert rel_err(acc, ref) < 1e-10 and rel_err(acc2, ref) < 1e-10
    assert rel_err(G, G128) < 1e-10


@pytest.mark.parametrize("N,nE", SIZES)
def test_other_kinds(N, nE):
    """Non-equilibrium charge with and without integrand samples, DOS and
    transmission, against segments of 128 sites."""
    lib = _lib.load()
    U = smooth_potential(N, seed=N + 3, lo=-0.3, hi=0.2)
    E = np.linspace(-2.5, 1.5, nE) + 1e-4j
    rng = np.random.default_rng(N + 1)
    dU, dE, dL, dR = (dev_array(a) for a in (U, E, rng.normal(size=nE), rng.normal(size=nE)))
    got = []
    for L in (0, 128):
        p = chain_params(N, BETA17, GAMMA, (U[0], U[-1]), segment_length=L)
        a, b, s, d, t = dev_zeros(N), dev_zeros(N), dev_zeros(3 * nE), dev_zeros(nE), dev_zeros(nE)
        _lib.check(lib.negf_rgf_noneq_accumulate(p, ptr(dU), nE, ptr(dE), ptr(dL), ptr(dR), None, None, ptr(a), None,
                                                 None))
        _lib.check(lib.negf_rgf_noneq_accumulate(p, ptr(dU), nE, ptr(dE), ptr(dL), ptr(dR), None, None, ptr(b),
                                                 ptr(s), None))
        _lib.check(lib.negf_rgf_dos(p, ptr(dU), nE, ptr(dE), ptr(d), ptr(t), None))
        got.append([to_np(x) for x in (a, b, s, d, t)])
    for x, y in zip(*got):
        assert rel_err(x, y) < 1e-10
