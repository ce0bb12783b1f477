"""Charge sweeps whose last segment is partial: it shares the launch of the full
ones, except where those run three wavefronts per SIMD and need them."""
import numpy as np
import pytest

from electrostatic_amd import _lib
from oracle import oracle as O
from tests.gpu_util import chain_params, dev_array, dev_zeros, ptr, smooth_potential, to_np
from tests.test_gpu_rgf import BETA17, GAMMA, energies, run_diag

pytestmark = pytest.mark.gpu


def rel_err(a, ref):
    return np.abs(a - ref).max() / np.abs(ref).max()


# (sites, segment length, energies): last segments of 1 site, of one less than full,
# below and above a sub-block; 1, 4, 5 and 8 sub-blocks; more items than two
# wavefronts per SIMD (short segments: a launch of its own; long ones: shared)
SIZES = [(17, 16, 5), (31, 16, 70), (65, 64, 64), (145, 80, 3), (129, 128, 65), (255, 128, 1), (1000, 48, 65),
         (33617, 16, 64), (8201, 128, 2100)]


@pytest.mark.parametrize("N,L,nE", SIZES)
def test_equilibrium(N, L, nE):
    U = smooth_potential(N, seed=N)
    E = energies(nE - nE // 2, nE // 2, seed=N)
    rng = np.random.default_rng(N)
    coef = rng.normal(size=E.size) + 1j * rng.normal(size=E.size)
    Uc = (U[0], U[-1])
    ref, _ = O.accumulate_diagG(U, BETA17, GAMMA, Uc, BETA17, GAMMA, E, coef)
    acc, _ = run_diag(U, BETA17, GAMMA, Uc, E, coef, want_G=False, segment_length=L)
    assert rel_err(acc, ref) < 1e-10


@pytest.mark.parametrize("N,L,nE", SIZES)
def test_nonequilibrium(N, L, nE):
    """Against the launch that also writes integrand samples, where the general
    sweep takes every segment."""
    lib = _lib.load()
    U = smooth_potential(N, seed=N + 3, lo=-0.3, hi=0.2)
    E = np.linspace(-2.5, 1.5, nE) + 1e-5j
    rng = np.random.default_rng(N + 1)
    cL, cR = rng.normal(size=nE), rng.normal(size=nE)
    p = chain_params(N, BETA17, GAMMA, (U[0], U[-1]), segment_length=L)
    dU, dE, dL, dR = dev_array(U), dev_array(E), dev_array(cL), dev_array(cR)
    acc, acc2, integ = dev_zeros(N), dev_zeros(N), dev_zeros(3 * nE)
    for a, i in ((acc, None), (acc2, integ)):
        _lib.check(lib.negf_rgf_noneq_accumulate(p, ptr(dU), nE, ptr(dE), ptr(dL), ptr(dR), None, None, ptr(a),
                                                 i if i is None else ptr(i), None))
    assert rel_err(to_np(acc), to_np(acc2)) < 1e-12
