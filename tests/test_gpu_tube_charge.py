"""A tube's solve: both plans in shared launches, row sums and charge in one kernel,
results through host memory; against the separate forms and the oracle."""
import numpy as np
import pytest
import torch

from electrostatic_amd import negf
from oracle import oracle as O
from tests.test_gpu_material import pair

pytestmark = pytest.mark.gpu


def charges(tube, U):
    """Charge by the host and the device entry point and its components."""
    tube.set_potential(U)
    Q, _ = tube.solve(0)
    parts = tube.charge_components()
    d = torch.full((tube.N,), float("nan"), dtype=torch.float64, device="cuda")
    tube.solve_device(0, d.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    tube.status()
    assert np.array_equal(Q, d.cpu().numpy())
    assert np.array_equal(Q, (parts[0] + parts[1]) - parts[2])
    return Q


# sites: 4 (one partial segment), 16 (one full), 64, 68, 272, 1024 (the pair's segments
# of 16 and 32), 2180 (of 128, last one partial), 4352 (not in the fused launch)
@pytest.mark.parametrize("cells", [1, 4, 16, 17, 68, 256, 545, 1088])
@pytest.mark.parametrize("mu", [(-1.0, -1.0), (-1.0, -1.12)])
def test_solve(cells, mu, monkeypatch):
    U = 0.15 * np.sin(np.arange(4 * cells) * 0.11) + 0.05
    tube, ot = pair(num_unitcells=cells, num_modes=2, mu=mu, noneq_pts=(96,))
    Q = charges(tube, U)
    if cells <= 256:
        Rho0, st0 = O.rho0(ot)
        ref, _, _, st = O.solve_negf(ot, U, U[[0, -1]], Rho0)
        assert st0 == 0 and st == 0
        assert np.abs(Q - ref).max() < 1e-10 * max(np.abs(ref).max(), 1e-3)
    # contacts moved to equilibrium and back: the non-equilibrium part goes and returns
    tube.set_contacts((-1.0, -1.0))
    q0 = charges(tube, U)
    tube.set_contacts(mu)
    assert np.array_equal(charges(tube, U), Q)
    if mu[0] == mu[1]:
        assert np.array_equal(q0, Q)
    tube.close()
    monkeypatch.setenv("NEGF_RGF_FUSED", "0")  # separate transfer and scan: no pair
    other, _ = pair(num_unitcells=cells, num_modes=2, mu=mu, noneq_pts=(96,))
    assert np.abs(charges(other, U) - Q).max() < 1e-11 * max(np.abs(Q).max(), 1e-3)
    other.close()


def test_many_rows():
    """More than 16 partial rows: the plans' own row sums."""
    tube, _ = pair(num_unitcells=20, num_modes=1, mu=(-1.0, -1.1), eq_pts=(400, 400, 419), noneq_pts=(1100,))
    few, _ = pair(num_unitcells=20, num_modes=1, mu=(-1.0, -1.1), eq_pts=(200, 200, 200), noneq_pts=(900,))
    U = 0.1 * np.cos(np.arange(80) * 0.2)
    a, b = charges(tube, U), charges(few, U)
    assert np.abs(a - b).max() < 1e-6 * np.abs(a).max()
    tube.close()
    few.close()
