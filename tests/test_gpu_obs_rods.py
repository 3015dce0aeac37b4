"""Pair energies of hard rods longer than the well is wide (a caller's theta may
make them so): rods that overlap have infinite energy also beyond the well."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("N", [5, 700, 1500])
def test_overlapping_rods_beyond_the_well(gpu, N, precision):
    import torch

    from jmmonedmc_amd.autograd import observables
    print(f"[gpu] long rods N={N} {precision}", flush=True)
    # rods of 1.8 with a well out to 1.5 (depth 0.7), partners looked at up to 2.5
    chain = Chain(N=N, rho=0.2, potential=nat.POT_HRSW, cutoff=2.5, pot_p=(1.8, 0.7, 1.5, 0.0))
    gaps = np.full((3, N), 3.0)
    gaps[1, N // 2] = 1.6  # overlapping, beyond the well
    gaps[2, N // 2] = 2.2  # not overlapping
    x = torch.tensor(np.cumsum(gaps, 1) - 1.5 * N, dtype=torch.float64, device="cuda")
    L = torch.full((3,), 3.0 * N + 10.0, dtype=torch.float64, device="cuda")
    obs = observables(x, L, chain, torch.tensor([1.8, 0.7]), precision).cpu().numpy()
    assert np.array_equal(obs[:, 0], [0.0, np.inf, 0.0])
    assert np.all(obs[:, 1:] == 0.0)
