"""Configurations of one to four whole tiles of 512 particles, one fewer and one
more, against the oracle (the check and its tolerances are those of the tiled
observables' own test)."""
import pytest

import test_gpu_obs_tiles as tiles
from jmmonedmc_amd import _native as nat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [511, 512, 513, 1535, 1536, 1537, 2047, 2048, 2049])
@pytest.mark.parametrize("boundary", [nat.PERIODIC, nat.WALLS])
@pytest.mark.parametrize("kind", ["lj", "yukawa"])
def test_tile_ends(gpu, oracle, N, boundary, kind):
    tiles.test_tiled_observables_equal_oracle(gpu, oracle, N, boundary, kind)
