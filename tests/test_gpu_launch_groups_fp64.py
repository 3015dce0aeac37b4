"""The two launches beside each other in the FP64 form, which takes the third
wave only where the queue is long against its longest bundle: the same bits as
the chains in small engines, with a captured graph and without."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import hrsw, lj

pytestmark = pytest.mark.gpu

BLOCK = 3


@pytest.mark.parametrize("graph", [False, True])
def test_two_fp64_launches_equal_small_engines(gpu, graph):
    print(f"[gpu] FP64 launch groups graph={graph}", flush=True)
    chains = [Chain(N=6200 + 67 * c if c < 30 else 1800 + (c * 7) % 500, rho=0.4, T=1.0, P=0.5, ensemble=nat.NPT,
                    max_dv=0.01, seed=7, chain_id=c, eci=5, **(lj() if c < 30 or c % 4 else hrsw()))
              for c in range(2200)]
    pick = [0, 14, 29, 30, 31, 1000, 2198, 2199]
    got = []
    for cs, g, lanes in ((chains, graph, 0), ([chains[c] for c in pick], False, 1)):
        with Engine(cs, form="batched_fp64", sample_capacity=3 * BLOCK, block_sweeps=BLOCK, use_graph=g,
                    block_lanes=lanes) as e:
            e.run(2 * BLOCK)
            first = e.read_samples(2 * BLOCK)
            obs = e.observables()
            e.run(BLOCK)
            got.append((first, obs, e.read_samples(BLOCK), e.states()))
    (a1, ao, a2, (ax, aL, aU)), (b1, bo, b2, (bx, bL, bU)) = got
    assert np.array_equal(a1[pick], b1) and np.array_equal(ao[pick], bo) and np.array_equal(a2[pick], b2)
    assert np.array_equal(aL[pick], bL) and np.array_equal(aU[pick], bU)
    assert all(np.array_equal(ax[c], bx[k]) for k, c in enumerate(pick))
