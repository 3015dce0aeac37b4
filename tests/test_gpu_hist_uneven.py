"""Histograms of engines whose chains differ widely in length: a sample costs
what the chains' own tiles cost, and counts every particle and pair."""
import time

import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import lj

pytestmark = pytest.mark.gpu

RHO = dict(rhonb=200, rbw=20.0)
SHORT, LONG = [32] * 512, [60000] * 4


def chains(Ns):
    return [Chain(N=N, L0=N / 0.48, boundary=nat.WALLS, seed=7, chain_id=c, **lj()) for c, N in enumerate(Ns)]


def sample_time(Ns):
    with Engine(chains(Ns), form="batched_fp64", sample_capacity=1) as e:
        e.hist_configure(1000, **RHO)
        best = np.inf
        for _ in range(6):
            e.sync()
            t = time.perf_counter()
            for _ in range(20):
                e.hist_sample()
            e.sync()
            best = min(best, (time.perf_counter() - t) / 20)
    return best


def test_short_chains_beside_long_ones_cost_their_own_tiles(gpu):
    """Three times the two parts' times: with a share of workgroups per chain
    as many as the longest needs, six times."""
    print("[gpu] histograms of uneven chains, time", flush=True)
    together, parts = sample_time(SHORT + LONG), sample_time(SHORT) + sample_time(LONG)
    assert together <= 3.0 * parts, (together, parts)


@pytest.mark.parametrize("g", [False, True])
def test_every_particle_and_pair_is_counted(gpu, g):
    Ns = [60, 64, 65, 128, 129, 257, 6000, 2]
    print(f"[gpu] histograms of uneven chains g={g}", flush=True)
    cs = chains(Ns)
    kw = dict(gns=1, gsw=50000.0, gnb=2, gbw=50000.0) if g else {}
    with Engine(cs, form="batched_fp64", sample_capacity=1) as e:
        e.hist_configure(1, rhonb=2, rbw=50000.0, **kw)
        e.run(1)
        e.hist_sample()
        rho, got, ns = e.hist_read()
        assert ns == 2
        # a second configuration of the same engine
        e.hist_configure(1, rhonb=2, rbw=50000.0)
        e.hist_sample()
        again = e.hist_read()[0]
    N = np.array(Ns, dtype=np.uint64)
    assert np.array_equal(rho.sum(1), 2 * N) and np.array_equal(again.sum(1), N)
    if g:
        assert np.array_equal(got.sum((1, 2)), 2 * N * (N - np.uint64(1)))
