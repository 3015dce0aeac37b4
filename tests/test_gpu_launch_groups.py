"""Engines whose chains run in two launches beside each other (three waves
per SIMD: more bundles than fit at two, some larger than a third of a CU's LDS)
against the same chains in small engines: the same bits per chain, over
several blocks, with a captured graph and without, and with reads, histograms
and state changes between the blocks (each must follow both launches)."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import hrsw, lj

pytestmark = pytest.mark.gpu

BLOCK = 4


def batch(ensemble=nat.NPT):
    """600 bundles: 30 chains of 6200 to 8190 (images above 45 KB) among 256-block chains of 1800 to 2300."""
    out = []
    for c in range(600):
        N = 6200 + 67 * c if c < 30 else 1800 + (c * 7) % 500
        out.append(Chain(N=N, rho=0.4, T=1.0, P=0.5, ensemble=ensemble, max_dv=0.01, seed=7, chain_id=c, eci=5,
                         **(lj() if c % 2 else hrsw())))
    return out


@pytest.mark.parametrize("form", ["batched_fp32", "batched_fp64"])
@pytest.mark.parametrize("graph", [False, True])
def test_two_launches_equal_small_engines(gpu, form, graph):
    print(f"[gpu] launch groups {form} graph={graph}", flush=True)
    chains = batch()
    with Engine(chains, form=form, sample_capacity=3 * BLOCK, block_sweeps=BLOCK, use_graph=graph) as e:
        e.run(2 * BLOCK)
        first = e.read_samples(2 * BLOCK)
        obs = e.observables()
        x0, L0, U0 = e.states()
        e.run(BLOCK)
        x1, L1, U1 = e.states()
        # back to the earlier state: the same block again
        e.set_states(x0, L0, U0, np.full(len(chains), 2 * BLOCK, dtype=np.uint64))
        second = e.read_samples(BLOCK)
        e.run(BLOCK)
        again = e.read_samples(BLOCK)
        x2, L2, U2 = e.states()
        cnt = e.all_counters()
    assert np.array_equal(second, again) and np.array_equal(L1, L2) and np.array_equal(U1, U2)
    pick = [0, 1, 14, 29, 30, 31, 311, 598, 599]
    with Engine([chains[c] for c in pick], form=form, sample_capacity=3 * BLOCK, block_sweeps=BLOCK,
                block_lanes=1) as e:
        e.run(2 * BLOCK)
        want = e.read_samples(2 * BLOCK)
        wobs = e.observables()
        e.run(BLOCK)
        wx, wL, wU = e.states()
        wc = e.all_counters()
    assert np.array_equal(first[pick], want) and np.array_equal(obs[pick], wobs)
    assert np.array_equal(L1[pick], wL) and np.array_equal(U1[pick], wU)
    for k, c in enumerate(pick):
        assert np.array_equal(x1[c], wx[k]) and np.array_equal(x2[c], wx[k])
    assert np.array_equal(cnt["sweeps"], np.full(len(chains), 3 * BLOCK)) and np.all(wc["vol_trials"] == 3 * BLOCK)


def test_histograms_follow_both_launches(gpu):
    print("[gpu] launch groups histograms", flush=True)
    chains = batch(nat.NLT)
    pick = [0, 29, 30, 599]
    got = []
    for cs, lanes in ((chains, 0), ([chains[c] for c in pick], 1)):
        with Engine(cs, form="batched_fp32", sample_capacity=2 * BLOCK, block_sweeps=BLOCK, block_lanes=lanes) as e:
            e.hist_configure(2, rhonb=200, rbw=50.0)
            e.run(2 * BLOCK)
            got.append(e.hist_read())
    assert got[0][2] == got[1][2] == BLOCK
    assert np.array_equal(got[0][0][pick], got[1][0])
