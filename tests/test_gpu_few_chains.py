"""Engines that take several lanes per block by themselves: where the launch,
with every workgroup as large as the largest chain's, ends before the chains
would with one lane per block; the same bits either way."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import hrsw, lj

pytestmark = pytest.mark.gpu


def npt(N, c, pot=None, bcap=256):
    return Chain(N=N, L0=max(N / 0.4, 9.0), T=1.0, P=0.5, ensemble=nat.NPT, max_dv=0.01, seed=7, chain_id=c, eci=3,
                 bcap=bcap, **(pot or lj()))


def uneven(n, pots):
    rng = np.random.default_rng(1)
    N = np.rint(np.exp(rng.uniform(np.log(20), np.log(256), n))).astype(int)
    return [npt(int(N[c]), c, pots[c % len(pots)]()) for c in range(n)]


# name: (chains, several lanes in FP32, in FP64); a workgroup of 512 lanes
# fills a CU, of 64 an eighth
CASES = {
    "512_lanes_all_resident": (lambda: [npt(250, c) for c in range(256)], True, True),
    "512_lanes_one_more": (lambda: [npt(250, c) for c in range(257)], False, False),
    "64_lanes_all_resident": (lambda: [npt(25, c) for c in range(2048)], True, True),
    "one_long_among_few": (lambda: [npt(25, c) for c in range(300)] + [npt(300, 300)], True, True),
    "one_long_among_many": (lambda: [npt(25, c) for c in range(1000)] + [npt(300, 1000)], False, False),
    "one_block_chains": (lambda: [npt(13, c) for c in range(2000)] + [npt(300, 2000)], False, False),
    "uneven_300": (lambda: uneven(300, [hrsw, lj]), True, True),
    "long_blocks": (lambda: [npt(3000 + 7 * c, c, bcap=64) for c in range(700)], False, False),
    "uneven_1500": (lambda: uneven(1500, [hrsw, lj]), False, False),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_choice_by_what_the_launch_takes(gpu, name):
    make, fp32, fp64 = CASES[name]
    for form, several in (("batched_fp32", fp32), ("batched_fp64", fp64)):
        with Engine(make(), form=form, sample_capacity=1) as e:
            assert (e.layout(0)["lanes"] > 1) == several, form


@pytest.mark.parametrize("form", ["batched_fp32", "batched_fp64"])
def test_chains_that_wait_for_others(gpu, form):
    """More chains than are resident, of every workgroup size in one launch."""
    print(f"[gpu] few chains, two rounds {form}", flush=True)
    chains = uneven(300, [hrsw, lj])
    got = []
    for lanes in (0, 1):
        with Engine(chains, form=form, sample_capacity=12, block_sweeps=4, block_lanes=lanes) as e:
            e.run(12)
            got.append((e.read_samples(12), e.states(), e.all_counters()))
    (s0, (x0, L0, U0), c0), (s1, (x1, L1, U1), c1) = got
    assert np.array_equal(s0, s1) and np.array_equal(L0, L1) and np.array_equal(U0, U1)
    assert all(np.array_equal(a, b) for a, b in zip(x0, x1))
    assert all(np.array_equal(c0[k], c1[k]) for k in c0)


def test_two_partners_a_side(gpu):
    """Two lanes per block (more than 128 blocks) gain in FP64 only."""
    for N, fp32, fp64 in ((64, 16, 16), (400, 4, 4), (800, 1, 2), (2000, 1, 2)):
        ch = Chain(N=N, L0=N / 0.48, T=0.8, P=0.7, boundary=nat.WALLS, ensemble=nat.NPT, max_dv=1.0, max_step=0.1,
                   nbn=2, seed=9, **lj(cutoff=np.inf, shifted=0))
        for form, lanes in (("batched_fp32", fp32), ("batched_fp64", fp64)):
            with Engine([ch], form=form, sample_capacity=1) as e:
                assert e.layout(0)["lanes"] == lanes, (N, form)
