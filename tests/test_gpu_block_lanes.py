"""Several lanes per block (a workgroup per chain, engines of few chains)
against one lane per block: the same bits, in both forms: samples, virials,
accept decisions, positions, lengths, energies and counters over two launches
with recomputes in between.  The cases are those of the oracle replays (walls,
periodic, NPT linear and log, every potential, the smallest chains, mixed
batches) and the block counts at which the layout changes (1, 64, 65 to 256
blocks; blocks cut in two from 40 particles on; windows of 0, 1 and 8
partners, remainders of the 2 G block positions drawn at once)."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import CASES, hrsw, lj

pytestmark = pytest.mark.gpu

SWEEPS, BLOCK = 18, 9


def npt(N, bcap=256, **kw):
    d = dict(N=N, rho=0.5, T=1.0, P=0.5, ensemble=nat.NPT, vol_move=nat.VOL_LOG, max_dv=0.01, seed=31, chain_id=N,
             eci=5, bcap=bcap, **lj())
    d.update(kw)
    return Chain(**d)


LAYOUTS = {
    "one_block": lambda: [npt(40, bcap=1), npt(300, bcap=1)],
    "blocks_16": lambda: [npt(129, bcap=16), npt(640, bcap=16), npt(700, bcap=16)],
    "blocks_64": lambda: [npt(448, bcap=64), npt(64 * 33 + 5, bcap=64)],
    "blocks_128_256": lambda: [npt(1000), npt(1900), npt(4001)],
    "well_256": lambda: [npt(700, **hrsw()), npt(513, T=0.7, **hrsw())],
    "window_0": lambda: [npt(50, nbn=0), npt(9, nbn=0, boundary=nat.WALLS, vol_move=nat.VOL_LINEAR, max_dv=0.5)],
    "window_8": lambda: [npt(333, cutoff=4.0), npt(9, cutoff=4.0, L0=20.0)],
    "nvt": lambda: [npt(200, ensemble=nat.NLT), npt(2000, ensemble=nat.NLT, eci=0)],
}
ALL = {**{f"case_{k}": v for k, v in CASES.items()}, **LAYOUTS}


def go(chains, form, lanes):
    with Engine(chains, form=form, sample_capacity=SWEEPS, block_sweeps=BLOCK, log_accepts=True, sample_virial=True,
                block_lanes=lanes) as e:
        lay = [e.layout(c) for c in range(len(chains))]
        e.run(SWEEPS)
        log = e.read_accept_log(SWEEPS)
        smp, vir = e.read_samples_virial(SWEEPS)
        x, L, U = e.states()
        return lay, log, smp, vir, x, L, U, e.all_counters()


@pytest.mark.parametrize("form", ["batched_fp64", "batched_fp32"])
@pytest.mark.parametrize("name", sorted(ALL))
def test_same_bits_as_one_lane_per_block(gpu, name, form):
    print(f"[gpu] block lanes {name} {form}", flush=True)
    chains = ALL[name]()
    one, many = go(chains, form, 1), go(chains, form, 16)
    assert all(l["lanes"] == 1 for l in one[0])
    if all(l["w"] <= 8 and l["B"] <= 256 for l in one[0]):
        assert all(l["lanes"] > 1 for l in many[0])
    for a, b in zip(one[1], many[1]):
        assert np.array_equal(a, b)
    assert np.array_equal(one[2], many[2])
    assert np.array_equal(one[3], many[3])
    for a, b in zip(one[4], many[4]):
        assert np.array_equal(a, b)
    assert np.array_equal(one[5], many[5]) and np.array_equal(one[6], many[6])
    for k in one[7]:
        assert np.array_equal(one[7][k], many[7][k]), k


def test_few_chains_choose_it(gpu):
    """By default: a few chains take several lanes per block, thousands one."""
    with Engine([npt(64)], form="batched_fp32", sample_capacity=1) as e:
        assert e.layout(0)["lanes"] == 16
    with Engine([npt(300, chain_id=c) for c in range(3000)], form="batched_fp32", sample_capacity=1) as e:
        assert e.layout(0)["lanes"] == 1
    # the longest chain decides: 256 blocks with six partners a side gain nothing
    with Engine([npt(64), npt(4000)], form="batched_fp32", sample_capacity=1) as e:
        assert e.layout(0)["lanes"] == e.layout(1)["lanes"] == 1
    with Engine([npt(64), npt(64, **hrsw())], form="batched_fp32", sample_capacity=1) as e:
        assert e.layout(0)["lanes"] == e.layout(1)["lanes"] == 16
