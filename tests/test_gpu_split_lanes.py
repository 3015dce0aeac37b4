"""Lanes per block of split chains where the caller leaves them to the engine:
an engine is accepted wherever its segments are resident with one lane per
block, two lanes are taken where they gain (FP32; not in segments of 256 short
blocks), and a chain's bits do not depend on the choice."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import lj, yukawa

pytestmark = pytest.mark.gpu


def npt(N, c, bcap, **kw):
    return Chain(N=N, rho=0.5, T=1.0, P=0.5, ensemble=nat.NPT, vol_move=nat.VOL_LOG, max_dv=0.001, seed=41,
                 chain_id=c, eci=2, bcap=bcap, **(kw or lj()))


def go(chains, lanes=0, seg_lds=0, form="batched_fp32"):
    with Engine(chains, form=form, sample_capacity=4, block_sweeps=2, seg_lds=seg_lds, seg_lanes=lanes) as e:
        lay = [e.layout(c) for c in range(len(chains))]
        e.run(4)
        return lay, e.read_samples(4), e.states()[0]


def test_more_segments_than_compute_units(gpu):
    """100 LJ chains of 22,000 at up to 1024 blocks: 400 segments of 256
    blocks, resident three to a CU with one lane per block and one with two."""
    print("[gpu] split lanes: 400 segments", flush=True)
    chains = [npt(22000, c, 1024) for c in range(100)]
    lay, smp, x = go(chains)
    assert all(l["mode"] == "split" and l["segments"] == 4 and l["lanes"] == 1 for l in lay)
    with pytest.raises(nat.JmmError):
        Engine(chains, form="batched_fp32", sample_capacity=4, seg_lanes=2)
    for c in (0, 99):
        for lanes in (1, 2):
            _, s1, x1 = go([chains[c]], lanes)
            assert np.array_equal(s1[0], smp[c]) and np.array_equal(x1[0], x[c])


def test_gives_two_lanes_up_where_they_are_not_resident(gpu):
    """A chain of long blocks (two lanes gain) among 80 chains of 256-block
    segments (322 segments in all): one lane."""
    print("[gpu] split lanes: fall back to one", flush=True)
    chains = [npt(8192, 0, 64)] + [npt(16384, c, 1024) for c in range(1, 81)]
    seg_lds = 36000
    lay, smp, x = go(chains, seg_lds=seg_lds)
    assert [l["segments"] for l in lay] == [2] + [4] * 80 and all(l["lanes"] == 1 for l in lay)
    with pytest.raises(nat.JmmError):
        Engine(chains, form="batched_fp32", sample_capacity=4, seg_lds=seg_lds, seg_lanes=2)
    for c in (0, 80):
        lay1, s1, x1 = go([chains[c]], 2, seg_lds)
        assert lay1[0]["lanes"] == 2
        assert np.array_equal(s1[0], smp[c]) and np.array_equal(x1[0], x[c])


@pytest.mark.parametrize("form", ["batched_fp32", "batched_fp64"])
def test_choice_by_segment_and_block_length(gpu, form):
    """(particles, most blocks, split threshold) -> blocks per segment, lanes."""
    cases = [(22000, 1024, 0, 256, 1), (65536, 1024, 0, 256, 2), (1024 * 39, 1024, 0, 256, 1),
             (1024 * 40, 1024, 0, 256, 2), (22000, 256, 0, 128, 2), (512 * 16, 512, 18000, 128, 2)]
    for N, bcap, seg_lds, blocks, lanes in cases:
        for pot in (lj(), yukawa(cutoff=4.0)):
            with Engine([npt(N, 0, bcap, **pot)], form=form, sample_capacity=1, seg_lds=seg_lds) as e:
                l = e.layout(0)
            assert l["mode"] == "split" and l["B"] // l["segments"] == blocks, (N, bcap, l)
            assert l["lanes"] == (lanes if form == "batched_fp32" else 1), (N, bcap, l)


@pytest.mark.parametrize("form", ["batched_fp32", "batched_fp64"])
@pytest.mark.parametrize("lanes", [0, 1, 2])
def test_largest_segment_image(gpu, form, lanes):
    """Segments whose images leave just the 512 bytes of LDS that the split
    threshold sets aside (8 blocks of 5099, 2 segments of 20,408 doubles of the
    20,416): accepted, and equal to the chain in more segments."""
    print(f"[gpu] split lanes: largest image {form} {lanes}", flush=True)
    ch = npt(8 * 5099, 0, 8)
    lay, smp, x = go([ch], lanes, form=form)
    assert lay[0]["mode"] == "split" and lay[0]["segments"] == 2 and lay[0]["lds_bytes"] == 8 * 20408
    lay4, smp4, x4 = go([ch], lanes, seg_lds=90000, form=form)
    assert lay4[0]["segments"] == 4
    assert np.array_equal(smp, smp4) and np.array_equal(x[0], x4[0])
