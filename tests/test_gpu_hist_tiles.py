"""The histogram kernel's tiles and its window of segments counted in LDS:
chain lengths around a tile and around the lengths where a tile has more
lanes per particle, folded periodic ends, windows that hold all segments, a
part of them, or none, against the oracle's all-pairs binning (whole numbers:
equal)."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import lj, oracle_spec

pytestmark = pytest.mark.gpu

NS = [20, 63, 64, 65, 128, 129, 256, 257, 1025]
# all segments in the window; 16 of 40; bins beyond the window's size; one wide
# segment whose pairs reach over most of the chain; segments narrower than a pair
SPECS = [dict(gns=6, gsw=30.0, gnb=40, gbw=0.25), dict(gns=40, gsw=5.0, gnb=1000, gbw=0.05),
         dict(gns=2, gsw=100.0, gnb=17000, gbw=0.001), dict(gns=1, gsw=4000.0, gnb=300, gbw=1.0),
         dict(gns=500, gsw=0.5, gnb=20, gbw=0.5), dict(gns=0, gsw=1.0, gnb=5, gbw=1.0)]


@pytest.mark.parametrize("boundary", [nat.PERIODIC, nat.WALLS])
@pytest.mark.parametrize("spec", range(len(SPECS)))
def test_tiled_histograms_equal_oracle(gpu, oracle, boundary, spec):
    hs = dict(SPECS[spec], rhonb=60, rbw=5.0)
    chains = [Chain(N=N, L0=max(1.5 * N, 30.0), boundary=boundary, seed=5, chain_id=c, **lj()) for c, N in enumerate(NS)]
    print(f"[gpu] tiled histograms boundary={boundary} {hs}", flush=True)
    with Engine(chains, form="batched_fp64", sample_capacity=8) as e:
        e.hist_configure(3, **hs)
        e.run(6)
        xs, Ls, _ = e.states()
        rho, g, ns = e.hist_read()
    assert ns == 2
    for c, ch in enumerate(chains):
        orc = oracle.Chain(oracle_spec(oracle, ch))
        want_r = np.zeros(hs["rhonb"], dtype=np.uint64)
        want_g = np.zeros((hs["gns"], hs["gnb"]), dtype=np.uint64)
        for _ in range(2):
            orc.sweeps(3)
            x, L, _, _ = orc.state()
            r1, g1 = oracle.hist_x(orc.spec, x, L, hs["rhonb"], hs["rbw"], hs["gns"], hs["gsw"], hs["gnb"], hs["gbw"])
            want_r += r1
            want_g += g1
        assert np.array_equal(x, xs[c]) and np.array_equal(rho[c], want_r), c
        if hs["gns"]:
            assert np.array_equal(g[c], want_g), c


def test_many_chains_beside_a_long_one(gpu):
    """A launch of 64 workgroups a chain whose lanes would pass 2^32 at 1024 a
    workgroup: every particle is counted all the same."""
    n = 66000
    chains = [Chain(N=17000 if c == 1000 else 2, L0=40000.0 if c == 1000 else 40.0, boundary=nat.WALLS, seed=5,
                    chain_id=c, **lj()) for c in range(n)]
    print(f"[gpu] histograms of {n} chains", flush=True)
    with Engine(chains, form="batched_fp64", sample_capacity=1) as e:
        e.hist_configure(1, rhonb=2, rbw=50000.0, gns=1, gsw=50000.0, gnb=2, gbw=50000.0)
        e.run(1)
        rho, g, ns = e.hist_read()
    assert ns == 1
    N = np.array([ch.N for ch in chains], dtype=np.uint64)
    assert np.array_equal(rho.sum(1), N)
    assert np.array_equal(g.sum((1, 2)), N * (N - np.uint64(1)))
