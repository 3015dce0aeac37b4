"""The same chain split over workgroups and run from HBM (a split threshold that
no segment fits): the same bits, also where they show: a lattice with zero
energy, so that the box-length moves' energy changes are not rounded to a large
total."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import lj

pytestmark = pytest.mark.gpu

SWEEPS = 30
# the spacing at which 4 (a^-12 - a^-6) + 4 ((2a)^-12 - (2a)^-6) = 0
SPACING = 0.9974598856126655


@pytest.mark.parametrize("form", ["batched_fp32", "batched_fp64"])
@pytest.mark.parametrize("N,bcap", [(24011, 256), (40000, 256), (30011, 1024)])
def test_split_chain_equals_chain_in_hbm(gpu, form, N, bcap):
    print(f"[gpu] split and HBM {form} N={N}", flush=True)
    ch = Chain(N=N, L0=N * SPACING, T=1.0, P=25.0, ensemble=nat.NPT, vol_move=nat.VOL_LOG, max_dv=1e-3, max_step=0.0,
               seed=31, bcap=bcap, **lj(cutoff=2.5, shifted=0))
    got = []
    for seg_lds, mode in ((0, "split"), (8, "hbm")):
        with Engine([ch], form=form, sample_capacity=SWEEPS, block_sweeps=10, seg_lds=seg_lds) as e:
            assert e.layout(0)["mode"] == mode
            e.run(SWEEPS)
            got.append((e.read_samples(SWEEPS), e.states()[0][0]))
    (s0, x0), (s1, x1) = got
    assert s0["acc_v"].sum() > 0
    assert np.array_equal(s0, s1) and np.array_equal(x0, x1)
