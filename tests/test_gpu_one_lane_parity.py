"""The batched kernel with one lane per block against the oracle at the sizes of
the oracle replays, where engines of few chains take several by themselves:
FP64 move for move (positions equal, energies to 1e-10), FP32 every decision
(energies to 1e-5, the rounding of its pair energies)."""
import numpy as np
import pytest

from jmmonedmc_amd.engine import Engine

from helpers import CASES, oracle_spec, rel

pytestmark = pytest.mark.gpu

SWEEPS = 40


@pytest.mark.parametrize("form,tol", [("batched_fp64", 1e-10), ("batched_fp32", 1e-5)])
@pytest.mark.parametrize("case", sorted(CASES))
def test_one_lane_per_block_replays_oracle(gpu, oracle, case, form, tol):
    print(f"[gpu] one lane per block {case} {form}", flush=True)
    chains = CASES[case]()
    with Engine(chains, form=form, log_accepts=True, sample_capacity=SWEEPS, block_sweeps=16, block_lanes=1) as e:
        assert all(e.layout(c)["lanes"] == 1 for c in range(len(chains)))
        e.run(SWEEPS)
        logs = e.read_accept_log(SWEEPS)
        smp = e.read_samples(SWEEPS)
        xs, Ls, Us = e.states()
        cnt = e.all_counters()
    for c, ch in enumerate(chains):
        orc = oracle.Chain(oracle_spec(oracle, ch))
        osmp, olog = orc.sweeps(SWEEPS, log=True)
        ox, oL, oU, osw = orc.state()
        assert np.array_equal(logs[c].ravel(), olog), c
        assert np.array_equal(xs[c], ox) and Ls[c] == oL and cnt["sweeps"][c] == osw, c
        assert rel(Us[c], oU) <= tol, c
        assert np.array_equal(smp[c]["acc_d"], osmp["acc_d"]) and np.array_equal(smp[c]["acc_v"], osmp["acc_v"]), c
        for k, ok in (("trials", "trials"), ("acc_d", "acc_d"), ("core_rejects", "hc_rej"),
                      ("wall_rejects", "wall_rej"), ("pair_terms", "pair_terms"), ("recomputes", "recomputes")):
            assert cnt[k][c] == orc.counter(ok), (c, k)
