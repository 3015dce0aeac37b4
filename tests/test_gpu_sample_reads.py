"""Sample reads at the sizes where their route changes (pinned staging up to
64 KiB, one device copy beyond; rows as wide as the read or wider), with and
without virials, drained repeatedly: the same values as one large read of the
same chains (exact), and the sweeps after a read land in the next one."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import hrsw, lj

pytestmark = pytest.mark.gpu


def chains(n):
    # two potentials in alternation: the engine's own chain order is not the caller's
    return [Chain(N=12 + c % 5, L0=40.0 + c, T=1.0, P=0.5, ensemble=nat.NPT, seed=5, chain_id=c,
                  **(lj() if c % 2 else hrsw())) for c in range(n)]


@pytest.mark.parametrize("n", [1, 3, 40])
@pytest.mark.parametrize("virial", [False, True])
def test_reads_by_every_route(gpu, n, virial):
    print(f"[gpu] sample reads n={n} virial={virial}", flush=True)
    total = 160
    with Engine(chains(n), form="batched_fp64", sample_capacity=total, sample_virial=True) as e:
        e.run(total)
        want, wvir = e.read_samples_virial(total)
    row = 24 + (16 if virial else 0)
    # per-chain sweeps below, at and above the staging limit (where n reaches it)
    edge = max(1, min(70, 65536 // (row * n)))
    counts = [1, edge, min(edge + 1, 71)]
    with Engine(chains(n), form="batched_fp64", sample_capacity=total, sample_virial=True) as e:
        at = 0
        for m in counts + counts[:1]:
            for room in (m, m + 3):
                if at + m > total:
                    break
                e.run(m)
                if virial:
                    got, vir = e.read_samples_virial(room)
                    assert np.array_equal(vir, wvir[:, at:at + m])
                else:
                    got = e.read_samples(room)
                assert got.shape == (n, m)
                assert np.array_equal(got, want[:, at:at + m])
                at += m
        x, L, U, sweep = e.state(n - 1)
        xs, Ls, Us = e.states()
        assert sweep == at and np.array_equal(x, xs[n - 1]) and L == Ls[n - 1] and U == Us[n - 1]
