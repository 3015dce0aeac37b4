"""Observables of configurations whose pairs reach past a wave of particles:
the force on a right-hand partner is handed over inside a wave, to the next
one, or evaluated again (across a tile's left edge, or beyond 64 partners).
No cutoff between walls, and rings dense enough for about 80 partners a side,
at sizes around one, two and four waves and around a tile, against the FP64
oracle.

Tolerances: as for the tiled kernel, FP64 terms differ from the oracle's by
their rounding and the order of the sums, 1e-11 of the sums' scale; FP32 terms
by their rounding, 1e-5 (dU/dx ten times that of its largest component, a
difference of two sides)."""
import math

import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, pair_observables, pair_observables_work

from helpers import lj, oracle_spec, yukawa
from test_gpu_obs_tiles import configs

pytestmark = pytest.mark.gpu


def case(kind, N):
    if kind == "no_cutoff":
        return Chain(N=N, L0=1.6 * N + 5.0, boundary=nat.WALLS, **dict(lj(), cutoff=math.inf, shifted=0)), 0.8
    pot = yukawa()
    pot["pot_p"] = (*pot["pot_p"][:2], 0.05, *pot["pot_p"][3:])
    return Chain(N=N, L0=max(0.25 * N, 45.0), boundary=nat.PERIODIC, **pot), 0.1


@pytest.mark.parametrize("N", [2, 63, 64, 65, 127, 129, 257, 321, 1025, 1100])
@pytest.mark.parametrize("kind", ["no_cutoff", "dense"])
def test_far_reaching_pairs_equal_oracle(gpu, oracle, N, kind):
    import torch
    chain, core = case(kind, N)
    L, n = chain.L0, 2
    X = configs(n, N, L, core, kind == "no_cutoff", N)
    print(f"[gpu] far-reaching pairs {kind} N={N}", flush=True)
    x = torch.tensor(X, dtype=torch.float64, device="cuda")
    Lt = torch.full((n,), L, dtype=torch.float64, device="cuda")
    need = pair_observables_work(chain, n)
    ref = [oracle.observables_x(oracle_spec(oracle, chain), X[c], L) for c in range(n)]
    for precision, tol in ((64, 1e-11), (32, 1e-5)):
        for work in ([0, need] if need else [0]):
            obs = torch.full((n, 6), float("nan"), dtype=torch.float64, device="cuda")
            grad = torch.full((n, N), float("nan"), dtype=torch.float64, device="cuda")
            ws = torch.full((max(work, 1),), float("nan"), dtype=torch.float64, device="cuda")
            pair_observables(chain, x.data_ptr(), Lt.data_ptr(), obs.data_ptr(), grad.data_ptr(), n, precision,
                             torch.cuda.current_stream().cuda_stream, ws.data_ptr() if work else None, work)
            torch.cuda.synchronize()
            for c in range(n):
                o, g = ref[c]
                scale = np.abs(o).max() + N
                assert np.all(np.abs(obs[c].cpu().numpy() - o) <= tol * scale), (precision, work, c)
                gs = np.abs(g).max() + 1.0
                assert np.all(np.abs(grad[c].cpu().numpy() - g) <= 10 * tol * gs), (precision, work, c)
