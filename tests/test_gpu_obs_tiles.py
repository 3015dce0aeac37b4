"""The observables kernel cut into tiles: configurations at the sizes where
the cut changes (one workgroup up to 1024 particles, tiles of 256 beyond),
with remainders of a tile, on both boundaries, with and without a work array,
and engine chains of mixed lengths, against the FP64 oracle.

Tolerances: FP64 pair terms differ from the oracle's by their rounding and
the order of the sums only, at most a few ulp of the sum of |terms|: 1e-11 of
that scale as for the untiled kernel; FP32 terms by their FP32 rounding, 1e-5
(dU/dx: ten times that of the largest component, a difference of two sides)."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine, pair_observables, pair_observables_work

from helpers import lj, oracle_spec, yukawa

pytestmark = pytest.mark.gpu


def configs(n, N, L, core, walls, seed):
    rng = np.random.default_rng(seed)
    e = rng.exponential(size=(n, N + 1))
    gaps = core + e * ((L - (N + 1) * core) / e.sum(1, keepdims=True))
    return np.cumsum(gaps[:, :N], 1) - L / 2.0 - (0.0 if walls else core / 2.0)


@pytest.mark.parametrize("N", [1, 2, 255, 1023, 1024, 1025, 1279, 1281, 3000])
@pytest.mark.parametrize("boundary", [nat.PERIODIC, nat.WALLS])
@pytest.mark.parametrize("kind", ["lj", "yukawa"])
def test_tiled_observables_equal_oracle(gpu, oracle, N, boundary, kind):
    import torch
    pot = lj() if kind == "lj" else yukawa()
    L, n = max(1.6 * N, 45.0), 3
    chain = Chain(N=N, L0=L, boundary=boundary, **pot)
    X = configs(n, N, L, 0.8 if kind == "lj" else 0.55, boundary == nat.WALLS, N)
    print(f"[gpu] tiled observables {kind} N={N} boundary={boundary}", flush=True)
    x = torch.tensor(X, dtype=torch.float64, device="cuda")
    Lt = torch.full((n,), L, dtype=torch.float64, device="cuda")
    need = pair_observables_work(chain, n)
    assert (need > 0) == (N > 1024)
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


def test_engine_chains_of_mixed_lengths(gpu, oracle):
    """Chains on both sides of the cut in one engine: every chain's row and
    gradient offset, and the energies of rescaled configurations."""
    Ns = [1300, 5, 1024, 257, 1025, 64]
    chains = [Chain(N=N, L0=max(1.7 * N, 12.0), seed=3, chain_id=c, **lj()) for c, N in enumerate(Ns)]
    print("[gpu] engine observables of mixed lengths", flush=True)
    with Engine(chains, form="batched_fp64", sample_capacity=4) as e:
        e.run(4)
        e.sync()
        xs, L, U = e.states()
        obs, grad = e.observables(want_grad=True)
        full, scaled = e.full_energy(), e.scaled_energy(L * 1.01)
    for c, ch in enumerate(chains):
        o, g = oracle.observables_x(oracle_spec(oracle, ch), xs[c], L[c])
        scale = np.abs(o).max() + ch.N
        assert np.all(np.abs(obs[c] - o) <= 1e-11 * scale)
        assert np.all(np.abs(grad[c] - g) <= 1e-11 * (np.abs(g).max() + 1.0))
        assert abs(full[c] - o[0]) <= 1e-11 * scale
        o2, _ = oracle.observables_x(oracle_spec(oracle, ch), xs[c] * 1.01, L[c] * 1.01)
        assert abs(scaled[c] - o2[0]) <= 1e-11 * scale
