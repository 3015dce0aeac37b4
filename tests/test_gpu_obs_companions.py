"""A chain's energies, observables and gradients do not depend on the chains it
shares an engine with (the workgroups of the observables kernel take their
shape from the longest): the same bits alone and beside shorter and longer
chains, at lengths around one and two tiles of 512 and a tile's waves."""
import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import Chain, Engine

from helpers import hrsw, lj, yukawa

pytestmark = pytest.mark.gpu

POTS = {"lj": lj, "hrsw": hrsw, "yukawa": yukawa}


def observed(N, beside, kind, boundary, form):
    def chain(n, c):
        return Chain(N=n, L0=max(1.6 * n, 45.0), T=1.0, seed=17, chain_id=c, boundary=boundary, **POTS[kind]())
    with Engine([chain(m, 1 + k) for k, m in enumerate(beside)] + [chain(N, 0)], form=form, sample_capacity=4) as e:
        U0 = e.states()[2][-1]
        e.run(4)
        smp = e.read_samples(4)[-1]
        obs, grad = e.observables(want_grad=True)
        L = e.states()[1]
        return U0, smp, obs[-1], np.array(grad[-1]), e.full_energy()[-1], e.scaled_energy(L * 0.999)[-1]


@pytest.mark.parametrize("form", ["batched_fp32", "batched_fp64"])
@pytest.mark.parametrize("boundary", [nat.PERIODIC, nat.WALLS])
@pytest.mark.parametrize("kind", sorted(POTS))
def test_same_bits_beside_any_chain(gpu, kind, boundary, form):
    for N in (40, 100, 511, 512, 513, 600, 1000, 1024, 1025, 1537):
        print(f"[gpu] observables beside others {kind} {boundary} {form} N={N}", flush=True)
        alone = observed(N, [], kind, boundary, form)
        for beside in ([64], [700], [1024], [1300], [30, 5000]):
            for a, b in zip(alone, observed(N, beside, kind, boundary, form)):
                assert np.array_equal(a, b), (N, beside)
