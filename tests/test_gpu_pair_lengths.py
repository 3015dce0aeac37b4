"""PairEnergy refuses lengths that do not hold one for each configuration (the
kernel reads n of them), without a copy from the device, and takes the shapes
that do."""
import pytest

from jmmonedmc_amd.configs import LJ
from jmmonedmc_amd.engine import Chain

pytestmark = pytest.mark.gpu


def test_lengths_one_a_configuration(gpu):
    import torch

    from jmmonedmc_amd.autograd import PairEnergy, observables
    print("[gpu] pair energy lengths", flush=True)
    N, n = 64, 3
    chain = Chain(N=N, rho=0.5, **LJ)
    x = (torch.arange(N, dtype=torch.float64, device="cuda") - 31.5).mul(2.0).repeat(n, 1) * 0.99
    th = torch.tensor([1.0, 1.0], dtype=torch.float64)

    def lengths(*shape):
        return torch.full(shape, 130.0, dtype=torch.float64, device="cuda")

    for shape in ((), (0,), (1,), (2,), (1, 3), (3, 2)):
        for call in (lambda L: PairEnergy.apply(x, L, th, chain, 64), lambda L: observables(x, L, chain, th)):
            with pytest.raises(ValueError):
                call(lengths(*shape))
    want = PairEnergy.apply(x, lengths(3), th, chain, 64)
    for shape in ((3, 1), (5,)):
        assert torch.equal(PairEnergy.apply(x, lengths(*shape), th, chain, 64), want)
