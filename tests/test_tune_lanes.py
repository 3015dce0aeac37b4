"""The tuner offers every choice of lanes per block (host logic, no GPU)."""
import pytest

from jmmonedmc_amd import configs, tune as t
from jmmonedmc_amd._native import JmmError


def test_split_lanes_at_every_threshold():
    big = t.candidates_for(configs.c5(2))
    for seg_lds in (None, 65536, 32768):
        assert {c["seg_lanes"] for c in big if "seg_lanes" in c and c.get("seg_lds") == seg_lds} == {1, 2}
    assert not any("seg_lds" in c and "seg_lanes" not in c for c in big)


def test_block_lanes_are_timed(monkeypatch):
    """Every candidate is created; the fastest wins, also among the lanes; a
    refused one is left out."""
    seen = []

    class Fake:
        def __init__(self, chains, form, device, sample_capacity, block_sweeps, **opts):
            seen.append(opts)
            if opts.get("seg_lanes") == 2:
                raise JmmError("not resident")
            self.ms = 1.0 if opts.get("block_lanes") == 1 else 2.0

        def __enter__(self):
            return self

        def __exit__(self, *exc):
            pass

        def run(self, n):
            pass

        def sync(self):
            pass

        def kernel_time(self, reset=False):
            return 1, self.ms, 1

    monkeypatch.setattr(t, "Engine", Fake)
    res = t.tune(configs.c5(2), candidates=t.candidates_for(configs.c5(2)) + t.lane_candidates())
    assert {o.get("block_lanes") for o in seen} == {None, 1, 2}
    assert res.best["block_lanes"] == 1
    assert len(seen) == len({str(sorted(o.items())) for o in seen})
    assert [res.ms_per_sweep[k] for k in res.ms_per_sweep if "seg_lanes=2" in k] == [None] * 3
    with pytest.raises(JmmError):
        t.tune(configs.c5(2), candidates=[dict(seg_lanes=2)])
