"""Reads into rows wider than the read (max_sweeps above the pending sweeps):
the same records as rows of just the read's width, nothing written behind
them, and no allocation by jmm_read_samples_noalloc."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from jmmonedmc_amd import _native as nat
from jmmonedmc_amd.engine import SAMPLE_DTYPE, Chain, Engine

from helpers import lj

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "jmmonedmc_amd", "build")


def read(e, how, width):
    out = np.full((e.n, width * SAMPLE_DTYPE.itemsize), 0x5A, dtype=np.uint8)
    n = C.c_uint32()
    f = nat.lib().jmm_read_samples_noalloc if how == "noalloc" else nat.lib().jmm_read_samples
    rc = f(e.h, out.ctypes.data_as(C.POINTER(nat.Sample)), width, C.byref(n))
    assert rc == 0, nat.lib().jmm_last_error()
    return out, n.value


# records of 24 bytes: rows of 240 bytes (many to a 128 KB buffer, the last part
# of it ragged), of 60 KB (two), of 72 KB (one) and of 144 KB (beyond the limit)
@pytest.mark.parametrize("n,sweeps", [(700, 10), (3, 2500), (3, 3000), (3, 6000)])
@pytest.mark.parametrize("how", ["read", "noalloc"])
def test_wide_rows(gpu, how, n, sweeps):
    print(f"[gpu] wide rows {how} {n} x {sweeps}", flush=True)
    chains = [Chain(N=2, L0=20.0, T=1.0, seed=3, chain_id=c, **lj()) for c in range(n)]
    got = []
    for width in (sweeps, sweeps + 7):
        with Engine(chains, form="batched_fp32", sample_capacity=sweeps) as e:
            e.run(sweeps)
            out, m = read(e, how, width)
        assert m == sweeps
        rec = sweeps * SAMPLE_DTYPE.itemsize
        got.append(out[:, :rec].copy())
        assert np.all(out[:, rec:] == 0x5A)
    assert np.array_equal(got[0], got[1])


def test_noalloc_makes_no_large_allocation(gpu, tmp_path):
    print("[gpu] noalloc with wide rows: allocations", flush=True)
    prog = str(tmp_path / "noalloc_rows")
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{ROOT}/include", os.path.join(ROOT, "tests", "native", "noalloc_rows.cpp"),
                    "-o", prog, f"-L{BUILD}", "-ljmm_engine", f"-Wl,-rpath,{BUILD}", "-Wl,-rpath,/opt/rocm/lib"],
                   check=True)
    r = subprocess.run([prog], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "sweeps 100 large allocations 0" in r.stdout, r.stdout + r.stderr
