"""The kinematic-wave solve of the kernels (straight updates with in-range divisions, then kw_end) on the
host: bit for bit the reference's loop over ordinary flows, dry cells, flows at the smallest value,
operands at the limits of the straight path and far beyond them; and the bounds that its comments
rest on: where the straight path takes a case no term leaves the normal range, and in the four
updates that run without a test f + C falls less than 3.6-fold in each."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("kw") / "libkw.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-mfma",
                    "-D__host__=", "-D__device__=", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "wflow.jl_amd", "csrc"), "-o", str(out),
                    os.path.join(HERE, "kw_host.cpp")], check=True)
    return ctypes.CDLL(str(out))


def solve(lib, q_in, q_prev, q_lat, alpha, dt, dx):
    z = np.ascontiguousarray(np.stack(np.broadcast_arrays(q_in, q_prev, q_lat, alpha, dt, dx), axis=1), dtype=float)
    out = np.empty((len(z), 10))
    lib.host_kw(z.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p), ctypes.c_long(len(z)))
    return z, out


def logs(rng, lo, hi, n):
    return 10.0 ** rng.uniform(lo, hi, n)


CASES = {
    # flows, roughness, step lengths and cell sizes of models, dry cells among them
    "model": lambda r, n: (logs(r, -9, 4, n) * (r.random(n) > 0.1), np.where(r.random(n) < 0.2, 1e-30, logs(r, -9, 4, n)),
                           logs(r, -9, -1, n) * r.choice([1.0, 0.0, -1.0], n), logs(r, -1, 2, n),
                           r.choice([900.0, 3600.0, 86400.0, 994.6119029285007], n), logs(r, 1, 4, n)),
    # nothing at all, or nothing before
    "dry": lambda r, n: (logs(r, -12, 2, n) * (r.random(n) > 0.5), np.zeros(n), logs(r, -12, -2, n) * (r.random(n) > 0.5),
                         logs(r, -1, 2, n), 3600.0, logs(r, 1, 4, n)),
    # the smallest flow with a large residual: the long way down, with both signs of C
    "fall": lambda r, n: (logs(r, -8, 2, n), np.full(n, 1e-30), logs(r, -8, 0, n) * r.choice([1.0, -1.0], n),
                          logs(r, -3, 3, n), logs(r, 2, 5, n), logs(r, 1, 4, n)),
    # the whole range that the straight path admits, and beyond
    "limits": lambda r, n: (logs(r, -5, 14, n) * r.choice([1.0, 1e-6], n),
                            np.where(r.random(n) < 0.3, 2.0 ** r.uniform(-101, -99, n), logs(r, -150, 10, n)),
                            logs(r, -9, 3, n) * r.choice([1.0, -1.0], n), 2.0 ** r.uniform(-31, 61, n),
                            2.0 ** r.uniform(-31, 61, n), 1.0),
}


@pytest.mark.parametrize("kind", sorted(CASES))
def test_the_solve_is_the_loop(lib, kind):
    n = 150_000 if kind != "limits" else 60_000
    rng = np.random.default_rng(sorted(CASES).index(kind))
    z, o = solve(lib, *CASES[kind](rng, n))
    same = (o[:, 0:2].view(np.uint64) == o[:, 2:4].view(np.uint64)).all(axis=1)
    assert same.all(), z[~same][:3]
    fast = o[:, 4] == 1.0
    if kind != "dry":
        assert fast.mean() > 0.1, fast.mean()
    assert (o[fast, 5] < 2.0 ** 130).all(), (o[fast, 5].max(), z[fast][np.argmax(o[fast, 5])])
    assert (o[fast, 6] < 2.0 ** 720).all() and (o[fast, 7] < 2.0 ** 590).all()
    assert (o[fast, 8] >= 2.0 ** -69).all()
    assert (o[:, 9] < 3.6).all(), (o[:, 9].max(), z[np.argmax(o[:, 9])])
    if kind == "fall":
        assert (o[:, 9] > 3.0).mean() > 0.5  # (the long way down was taken)
