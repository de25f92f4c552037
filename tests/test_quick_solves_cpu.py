"""The prepared forms of the routing solves against the forms they stand for, on the host: the
subsurface solve with its inflow-independent part formed beforehand (ssf_quick_solve) against
kinematic_wave_ssf, and in-range quotients against IEEE division. Both are the same operations, so
the results must be equal bit for bit wherever the prepared form takes a case."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("quick") / "libquick.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-mfma",
                    "-D__host__=", "-D__device__=", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "wflow.jl_amd", "csrc"), "-o", str(out),
                    os.path.join(HERE, "quick_host.cpp")], check=True)
    return ctypes.CDLL(str(out))


def rows(rng, n):
    """Subsurface solves over the ranges of real columns, dry cells, water tables at the surface and at
    the soil's bottom, full layers and values far out of range among them."""
    z = np.zeros((n, 16))
    z[:, 0] = 10.0 ** rng.uniform(-9, 1, n) * (rng.random(n) > 0.1)                 # q_in
    z[:, 1] = np.where(rng.random(n) < 0.1, 0.0, 10.0 ** rng.uniform(-9, 1, n))      # q_prev
    z[:, 6] = rng.uniform(0.4, 2.5, n)                                              # soil thickness
    u = rng.random(n)
    z[:, 2] = np.where(u < 0.1, 0.0, np.where(u > 0.9, z[:, 6], z[:, 6] * rng.random(n)))  # water table
    z[:, 3] = 10.0 ** rng.uniform(-8, -1, n) * rng.choice([-1.0, 0.0, 1.0], n)      # lateral net flux
    z[:, 4] = 10.0 ** rng.uniform(-5, 0, n)
    z[:, 5] = rng.uniform(0.02, 0.4, n)
    z[:, 7] = rng.choice([600.0, 3600.0, 86400.0, 994.6119029285007], n)
    z[:, 8] = rng.uniform(30.0, 1500.0, n)
    z[:, 9] = rng.uniform(30.0, 1500.0, n)
    z[:, 10] = 10.0 ** rng.uniform(-6, 0, n)
    z[:, 11] = 10.0 ** rng.uniform(-6, -2, n)
    z[:, 12] = rng.uniform(0.1, 5.0, n)
    z[:, 13] = np.where(rng.random(n) < 0.5, np.inf, rng.uniform(0.1, 1.0, n))
    z[:, 14] = rng.uniform(0.1, 0.5, n)
    z[:, 15] = rng.random(n)
    odd = rng.random(n) < 0.02
    z[odd, 0] = rng.choice([1e-310, 1e200, -0.0, 5e-324, np.inf], int(odd.sum()))
    odd = rng.random(n) < 0.02
    z[odd, 1] = rng.choice([1e-310, 1e200, 1e-30, 5e-324], int(odd.sum()))
    return z


def test_prepared_subsurface_solve_is_the_solve(lib):
    n = 400_000
    z = rows(np.random.default_rng(3), n)
    out = np.empty((n, 9))
    lib.host_ssf_pair(z.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p), ctypes.c_long(n))
    assert not (out[:, 0] < 0).any(), "the column's update is deferred differently"
    taken = out[:, 0] == 1.0
    assert 0.2 < taken.mean() < 0.99, taken.mean()
    a, b = out[taken, 1:5], out[taken, 5:9]
    assert np.array_equal(a + 0.0, b + 0.0)  # (+ 0.0: a zero's sign is not compared)
    for name, cond in (("dry", (z[:, 0] + z[:, 1] == 0.0) & (z[:, 3] <= 0.0)), ("falling", out[:, 8] < 0.0),
                       ("rising", out[:, 8] > 0.0), ("surface", z[:, 2] == 0.0)):
        assert (taken & cond).sum() > 200, name


def test_in_range_quotients_are_ieee_quotients(lib):
    rng = np.random.default_rng(4)
    n = 2_000_000
    a = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-200, 200, n)
    b = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-200, 200, n)
    # mantissas next to 1 and 2, and quotients next to a rounding boundary
    b[: n // 4] = np.nextafter(2.0, 0.0) - rng.integers(0, 50, n // 4) * 2.0 ** -52
    a[n // 4: n // 2] = 1.0 + rng.integers(0, 50, n // 2 - n // 4) * 2.0 ** -52
    m = slice(n // 2, 3 * n // 4)
    q = 1.0 + (rng.integers(0, 2 ** 52, n // 4) + 0.5) * 2.0 ** -52
    b[m] = rng.uniform(1.0, 2.0, n // 4)
    a[m] = q * b[m]
    out = np.empty(n)
    lib.host_div(a.ctypes.data_as(ctypes.c_void_p), b.ctypes.data_as(ctypes.c_void_p),
                 out.ctypes.data_as(ctypes.c_void_p), ctypes.c_long(n))
    assert np.array_equal(out, a / b)
