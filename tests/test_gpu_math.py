"""The device forms of the elementary functions (include/wfh_math.h) against the host's, bit for bit: the
device splits and joins exponents with v_frexp / v_ldexp, selects the range cases at the end, takes
v_min / v_max and divides in range through a refined reciprocal estimate. Arguments are random bit
patterns, the ranges the model uses, the limits of each range case, subnormals, signed zeros,
infinities, NaN, mantissas next to the series' split, and quotients next to a rounding boundary over
the exponents that in-range division admits. (NaN results are compared as NaN.)"""
import ctypes

import numpy as np
import pytest

import oracle as O
from wflowhip.model import load_library

pytestmark = pytest.mark.gpu

OPS = {"exp": 0, "log": 1, "pow": 2, "cbrt": 3, "min": 4, "max": 5, "div": 6}
SPECIAL = np.array([0.0, -0.0, 1.0, -1.0, np.inf, -np.inf, np.nan, -np.nan, 5e-324, -5e-324, 2.2250738585072014e-308,
                    1.7976931348623157e308, -1.7976931348623157e308, 1e-310, 0.5, 2.0, 1e-30, 1e-6])


def device(name, a, b=None):
    a = np.ascontiguousarray(a, dtype=float)
    b = np.zeros_like(a) if b is None else np.ascontiguousarray(b, dtype=float)
    out = np.empty_like(a)
    print(f"{name}: {a.size} values", flush=True)
    rc = load_library().wfh_test_math(0, OPS[name], a.ctypes.data, b.ctypes.data, out.ctypes.data, a.size)
    assert rc == 0, rc
    return out


def same(got, want, *args):
    ok = (got.view(np.uint64) == want.view(np.uint64)) | (np.isnan(got) & np.isnan(want))
    k = np.nonzero(~ok)[0][:3]
    assert ok.all(), [(float(got[i]).hex(), float(want[i]).hex(), [float(x[i]).hex() for x in args]) for i in k]


def around(x, steps=40):
    """The doubles next to each of the values."""
    x = np.asarray(x, dtype=float)
    return (x.view(np.int64)[:, None] + np.arange(-steps, steps + 1)[None, :]).ravel().view(float)


def bits(rng, n):
    return rng.integers(0, 2 ** 64, n, dtype=np.uint64).view(float)


def test_exp():
    rng = np.random.default_rng(1)
    half_ln2 = (np.arange(-1074, 1024) + 0.5) * np.log(2.0)
    x = np.concatenate([SPECIAL, bits(rng, 400_000), rng.uniform(-760.0, 720.0, 600_000), rng.uniform(-746.0, -707.0, 200_000),
                        rng.uniform(-1.0, 1.0, 200_000), around([709.782712893384, -745.1332191019412, -708.3964185322641]),
                        around(half_ln2, 3)])
    same(device("exp", x), O.math("exp", x), x)


def test_log():
    rng = np.random.default_rng(2)
    split = np.ldexp(np.sqrt(0.5), np.arange(-1073, 1024))
    x = np.concatenate([SPECIAL, bits(rng, 400_000), np.abs(bits(rng, 600_000)), 10.0 ** rng.uniform(-323.5, 308.2, 400_000),
                        rng.integers(1, 2 ** 52, 100_000).view(float), 1.0 + rng.uniform(-1e-3, 1e-3, 200_000),
                        around([1.0, 2.2250738585072014e-308]), around(split, 3), around(np.ldexp(1.0, np.arange(-1022, 1024)), 3)])
    same(device("log", x), O.math("log", x), x)


@pytest.mark.parametrize("y", [0.2, 0.6 - 1.0, 0.6, 1.5, 5.0 / 3.0, None])
def test_pow(y):
    rng = np.random.default_rng(3)
    x = np.concatenate([SPECIAL, bits(rng, 200_000), 10.0 ** rng.uniform(-30, 12, 400_000), rng.uniform(0.0, 1.0, 200_000)])
    b = np.full_like(x, y) if y is not None else rng.uniform(-12.0, 12.0, x.size)
    same(device("pow", x, b), O.math("pow", x, b), x, b)


def test_cbrt():
    rng = np.random.default_rng(4)
    x = np.concatenate([SPECIAL, bits(rng, 300_000), rng.choice([1.0, -1.0], 300_000) * 10.0 ** rng.uniform(-30, 12, 300_000)])
    same(device("cbrt", x), O.math("cbrt", x), x)


@pytest.mark.parametrize("name", ["min", "max"])
def test_min_max(name):
    rng = np.random.default_rng(5)
    s = np.array(np.meshgrid(SPECIAL, SPECIAL)).reshape(2, -1)
    near = rng.uniform(-2.0, 2.0, 100_000)
    x = np.concatenate([s[0], bits(rng, 400_000), near, near])
    y = np.concatenate([s[1], bits(rng, 400_000), near, np.nextafter(near, 3.0)])
    same(device(name, x, y), O.math(name, x, y), x, y)


def test_in_range_division_is_ieee_division():
    """Divisors as the solves have them: f' and the log's 2 + f (2^-230 .. 2^590), the subsurface's
    (2^-100 .. 2^100); dividends 0 or 2^-400 .. 2^720 where the quotient is in range."""
    rng = np.random.default_rng(6)
    n = 600_000

    def mantissas(k):
        return rng.uniform(1.0, 2.0, k)

    eb = rng.integers(-230, 590, n)
    ea = np.clip(eb + rng.integers(-400, 400, n), -400, 720)
    sign = rng.choice([1.0, -1.0], n)
    b, a = np.ldexp(mantissas(n), eb), sign * np.ldexp(mantissas(n), ea)
    parts = [(a, b), (np.zeros(1000), b[:1000])]
    # both mantissas next to 1 or 2
    edge = np.concatenate([1.0 + np.arange(60) * 2.0 ** -52, 2.0 - np.arange(1, 60) * 2.0 ** -52])
    g = np.array(np.meshgrid(edge, edge)).reshape(2, -1)
    parts.append((g[0], g[1]))
    # quotients next to halfway between two doubles
    bm = mantissas(n)
    q = 1.0 + (rng.integers(0, 2 ** 51, n) * 2 + 1) * 2.0 ** -52
    near = (q * bm)
    for step in (-1, 0, 1):
        parts.append(((near.view(np.int64) + step).view(float), bm))
    # a / b with few bits in b: exact halves and their neighbours
    bi = rng.integers(1, 2 ** 26, n).astype(float)
    qi = (rng.integers(2 ** 26, 2 ** 27, n) * 2 + 1).astype(float)
    parts.append((bi * qi, bi))
    parts.append((np.nextafter(bi * qi, np.inf), bi))
    a, b = np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts])
    same(device("div", a, b) + 0.0, a / b + 0.0, a, b)
