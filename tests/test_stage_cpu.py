"""The staged upload of host forcing (wfh_stage.h) on the host: pieces of every size arrive whole and in
place, a slot is waited for before it is filled again, a failing wait or transfer ends the call with its
threads, and an allocation or event that could not be made is made by the next call. The call has no
more threads than CPUs it may use, and they sleep while it waits for transfers."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("stage") / "libstage.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-pthread",
                    "-I", os.path.join(ROOT, "wflow.jl_amd", "csrc"), "-o", str(out),
                    os.path.join(HERE, "stage_host.cpp")], check=True)
    return ctypes.CDLL(str(out))


def stage(lib, n, fail_wait=-1, fail_send=-1, wait_us=0):
    a = np.random.default_rng(n).random(3 * n)
    out = np.full(3 * n, np.nan)
    info = np.zeros(5)
    ok = lib.host_stage(a.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p), ctypes.c_long(n),
                        fail_wait, fail_send, wait_us, info.ctypes.data_as(ctypes.c_void_p))
    return ok, a, out, info


@pytest.mark.parametrize("n", [1, 7, 2 ** 18 - 1, 2 ** 18, 2 ** 18 + 1, 3 * 2 ** 18 + 5, 1_000_003])
def test_everything_arrives(lib, n):
    for wait_us in (0, 50):
        ok, a, out, info = stage(lib, n, wait_us=wait_us)
        assert ok == 1 and np.array_equal(a, out) and info[3] == 0
        assert info[2] == 3 * -(-n // 2 ** 18)


@pytest.mark.parametrize("where", ["fail_wait", "fail_send"])
@pytest.mark.parametrize("piece", [0, 1, 5, 8])
def test_a_failure_ends_the_call(lib, where, piece):
    for _ in range(5):
        ok, a, out, info = stage(lib, 3 * 2 ** 18, **{where: piece})
        assert ok == 0
        sent = piece * 2 ** 18
        assert np.array_equal(a[:sent], out[:sent]) and np.isnan(out[sent:]).all()


@pytest.mark.parametrize("fail", [-1, 0, 1, 2, 4])
def test_what_could_not_be_made_is_made_by_the_next_call(lib, fail):
    rc, made, count = (ctypes.c_int * 2)(), (ctypes.c_int * 2)(), (ctypes.c_int * 2)()
    lib.host_ready(fail, rc, made, count)
    assert list(rc) == [int(fail < 0), 1]
    assert list(made) == [int(fail < 0), 1]
    assert list(count) == [1, 4]


def test_no_more_threads_than_usable_cpus(lib):
    cpus = os.sched_getaffinity(0)
    try:
        for use in (1, 2, 3):
            if len(cpus) >= use:
                os.sched_setaffinity(0, sorted(cpus)[:use])
                ok, a, out, info = stage(lib, 1_000_003)
                assert ok == 1 and np.array_equal(a, out)
                assert info[4] == use
    finally:
        os.sched_setaffinity(0, cpus)
    assert stage(lib, 1_000_003)[3][4] == min(8, len(cpus))


def test_threads_sleep_while_the_call_waits(lib):
    ok, _, _, info = stage(lib, 3 * 2 ** 18, wait_us=30_000)  # nine pieces, a wait of 30 ms before each
    assert ok == 1 and info[1] > 0.27
    assert info[0] < 0.5 * info[1], info  # CPU time of all threads; spinning helpers take seven seconds a second
