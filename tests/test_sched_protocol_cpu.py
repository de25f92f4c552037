"""The routing exchange of the kernels (run_sched, chunk_ranks: the same source, built for the host) under
random interleavings of the lanes and waves, a limited number of resident waves and outflow that
becomes visible late.

  - With tickets in chunk order every step drains for any interleaving and any number of resident
    waves down to one, the results are the sequential sweep's bit for bit, each cell publishes its
    outflow once, and every slot is empty again at the end (the next launch starts clean). That
    covers one and several sub-steps (more than the inbox has rows), the inbox of one row and of
    four, cells with up to nine upstream cells (the inbox has places for four), solves that end
    late, and chunks of which only some cells take part.
  - A cell of a chunk has the rank next above its upstream cells of the chunk.
  - A wait that is never met (of an edge with a place in the inbox, or of one beyond) ends by the spin
    limit, and nothing but right values has been published, by no wave: one that has given up, or
    was told to, has not passed on what it computed without its inflow.
  - The check is not vacuous: tickets in the reverse order do not drain, and wrong ranks are seen.
"""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
WAVE = 64
SSF, OL, RIV, RIV_RES, SNOW = range(5)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("sched") / "libsched.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-mfma", "-w", "-U_FORTIFY_SOURCE",
                    "-D__host__=", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "wflow.jl_amd", "csrc"), "-o", str(out),
                    os.path.join(HERE, "sched_host.cpp")], check=True)
    return ctypes.CDLL(str(out))


class Net:
    """n positions, upstream cells before their downstream cell. reach: mean distance to the downstream
    cell; chain: positions from there on form one chain; hubs: cells that draw up to nine upstream
    cells from the 150 positions before them; share: part of the positions that take part."""

    def __init__(self, n, seed, reach=128, chain=None, hubs=0, share=1.0):
        rng = random.Random(seed)
        self.n = n
        self.part = np.array([rng.random() < share for _ in range(n)], np.uint8)
        down = np.full(n, -1, np.int32)
        for v in range(n - 1):
            if not self.part[v] or rng.random() < 0.05:
                continue
            down[v] = v + 1 if chain is not None and v >= chain else min(n - 1, v + 1 + int(rng.expovariate(1 / reach)))
        for _ in range(hubs):
            v = rng.randrange(10, n)
            for u in rng.sample(range(max(0, v - 150), v), min(v, 9)):
                if self.part[u]:
                    down[u] = v
        down[[v for v in range(n) if down[v] >= 0 and not self.part[down[v]]]] = -1
        self.down = down
        self.ups = [[] for _ in range(n)]
        for v in range(n):
            if down[v] >= 0:
                self.ups[down[v]].append(v)
        self.level = np.zeros(n, np.int32)
        for v in range(n):
            if down[v] >= 0:
                self.level[down[v]] = max(self.level[down[v]], self.level[v] + 1)
        self.up_ptr = np.concatenate([[0], np.cumsum([len(u) for u in self.ups])]).astype(np.int32)
        self.up_idx = np.array([u for us in self.ups for u in us] + [0], np.int32)
        self.frac = np.array([rng.choice([0.0, 0.25, 1.0, rng.random()]) for _ in range(n)])
        self.up_f = np.ascontiguousarray(self.frac[self.up_idx])
        self.opens = np.array([rng.random() < 0.3 for _ in range(n)], np.uint8)


def _p(a):
    return None if a is None else a.ctypes.data_as(ctypes.c_void_p)


def ranks(lib, net, gap):
    nch = (net.n + WAVE - 1) // WAVE
    rank, nrank = np.zeros(net.n, np.uint8), np.zeros(nch, np.uint8)
    lib.host_ranks(ctypes.c_long(net.n), _p(net.part), _p(net.down), _p(net.level), gap, _p(rank), _p(nrank))
    return rank, nrank


def sequential(net, fold, S, fams, q0, lat, acc0):
    """Outflow of every cell and sub-step, the last outflow and the sum of the first fold."""
    pub, q_out, acc_out = np.zeros((fams, S, net.n)), np.zeros((fams, net.n)), np.zeros((fams, net.n))
    for fam in range(fams):
        q = q0[fam].tolist()
        total = [0.0] * net.n
        for k in range(S):
            out = [0.0] * net.n
            for v in range(net.n):
                if not net.part[v]:
                    continue
                a1, a2 = (float(acc0[fam, v]) if acc0 is not None else 0.0), 0.0
                for u in net.ups[v]:
                    f = float(net.frac[u])
                    if fold == SSF:
                        a1, a2 = a1 + out[u] * (1.0 - f), a2 + out[u] * f
                    elif fold == OL:
                        a1, a2 = a1 + out[u] * f, a2 + out[u] * (1.0 - f)
                    elif fold == RIV_RES and f != 0.0:
                        a2 = out[u]
                    else:
                        a1 = a1 + out[u]
                total[v] = total[v] + a1
                out[v] = 0.5 * q[v] + 0.25 * a1 + 0.125 * a2 + float(lat[fam, v]) * (1.0 + k)
            q = out
            pub[fam, k] = out
        q_out[fam], acc_out[fam] = q, total
    q_out[:, net.part == 0] = 0.0
    return pub, q_out, acc_out


def run(lib, net, fold, ring, S, fams=2, seed=0, resident=4, delay=30, limit=10 ** 9, reverse=False, unmet=None,
        spoil_ranks=False, gap=None):
    rng = np.random.default_rng(seed)
    q0, lat = rng.random((fams, net.n)), rng.random((fams, net.n))
    acc0 = rng.random((fams, net.n)) if fold == SNOW else None
    want = sequential(net, fold, S, fams, q0, lat, acc0)
    rank, nrank = ranks(lib, net, (4 if S > 1 else 1) if gap is None else gap)
    if spoil_ranks:
        rank[:] = 0
    up_node, up_slot = net.up_idx.copy(), net.up_idx.copy()
    if unmet is not None:  # this edge looks like one from another chunk whose outflow never comes
        e, v = unmet
        up_node[e] = v + WAVE if v + WAVE < net.n else v - WAVE
        up_slot[e] = net.n
    q, acc = np.zeros((fams, net.n)), np.zeros((fams, net.n))
    rc = lib.host_step(fold, ring, ctypes.c_long(net.n), S, fams, _p(net.part), _p(net.up_ptr), _p(up_node),
                       _p(up_slot), _p(net.up_f), _p(net.down), _p(rank), _p(nrank), _p(q0), _p(lat), _p(net.opens),
                       _p(want[0]), _p(acc0), ctypes.c_long(net.n + 1), resident, ctypes.c_uint(seed), delay,
                       ctypes.c_long(limit), int(reverse), _p(q), _p(acc))
    return rc, (q, acc), want[1:]


NETS = {
    "random": lambda s: Net(700, s),
    "hubs": lambda s: Net(500, s, reach=40, hubs=25),
    "chain": lambda s: Net(300, s, reach=60, chain=150),
    "chain_hubs": lambda s: Net(321, s, reach=30, chain=180, hubs=8),
    "some": lambda s: Net(450, s, reach=30, hubs=6, share=0.6),
    "small": lambda s: Net(17, s, reach=3),
    "full_chunk": lambda s: Net(128, s, reach=20, chain=40),
    "one_over": lambda s: Net(129, s, reach=20, hubs=3),
}


@pytest.mark.parametrize("kind", sorted(NETS))
@pytest.mark.parametrize("gap", [1, 4])
def test_a_cell_has_the_rank_above_its_upstream_cells_of_the_chunk(lib, kind, gap):
    for seed in range(5):
        net = NETS[kind](seed)
        rank, nrank = ranks(lib, net, gap)
        for v in range(net.n):
            if net.part[v]:
                assert rank[v] < nrank[v // WAVE] <= 255
                for u in net.ups[v]:
                    if u // WAVE == v // WAVE:
                        assert rank[u] + 1 == rank[v]


@pytest.mark.parametrize("kind", sorted(NETS))
@pytest.mark.parametrize("fold,ring,S", [(SSF, 4, 1), (OL, 4, 2), (SSF, 4, 5), (RIV_RES, 4, 11), (SSF, 1, 1), (SNOW, 1, 1)])
def test_steps_drain_and_equal_the_sequential_sweep(lib, kind, fold, ring, S):
    for seed, resident, delay in ((1, 1, 0), (2, 3, 60), (3, 7, 500)):
        net = NETS[kind](seed + 10 * S)
        rc, got, want = run(lib, net, fold, ring, S, seed=seed, resident=resident, delay=delay)
        assert rc == 0, (seed, rc)
        for a, b in zip(got, want):
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), seed


def _edges(net, place):
    """Edges that are the `place`-th of their cell, with the cell, where another chunk can stand in."""
    return [(int(net.up_ptr[v]) + place, v) for v in range(net.n)
            if len(net.ups[v]) > place and (v + WAVE < net.n or v >= WAVE)]


@pytest.mark.parametrize("fold,ring,S", [(SSF, 4, 1), (SSF, 4, 5), (SSF, 1, 1)])
@pytest.mark.parametrize("kind,place", [("random", 0), ("chain", 0), ("hubs", 0), ("hubs", 4), ("hubs", 6),
                                        ("chain_hubs", 0), ("chain_hubs", 4)])
def test_a_wait_that_is_never_met_ends_the_step(lib, kind, place, fold, ring, S):
    net = NETS[kind](4)
    edges = _edges(net, place)
    for k, edge in enumerate((edges[0], edges[len(edges) // 2], edges[-1])):
        rc, _, _ = run(lib, net, fold, ring, S, seed=k, limit=400, unmet=edge)
        assert rc == 1, (edge, rc)


def test_tickets_in_the_reverse_order_do_not_drain(lib):
    rc, _, _ = run(lib, NETS["random"](2), SSF, 4, 2, resident=1, limit=400, reverse=True)
    assert rc == 1


def test_wrong_ranks_are_seen(lib):
    rc, _, _ = run(lib, NETS["chain"](2), SSF, 4, 3, spoil_ranks=True, limit=400)
    assert rc in (-4, -5, 1), rc
    assert rc != 0
