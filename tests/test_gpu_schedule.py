"""The passes of the routing families (run_sched) at the sizes where a schedule can go wrong, against
the oracle: chunks of 64 cells just filled, one short and one over; cells with seven upstream cells
(more than the inbox has places), also across chunks; one, two, three, four, five and many
sub-steps of land and river (the inbox holds four); reservoirs among them, per-sub-step launches,
and overland cells that fall wet from nothing and from the smallest flow."""
import sys

import numpy as np
import pytest

from test_gpu_parity import run_pair
from wflowhip import synth

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, file=sys.__stderr__, flush=True)


def comb(m, dt=3600.0, cell=250.0, river=True):
    """m junctions in a row: three cells above and three below drain into each, and so does the row
    itself, so a junction has seven upstream cells; between two junctions lie two plain cells."""
    nx = 3 * m
    c = synth.make_catchment(nx, 3, cell=cell, dt=dt, river_threshold=10 ** 9, seed=7)
    A = c.arrays
    y, x = np.divmod(np.arange(c.n), nx)
    code = np.full(c.n, 6, np.uint8)
    ox = x % 3 - 1
    top, bottom = y == 0, y == 2
    code[top] = np.choose(ox[top] + 1, [9, 8, 7])
    code[bottom] = np.choose(ox[bottom] + 1, [3, 2, 1])
    code[(y == 1) & (x == nx - 1)] = 5
    A["ldd"] = code
    A["land_slope"] = np.ascontiguousarray(np.random.default_rng(8).uniform(1e-3, 0.05, c.n))
    row = (y == 1) & (x >= 4) if river else np.zeros(c.n, bool)
    A["river_location"] = row.astype(np.uint8)
    k = int(row.sum())
    A["river_width_land"] = np.where(row, 6.0, 0.0)
    A["river_length_land"] = np.where(row, float(cell), 0.0)
    A["river_slope"] = np.ascontiguousarray(A["land_slope"][row])
    A["river_manning_n"] = np.full(k, 0.036)
    A["river_bankfull_depth"] = np.full(k, 1.0)
    A["river_length"] = np.full(k, float(cell))
    A["river_width"] = np.full(k, 6.0)
    return c


@pytest.mark.parametrize("m", [1, 7, 22, 60])
@pytest.mark.parametrize("kw", [{}, {"river_dt": 3600.0}, {"river_dt": 600.0, "land_dt": 720.0}, {"adaptive": True}])
def test_cells_with_seven_upstream_cells(m, kw):
    _say(f"comb of {m} junctions, {kw}")
    gpu, ref = run_pair(comb(m), 5, **kw)
    gpu.close()
    ref.close()


@pytest.mark.parametrize("shape", [(8, 8), (9, 7), (13, 5), (16, 8), (43, 3)])
def test_chunk_edges(shape):
    _say(f"{shape[0]}x{shape[1]} cells")
    c = synth.make_catchment(shape[0], shape[1], cell=500.0, dt=3600.0, river_threshold=6, seed=31)
    gpu, ref = run_pair(c, 6)
    gpu.close()
    ref.close()


@pytest.mark.parametrize("land,river", [(1, 2), (1, 3), (2, 5), (4, 4), (5, 7), (3, 1), (30, 60)])
def test_sub_step_counts(land, river):
    _say(f"67x59, {land} land and {river} river sub-steps")
    c = synth.make_catchment(67, 59, cell=250.0, dt=3600.0, river_threshold=20, seed=32)
    gpu, ref = run_pair(c, 4, land_dt=3600.0 / land, river_dt=3600.0 / river)
    gpu.close()
    ref.close()


def test_subsurface_sub_steps_and_reservoirs():
    _say("61x57, 3 subsurface sub-steps, 6 reservoirs")
    c = synth.make_catchment(61, 57, cell=250.0, dt=3600.0, river_threshold=20, seed=33)
    synth.add_reservoirs(c, 6, seed=2, curves=True)
    gpu, ref = run_pair(c, 4, subsurface_dt=1200.0)
    gpu.close()
    ref.close()


def test_overland_flow_from_dry_and_from_the_smallest_flow():
    """Storms over part of the cells, then dry hours, then storms again: overland solves that start
    from the inflow (no flow before) and from KIN_WAVE_MIN_FLOW (which take over a hundred updates)."""
    _say("96x88 storms")
    c = synth.make_catchment(96, 88, cell=250.0, dt=3600.0, river_threshold=40, seed=34)

    def storms(cc, k):
        P, E, T = synth.forcing_numpy(cc, k)
        wet = np.random.default_rng(100 + k).random(cc.n) < 0.3
        return np.ascontiguousarray(np.where(wet & (k % 4 < 2), 60.0e-3 / 3600.0, 0.0)), E, np.full(cc.n, 290.0)

    gpu, ref = run_pair(c, 10, forcing=storms)
    gpu.close()
    ref.close()
