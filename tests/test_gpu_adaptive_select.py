"""The stable time step's selection in one block: keys in registers (up to 8192 cells), keys read
from memory (up to 65536) and the grid-wide passes beyond. The sub-step counts, states and
fluxes are the oracle's."""
import numpy as np
import pytest

import oracle as O
from wflowhip import Model, Var, synth
from test_gpu_adaptive import run_adaptive
from test_gpu_parity import FLUX_VARS, STATE_VARS, compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,river", [
    (3, 2, 1),       # a handful of cells: no or one eligible river cell at first
    (32, 32, 1000),  # (almost) no river
    (128, 64, 30),   # 8192 cells: the most that registers hold
    (91, 91, 1),     # 8281: overland and river from memory
    (256, 256, 9),   # 65536: the last size of the block
    (257, 256, 50),  # 65792: the grid-wide passes
])
def test_selection_by_size(nx, ny, river):
    c = synth.make_catchment(nx, ny, cell=250.0, dt=3600.0, river_threshold=river, seed=31)
    run_adaptive(c, 2)


def test_selection_with_equal_keys():
    """Every cell the same state and geometry: all keys equal, then few distinct ones."""
    c = synth.make_catchment(60, cell=250.0, dt=3600.0, river_threshold=20, seed=32)
    q = np.full(c.n, 0.125)
    q[::7] = 0.25
    gpu, ref = Model(c, adaptive=True), O.OracleModel(c, adaptive=True)
    gpu.set_value(Var.LAND_Q, q)
    ref.set(Var.LAND_Q, q)
    P, E, T = synth.forcing_numpy(c, 0)
    gpu.run_timestep(P, E, T)
    ref.step(P, E, T)
    assert gpu.last_substeps() == ref.last_substeps()
    compare(gpu, ref, STATE_VARS + FLUX_VARS, "equal keys")
    gpu.close()
    ref.close()
