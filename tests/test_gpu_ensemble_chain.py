"""Chain stages of the ensemble pipelined over the families (2 + S_r waves a block, up to six river
sub-steps and 256 blocks) against one wave per strand. The solves with the Newton histogram switched
on take the second path and give kw_solve's results bit for bit, so every state has to be equal."""
import numpy as np
import pytest

from wflowhip import Ensemble, Var, synth
from test_gpu_ensemble import ENS_STATES, factors

pytestmark = pytest.mark.gpu


# seeds 3 and 16: confluences of five and seven upstream cells (a record holds four)
@pytest.mark.parametrize("side,seed,members,river_dt,river", [
    (33, 3, 64, 3600.0, 8),     # one river sub-step
    (33, 16, 128, 1800.0, 3),   # two, rivers from three cells upstream
    (64, 5, 192, 900.0, 60),    # four, three member groups, stages of more and of fewer than 256 blocks
    (40, 6, 64, 600.0, 30),     # six: the most a block takes
    (40, 6, 64, 500.0, 30),     # more than six: one wave per strand
])
def test_pipelined_chains_equal_the_serial_ones(side, seed, members, river_dt, river):
    c = synth.make_catchment(side, cell=250.0, dt=3600.0, river_threshold=river, seed=seed)
    fac = factors(members, seed)
    ens = [Ensemble(c, *fac, river_dt=river_dt) for _ in range(2)]
    ens[1].kw_histogram(True)
    for k in range(5):
        P, E, T = synth.forcing_numpy(c, k)
        bal = []
        for x in ens:
            x.run_timestep(P, E, T)
            bal.append(np.asarray(x.balance()).copy())
        assert np.array_equal(bal[0], bal[1])
    for m in (0, members // 2, members - 1):
        for v in ENS_STATES:
            a, b = (x.get(v, m) for x in ens)
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), (v, m)
    assert np.any(ens[0].get(Var.RIVER_Q, 0) > 0.0)
    for x in ens:
        x.close()
