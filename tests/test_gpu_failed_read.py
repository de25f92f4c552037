"""Reads after a step that failed (non-finite forcing; a routing wait that is never met): wfh_get reports
the failure and leaves the destination as it was, in device memory as in host memory, for every kind
of variable and order, at the read that finds the failure and at the ones after it."""
import numpy as np
import pytest

from wflowhip import Model, Var, _abi, synth
from wflowhip.model import WflowError

pytestmark = pytest.mark.gpu

READS = [(Var.RIVER_Q_AVERAGE, False), (Var.SATWATERDEPTH, False), (Var.SATWATERDEPTH, True),
         (Var.USTORELAYERDEPTH, False), (Var.USTORELAYERDEPTH, True), (Var.RESERVOIR_STORAGE, False)]


def _failed(c, kind):
    m = Model(c)
    f = list(synth.forcing_numpy(c, 0))
    m.run_timestep(*f)
    m.sync()
    if kind == "nonfinite":
        f[2] = f[2].copy()
        f[2][c.n // 2] = np.nan
    else:
        down = synth.land_downstream(c)
        has_up = np.zeros(c.n, bool)
        has_up[down[down >= 0]] = True
        nodes = np.nonzero(has_up[m.node_order()])[0]
        m.test_route_stall(20_000, int(nodes[len(nodes) // 2]))
    m.set_forcing(*f)
    m.update_model()
    return m


@pytest.mark.parametrize("kind,code", [("nonfinite", -4), ("stall", -5)])
@pytest.mark.parametrize("first", range(len(READS)))
def test_a_failed_step_leaves_the_destination(kind, code, first):
    import torch

    c = synth.make_catchment(96, cell=250.0, dt=3600.0, river_threshold=40, seed=31)
    synth.add_reservoirs(c, 3, seed=31, radius=1, curves=False)
    print(f"{kind}, first read {READS[first]}", flush=True)
    m = _failed(c, kind)
    for var, node in READS[first:] + READS[:first]:
        count = _abi.var_count(var, c.n, c.nriv, c.nlayers, c.nres)
        assert count > 0
        out = torch.full((count,), -7.25, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        with pytest.raises(WflowError) as e:
            m.get_value_device(var, out, node_order=node)
        assert e.value.code == code
        assert bool((out == -7.25).all()), (var, node)
    m.close()
