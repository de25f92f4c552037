"""Host forcing through the pinned slots (arrays of 2 MiB and more: several pieces, an odd last one),
below that size, and from pinned arrays: the step is the one from device arrays bit for bit, also when
the caller overwrites its arrays right after the call."""
import numpy as np
import pytest

from wflowhip import Model, Var, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,pinned", [(511, 513, False), (512, 512, False), (773, 701, False), (773, 701, True)])
def test_host_forcing_equals_device_forcing(nx, ny, pinned):
    import torch

    c = synth.make_catchment(nx, ny, cell=250.0, dt=3600.0, river_threshold=200, seed=9)
    host, dev = Model(c), Model(c)
    for k in range(3):
        fr = [np.ascontiguousarray(f) for f in synth.forcing_numpy(c, k)]
        on_dev = [torch.as_tensor(f, device="cuda") for f in fr]
        if pinned:
            fr = [torch.as_tensor(f).pin_memory().numpy() for f in fr]
        host.set_forcing(*fr)
        for f in fr:
            f.fill(np.nan)
        host.update_model()
        dev.set_forcing(*on_dev)
        dev.update_model()
    for v in (Var.CANOPY_STORAGE, Var.SATWATERDEPTH, Var.SNOW_STORAGE, Var.LAND_Q, Var.RIVER_Q):
        assert np.array_equal(host.get(v).view(np.uint64), dev.get(v).view(np.uint64)), v
    host.close()
    dev.close()
