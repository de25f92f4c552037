"""Host forcing on both sides of the line from which it is staged (arrays of 5 MiB): just below, exactly on
it and above, with an odd last piece, pageable and pinned. The step is the one from device arrays bit for
bit, also when the caller overwrites its arrays right after the call."""
import pytest

from test_gpu_host_forcing import test_host_forcing_equals_device_forcing as _equals

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,pinned", [(809, 809, False), (1024, 640, False), (1021, 997, False), (1021, 997, True)])
def test_staged_forcing_equals_device_forcing(nx, ny, pinned):
    print(f"{nx} x {ny}, pinned {pinned}", flush=True)
    _equals(nx, ny, pinned)
