"""A handle's transfers run on its own device whatever device is current in the
calling thread (a new thread starts with device 0)."""
import threading

import numpy as np
import pytest
import torch

from opencl_dpm_amd import capi
from opencl_dpm_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two devices")
def test_transfers_from_a_thread_with_another_current_device():
    m = W.monolayer3d(3, 2.4, subdiv=1)
    with torch.cuda.device(1):
        t = capi.Tissues3D(m.mesh.faces, [0, m.C], m.Kv, m.Ka, m.Ks, m.v0, m.a0, m.L, m.Kre, nv=m.mesh.nv)
    got = []

    def work():
        t.set_positions(m.X)
        got.append(t.positions())

    th = threading.Thread(target=work)
    th.start()
    th.join()
    np.testing.assert_array_equal(got[0], m.X)
    assert torch.cuda.current_device() == 0
