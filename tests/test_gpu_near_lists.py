"""The step's candidate lists (tissues of more than 512 cells) give the
candidates of the searches that are made anew every step: the same positions,
bit for bit, while cells move far enough that the lists go stale on the way.
"""
import numpy as np
import pytest

from opencl_dpm_amd import capi
from opencl_dpm_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [1, 2])
@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("n,spacing", [(23, 1.6), (24, 1.7)])
def test_listed_steps_equal_scanned_steps(n, spacing, bits, kernel):
    m = W.monolayer3d(n, spacing, seed=11)  # in a box twice its size: the sheet spreads
    t = capi.Tissues3D(m.mesh.faces, [0, m.C], m.Kv, m.Ka, m.Ks, m.v0, m.a0, 2 * m.L, 40.0, Kat=2.0, Kb=m.Kb,
                       mask=capi.DPM3D_ALL, nv=m.mesh.nv, precision=bits)
    t.set_step_kernel(kernel)
    X = np.asarray(m.X, np.float64 if bits == 64 else np.float32)
    steps, dt = 140, 0.05
    t.set_positions(X)
    t.euler(steps, dt)  # 128 of them from a step graph
    listed = t.positions()
    moved = np.linalg.norm((listed - X.reshape(-1, 3)).reshape(m.C, -1, 3).mean(1), axis=1).max()
    r = (3 / (4 * np.pi) * np.min(m.v0)) ** (1 / 3)
    print(f"largest centre displacement {moved:.3f}, skin {0.15 * r:.3f}")
    assert moved > 0.49 * 0.15 * r  # the lists went stale at least once
    # the bins' candidates are the scan's (test_gpu_parity), made anew every step
    t.set_cell_list(1)
    t.set_positions(X)
    t.euler(steps, dt)
    np.testing.assert_array_equal(listed, t.positions())
    # lists of before the steps with bins are not used after them
    t.set_positions(X)
    t.set_cell_list(0)
    t.euler(10, dt)
    t.set_cell_list(1)
    t.euler(100, dt)
    t.set_cell_list(0)
    t.euler(steps - 110, dt)
    np.testing.assert_array_equal(listed, t.positions())
