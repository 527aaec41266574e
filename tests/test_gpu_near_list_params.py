"""The candidate lists' skin follows the smallest rest volume.  Steps replayed
from a captured graph and steps launched one by one use the same skin after
dpm3d_set_cell_params changed it: the positions are those of the search made
anew every step (the bins), bit for bit.  The cells grow towards rest volumes
far above their own, so that pairs out of reach come into it all the time."""
import numpy as np
import pytest

from opencl_dpm_amd import capi
from opencl_dpm_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [1, 2])
@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("first", [1, 2, 4])  # where the steps before the change leave buffers and marks
@pytest.mark.parametrize("change", ["wider", "narrower"])
def test_lists_after_a_change_of_the_skin(change, first, bits, kernel):
    m = W.monolayer3d(24, 2.9, jitter=0.35, seed=11)
    X = np.asarray(m.X, np.float64 if bits == 64 else np.float32)
    before, after = m.v0, 1000 * m.v0  # ten times the skin
    if change == "narrower":  # by one cell
        before, after = after, after.copy()
        after[m.C // 2] = m.v0[m.C // 2]

    def run(mode):
        t = capi.Tissues3D(m.mesh.faces, [0, m.C], 2.0, 0.5, m.Ks, before, m.a0, m.L, 10.0, Kat=2.0, Kb=m.Kb,
                           mask=capi.DPM3D_ALL, nv=m.mesh.nv, precision=bits)
        t.set_step_kernel(kernel)
        t.set_cell_list(mode)
        t.set_positions(X)
        t.euler(70, 0.05)  # a graph of 64 steps is captured
        t.euler(first, 0.05)
        t.set_cell_params(v0=after)
        out = []
        for _ in range(2):  # a graph each, up to three steps before it, the rest after it
            t.euler(124, 0.05)
            out.append(t.positions())
        t.close()
        return out

    listed, binned = run(0), run(1)
    assert np.isfinite(binned[-1]).all()
    for a, b in zip(listed, binned):
        np.testing.assert_array_equal(a, b)
