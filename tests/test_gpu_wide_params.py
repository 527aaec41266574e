"""The wide 2D form's captured steps follow a change of the tissue's terms: as
k2d_run (which reads them at every call), bit for bit."""
import numpy as np
import pytest

from opencl_dpm_amd import capi
from opencl_dpm_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_captured_steps_take_the_new_terms():
    p = W.tissue2d(40, 0, 1.4, 0.88, Kb=0.01, Kat=0.3, seed=2, nv_range=(16, 40))
    got = []
    for kind in (1, 2):
        t = capi.Tissues2D([0, p.C], p.nv, p.Ka, p.Kl, p.Kb, p.a0, p.l0, p.r0, p.L, Kre=p.Kre, Kat=p.Kat)
        t.set_step_kernel(kind)
        t.set_positions(p.X)
        t.euler(70, 0.005)  # 64 of them from a graph
        t.set_tissue_params(mask=capi.DPM2D_ALL & ~capi.DPM2D_REPULSION)
        t.euler(70, 0.005)
        got.append((t.positions(), t.forces()))
    np.testing.assert_array_equal(got[0][0], got[1][0])
    np.testing.assert_array_equal(got[0][1], got[1][1])
