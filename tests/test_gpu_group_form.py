"""The workgroup form of the 3D step against the wave form and the oracle at
the sizes where its passes change: more vertices than threads, one to four
vertices a thread, the instances with fixed sizes, candidates beyond the kept
lists (small boxes, where every vertex pair is tested; many neighbours) and
more cells than are tested ahead of its first barrier."""
import numpy as np
import pytest

import oracle
from opencl_dpm_amd import capi
from opencl_dpm_amd import workloads as W

pytestmark = pytest.mark.gpu


def check(m, faces, bits, mask=capi.DPM3D_ALL):
    """One step of the workgroup form; force error against the oracle in double
    (which takes the parameters the device holds, in float)."""
    t = capi.Tissues3D(faces, [0, m.C], m.Kv, m.Ka, m.Ks, m.v0, m.a0, m.L, m.Kre, Kat=m.Kat, Kb=m.Kb,
                       mask=mask, nv=m.mesh.nv, precision=bits)
    t.set_step_kernel(1)
    t.set_positions(np.asarray(m.X, np.float64))
    t.euler(1, m.dt)
    f = lambda v: np.asarray(v, np.float32).astype(np.float64)
    X64, F64 = oracle.run3d(m.X, faces, m.mesh.nv, f(m.Kv), f(m.Ka), f(m.Ks), f(m.v0), f(m.a0), float(f(m.L)),
                            float(f(m.Kre)), 1, float(f(m.dt)), Kat=float(f(m.Kat)), Kb=f(m.Kb), mask=mask,
                            prec=64)
    err = np.linalg.norm(t.forces() - F64) / np.linalg.norm(F64)
    print(f"{m.C} cells of {m.mesh.nv} vertices, {bits} bits: force error {err:.2e}", flush=True)
    # a float force term's rounding is about 1e-7 of its size, cancelled
    # against its neighbours by up to 100; the same bound times the ratio of
    # the roundings would be 1e-13 in double, 1e-9 allows for sums of another
    # grouping near a cut-off
    assert err < (1e-5 if bits == 32 else 1e-9)
    assert np.abs(t.positions() - X64).max() < 1e-5


# cells per side, spacing, subdivision (12, 42, 162, 642 vertices)
CASES = [(3, 1.8, 0), (3, 1.9, 1), (2, 1.7, 2), (3, 1.6, 2), (17, 1.9, 1), (3, 1.9, 3), (2, 1.6, 3)]


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("n,spacing,subdiv", CASES)
def test_one_step_against_the_oracle(n, spacing, subdiv, bits):
    m = W.monolayer3d(n, spacing, subdiv=subdiv, seed=21)
    check(m, m.mesh.faces, bits)


# A mesh with a face removed has no instance of its own and takes its faces one
# by one.  Without volume and contact: the library's volume is taken about the
# centre of mass and its contact search culls by the convex hull, both equal to
# the reference's for closed surfaces only.
@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("subdiv", [1, 2, 3])
def test_open_mesh_against_the_oracle(subdiv, bits):
    m = W.monolayer3d(3, 1.9, subdiv=subdiv, seed=22)
    check(m, np.ascontiguousarray(m.mesh.faces[1:]), bits, capi.DPM3D_ALL & ~(capi.DPM3D_VOLUME | capi.DPM3D_CONTACT))
