"""The double adjoint takes closed meshes up to the LDS of one workgroup, 706
vertices, and refuses one more.  One step's J_x^T lambda there against central
differences of the oracle's forces in double, with and without bending (the
kernel's last sums lie in other scratch then)."""
import numpy as np
import pytest

import oracle
from opencl_dpm_amd import capi
from opencl_dpm_amd import workloads as W

pytestmark = pytest.mark.gpu

SHAPE = capi.DPM3D_VOLUME | capi.DPM3D_SURFACE | capi.DPM3D_SUBSTRATE


def sphere(nv):
    """The icosphere of 642 vertices with a vertex more inside some faces, no
    two of which share a vertex (degrees 3, 6 and 7)."""
    m = W.icosphere(3)
    V, F, used = [*m.unit.astype(np.float64)], [tuple(f) for f in m.faces], set()
    for f in list(F):
        if len(V) == nv:
            break
        if used.isdisjoint(f):
            used.update(f)
            c = sum(V[i] for i in f)
            V.append(c / np.linalg.norm(c))
            F.remove(f)
            a, b, d = f
            n = len(V) - 1
            F += [(a, b, n), (b, d, n), (d, a, n)]
    assert len(V) == nv and len(F) == 2 * nv - 4
    return np.array(V), np.array(F, np.int32)


def tissue(nv, mask):
    V, F = sphere(nv)
    X = np.concatenate([V * 1.03 + [2.4 * k + 1.2, 1.2, 1.0] for k in range(2)])
    v0, a0 = W.sphere_targets(np.ones(2, np.float32), 1.0, len(F))
    t = capi.Tissues3D(F, [0, 2], 1.0, 0.5, 0.25, v0, a0, 4.75, 1.0, Kb=0.5, mask=mask, nv=nv, precision=64)
    force = lambda x: oracle.forces3d(x, F, nv, np.ones(2), np.full(2, 0.5), np.full(2, 0.25), v0.astype(np.float64),
                                      a0.astype(np.float64), 4.75, 1.0, Kat=0.0, Kb=np.full(2, 0.5), mask=mask,
                                      ks_grad=0.0, prec=64)["forces"]
    return t, X, force


@pytest.mark.parametrize("mask", [SHAPE, SHAPE | capi.DPM3D_BENDING])
def test_largest_mesh(mask):
    t, X, force = tissue(706, mask)
    t.set_positions(X)
    dt = 0.002
    t.trajectory(1, dt, 1)
    rng = np.random.default_rng(0)
    lam = rng.normal(size=X.shape)
    _, l0 = t.adjoint(lam)
    mu = (l0 - lam) / dt
    for _ in range(2):
        v = rng.normal(size=X.shape)
        cd = lambda e: np.sum(lam * (force(X + e * v) - force(X - e * v))) / (2 * e)
        fd, ad = (4 * cd(1e-6) - cd(2e-6)) / 3, float(np.sum(mu * v))
        print(f"mask {mask}: adjoint {ad:.10e} differences {fd:.10e}", flush=True)
        # the differences' rounding: forces of order 1 with 1e-16 over 1e-6, about 4000 terms
        assert abs(ad - fd) < 1e-6 * abs(fd) + 1e-7


def test_a_vertex_more_is_refused_by_the_adjoint_only():
    t, X, force = tissue(707, SHAPE)
    t.set_positions(X)
    t.euler(1, 0.002)
    # grouping of the sums, forces of order 1 (test_gpu_group_form's bound)
    np.testing.assert_allclose(t.forces(), force(X), atol=1e-9)
    with pytest.raises(capi.DPMError, match="adjoint kernel"):
        t.trajectory(1, 0.002, 1)
