"""The workgroup form's instances for handles with few and with many cells
(registers, waves at the winding numbers, all waves on one point) give the same
step: a tissue alone against the same tissue many times over, cells in contact.
Forces agree to rounding, contact sets are the same, and every copy of the
tissue is the same bit for bit."""
import numpy as np
import pytest
from scipy.spatial import ConvexHull

from opencl_dpm_amd import capi
from opencl_dpm_amd import workloads as W

pytestmark = pytest.mark.gpu


def mesh(nv):
    """An icosphere, or the hull of nv points along a spiral."""
    if nv in (12, 42, 162, 642):
        m = W.icosphere({12: 0, 42: 1, 162: 2, 642: 3}[nv])
        return m.unit.astype(np.float64), m.faces
    z = 1 - (2 * np.arange(nv) + 1) / nv
    phi = np.arange(nv) * np.pi * (3 - 5**0.5)
    V = np.stack([np.cos(phi) * np.sqrt(1 - z * z), np.sin(phi) * np.sqrt(1 - z * z), z], 1)
    F = ConvexHull(V).simplices
    inward = np.einsum("ij,ij->i", np.cross(V[F[:, 1]] - V[F[:, 0]], V[F[:, 2]] - V[F[:, 0]]), V[F[:, 0]]) < 0
    F[inward] = F[inward][:, ::-1]
    return V, np.ascontiguousarray(F, dtype=np.int32)


# vertices, and copies of the tissue of 9 cells: beyond 1024 cells (642 vertices: the
# instance that keeps three cells on a compute unit; 162 and general: four), beyond 256
# (a cell a compute unit: general meshes over 690 vertices, doubles over 256, 257 to 512
# vertices on 512 threads)
@pytest.mark.parametrize("nv,T,bits", [(12, 120, 32), (42, 120, 32), (162, 120, 32), (190, 120, 32), (257, 40, 32),
                                       (330, 40, 32), (512, 40, 32), (700, 40, 32), (642, 120, 32), (42, 60, 64),
                                       (190, 60, 64), (257, 40, 64), (512, 40, 64), (642, 40, 64)])
def test_few_and_many_cells(nv, T, bits):
    V, F = mesh(nv)
    rng = np.random.default_rng(nv)
    c = np.stack([np.arange(9) % 3, np.arange(9) // 3, np.zeros(9)], 1) * 1.75 + [0.9, 0.9, 1.0]
    X = (V[None] + (c + rng.uniform(-0.1, 0.1, (9, 3)))[:, None]).reshape(-1, 3)
    v0, a0 = W.sphere_targets(np.ones(9, np.float32), 1.0, len(F))
    got = []
    for k in (1, T):
        t = capi.Tissues3D(F, [9 * i for i in range(k + 1)], 1.0, 0.5, 0.2, np.tile(v0, k), np.tile(a0, k), 5.25, 1.0,
                           Kat=0.1, Kb=0.01, mask=capi.DPM3D_ALL, nv=nv, precision=bits)
        t.set_step_kernel(1)
        t.set_positions(np.tile(X, (k, 1)))
        n, keys = t.probe_contact()
        t.euler(1, 0.002)
        got.append([np.asarray(a).reshape(k, 9 * nv, -1) for a in (t.forces(), n, keys)])
        t.close()
    (f1, n1, k1), (ft, nt, kt) = got
    assert n1.any()
    for a in (ft, nt, kt):
        assert (a == a[:1]).all()
    np.testing.assert_array_equal(n1[0], nt[0])
    np.testing.assert_array_equal(k1[0], kt[0])
    # a force term's rounding is about 1e-7 (1e-16) of its size, cancelled by up to 100, and
    # a winding number's is that times the root of its faces
    err = np.linalg.norm(f1[0] - ft[0]) / np.linalg.norm(f1[0])
    print(f"{nv} vertices, {bits} bits: {int(n1.sum())} contacts, forces differ by {err:.1e}")
    assert err < (1e-5 if bits == 32 else 1e-13)
