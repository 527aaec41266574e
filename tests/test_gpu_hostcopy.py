"""Positions go to the device and come back unchanged at the sizes where the
transfer changes its way: one workgroup of vertices, one pinned slot, two
alternating slots, four threads; float and double host arrays, float, double
and compensated tissues; a refused array leaves the state."""
import numpy as np
import pytest

from opencl_dpm_amd import capi
from opencl_dpm_amd import workloads as W

pytestmark = pytest.mark.gpu


def handle(m, bits):
    return capi.Tissues3D(m.mesh.faces, [0, m.C], m.Kv, m.Ka, m.Ks, m.v0, m.a0, m.L, m.Kre, nv=m.mesh.nv,
                          precision=bits)


# 162 x 1 vertices; 8 x 8 cells: 10,368 (124 KB); 17 x 17: 46,818 (562 KB,
# two slots); 66 x 66: 705,672 (8.5 MB in float, four threads)
@pytest.mark.parametrize("n", [1, 8, 17, 66])
@pytest.mark.parametrize("bits", [32, 64])
def test_positions_round_trip(n, bits):
    m = W.monolayer3d(n, 2.4, seed=5)
    t = handle(m, bits)
    X = np.asarray(m.X, np.float32).reshape(-1, 3)
    X64 = X.astype(np.float64) * (1.0 + 1e-9)
    for host in (X, X64):
        t.set_positions(host)
        for dtype in (np.float32, np.float64):
            got = t.positions(dtype)
            want = host.astype(np.float64 if bits == 64 else np.float32).astype(dtype)
            np.testing.assert_array_equal(got, want)
    if bits == 32:
        t.set_compensated(True)
        t.set_positions(X64)
        np.testing.assert_array_equal(t.positions(np.float32), X64.astype(np.float32))
        hi = X64.astype(np.float32).astype(np.float64)
        np.testing.assert_array_equal(t.positions(np.float64), hi + (X64 - hi).astype(np.float32))


@pytest.mark.parametrize("n", [1, 17, 66])
def test_a_refused_array_leaves_the_state(n):
    m = W.monolayer3d(n, 2.4, seed=6)
    t = handle(m, 32)
    X = np.asarray(m.X, np.float32).reshape(-1, 3)
    t.set_positions(X)
    for where, value in ((0, np.nan), (len(X) // 2, np.inf), (len(X) - 1, -np.inf)):
        bad = X + np.float32(1)
        bad[where, 2] = value
        with pytest.raises(capi.DPMError, match="Non-finite"):
            t.set_positions(bad)
        np.testing.assert_array_equal(t.positions(), X)


@pytest.mark.parametrize("cells", [3, 700, 40000])
@pytest.mark.parametrize("bits", [32, 64])
def test_2d_positions_round_trip(cells, bits):
    # 30 vertices a cell: 90; 21,000; 1,200,000 vertices (9.6 MB in float)
    nv = np.full(cells, 30, np.int32)
    one = np.ones(cells, np.float32)
    begin = np.arange(0, cells + 1, 1 if cells < 700 else 100, dtype=np.int32)
    L = np.full(len(begin) - 1, 50.0, np.float32)
    t = capi.Tissues2D(begin, nv, 1.0, 1.0, 0.0, one, one, one, L, precision=bits)
    X = np.random.default_rng(cells).uniform(-5, 5, (30 * cells, 2))
    for host in (X, X.astype(np.float32)):
        t.set_positions(host)
        want = host.astype(np.float64 if bits == 64 else np.float32)
        np.testing.assert_array_equal(t.positions(), want)
