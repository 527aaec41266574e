"""The candidate lists where their bookkeeping can go wrong, against the bins,
which are made anew every step, bit for bit: several tissues in one handle that
go stale at different steps, tissues without lists beside ones with them, lists
of more entries than are kept, lists that are stale as soon as they are made,
and calls of one step (the first of them makes no lists)."""
import numpy as np
import pytest

from opencl_dpm_amd import capi
from opencl_dpm_amd import workloads as W

pytestmark = pytest.mark.gpu


def same(make, X, steps, dt, kernel, between=lambda t: None):
    got = []
    for mode in (0, 1):
        t = make()
        t.set_step_kernel(kernel)
        t.set_cell_list(mode)
        t.set_positions(X)
        out = []
        for k, n in enumerate(steps):
            t.euler(n, dt)
            out += [t.positions(), t.forces()]
            if k == len(steps) // 2:
                between(t)
        got.append(out)
        t.close()
    assert np.isfinite(got[1][-1]).all()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("kernel", [1, 2])
@pytest.mark.parametrize("bits", [32, 64])
def test_tissues_of_one_handle(bits, kernel):
    ms = [W.monolayer3d(n, 1.7, subdiv=1, seed=n) for n in (24, 3, 25, 9)]
    cat = lambda k: np.concatenate([getattr(m, k) for m in ms])
    cb = np.concatenate([[0], np.cumsum([m.C for m in ms])])
    X = cat("X").astype(np.float64 if bits == 64 else np.float32)
    make = lambda: capi.Tissues3D(ms[0].mesh.faces, cb, 1.0, 0.5, 0.2, cat("v0"), cat("a0"),
                                  [2 * m.L for m in ms], [40.0, 5.0, 2.0, 40.0], Kat=[2.0, 0.1, 0.5, 1.0], Kb=0.01,
                                  mask=capi.DPM3D_ALL, nv=42, precision=bits)
    same(make, X, [1, 1, 70, 3, 64, 130], 0.05, kernel)


@pytest.mark.parametrize("kernel", [1, 2])
@pytest.mark.parametrize("spacing", [1.12, 1.2])  # most lists past 64 entries; some of them
def test_more_entries_than_a_list_keeps(spacing, kernel):
    mesh = W.icosphere(0)
    rng = np.random.default_rng(3)
    c = np.stack(np.meshgrid(*[np.arange(9)] * 3), -1).reshape(-1, 3) * spacing + rng.uniform(-0.1, 0.1, (729, 3))
    X = (mesh.unit[None] * np.float32(0.9) + c[:, None].astype(np.float32)).reshape(-1, 3)
    v0, a0 = W.sphere_targets(np.full(729, 0.9, np.float32), 1.0, mesh.nf)
    reach = 2 * 0.9 + max(0.4 * 0.95, 2 * np.sqrt(4 * a0[0] / 3)) + 0.15 * (0.2387 * v0[0]) ** (1 / 3)
    d = c[:, None] - c[None]
    d -= 9 * spacing * np.round(d / (9 * spacing))
    n = (np.linalg.norm(d, axis=2) < reach).sum(1) - 1
    print(f"entries {n.min()} to {n.max()}")
    assert n.max() > 64
    make = lambda: capi.Tissues3D(mesh.faces, [0, 729], 1.0, 0.5, 0.2, v0, a0, 9 * spacing, 1.0, Kat=0.1, Kb=0.01,
                                  mask=capi.DPM3D_ALL & ~capi.DPM3D_SUBSTRATE, nv=mesh.nv)
    same(make, X, [20, 70], 0.01, kernel)


@pytest.mark.parametrize("kernel", [1, 2])
@pytest.mark.parametrize("bits", [32, 64])
def test_lists_stale_at_once(bits, kernel):
    m = W.monolayer3d(24, 1.7, subdiv=1, seed=5)
    X = np.asarray(m.X, np.float64 if bits == 64 else np.float32)
    Kv, v0 = np.full(m.C, 1.0, np.float32), m.v0.copy()
    v0[100], Kv[100] = 1e-9, 1e-9  # the skin follows the smallest rest volume
    make = lambda: capi.Tissues3D(m.mesh.faces, [0, m.C], Kv, m.Ka, m.Ks, v0, m.a0, 2 * m.L, 40.0, Kat=2.0, Kb=m.Kb,
                                  mask=capi.DPM3D_ALL, nv=42, precision=bits)
    # stale at every step, then (the cell's volume back) lists that serve
    same(make, X, [1, 5, 90, 1, 100, 70], 0.05, kernel, between=lambda t: t.set_cell_params(v0=m.v0))
