"""k2d_wide_step with 32, 16 and 8 lanes per vertex (chosen by the handle's vertex count) against k2d_run, bit for
bit: forces, pair sets and 5 steps, with polygons of 3 to 70 vertices (remainders of every group), the reference's
terms and every term, cells across the sides of the box."""
import numpy as np
import pytest

from opencl_dpm_amd import capi

pytestmark = pytest.mark.gpu


def tissues(T, n, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    cols = int(np.ceil(np.sqrt(n)))
    L = np.float32(2.15 * cols)
    nv = rng.integers(3, 71, T * n).astype(np.int32)
    r = np.where(np.arange(T * n) % 2, 1.18, 1.0)
    c = np.stack([np.arange(T * n) % n % cols, np.arange(T * n) % n // cols], 1) * 2.15 + rng.uniform(-0.2, 0.2, (T * n, 2))
    own = np.repeat(np.arange(T * n), nv)
    th = 2 * np.pi * (np.arange(len(own)) - np.repeat(np.cumsum(nv) - nv, nv)) / nv[own] + own
    X = (c[own] + r[own, None] * np.stack([np.cos(th), np.sin(th)], 1)).astype(np.float32)
    a0 = (0.5 * nv * r * r * np.sin(2 * np.pi / nv)).astype(np.float32)
    l0 = (2 * r * np.sin(np.pi / nv)).astype(np.float32)
    return dict(cb=np.arange(T + 1) * n, nv=nv, X=X, a0=a0, l0=l0, r0=r, L=L)


@pytest.mark.parametrize("mask", [capi.DPM2D_ALL, capi.DPM2D_ALL_TERMS])
@pytest.mark.parametrize("T,n", [(1, 7), (2, 150), (10, 150), (40, 120)])
def test_groups_equal_one_workgroup(T, n, mask):
    m = tissues(T, n, seed=T + n)
    got = []
    for kind in (1, 2):
        t = capi.Tissues2D(m["cb"], m["nv"], 1.0, 1.0, 0.01, m["a0"], m["l0"], m["r0"], [m["L"]] * T, Kat=0.4, mask=mask)
        t.set_step_kernel(kind)
        t.set_positions(m["X"])
        g = t.probe()
        t.euler(5, 0.002)
        got.append({**g, "X": t.positions(), "F": t.forces()})
    assert got[0]["overlap"].any() and got[0]["attraction"].any()
    for key in got[0]:
        np.testing.assert_array_equal(got[0][key], got[1][key], err_msg=key)
