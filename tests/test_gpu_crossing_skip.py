"""The crossing parity on the device, with its box rules, where those decide:
cells across the sides of the box, vertices that share rows and columns with
other cells' vertices or lie a margin beside their boxes (the geometries of
test_crossing_skip).  Every vertex's overlap against the plain parity, in k2d_run
with the pair list and with the loop per vertex over arc boxes, and in the wide
form."""
import numpy as np
import pytest
from test_crossing_skip import parity

from opencl_dpm_amd import capi

f = np.float32


def cells(count, n, L, rng):
    out = []
    while len(out) < count:  # a polygon near a side or a corner, then triangles at its ties
        c = rng.choice([0.0, 0.5, 1.0], 2) * float(L) + rng.normal(0, 0.03 * float(L), 2)
        th = np.sort(rng.uniform(0, 2 * np.pi, n))
        r = 0.12 * float(L) * rng.uniform(0.6, 1.0, n)
        x, y = (c[0] + r * np.cos(th)).astype(f), (c[1] + r * np.sin(th)).astype(f)
        out.append((x, y))
        for k in range(3):
            px, py = (rng.uniform(-0.2, 1.2, 3).astype(f) * L for _ in "xy")
            if k == 0:
                px = rng.choice(x, 3)
            elif k == 1:
                py = rng.choice(y, 3)
            else:
                px = rng.choice([x.min(), x.max()], 3) + rng.choice([-1, 1], 3).astype(f) * f(2e-5) * (1 + L)
                py = np.nextafter(rng.choice([y.min(), y.max()], 3), f(0))
            out.append((px.astype(f), py.astype(f)))
    return out[:count]


@pytest.mark.gpu
@pytest.mark.parametrize("pbc", [1, 0])
@pytest.mark.parametrize("L", [0.7, 9.3, 153.6])
@pytest.mark.parametrize("count,n", [(12, 16), (90, 70)])  # the pair list; a loop per vertex
def test_overlaps_are_the_parity(count, n, L, pbc):
    L = f(L)
    rng = np.random.default_rng(count + int(L))
    cs = cells(count, n, L, rng)
    nv = np.array([len(x) for x, _ in cs], np.int32)
    assert (nv.sum() * count <= 16 * 1024) == (count == 12)
    X = np.concatenate([np.stack(c, 1) for c in cs])
    expect = np.zeros(len(X), bool)
    own = np.repeat(np.arange(count), nv)
    for c, (x, y) in enumerate(cs):
        odd = parity(X[:, 0], X[:, 1], x, y, L if pbc else f(1e30))
        expect |= odd & (own != c)
    assert expect.any() and not expect.all()
    one = np.ones(count, np.float32)
    for kind in (1, 2):
        t = capi.Tissues2D([0, count], nv, 1.0, 1.0, 0.0, one, one * f(1e-6), one, float(L), pbc=pbc,
                           mask=capi.DPM2D_REPULSION)
        t.set_step_kernel(kind)
        t.set_positions(X)
        got = t.probe()["overlap"].astype(bool)
        np.testing.assert_array_equal(got, expect, err_msg=f"form {kind}")
