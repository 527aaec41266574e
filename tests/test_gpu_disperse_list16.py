"""k_disperse_list with lists of 16 entries (377 to 768 centres, whose lists of
32 do not fit the LDS) against the reference's serial loop, bit for bit: more
segments than waves, and a run whose lists fit at first and overflow after some
iterations, so that k_disperse2d goes on from the middle of it; 769 centres run
in k_disperse2d alone."""
import numpy as np
import pytest
from test_gpu_disperse_list import reference

from opencl_dpm_amd import capi

f, d = np.float32, np.float64


def centres(n, spread, seed):
    rng = np.random.default_rng(seed)
    r = np.where(np.arange(n) % 2, 1.3, 1.0).astype(f)
    L = f(np.sqrt((np.pi * r.astype(d) ** 2).sum()) / 0.9)
    X, Y = (rng.uniform(0, 1, (2, n)) * spread * L + (1 - spread) * 0.4 * L).astype(f)
    return r, L, X, Y


def most_entries(r, L, X, Y):
    dx, dy = (p[None].astype(d) - p[:, None] for p in (X, Y))
    dist = np.hypot(dx - L * np.round(dx / L), dy - L * np.round(dy / L))
    return ((dist <= r[:, None] + r[None] + 0.2 * r.max()).sum(1) - 1).max()


@pytest.mark.gpu
@pytest.mark.parametrize("n,spread,seed,most,overflows", [(377, 1.0, 0, 40, False), (400, 0.74, 5, 30, True),
                                                          (640, 1.0, 1, 20, False), (768, 1.0, 2, 15, False),
                                                          (769, 1.0, 2, 10, False)])
def test_list_of_16_is_the_serial_loop(n, spread, seed, most, overflows):
    r, L, X, Y = centres(n, spread, seed)
    if overflows:
        assert most_entries(r, L, X, Y) == 16
        assert most_entries(r, L, *reference(r, L, X, Y, 5)[:2]) > 16
    elif n <= 768:
        assert most_entries(r, L, X, Y) <= 16
    x, y, it, cap = reference(r, L, X, Y, most)
    gx, gy, (git, gcap) = capi.disperse(r, L, X, Y, max_count=most)
    assert (git, gcap) == (it, cap)
    np.testing.assert_array_equal(gx, x)
    np.testing.assert_array_equal(gy, y)
