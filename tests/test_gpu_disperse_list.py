"""k_disperse_list against the reference's serial loop in numpy float32, bit for bit (centres, iteration count, cap):
one to nine segments of eight centres, lists of more than 16 and of more than 32 centres (the run then goes on in
k_disperse2d), coincident centres (NaN)."""
import numpy as np
import pytest

from opencl_dpm_amd import capi

f, d = np.float32, np.float64


def reference(r, L, X, Y, most):
    X, Y, n, L = X.copy(), Y.copy(), len(r), f(L)
    old, dU, it = f(100), f(100), 0
    rnd = lambda q: np.copysign(np.floor(np.abs(q) + f(0.5)), q)
    with np.errstate(all="ignore"):
        while d(dU) > 1e-6:
            dx, dy = (p[None] - p[:, None] for p in (X, Y))
            dx, dy = (q - L * rnd(q / L) for q in (dx, dy))
            dist = np.sqrt(dx * dx + dy * dy)
            rr = r[:, None] + r[None]
            q = dist / rr
            ft = ((1.0 - q.astype(d)) / rr.astype(d)).astype(f)
            fx, fy, u = ft * (dx / dist), ft * (dy / dist), f(1) - q * (f(1) - q)
            Fx, Fy, U = np.zeros(n, f), np.zeros(n, f), f(0)
            for i, j in zip(*np.nonzero((dist <= rr) & ~np.eye(n, dtype=bool))):
                Fx[i], Fy[i] = Fx[i] - fx[i, j], Fy[i] - fy[i, j]
                Fx[j], Fy[j] = Fx[j] + fx[i, j], Fy[j] + fy[i, j]
                U = f(d(U) + 0.5 * d(u[i, j]))
            X, Y = ((p.astype(d) + 0.01 * F.astype(d)).astype(f) for p, F in ((X, Fx), (Y, Fy)))
            dU = np.abs(f(U - old))
            old, it = U, it + 1
            if it > most:
                return X, Y, it, True
    return X, Y, it, False


@pytest.mark.gpu
@pytest.mark.parametrize("n,spread,most", [(1, 1.0, 50), (2, 0.1, 400), (8, 0.4, 200), (9, 0.5, 200), (33, 0.9, 150),
                                           (40, 0.25, 60), (70, 0.3, 40), (70, 1.0, 120), (12, 0.0, 20)])
def test_list_form_is_the_serial_loop(n, spread, most):
    rng = np.random.default_rng(n + most)
    r = np.where(np.arange(n) % 2, 1.3, 1.0).astype(f)
    L = f(np.sqrt((np.pi * r.astype(d) ** 2).sum()) / 0.9)
    X, Y = (rng.uniform(0, 1, (2, n)) * spread * L + (1 - spread) * 0.4 * L).astype(f)
    x, y, it, cap = reference(r, L, X, Y, most)
    gx, gy, (git, gcap) = capi.disperse(r, L, X, Y, max_count=most)
    assert (git, gcap) == (it, cap)
    np.testing.assert_array_equal(gx, x)
    np.testing.assert_array_equal(gy, y)
