"""The bounding-box rules that skip a crossing test (dpm2d.hip, outside_box_even and maybe_pair's repulsion part),
restated in float32, against the crossing parity they replace: a pair that a rule skips has even parity.  Cells lie
across the sides of the periodic box, points on either side of it, rows and columns shared with the cell's vertices."""
import numpy as np
import pytest

f = np.float32


def parity(px, py, x, y, L):
    """Crossing parity of points [P] about one polygon [n], the reference's float operations (Cell2D_kernel.cl:171-196)."""
    xj, yj = np.roll(x, 1), np.roll(y, 1)
    dix, diy, djx, djy = (p[:, None] - q[None] for p, q in ((px, x), (py, y), (px, xj), (py, yj)))
    big = (np.abs(dix) > L) | (np.abs(djx) > L)
    rnd = lambda q: np.copysign(np.floor(np.abs(q) + f(0.5)), q)
    dix, djx = (np.where(big, d - L * np.floor(d / L), d) for d in (dix, djx))
    big = (np.abs(diy) > L) | (np.abs(djy) > L)
    diy, djy = (np.where(big, d - L * rnd(d / L), d) for d in (diy, djy))
    straddle = (diy > 0) != (djy > 0)
    with np.errstate(divide="ignore", invalid="ignore"):
        tt = (djx - dix) * (f(0) - diy) / (djy - diy) + dix
    assert tt.dtype == np.float32
    return ((straddle & (f(0) < tt)).sum(1) & 1).astype(bool)


def skip_point(px, py, x, y, pbc, L):
    x0, x1, y0, y1 = x.min(), x.max(), y.min(), y.max()
    xin = (~pbc) | ((np.abs(px - x0) <= L) & (np.abs(px - x1) <= L))
    yin = (~pbc) | ((np.abs(py - y0) <= L) & (np.abs(py - y1) <= L))
    m = f(1e-5) * (f(1) + L)
    return (yin & ((py < y0) | (py > y1))) | (xin & ((px < x0 - m) | (yin & (px > x1 + m))))


def skip_cell(b, x, y, pbc, L):
    x0, x1, y0, y1 = x.min(), x.max(), y.min(), y.max()
    bx0, bx1, by0, by1 = b
    sx, sy = max(bx1 - x0, x1 - bx0), max(by1 - y0, y1 - by0)
    xin, yin = not pbc or sx < L * f(0.999), not pbc or sy < L * f(0.999)
    m = f(1e-5) * (f(1) + max(abs(x0), abs(x1)) + max(abs(y0), abs(y1)))
    return (yin and (by1 < y0 - m or by0 > y1 + m)) or (xin and (bx1 < x0 - m or (yin and bx0 > x1 + m)))


@pytest.mark.parametrize("n", [3, 5, 16, 64])
@pytest.mark.parametrize("L", [0.7, 9.3, 153.6])
def test_skipped_pairs_have_even_parity(n, L):
    rng = np.random.default_rng(1000 * n + int(L))
    L = f(L)
    skipped = odd = kept = cells = 0
    for _ in range(60):
        # a polygon near a side or a corner of the box as often as inside it, uneven so that rows repeat
        c = rng.choice([0.0, 0.5, 1.0], 2) * float(L) + rng.normal(0, 0.03 * float(L), 2)
        th = np.sort(rng.uniform(0, 2 * np.pi, n))
        r = 0.12 * float(L) * rng.uniform(0.6, 1.0, n)
        x, y = (c[0] + r * np.cos(th)).astype(f), (c[1] + r * np.sin(th)).astype(f)
        px = rng.uniform(-0.2, 1.2, 400).astype(f) * L
        py = rng.uniform(-0.2, 1.2, 400).astype(f) * L
        px[:60], py[60:120] = rng.choice(x, 60), rng.choice(y, 60)  # exact ties with vertices
        px[120:160], py[120:160] = rng.choice(x, 40), rng.choice(y, 40)
        px[160:200] = rng.choice([x.min(), x.max()], 40) + rng.choice([-1, 1], 40).astype(f) * f(2e-5) * (1 + L)
        py[200:240] = np.nextafter(rng.choice([y.min(), y.max()], 40), f(0))
        mid = rng.uniform(-0.2, 1.2, (20, 2)).astype(f) * L  # the last 160: clusters of eight, other cells
        px[240:], py[240:] = (np.repeat(mid[:, k], 8) + (0.06 * L * rng.normal(0, 1, 160)).astype(f) for k in (0, 1))
        for pbc in (True, False):
            par = parity(px, py, x, y, L if pbc else f(np.inf)) if pbc else parity(px, py, x, y, f(1e30))
            s = skip_point(px, py, x, y, np.bool_(pbc), L)
            assert not (s & par).any()
            skipped, odd, kept = skipped + int(s.sum()), odd + int(par.sum()), kept + int((~s).sum())
            for q in range(240, 400, 8):
                bx, by = px[q:q + 8], py[q:q + 8]
                if skip_cell((bx.min(), bx.max(), by.min(), by.max()), x, y, pbc, L):
                    assert not par[q:q + 8].any()
                    cells += 1
    assert cells > 500 and odd > 100 and kept > 1000 and skipped > 10000
