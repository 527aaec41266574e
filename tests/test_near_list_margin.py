"""The candidate lists' rules (near_list_takes, near_list_moved in dpm3d_pairs.h,
compiled for the host) against the scan's test: a pair that was not listed, and
neither of whose cells has marked the lists stale, is out of the scan's reach.
Adversarial pairs: just past the list's limit, then as close as the cells may
come, across a side of the box, far from the origin and with skins far below
the cells' size."""
import ctypes
import subprocess

import pytest

from opencl_dpm_amd import build

SRC = r"""
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <random>
#include "dpm3d_pairs.h"

// the scan's test (in_reach of dpm3d_group.hip)
template <typename R>
static bool in_reach(const CellStat<R>& i, const CellStat<R>& j, bool pbc, R L, R invL, bool contact, bool adh) {
  V3<R> sh = {R(0), R(0), R(0)};
  if (pbc)
    sh = v3(image_shift(i.cx - j.cx, L, invL), image_shift(i.cy - j.cy, L, invL), image_shift(i.cz - j.cz, L, invL));
  const V3<R> d = {j.cx + sh.x - i.cx, j.cy + sh.y - i.cy, j.cz + sh.z - i.cz};
  R reach = R(0);
  if (contact) reach = i.r + j.r + contact_margin(j.r, j.em);
  if (adh) {
    const R l0m = fmax(i.l0, fmax(j.l0, R(1e-12f)));
    reach = fmax(reach, i.r + j.r + R(2) * l0m);
  }
  const R rr = reach * R(1.0001f) + R(1e-6f);
  return vdot(d, d) <= rr * rr;
}

template <typename R>
static void search(double at, double skin_d, int pbc, int n, unsigned seed, long* out) {
  std::mt19937_64 g(seed);
  auto u = [&](double a, double b) { return a + (b - a) * std::uniform_real_distribution<double>(0, 1)(g); };
  const R skin = (R)skin_d;
  for (int q = 0; q < n; q++) {
    const R L = (R)u(20, 60), invL = R(1) / L;
    auto cell = [&](double x, double y, double z) {
      const R em = (R)u(0.2, 0.4);
      return make_cell_stat<R>((R)x, (R)y, (R)z, (R)u(0.8, 1.2), em, (R)u(0.2, 0.4));
    };
    const double far[3] = {at * u(-1, 1), at * u(-1, 1), at * u(-1, 1)};
    const CellStat<R> i0 = cell(far[0], far[1], far[2]);
    double e[3] = {u(-1, 1), u(-1, 1), u(-1, 1)};
    if (u(0, 1) < 0.5) e[(int)u(0, 3)] = 0.0;
    const double en = std::sqrt(e[0] * e[0] + e[1] * e[1] + e[2] * e[2]);
    if (!(en > 0.1)) continue;
    const bool contact = u(0, 1) < 0.7, adh = !contact || u(0, 1) < 0.5;
    // j an image away (periodic) along each axis, at distance D along e
    double img[3];
    for (double& k : img) k = pbc ? std::floor(u(-1, 2)) * (double)L : 0.0;
    CellStat<R> j0 = cell(0, 0, 0);
    auto put = [&](double D) {
      j0.cx = (R)((double)i0.cx + e[0] / en * D + img[0]);
      j0.cy = (R)((double)i0.cy + e[1] / en * D + img[1]);
      j0.cz = (R)((double)i0.cz + e[2] / en * D + img[2]);
    };
    double lo = 0.5, hi = 9.0;  // the closest place that is not listed
    for (int k = 0; k < 80; k++) {
      const double m = 0.5 * (lo + hi);
      put(m);
      (near_list_takes(i0, j0, pbc, L, invL, contact, adh, skin) ? lo : hi) = m;
    }
    put(hi);
    if (near_list_takes(i0, j0, pbc, L, invL, contact, adh, skin)) continue;
    out[0]++;
    // each as far towards the other as it may go without a mark, part of it by growing
    auto closer = [&](const CellStat<R>& s, double sign) {
      CellStat<R> best = s;
      const double grow = u(0, 1) < 0.5 ? 0.0 : u(0, 0.5);
      double a = 0, b = skin_d;
      bool any = false;
      for (int k = 0; k < 60; k++) {
        const double m = 0.5 * (a + b);
        CellStat<R> c = s;
        c.cx = (R)((double)s.cx + sign * e[0] / en * m * (1 - grow));
        c.cy = (R)((double)s.cy + sign * e[1] / en * m * (1 - grow));
        c.cz = (R)((double)s.cz + sign * e[2] / en * m * (1 - grow));
        c.r = (R)((double)s.r + m * grow);
        if (near_list_moved(s, v3(c.cx, c.cy, c.cz), c.r, c.em, pbc != 0, L, skin)) {
          b = m;
        } else {
          a = m;
          best = c;
          any = true;
        }
      }
      if (!any && near_list_moved(s, v3(s.cx, s.cy, s.cz), s.r, s.em, pbc != 0, L, skin)) best.r = R(-1);
      return best;
    };
    const CellStat<R> i1 = closer(i0, 1.0), j1 = closer(j0, -1.0);
    if (i1.r < R(0) || j1.r < R(0)) continue;  // marked stale where they are
    out[1]++;
    if (in_reach(i1, j1, pbc, L, invL, contact, adh)) out[2]++;
  }
}
extern "C" void search_pairs(int bits, double at, double skin, int pbc, int n, unsigned seed, long* out) {
  out[0] = out[1] = out[2] = 0;
  if (bits == 64) search<double>(at, skin, pbc, n, seed, out);
  else search<float>(at, skin, pbc, n, seed, out);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("near")
    src, so = str(d / "near.hip"), str(d / "near.so")
    with open(src, "w") as f:
        f.write(SRC)
    subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--offload-host-only", "-w", "-shared", f"-I{build.CSRC}", src, "-o",
                    so], check=True, cwd=str(d))
    return ctypes.CDLL(so)


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("pbc", [0, 1])
@pytest.mark.parametrize("at", [0.0, 30.0, 1e3, 1e4, 1e5, 1e6])
@pytest.mark.parametrize("skin", [0.15, 1e-2, 1e-4, 1e-6])
def test_no_pair_in_reach_is_missing_from_the_lists(lib, skin, at, pbc, bits):
    out = (ctypes.c_long * 3)()
    lib.search_pairs(bits, ctypes.c_double(at), ctypes.c_double(skin), pbc, 20000, 7, out)
    print(f"skin {skin} at {at} pbc {pbc} {bits} bits: {out[0]} pairs, {out[1]} with lists in force, {out[2]} missing")
    assert out[0] > 10000
    assert out[2] == 0
    if skin == 0.15 and at <= 1e3:
        assert out[1] > 10000  # the lists serve tissues near the origin
