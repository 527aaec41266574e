// Cell statistics of the 3D step and the rules that select pairs of cells by
// them.  No kernels here: the host can compile these rules too.
#pragma once
#include "dpm_device.h"

using namespace dpm;

// Per-cell statistics of a step's input positions (written by the previous
// step's epilogue or k3d_stats): centre of mass, bounding radius, longest
// edge, target edge length l0, and 1 / max(l0, 1e-12) in double (the
// adhesion term's, divided once per cell instead of once per pair).  Eight
// reals either way (32 bytes in float, 64 in double).
template <typename R>
struct CellStat;
template <>
struct CellStat<float> {
  float cx, cy, cz, r;
  float em, l0;
  double inv_l0;
};
template <>
struct CellStat<double> {
  double cx, cy, cz, r;
  double em, l0;
  double inv_l0, pad;
};
template <typename R>
__host__ __device__ inline CellStat<R> make_cell_stat(R cx, R cy, R cz, R r, R em, R l0) {
  CellStat<R> s{};
  s.cx = cx;
  s.cy = cy;
  s.cz = cz;
  s.r = r;
  s.em = em;
  s.l0 = l0;
  s.inv_l0 = 1.0 / (double)(l0 > R(1e-12f) ? l0 : R(1e-12f));
  return s;
}

// Periodic shift of cell j toward cell i along one axis, L round(d / L)
// with d = C_i - C_j (Cell3D_Kernel.cl:279-281).  The quotient is taken as
// a product with 1/L (within two ulp of the quotient); only where that
// product lies within 1e-5 (relative) of a half-integer can the two round
// differently, and there the division itself decides.
template <typename R>
__host__ __device__ __forceinline__ R image_shift(R d, R L, R invL) {
  const R q = d * invL;
  R n = round(q);
  if (fabs(fabs(q - n) - R(0.5f)) < R(1e-5f) * (R(1) + fabs(q))) n = round(d / L);
  return L * n;
}

// Culling reach added to a cell's bounding radius for the winding-number
// test.  Every face of cell j lies inside its bounding sphere R_j, so a
// point p outside R_j + m_j is at least m_j from every face and edge of j,
// and outside j's convex hull: its exact winding number is 0.  An edge of
// length <= e seen from distance >= d subtends at most 2 atan(e / 2d); with
// d >= 0.4 e that is <= 102.7 degrees, so every pair of the unit vectors
// u, v, w toward a face's corners has a dot product >= -0.2195 and the
// reference's denominator 1 + u.v + v.w + w.u (Cell3D_Kernel.cl:293) is
// >= 0.34: no face is skipped (denom < 1e-8), and the float sum of the
// face angles is rounding noise about a true 0, far below the 1e-6 pair
// threshold (Cell3D_Kernel.cl:303) — the pair is absent in the reference
// arithmetic too.  m_j = 0.4 e_max(j) (with slack for float rounding).
template <typename R>
__host__ __device__ __forceinline__ R contact_margin(R Rj, R emax_j) {
  return emax_j * R(0.4004f) + R(1e-6f) * Rj;
}

// ---------------------------------------------------------- candidate lists
//
// The scan tests every cell of the tissue for every cell and step: at 4096
// cells of 642 vertices a third of the step (27 of 86 kcycles of a
// workgroup).  A step that finds its tissue's lists stale scans as before and
// also keeps, per cell, the cells within `skin` of its reach; the following
// steps apply the scan's own test to those entries, in the same ascending
// order, so the candidates are the scan's, bit for bit.
// The lists hold as long as no pair can have come closer than the skin: a
// cell's excess is its centre's displacement since the lists were made plus
// what its radius and contact margin grew; the reach of a pair grows by no
// more than both excesses, its minimum-image distance shrinks by no more.
// The step that moves a cell past 0.49 of the skin marks the tissue's lists
// stale for the next one, and so does a cell whose tests may round by more than
// the 0.02 of the skin that both halves leave: with u half an ulp of 1, each of
// two tests of a pair rounds C_j + shift (u |C|, the shift is the same number
// both times), the image may be the other of two equal ones (u L), and the
// differences, squares and the reach round by u times a few reaches.  Without
// periodic images the coordinates' size does not enter.  A tissue far from the
// origin, or with one cell far smaller than the others (the skin follows the
// smallest), thus scans.  A tissue whose lists went stale in the step that made
// them has kNearPause - 1 steps without them: there the entries cost and serve
// nothing (10000 cells of 162 vertices that pass the skin at every step: 1062 us
// a step with lists made at each, 924 now, 925 by the scan alone).  Four sets of
// marks in turn: the one read, the one written for the next step, the
// one cleared for the step after.
constexpr int kNearList = DPM_WAVE;
constexpr int kNearPause = 8;

// The mark that a cell past the skin leaves for the next step: 0 lists in
// force, 1 the step makes them, more: it scans, and the mark counts down.
__host__ __device__ __forceinline__ int near_list_mark(bool made_now) { return made_now ? kNearPause : 1; }

template <typename R>
__host__ __device__ __forceinline__ bool near_list_moved(const CellStat<R>& ref, V3<R> C, R r, R em, bool pbc, R L,
                                                         R skin) {
  const V3<R> d = {C.x - ref.cx, C.y - ref.cy, C.z - ref.cz};
  const R zero = R(0);
  const R excess = sqrt(vdot(d, d)) + R(1.0002f) * fmax(zero, r - ref.r) + R(0.41f) * fmax(zero, em - ref.em);
  const R ulp = sizeof(R) == 4 ? R(0x1p-23) : R(0x1p-52);
  R size = R(16) * ((r + em) + ref.l0);
  if (pbc) size += R(2) * (((fabs(C.x) + fabs(C.y)) + fabs(C.z)) + L);
  return !(excess <= R(0.49f) * skin && ulp * size <= R(0.02f) * skin);  // a NaN is stale
}

// The scan's test with the skin: within reach + skin by either contact or
// adhesion, or the pair takes every image.
template <typename R>
__host__ __device__ __forceinline__ bool near_list_takes(const CellStat<R>& sti, const CellStat<R>& stj, bool pbc, R L, R invL,
                                                bool contact, bool adhesion, R skin) {
  V3<R> sh = {R(0), R(0), R(0)};
  if (pbc)
    sh = v3(image_shift(sti.cx - stj.cx, L, invL), image_shift(sti.cy - stj.cy, L, invL),
            image_shift(sti.cz - stj.cz, L, invL));
  const V3<R> d = {stj.cx + sh.x - sti.cx, stj.cy + sh.y - sti.cy, stj.cz + sh.z - sti.cz};
  R reach = R(0);
  if (contact) reach = sti.r + stj.r + contact_margin(stj.r, stj.em);
  if (adhesion) reach = fmax(reach, sti.r + stj.r + R(2) * fmax(sti.l0, fmax(stj.l0, R(1e-12f))));
  const R rr = (reach + skin) * R(1.0001f) + R(1e-6f);
  return vdot(d, d) <= rr * rr || (pbc && R(2) * rr >= R(0.999f) * L);
}
