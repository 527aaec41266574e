// The 2D step for tissues beyond one workgroup (float).
//
// k2d_run keeps a whole tissue in one workgroup's LDS; a tissue larger than
// that (the reference's Tissue2D has no size limit: its NDRange covers every
// cell, Tissue2D.cpp:212) runs here over the whole device, three launches
// per step on global arrays laid out as k2d_run's LDS (the same Lds2D view,
// pointing at global memory, and the same per-cell, candidate and per-vertex
// functions, so every decision and every force is k2d_run's):
//   k2d_wide_cells  eight lanes per cell: strain, orientation, centre of mass,
//                   bounds of the input positions;
//   k2d_wide_cand   one wave per cell: its candidate cells, ascending (the
//                   lanes test 64 cells at a time, a ballot keeps the order);
//   k2d_wide_step   a group of lanes per vertex: all force terms, then
//                   x + F dt into the other position buffer (positions are
//                   double-buffered, so every vertex reads the step's input
//                   positions).
#pragma once

struct Wide2D {
  Geom2D<float> g;
  const float* xin;
  const float* yin;
  float* xout;
  float* yout;
  float* fx;  // forces of the step (written with W2_FORCES)
  float* fy;
  const int* cell_tissue;  // [C]
  const int* vbl;          // [C + T]: tissue-local vertex offsets; tissue t's nc + 1 at c0 + t
  float* cellq;            // [8 * C]: strain, orientation, com x, com y, x0, x1, y0, y1
  int* ncand;              // [C]
  short* cand;             // [C * DPM2D_MAXCAND]
  int C, V;
  float dt;
  int flags;
  unsigned long long* counters;  // [4 * DPM_COUNTER_SLOTS] (may be nullptr)
  int* p_overlap;          // diagnostics per vertex (nullptr normally)
  int* p_attr;
  unsigned* p_attr_key;
  const int* vcell;        // [V] cell of each vertex
};

enum : int {
  W2_FORCES = 1,  // write the forces
  W2_MOVE = 2,    // write x + F dt
};

// The Lds2D view of tissue t over the global arrays and positions x, y.
__device__ __forceinline__ Lds2D<float> wide_view(const Wide2D& a, const Tissue2DCtx<float>& T, int t, const float* x,
                                                  const float* y) {
  Lds2D<float> l;
  l.x = const_cast<float*>(x) + T.v0;
  l.y = const_cast<float*>(y) + T.v0;
  l.vb = const_cast<int*>(a.vbl) + T.c0 + t;
  float* q = a.cellq + T.c0;
  l.strain = q;
  l.orient = q + a.C;
  l.comx = q + 2 * (size_t)a.C;
  l.comy = q + 3 * (size_t)a.C;
  l.ax0 = q + 4 * (size_t)a.C;
  l.ax1 = q + 5 * (size_t)a.C;
  l.ay0 = q + 6 * (size_t)a.C;
  l.ay1 = q + 7 * (size_t)a.C;
  l.l0c = const_cast<float*>(a.g.l0) + T.c0;
  l.ncand = a.ncand + T.c0;
  l.cand = a.cand + (size_t)T.c0 * DPM2D_MAXCAND;
  l.cbits = nullptr;
  l.red = nullptr;
  l.has_arc = l.has_vc = false;
  l.arc = nullptr;
  l.vc = nullptr;
  return l;
}

extern "C" __global__ void __launch_bounds__(256) k2d_wide_cells(const Wide2D a) {
  const int gc = (int)((blockIdx.x * blockDim.x + threadIdx.x) / 8);
  if (a.counters && blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&a.counters[0], 1ull);
  if (gc >= a.C) return;  // whole groups
  const int t = a.cell_tissue[gc];
  const Tissue2DCtx<float> T = tissue_ctx(a.g, t);
  cell_group(a.g, T, wide_view(a, T, t, a.xin, a.yin), gc - T.c0, threadIdx.x & 7);
}

// The list cand_one makes (maybe_pair over the tissue's cells, ascending,
// the count past DPM2D_MAXCAND meaning "scan every cell"), by one wave.
extern "C" __global__ void __launch_bounds__(256) k2d_wide_cand(const Wide2D a) {
  const int lane = threadIdx.x & (DPM_WAVE - 1);
  const int gc = blockIdx.x * (blockDim.x / DPM_WAVE) + (int)(threadIdx.x / DPM_WAVE);
  if (gc >= a.C) return;  // whole wave
  const int t = a.cell_tissue[gc];
  const Tissue2DCtx<float> T = tissue_ctx(a.g, t);
  const Lds2D<float> l = wide_view(a, T, t, a.xin, a.yin);
  const int ci = gc - T.c0;
  int n = 0;
  for (int c0 = 0; c0 < T.nc; c0 += DPM_WAVE) {  // wave-uniform
    const int cj = c0 + lane;
    const bool hit = cj < T.nc && cj != ci && maybe_pair(a.g, T, l, ci, cj);
    const unsigned long long m = __ballot(hit);
    const int slot = n + (int)__popcll(m & ((1ull << lane) - 1ull));
    if (hit && slot < DPM2D_MAXCAND) l.cand[ci * DPM2D_MAXCAND + slot] = (short)cj;
    n += (int)__popcll(m);
  }
  if (lane == 0) l.ncand[ci] = n;
}

// A group of G lanes per vertex (G a power of two; the groups of a wave are
// aligned, every lane of a group takes the same branches).  The group's lanes
// test G candidate cells at a time against the vertex, then share the near
// cells' vertices (attraction, vertex repulsion) or edges (crossing parity)
// between them; the terms of accepted pairs are added in ascending vertex
// order, one lane's after the other's, so every sum is force_vertex's, bit
// for bit.
//
// One thread per vertex, the form before this one, is 37 workgroups for the
// 9,400 vertices of the reference's test2D.py tissue: 127 us of a 155 us
// step, a chain of dependent loads on an idle chip, beside 15 us for a pass
// of its own over (vertex, candidate slot) for the crossing parity.
template <int G>
struct VertexGroup {
  int lane, base;  // lane in the group, first lane of the group in the wave
  __device__ __forceinline__ VertexGroup()
      : lane(threadIdx.x & (G - 1)), base((threadIdx.x & (DPM_WAVE - 1)) & ~(G - 1)) {}
  __device__ __forceinline__ unsigned long long bits(bool p) const {
    const unsigned long long m = __ballot(p) >> base;
    return G == DPM_WAVE ? m : m & ((1ull << G) - 1ull);
  }
  template <typename V>
  __device__ __forceinline__ V from(V v, int src) const { return __shfl(v, base + src); }
};

// Calls cell(cj) for the candidates of ci that pass keep(cj), ascending,
// while it returns true.
template <int G, typename Keep, typename Cell>
__device__ __forceinline__ void group_candidates(const VertexGroup<G>& w, const Lds2D<float>& l, int ci, int nc,
                                                 Keep keep, Cell cell) {
  const int ncd = l.ncand[ci];
  const bool scan_all = ncd > DPM2D_MAXCAND;
  const int ncl = scan_all ? nc : ncd;
  for (int q0 = 0; q0 < ncl; q0 += G) {
    const int q = q0 + w.lane;
    const int cj = q < ncl ? (scan_all ? q : (int)l.cand[ci * DPM2D_MAXCAND + q]) : ci;
    for (unsigned long long m = w.bits(cj != ci && keep(cj)); m; m &= m - 1ull)
      if (!cell(w.from(cj, __ffsll((long long)m) - 1))) return;
  }
}

template <int G>
__global__ void __launch_bounds__(256) k2d_wide_step(const Wide2D a) {
  const VertexGroup<G> w;
  const int gv = (int)((blockIdx.x * blockDim.x + threadIdx.x) / G);
  if (gv >= a.V) return;  // whole groups
  const int gc = a.vcell[gv];
  const int t = a.cell_tissue[gc];
  const Tissue2DCtx<float> T = tissue_ctx(a.g, t);
  const Lds2D<float> l = wide_view(a, T, t, a.xin, a.yin);
  const int k = gv - T.v0, ci = gc - T.c0;
  const float px = l.x[k], py = l.y[k], L = T.L, half_l = 0.49f * L;
  const unsigned mask = a.g.mask;
  float fx, fy;
  shape_vertex(a.g, T, l, ci, k, fx, fy, (double*)nullptr);
  // the accepted pairs of one stride of G vertices, in order
  auto add = [&](bool hit, float tx, float ty) {
    const unsigned long long hits = w.bits(hit);
    for (unsigned long long m = hits; m; m &= m - 1ull) {
      const int src = __ffsll((long long)m) - 1;
      fx += w.from(tx, src);
      fy += w.from(ty, src);
    }
    return (int)__popcll(hits);
  };
  int na = 0;
  if ((mask & M2_ATTRACTION) && (T.Kat != 0.0f || a.p_attr || a.p_attr_key)) {
    const float l0 = a.g.l0[gc];
    const float kat = T.Kat / (float)(l.vb[ci + 1] - l.vb[ci]);
    const float lim = l0 * l0 * 1.00001f;
    const double kk = (double)kat / (double)l0;
    group_candidates(w, l, ci, T.nc, [&](int cj) { return !vertex_far_from_box(l, T, cj, px, py, l0); }, [&](int cj) {
      const int e = l.vb[cj + 1];
      for (int j0 = l.vb[cj]; j0 < e; j0 += G) {
        const int j = j0 + w.lane;
        bool hit = false;
        float tx = 0.0f, ty = 0.0f;
        if (j < e) {  // force_vertex's pair test and term
          const float xj = l.x[j], yj = l.y[j];
          float rx = xj - px, ry = yj - py, nx = 0.0f, ny = 0.0f;
          if (T.pbc && !(fabs(rx) < half_l && fabs(ry) < half_l)) {
            nx = round(rx / L);
            ny = round(ry / L);
            rx -= L * nx;
            ry -= L * ny;
          }
          const float d2 = rx * rx + ry * ry;
          hit = d2 < lim && sqrt(d2) < l0;
          if (hit) {
            tx = (float)(kk * (((double)xj - (double)px) - (double)L * (double)nx));
            ty = (float)(kk * (((double)yj - (double)py) - (double)L * (double)ny));
            if (a.p_attr_key) atomicAdd(&a.p_attr_key[gv], vertex_key(xj, yj));
          }
        }
        na += add(hit, tx, ty);
      }
      return true;
    });
  }
  if (mask & M2_VREPULSION) {
    const float l0i = a.g.l0[gc];
    auto sigma = [&](int cj) { return 0.5f * (l0i + a.g.l0[T.c0 + cj]); };
    group_candidates(w, l, ci, T.nc, [&](int cj) { return !vertex_far_from_box(l, T, cj, px, py, sigma(cj)); },
                     [&](int cj) {
      const float sig = sigma(cj);
      const int e = l.vb[cj + 1];
      for (int j0 = l.vb[cj]; j0 < e; j0 += G) {
        const int j = j0 + w.lane;
        bool hit = false;
        float tx = 0.0f, ty = 0.0f;
        if (j < e) {
          float rx = l.x[j] - px, ry = l.y[j] - py;
          if (T.pbc && !(fabs(rx) < half_l && fabs(ry) < half_l)) {
            rx -= L * round(rx / L);
            ry -= L * round(ry / L);
          }
          const float d2 = rx * rx + ry * ry;
          hit = d2 < sig * sig && d2 != 0.0f;
          if (hit) {
            const float dist = sqrt(d2);
            const float ov = 1.0f - dist / sig;
            const float ft = T.Kre / sig * ov / dist;
            tx = -(ft * rx);
            ty = -(ft * ry);
          }
        }
        (void)add(hit, tx, ty);
      }
      return true;
    });
  }
  bool over = false;
  if (mask & M2_REPULSION) {
    group_candidates(w, l, ci, T.nc, [&](int cj) { return !outside_box_even(l, cj, px, py, T.pbc, L); }, [&](int cj) {
      over = __popcll(w.bits(crossing_odd(l, cj, px, py, T.pbc, L, T.invL, w.lane, G))) & 1;
      return !over;
    });
    if (over) repulsion_push(a.g, T, l, ci, px, py, fx, fy);
  }
  if (w.lane != 0) return;
  if (a.p_overlap) a.p_overlap[gv] = over ? 1 : 0;
  if (a.p_attr) a.p_attr[gv] = na;
  if (a.flags & W2_FORCES) {
    a.fx[gv] = fx;
    a.fy[gv] = fy;
  }
  if (a.flags & W2_MOVE) {
    a.xout[gv] = fmaf(fx, a.dt, px);
    a.yout[gv] = fmaf(fy, a.dt, py);
  }
  if (a.counters && over) atomicAdd(&a.counters[4 * (gv % DPM_COUNTER_SLOTS) + 2], 1ull);
}

// Lanes per vertex for V vertices: a small tissue is bound by one vertex's
// chain of loads and loops (more lanes shorten it), a large one by issue
// (fewer lanes idle in the last stride of a cell).  us per step at 32 / 16 /
// 8 lanes (one thread per vertex): 9,400 vertices 34 / 40 / 54 (155); 17,500
// 41 / 46 / 59 (376); 48,000 50 / 45 / 54 (204); 215,000 145 / 109 / 96
// (299); 328,000 213 / 150 / 133 (350).  64 lanes lose to 32 at every size
// above 3,000 vertices.
inline int wide_group(int V) { return V <= 32768 ? 32 : V <= 131072 ? 16 : 8; }
