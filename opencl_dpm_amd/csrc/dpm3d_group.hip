// Workgroup-per-cell form of the 3D step: 256 threads own one cell, thread t
// its vertices t, t + 256, ... (VPT of them); 512 threads in small handles of
// 257 to 512 vertices.
//
// The form serves what the wave-per-cell form does not: handles of few or a
// middling number of cells, where a step is one chain of dependent passes on a
// device that has room for more waves, and meshes over 256 vertices.  Both are
// bound by latency, so the passes are arranged for few barriers and independent
// loads:
//   loads and the candidate test of up to 256 cells | barrier | facing-down
//   faces, ring walk, separation and vertex lists of the candidates (a wave
//   each) | barrier | substrate, bending, the pair tests of all kept
//   candidates together | barrier | their sums, in order | barrier | Euler
//   step | barrier | volume, radius, longest edge | barrier | statistics.
// Long lists, many candidates and contact of many points or of cells with more
// than a vertex a thread take the candidates one by one.
// Four waves, not one thread per vertex: 11 waves of a 642-vertex cell at 141
// registers filled a compute unit alone, and every barrier idled it.
// Against one thread per vertex, a face pass of its own and five barriers per
// candidate, us per step: 9 x 162 vertices 12.9 -> 9.9, 256 x 162 23.5 ->
// 17.1, 4096 x 642 375 -> 133, in double 256 x 162 30.0 -> 23.7 and 1024 x 642
// 158 -> 97.
#pragma once

constexpr int kGrpThreads = 256;
constexpr int kGrpWaves = kGrpThreads / DPM_WAVE;
constexpr int kGrpSeg = 16;     // candidates of one wave's 64 cells kept ahead of the first barrier
constexpr int kGrpSlots = 4;    // candidates whose vertex lists are kept at once
constexpr int kGrpCap = 64;     // entries of such a list
constexpr int kGrpTasks = 512;  // partial sums of the adhesion pairs kept at once
// (candidate, vertex) points whose winding numbers are taken together: beyond
// that, re-reading a candidate's vertices from the L2 for every point costs more
// than staging it.  16 to 512 cells of 12 to 252 vertices packed into contact, 120
// workloads: a limit of 64 loses up to 8 per cent (92 vertices, 16 cells 45.8 ->
// 49.6 us a step), one of 1 up to 16 (12 vertices, 64 cells 19.1 -> 22.1); the
// means are alike.
constexpr int kGrpPoints = 16;
constexpr int kGrpSlices = 256;  // partial sums a candidate is cut into, at most
static_assert(kGrpSlots == 4 && kGrpCap <= 127 && kGrpSlices <= kGrpTasks, "the task search and the records' fields");

// LDS.  Three users of the last bytes, one after the other: the kept
// candidates' lists and partial sums; a candidate taken by itself (its own
// vertices over the bending sums); within that, winding directions, then
// partial sums.
struct LdsGroup {
  size_t own, sb, faces, down, rec, seg, segst, clist, glist, plist, gath, cnt, red, slots, slot, pw, acc, wb, nlist, mlist,
      smap, ut, total;
};
__host__ __device__ inline LdsGroup ldsg_layout(int nv, int nf, int ww, int rsize, int nt = kGrpThreads) {
  LdsGroup L;
  const size_t threads = (size_t)nt, waves = threads / DPM_WAVE;
  const size_t rs = (size_t)rsize, n = (size_t)nv;
  auto al = [](size_t o) { return (o + 31u) & ~(size_t)31u; };
  size_t o = 0;
  L.own = o;   o = al(o + 3u * rs * n);
  L.sb = o;    o = al(o + 3u * rs * n);
  L.faces = o; o = al(o + 4u * (size_t)nf);
  L.down = o;  o = al(o + (n + 3u) / 4u * 4u);  // facing-down faces per vertex, a byte each
  L.rec = o;   o = al(o + 4u * DPM_WAVE);
  L.seg = o;   o = al(o + 4u * waves * kGrpSeg);
  L.segst = o; o = al(o + 8u * rs * waves * kGrpSeg);
  L.clist = o; o = al(o + 4u * threads);
  L.glist = o; o = al(o + 4u * threads);
  L.plist = o; o = al(o + 4u * threads);
  L.gath = o;  o = al(o + 4u * 96u);
  L.cnt = o;   o = al(o + 4u * 48u);
  L.red = o;   o = al(o + 8u * 6u * waves);
  const size_t z = o;
  const size_t wind = 4u * rs * n * (size_t)ww;
  const bool points = nv <= nt;  // contact points of all candidates together
  L.slots = o;
  L.slot = al(3u * rs * kGrpCap + 2u * kGrpCap + 2u * n);  // positions, own vertices, vertex -> place
  L.pw = al(o + kGrpSlots * L.slot);  // the points' winding numbers
  L.acc = al(L.pw + (points ? rs * kGrpPoints : 0u));  // winding directions, then partial sums
  const size_t fast = L.acc + (points && wind > 4u * rs * kGrpTasks ? wind : 4u * rs * kGrpTasks);
  o = z;
  L.wb = o;    o = al(o + rs * n);
  L.nlist = o; o = al(o + 2u * n);
  L.mlist = o; o = al(o + 2u * n);
  L.smap = o;  o = al(o + 2u * n);
  L.ut = o;
  const size_t sums = 4u * rs * (n > (size_t)kGrpSlices ? n : (size_t)kGrpSlices);
  o += wind > sums ? wind : sums;
  L.total = al(o > fast ? o : fast);
  return L;
}

// Waves that take winding numbers, a point each; 1: all four on one point at a
// time.  A cell in contact waits for hundreds of them: the more waves the
// better, as long as their directions (four reals a vertex) do not keep cells
// off a compute unit that its registers would hold.  Meshes of up to 256
// vertices have room for four.  Above, floats take four where two cells still
// fit a compute unit or the device holds all cells one a unit; doubles, the
// instance that keeps three cells, and larger meshes have all waves on one
// point, a barrier more each.  us per step, cells packed into contact, with one
// to three waves at them (in brackets) | with these: 252 vertices, 256 cells (3)
// 207 | 158, in double (1) 690 | 208; 162 in double (2) 192 | 113; 642 vertices,
// 256 cells (1) 2705 | 768 (all on one point 863), in double (1) 3660 | 1111;
// 4096 cells (1) 6853 | 2696.
// Workgroups of 512 threads take what fits.
inline int group_winding_waves(int nv, int nf, int rsize, bool many, int cells, int cus, int lds_max, int nt) {
  if (nv <= kGrpThreads) return kGrpWaves;
  if (nt > kGrpThreads) {
    int n = nt / DPM_WAVE;
    while (n > 1 && (int)ldsg_layout(nv, nf, n, rsize, nt).total > lds_max) n--;
    return n;
  }
  if (rsize == 8 || (many && nv == 642 && nf == 1280)) return 1;
  const int fit = lds_max / (int)ldsg_layout(nv, nf, kGrpWaves, rsize).total;  // cells per compute unit
  return fit >= 2 || cells <= fit * cus ? kGrpWaves : 1;
}

__device__ __forceinline__ int from_lane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float from_lane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double from_lane(double v, int l) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <typename R>
__device__ __forceinline__ CellStat<R> from_lane(const CellStat<R>& s, int l) {
  CellStat<R> q{};
  q.cx = from_lane(s.cx, l);
  q.cy = from_lane(s.cy, l);
  q.cz = from_lane(s.cz, l);
  q.r = from_lane(s.r, l);
  q.em = from_lane(s.em, l);
  q.l0 = from_lane(s.l0, l);
  q.inv_l0 = from_lane(s.inv_l0, l);
  return q;
}

// One overdamped Euler step of every cell (or, without F_MOVE, one force
// evaluation for diagnostics), nv <= VPT * 256.
// NVC, NFC, WWC: vertex and face counts and winding waves fixed at compile
// time (0: taken from the arguments).  NT threads.
template <typename R, int NVC, int NFC, int VPT, int WWC, bool PROBE = true, int NT = kGrpThreads>
__device__ __forceinline__ void k3d_step_body() {
  Step3DArgs<R>* a = step_args_here<R>();
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int W = NT / DPM_WAVE;
  static_assert(W <= 8, "the counters' words");
  const int nv = NVC > 0 ? NVC : a->nv, nf = NFC > 0 ? NFC : a->nf, ww = WWC > 0 ? WWC : a->ww;
  const int tid = threadIdx.x, lane = tid & (DPM_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / DPM_WAVE);
  const int ci = xcd_remap(blockIdx.x, gridDim.x);
  const LdsGroup LG = ldsg_layout(nv, nf, ww, (int)sizeof(R), NT);
  R* sx = reinterpret_cast<R*>(smem + LG.own);
  R* sy = sx + nv;
  R* sz = sy + nv;
  R* bx = reinterpret_cast<R*>(smem + LG.sb);  // bending sums; a single candidate's vertices
  R* by = bx + nv;
  R* bz = by + nv;
  unsigned* sf = reinterpret_cast<unsigned*>(smem + LG.faces);
  unsigned* down4 = reinterpret_cast<unsigned*>(smem + LG.down);
  const unsigned char* down = smem + LG.down;
  int* rec = reinterpret_cast<int*>(smem + LG.rec);
  int* seg = reinterpret_cast<int*>(smem + LG.seg);
  CellStat<R>* segst = reinterpret_cast<CellStat<R>*>(smem + LG.segst);
  int* cnt = reinterpret_cast<int*>(smem + LG.cnt);  // [0..16): compaction, then [16..) below
  int* seg_n = cnt + 16;  // per wave: candidates among its cells
  int* short_edge = cnt + 24;
  int* one = cnt + 28;  // counts of a candidate taken by itself
  double* red = reinterpret_cast<double*>(smem + LG.red);

  const Lds3DWave LT = ldsw_layout(nv, nf, 1, (int)sizeof(R));  // the topology image's offsets
  const uint4* rows = a->wtopo;
  const size_t base = (size_t)ci * nv;
  const V3<R> zero = {R(0), R(0), R(0)};

  // every load in flight before the first LDS store: own positions and
  // neighbour rows, faces, parameters, and the cell this thread tests
  V3<R> P[VPT];
  uint4 arow[VPT];
#pragma unroll
  for (int k = 0; k < VPT; k++) {
    const int v = tid + k * NT;
    P[k] = zero;
    arow[k] = make_uint4(~0u, ~0u, ~0u, ~0u);
    if (v < nv) {
      P[k] = v3(a->xin[base + v], a->yin[base + v], a->zin[base + v]);
      arow[k] = rows[LT.adj / 16 + v];
    }
  }
  // (a handle of one tissue needs no look-up: two dependent loads less)
  int t = 0, cb = 0, ce = a->ncells;
  if (!a->one_tissue) {
    t = a->cell_tissue[ci];
    cb = a->tissue_begin[t];
    ce = a->tissue_begin[t + 1];
  }
  const R L = (R)a->tL[t];
  const int pbc = a->tpbc[t];
  const R Kre = (R)a->tKre[t], Kat = (R)a->tKat[t], ksg = (R)a->tksg[t];
  const CellStat<R> sti = a->st_in[ci];
  const V3<R> Ci = {sti.cx, sti.cy, sti.cz};
  const R Ri = sti.r;
  const R Kvi = (R)a->Kv[ci], Kai = (R)a->Ka[ci], Ksi = (R)a->Ks[ci], Kbi = (R)a->Kb[ci];
  const R v0i = (R)a->v0[ci], a0i = (R)a->a0[ci], l0i = cell_l0<R>(a->a0, ci);
  const unsigned mask = a->mask;
  const bool do_contact = (mask & M_CONTACT) && Kre != R(0);
  const bool do_adh = (mask & M_ADHESION) && Kat != R(0);
  const bool pairs_on = do_contact || do_adh;  // block-uniform, as all of these
  // candidate lists: made by this step, or read (nlist entries; not when
  // there are more than a list holds)
  const bool nl_on = a->nl_cnt && !a->bin_list && ce - cb > kNearList;
  const int stale = nl_on ? a->nl_stale[t] : 0;  // 1: make them; more: scan
  const bool relist = stale == 1;
  const int nlist = nl_on && stale == 0 ? a->nl_cnt[ci] : -1;
  const bool listed = nlist >= 0;
  CellStat<R> nl_ref = sti;  // where this step makes the lists
  if (nl_on && stale == 0) nl_ref = a->nl_ref[ci];
  const bool binned = a->bin_list && a->tbin_nb[t] > 0;
  // the candidates among at most 256 cells are found ahead of the first
  // barrier: each wave keeps those among its 64 cells
  const int nahead = !pairs_on || binned || relist ? 0 : listed ? nlist : ce - cb <= NT ? ce - cb : 0;
  int cj_l = ce;
  CellStat<R> st_l{};
  if (tid < nahead) {
    cj_l = listed ? a->nl_idx[(size_t)ci * kNearList + tid] : cb + tid;
    if (cj_l != ci) st_l = a->st_in[cj_l];
  }
  for (int f = tid; f < nf; f += NT) sf[f] = reinterpret_cast<const unsigned*>(rows)[f];
  for (int i = tid; i < (nv + 3) / 4; i += NT) down4[i] = 0u;
  if (tid == 0) {
    *short_edge = 0;
    one[3] = 0;
  }
#pragma unroll
  for (int k = 0; k < VPT; k++) {
    const int v = tid + k * NT;
    if (v < nv) {
      sx[v] = P[k].x;
      sy[v] = P[k].y;
      sz[v] = P[k].z;
    }
  }
  const R L0i = fmax(l0i, R(1e-12f));
  const R invL = R(1) / L;
  // the scan's test: centres within both radii and the contact margin, or
  // 2 l0; adhesion takes the minimum image per vertex pair
  // (Cell3D_Kernel.cl:341-346), which can differ from the centre-of-mass
  // image when the box is small: then no culling
  auto in_reach = [&](const CellStat<R>& stj) __attribute__((always_inline)) -> bool {
    V3<R> sh = zero;
    if (pbc)
      sh = v3(image_shift(Ci.x - stj.cx, L, invL), image_shift(Ci.y - stj.cy, L, invL),
              image_shift(Ci.z - stj.cz, L, invL));
    const V3<R> d = {stj.cx + sh.x - Ci.x, stj.cy + sh.y - Ci.y, stj.cz + sh.z - Ci.z};
    R reach = R(0);
    if (do_contact) reach = Ri + stj.r + contact_margin(stj.r, stj.em);
    bool all = false;
    if (do_adh) {
      const R l0m = fmax(L0i, fmax(stj.l0, R(1e-12f)));
      const R r2 = Ri + stj.r + R(2) * l0m;
      reach = fmax(reach, r2);
      all = pbc && R(2) * r2 >= R(0.999f) * L;
    }
    const R rr = reach * R(1.0001f) + R(1e-6f);
    return all || vdot(d, d) <= rr * rr;
  };
  {
    bool cand = false;
    if (cj_l < ce && cj_l != ci) cand = in_reach(st_l);
    const unsigned long long m = __ballot(cand);
    const int slot = lanes_below(m);
    if (cand && slot < kGrpSeg) {
      seg[wave * kGrpSeg + slot] = cj_l;
      segst[wave * kGrpSeg + slot] = st_l;
    }
    if (lane == 0) seg_n[wave] = __popcll(m);
  }
  __syncthreads();
  step_args_again<R>(a);

  // the kept candidates, one per lane in every wave, ascending
  unsigned long long cmask = 0;  // lanes that hold one
  bool ahead = nahead > 0;       // found ahead (otherwise searched for below)
  {
    int off = 0, src = -1;
#pragma unroll
    for (int w = 0; w < W; w++) {
      const int n = seg_n[w];
      if (n > kGrpSeg) ahead = false;
      if (src < 0 && lane < off + n && n <= kGrpSeg) src = w * kGrpSeg + (lane - off);
      off += n;
    }
    if (off > DPM_WAVE) ahead = false;
    if (ahead && lane < off) {
      cj_l = seg[src];
      st_l = segst[src];
    }
    if (ahead) cmask = off == DPM_WAVE ? ~0ull : (1ull << off) - 1ull;
  }

  V3<R> F[VPT];
  const bool shape_on = (mask & (M_VOLUME | M_SURFACE | M_SUBSTRATE)) != 0;
  // Volume strain of the current volume, in double (the residual V/v0 - 1
  // cancels when the cell is near its target).
  const R strain = (R)(a->vol_in[ci] / (double)v0i - 1.0);
  const R kvol = -Kvi * strain / R(6);
  const bool vol_on = (mask & M_VOLUME) && Kvi != R(0);
  const bool surf_on = (mask & M_SURFACE) && !(Kai < R(1e-8f));
  const bool sub_on = (mask & M_SUBSTRATE) && !(Ksi < R(1e-12f));
  const bool bend_on = (mask & M_BENDING) && Kbi != R(0);
  const R sc = Kai * sqrt(a0i) / l0i * R(0.3f);
  const R inv_l0 = R(1) / l0i;
  const double sub_inv_l0 = 1.0 / (double)l0i;

  // Facing-down faces (Cell3D_Kernel.cl:206-246), counted per vertex (integer
  // LDS atomics: the counts do not depend on their order).
  if (shape_on && sub_on) {
#pragma unroll
    for (int f = tid; f < nf; f += NT) {
      int i0, i1, i2;
      wface(sf, f, i0, i1, i2);
      const V3<R> P0 = lds_v(sx, sy, sz, i0);
      if (facing_down(vcross(vsub(lds_v(sx, sy, sz, i1), P0), vsub(lds_v(sx, sy, sz, i2), P0)))) {
        atomicAdd(&down4[i0 >> 2], 1u << (8 * (i0 & 3)));
        atomicAdd(&down4[i1 >> 2], 1u << (8 * (i1 & 3)));
        atomicAdd(&down4[i2 >> 2], 1u << (8 * (i2 & 3)));
        if (PROBE && a->p_down) a->p_down[(size_t)ci * nf + f] = 1;
      }
    }
  }
  // One walk around each vertex's ring u_0 .. u_(k-1) (closed mesh: face q is
  // (v, u_q, u_(q+1))), d_q = u_q - p: volume kvol sum_q d_q x d_(q+1), edge
  // springs 2 sc sum_q s(d_q), bending's first sum, as the wave-per-cell step
  // takes it.  The loads of six neighbours are issued together and an absent
  // one is the vertex itself (d = 0 adds nothing): with a branch per
  // neighbour each waited for the one before.
  bool bad = false;
  const bool ring = a->closed != 0;
  auto walk = [&](int k, auto degc) __attribute__((always_inline)) {
    constexpr int D = decltype(degc)::value;
    const int v = tid + k * NT;
    V3<R> d[D];
    bool has[D];
#pragma unroll
    for (int q = 0; q < D; q++) {
      const int u = row16(arow[k], q);
      has[q] = u != 0xffff;
      d[q] = vsub(lds_v(sx, sy, sz, has[q] ? u : v), P[k]);
    }
    V3<R> Fv = zero, Fs = zero, sb = zero;
#pragma unroll
    for (int q = 0; q < D; q++) {
      if (surf_on) {
        const R d2 = vdot_f(d[q], d[q]);
        bad = bad || (has[q] && d2 < R(4e-24f));
        R s = R(0);
        if (has[q]) s = spring_factor(d2, inv_l0);
        Fs = vmadd_f(d[q], s, Fs);
      }
      sb = vadd(sb, d[q]);
      if (vol_on) {
        const bool next = q + 1 < D && has[q + 1 < D ? q + 1 : 0];
        const V3<R> dn = next ? d[q + 1 < D ? q + 1 : 0] : d[0];
        Fv = vcross_add_f(d[q], dn, Fv);
      }
    }
    F[k] = vadd(vscale(Fv, kvol), vscale(Fs, R(2) * sc));
    if (bend_on) {
      bx[v] = sb.x;
      by[v] = sb.y;
      bz[v] = sb.z;
    }
  };
#pragma unroll
  for (int k = 0; k < VPT; k++) {
    const int v = tid + k * NT;
    F[k] = zero;
    if (ring && v < nv && (shape_on || bend_on)) {
      if (__ballot(row16(arow[k], 6) != 0xffff) != 0ull)
        walk(k, std::integral_constant<int, DPM3D_MAXDEG>{});
      else
        walk(k, std::integral_constant<int, 6>{});
      if (!shape_on) F[k] = zero;
    }
  }
  if (__ballot(bad) != 0ull && lane == 0) *short_edge = 1;

  // The kept candidates of a mask (cj_l, st_l per lane), the waves in turn:
  // the separation along the centre line n = (C_j - C_i) / D and the lists
  // of vertices in reach, in one pass over both cells' vertices.
  // Separation: every vertex p of this cell has (p - C_i).n <= hi and every
  // point x of cell j's (shifted) hull has (C_j - x).n <= hj, so
  // |x - p| >= D - hi - hj, less slack for the float sums (1e-4 of the cells'
  // extent, 1e-6 of the coordinates).  Contact needs a point closer than the
  // culling margin m_j to a face of j (contact_margin), adhesion a vertex
  // pair closer than 2 l0 on pairs that take no periodic image (the unshifted
  // centres and radii keep every component below 0.48 L; the shift is 0 then).
  // Lists: a pair closer than 2 l0 has |q - C_i| <= |q - p| + |p - C_i| <
  // 2 l0 + R_i, and the same bound reversed.
  // rec: 1 contact | 2 adhesion | 4 the lists fit, then near << 3 | own << 10
  // | slices << 17 | near vertices per slice << 24 (each at most 64): the
  // adhesion pairs are (own vertex, slice of near vertices) tasks, at most
  // kGrpSlices of them.
  auto separate = [&](unsigned long long m) __attribute__((always_inline)) {
    int o = 0;
    for (unsigned long long w = m; w; w &= w - 1ull, o++) {
      if (o % W != wave) continue;  // wave-uniform
      const int b = __ffsll((long long)w) - 1;
      const int cjq = from_lane(cj_l, b);
      const size_t bj = (size_t)cjq * nv;
      constexpr int kAtOnce = 4;  // 64-vertex chunks whose loads are issued together
      V3<R> q[kAtOnce];
      auto load = [&](int v0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kAtOnce; k++) {
          const int v = v0 + k * DPM_WAVE + lane;
          q[k] = zero;
          if (v < nv) q[k] = v3(a->xin[bj + v], a->yin[bj + v], a->zin[bj + v]);
        }
      };
      load(0);
      const CellStat<R> stj = from_lane(st_l, b);
      V3<R> sh = zero;
      if (pbc)
        sh = v3(image_shift(Ci.x - stj.cx, L, invL), image_shift(Ci.y - stj.cy, L, invL),
                image_shift(Ci.z - stj.cz, L, invL));
      const V3<R> Cj = {stj.cx + sh.x, stj.cy + sh.y, stj.cz + sh.z};
      const R l0m = fmax(L0i, fmax(stj.l0, R(1e-12f)));
      const bool all_images = pbc && R(2) * (Ri + stj.r + R(2) * l0m) >= R(0.999f) * L;
      const bool no_image = !pbc || (fabs(Ci.x - stj.cx) + (Ri + stj.r) < R(0.48f) * L &&
                                     fabs(Ci.y - stj.cy) + (Ri + stj.r) < R(0.48f) * L &&
                                     fabs(Ci.z - stj.cz) + (Ri + stj.r) < R(0.48f) * L);
      const V3<R> dC = vsub(Cj, Ci);
      const R D = sqrt(vdot(dC, dC));
      const V3<R> nC = D > R(0) ? vscale(dC, R(1) / D) : zero;
      const R rk = (Ri + R(2) * l0m) * R(1.0001f) + R(1e-6f);
      const R r2 = (stj.r + R(2) * l0m) * R(1.0001f) + R(1e-6f);
      unsigned char* sl = smem + LG.slots + (size_t)(o < kGrpSlots ? o : 0) * LG.slot;
      R* qx = reinterpret_cast<R*>(sl);
      R* qy = qx + kGrpCap;
      R* qz = qy + kGrpCap;
      unsigned short* own = reinterpret_cast<unsigned short*>(qz + kGrpCap);
      unsigned short* place = own + kGrpCap;
      const bool keep = o < kGrpSlots;
      R hi = R(-3.0e38f), hj = R(-3.0e38f);
      int nnear = 0, nmine = 0;
      for (int v0 = 0; v0 < nv; v0 += kAtOnce * DPM_WAVE) {
        if (v0 > 0) load(v0);
#pragma unroll
        for (int k = 0; k < kAtOnce; k++) {
          const int v = v0 + k * DPM_WAVE + lane;
          if (v0 + k * DPM_WAVE >= nv) break;  // wave-uniform
          bool near = false, mine = false;
          if (v < nv) {
            const V3<R> Pv = lds_v(sx, sy, sz, v);
            hi = fmax(hi, vdot(vsub(Pv, Ci), nC));
            hj = fmax(hj, vdot(v3(stj.cx - q[k].x, stj.cy - q[k].y, stj.cz - q[k].z), nC));
            if (do_adh) {
              const V3<R> ds = {q[k].x + sh.x - Ci.x, q[k].y + sh.y - Ci.y, q[k].z + sh.z - Ci.z};
              near = all_images || vdot(ds, ds) <= rk * rk;
              const V3<R> dp = {Pv.x - stj.cx - sh.x, Pv.y - stj.cy - sh.y, Pv.z - stj.cz - sh.z};
              mine = all_images || vdot(dp, dp) <= r2 * r2;
            }
          }
          if (do_adh) {
            const unsigned long long mn = __ballot(near), mm = __ballot(mine);
            const int jn = nnear + lanes_below(mn), jm = nmine + lanes_below(mm);
            if (keep && near && jn < kGrpCap) {
              qx[jn] = q[k].x;
              qy[jn] = q[k].y;
              qz[jn] = q[k].z;
            }
            if (keep && mine && jm < kGrpCap) own[jm] = (unsigned short)v;
            if (keep && v < nv) place[v] = mine ? (unsigned short)jm : (unsigned short)0xffff;
            nnear += __popcll(mn);
            nmine += __popcll(mm);
          }
        }
      }
      hi = wave_max_all(hi);
      hj = wave_max_all(hj);
      bool skip_contact = false, skip_adh = nnear == 0 || nmine == 0;
      const R Mc = ((fabs(Ci.x) + fabs(Ci.y)) + fabs(Ci.z)) + ((fabs(Cj.x) + fabs(Cj.y)) + fabs(Cj.z));
      if (D > R(0)) {
        const R gap = ((D - hi) - hj) - (R(1e-4f) * ((Ri + stj.r) + D) + R(1e-6f) * Mc);
        skip_contact = gap >= contact_margin(stj.r, stj.em);
        skip_adh = skip_adh || (!all_images && no_image && gap >= R(2) * l0m);
      }
      const int bits = ((do_contact && !skip_contact) ? 1 : 0) | ((do_adh && !skip_adh) ? 2 : 0);
      const bool fit = keep && nnear <= kGrpCap && nmine <= kGrpCap;
      if (lane == 0) {
        int e = bits;
        if (fit && nnear > 0 && nmine > 0) {
          const int S = max(1, min(nnear, kGrpSlices / nmine));
          e |= 4 | nnear << 3 | nmine << 10 | S << 17 | (nnear + S - 1) / S << 24;
        }
        rec[b] = e;
      }
    }
  };
  if (cmask) separate(cmask);
  __syncthreads();
  step_args_again<R>(a);

  const bool ring_ok = ring && !(surf_on && *short_edge);  // block-uniform
  if (!ring_ok && shape_on) {
    // an open mesh, one whose vertex faces are not one oriented cycle, or a
    // cell with an edge shorter than 2e-12 (an edge below 1e-12 makes the
    // reference skip its faces' springs): the vertex's faces one by one, in
    // ascending order
#pragma unroll 1
    for (int k = 0; k < VPT; k++) {
      const int v = tid + k * NT;
      V3<R> Fk = zero;
      if (v < nv) {
        const uint4 vrow = rows[LT.vf / 16 + v];
        for (int q = 0; q < DPM3D_MAXDEG; q++) {
          const int e = row16(vrow, q);
          if (e == 0xffff) break;
          const int f = e / 3, c = e - 3 * f;
          int i0, i1, i2;
          wface(sf, f, i0, i1, i2);
          const V3<R> P0 = lds_v(sx, sy, sz, i0), P1 = lds_v(sx, sy, sz, i1), P2 = lds_v(sx, sy, sz, i2);
          V3<R> cc = zero;
          if (vol_on) {  // Cell3D_Kernel.cl:95-111
            const V3<R> A = vsub(P1, Ci), B = vsub(P2, Ci), Cc = vsub(P0, Ci);
            cc = c == 0 ? vscale(vcross(A, B), kvol) : c == 1 ? vscale(vcross(B, Cc), kvol)
                                                              : vscale(vcross(Cc, A), kvol);
          }
          if (surf_on) {  // Cell3D_Kernel.cl:140-176
            const V3<R> lv0 = vsub(P1, P0), lv1 = vsub(P2, P1), lv2 = vsub(P0, P2);
            const R len0 = sqrt(vdot(lv0, lv0)), len1 = sqrt(vdot(lv1, lv1)), len2 = sqrt(vdot(lv2, lv2));
            if (!(len0 < R(1e-12f) || len1 < R(1e-12f) || len2 < R(1e-12f))) {
              const V3<R> la = c == 0 ? lv0 : c == 1 ? lv1 : lv2;
              const V3<R> lb = c == 0 ? lv2 : c == 1 ? lv0 : lv1;
              const R na = c == 0 ? len0 : c == 1 ? len1 : len2;
              const R nb = c == 0 ? len2 : c == 1 ? len0 : len1;
              const V3<R> ea = vscale(la, (na * inv_l0 - R(1)) / na);
              const V3<R> eb = vscale(lb, (nb * inv_l0 - R(1)) / nb);
              cc = vadd(cc, vscale(vsub(ea, eb), sc));
            }
          }
          if (sub_on && facing_down(vcross(vsub(P1, P0), vsub(P2, P0)))) {
            const V3<R> Pv = c == 0 ? P0 : c == 1 ? P1 : P2;
            cc = vadd(cc, substrate_corner(Pv, Ci, Ksi, ksg, L, l0i, sub_inv_l0));
          }
          Fk = vadd(Fk, cc);
        }
      }
#pragma unroll
      for (int j = 0; j < VPT; j++)
        if (j == k) F[j] = Fk;
    }
  } else if (shape_on && sub_on) {
#pragma unroll
    for (int k = 0; k < VPT; k++) {
      const int v = tid + k * NT;
      if (v < nv) {
        const unsigned n = down[v];
        if (n) F[k] = vadd(F[k], vscale(substrate_corner(P[k], Ci, Ksi, ksg, L, l0i, sub_inv_l0), (R)n));
      }
    }
  }
  if (bend_on) {
    if (!ring) {  // the first sums (a ring walk has them)
      for (int v = tid, k = 0; v < nv; v += NT, k++) {
        const V3<R> Pv = lds_v(sx, sy, sz, v);
        const uint4 row = rows[LT.adj / 16 + v];
        V3<R> s = zero;
        for (int q = 0; q < DPM3D_MAXDEG; q++) {
          const int u = row16(row, q);
          if (u == 0xffff) break;
          s = vadd(s, vsub(lds_v(sx, sy, sz, u), Pv));
        }
        bx[v] = s.x;
        by[v] = s.y;
        bz[v] = s.z;
      }
      __syncthreads();
    }
    auto second = [&](int k, auto degc) __attribute__((always_inline)) {
      constexpr int D = decltype(degc)::value;
      const int v = tid + k * NT;
      V3<R> acc = zero;
      int deg = 0;
#pragma unroll
      for (int q = 0; q < D; q++) {
        const int u = row16(arow[k], q);
        const bool has = u != 0xffff;
        const V3<R> s = lds_v(bx, by, bz, has ? u : v);
        acc = has ? vadd(acc, s) : acc;
        deg += has;
      }
      const V3<R> lap = vsub(acc, vscale(lds_v(bx, by, bz, v), (R)deg));
      F[k] = vadd(F[k], vscale(lap, -Kbi));
    };
#pragma unroll
    for (int k = 0; k < VPT; k++)
      if (tid + k * NT < nv) {
        if (__ballot(row16(arow[k], 6) != 0xffff) != 0ull)
          second(k, std::integral_constant<int, DPM3D_MAXDEG>{});
        else
          second(k, std::integral_constant<int, 6>{});
      }
  }

  // ------------------------------------------- contact and vertex adhesion
  unsigned n_wind = 0, n_contact = 0, n_cand = 0;
  R wsum[VPT];  // the contact force is wsum * Kre/2 * normalize(C_i - p)
  int npart[VPT];
#pragma unroll
  for (int k = 0; k < VPT; k++) {
    wsum[k] = R(0);
    npart[k] = 0;
  }
  // One own vertex against partners m0 .. m1 of a candidate: partner(m) is
  // the position of the m-th.
  auto pair_sum = [&](int v, int m0, int m1, R L0j, double inv_l0j, auto partner) __attribute__((always_inline)) -> Q4<R> {
    const V3<R> Pv = lds_v(sx, sy, sz, v);
    V3<R> Fa = zero;
    int cnt_own = 0;
    const R half_l = R(0.49f) * L;
    const AdhCut<R> cut_own(L0i * R(2)), cut_rev(L0j * R(2));
    const double kh = 0.5 * (double)Kat, inv_l0i = sti.inv_l0;
    const float kh_f = (float)kh, inv_l0i_f = (float)inv_l0i, inv_l0j_f = (float)inv_l0j;
    for (int m = m0; m < m1; m++) {
      const V3<R> pj = partner(m);
      // the own vertex's loop: delta = pj - p, minimum image per component
      // (Cell3D_Kernel.cl:341-346); a component below 0.49 L rounds to image
      // 0, which leaves it unchanged
      V3<R> dl = vsub(pj, Pv);
      V3<R> dr = vsub(Pv, pj);  // the partner's loop: delta = p - pj
      V3<R> nl = zero, nr = zero;
      bool imaged = false;
      if (pbc && !(fabs(dl.x) < half_l && fabs(dl.y) < half_l && fabs(dl.z) < half_l)) {
        nl = V3<R>{R(round(dl.x / L)), R(round(dl.y / L)), R(round(dl.z / L))};
        nr = V3<R>{R(round(dr.x / L)), R(round(dr.y / L)), R(round(dr.z / L))};
        dl = vsub(dl, v3(L * nl.x, L * nl.y, L * nl.z));
        dr = vsub(dr, v3(L * nr.x, L * nr.y, L * nr.z));
        imaged = true;
      }
      // The decisions are the reference's (AdhCut).  The force of an
      // accepted pair across the periodic boundary is evaluated in double on
      // the same image, since there the float difference of two near-L
      // numbers keeps few digits of a short vector; without an image
      // (dr = -dl exactly, the same squared distance) a float step takes it
      // in float (adhesion_term_near).
      const R d2 = vdot(dl, dl);
      if constexpr (sizeof(R) == 4) {
        if (!imaged) {
          const bool own_on = cut_own(d2), rev_on = cut_rev(d2);
          if (own_on || rev_on) {
            const R y = __builtin_amdgcn_rsqf(d2);
            if (own_on) {
              Fa = adhesion_term_near(dl, y, kh_f, inv_l0i_f, Fa);
              cnt_own++;
              if (PROBE && a->p_adh_hash) atomicAdd(&a->p_adh_hash[2 * (base + v)], vertex_key(pj.x, pj.y, pj.z));
            }
            if (rev_on) {
              Fa = adhesion_term_near(dl, y, kh_f, inv_l0j_f, Fa);
              if (PROBE && a->p_adh_hash) atomicAdd(&a->p_adh_hash[2 * (base + v) + 1], vertex_key(pj.x, pj.y, pj.z));
            }
          }
          continue;
        }
      }
      if (cut_own(d2)) {
        Fa = vsub(Fa, adhesion_term(pj, Pv, nl, L, Kat, L0i, kh, inv_l0i));
        cnt_own++;
        if (PROBE && a->p_adh_hash) atomicAdd(&a->p_adh_hash[2 * (base + v)], vertex_key(pj.x, pj.y, pj.z));
      }
      if (cut_rev(vdot(dr, dr))) {
        Fa = vadd(Fa, adhesion_term(Pv, pj, nr, L, Kat, L0j, kh, inv_l0j));
        if (PROBE && a->p_adh_hash) atomicAdd(&a->p_adh_hash[2 * (base + v) + 1], vertex_key(pj.x, pj.y, pj.z));
      }
    }
    return Q4<R>{Fa.x, Fa.y, Fa.z, (R)cnt_own};
  };
  // Own vertex k's contact with cell cj2 at winding number wv.
  auto touch = [&](int k, int cj2, R wv, V3<R> sh) __attribute__((always_inline)) {
    const int v = tid + k * NT;
    const size_t pidx = (base + v) * (size_t)a->ncmax + (size_t)(cj2 - cb);
    if (PROBE && a->p_winding) a->p_winding[pidx] = (float)wv;
    if (fabs(wv) < R(1e-6f)) return;
    const V3<R> dir = vnormalize(vsub(Ci, P[k]));
    const R mag = fabs(wv) * R(0.5f) * Kre;
    F[k] = vadd(F[k], vscale(dir, mag));
    n_contact++;
    wsum[k] += fabs(wv);
    if (a->rec_cell) {
      if (npart[k] < DPM3D_MAXPART) {
        const size_t r = (base + v) * DPM3D_MAXPART + npart[k];
        a->rec_cell[r] = cj2;
        a->rec_w[r] = wv;
        a->rec_shift[3 * r] = sh.x;
        a->rec_shift[3 * r + 1] = sh.y;
        a->rec_shift[3 * r + 2] = sh.z;
      } else {
        atomicOr(a->rec_overflow, 1);
      }
      npart[k]++;
    }
    if (PROBE && a->p_contact) a->p_contact[pidx] = 1;
    if (PROBE && a->p_contact_key) {  // count, then key sum of the partner cells
      atomicAdd(&a->p_contact_key[2 * (base + v)], 1u);
      atomicAdd(&a->p_contact_key[2 * (base + v) + 1], cell_key(cj2 - cb));
    }
  };
  auto shift_to = [&](const CellStat<R>& stj) __attribute__((always_inline)) -> V3<R> {
    if (!pbc) return V3<R>{R(0), R(0), R(0)};
    return V3<R>{image_shift(Ci.x - stj.cx, L, invL), image_shift(Ci.y - stj.cy, L, invL),
                 image_shift(Ci.z - stj.cz, L, invL)};
  };
  // A candidate by itself: lane b of cj_l, st_l; passes 1 contact, 2 adhesion.
  auto take_one = [&](int b, int passes) __attribute__((always_inline)) {
    const int cj2 = from_lane(cj_l, b);
    const CellStat<R> stj = from_lane(st_l, b);
    R* wb = reinterpret_cast<R*>(smem + LG.wb);
    unsigned short* nl = reinterpret_cast<unsigned short*>(smem + LG.nlist);
    unsigned short* ml = reinterpret_cast<unsigned short*>(smem + LG.mlist);
    unsigned short* sm = reinterpret_cast<unsigned short*>(smem + LG.smap);
    V3<R> sh = zero;
    if (pbc)
      sh = v3(image_shift(Ci.x - stj.cx, L, invL), image_shift(Ci.y - stj.cy, L, invL),
              image_shift(Ci.z - stj.cz, L, invL));
    __syncthreads();  // the bending sums, the lists and the candidate before are done with
    for (int v = tid; v < nv; v += NT) {
      bx[v] = a->xin[(size_t)cj2 * nv + v];
      by[v] = a->yin[(size_t)cj2 * nv + v];
      bz[v] = a->zin[(size_t)cj2 * nv + v];
    }
    if (tid == 0) one[0] = one[1] = 0;
    __syncthreads();
    if (passes & 1) {  // block-uniform
      const V3<R> Cj = {stj.cx + sh.x, stj.cy + sh.y, stj.cz + sh.z};
      const R mj = contact_margin(stj.r, stj.em);
      const R rj = (stj.r + mj) * R(1.0001f) + R(1e-6f);
      bool need[VPT];
#pragma unroll
      for (int k = 0; k < VPT; k++) {
        const int v = tid + k * NT;
        need[k] = false;
        if (v < nv) {
          const V3<R> d = vsub(P[k], Cj);
          need[k] = vdot(d, d) <= rj * rj;
        }
        const unsigned long long m = __ballot(need[k]);
        if (m) {  // the points, in any order (each has its own winding number)
          int at = 0;
          if (lane == 0) at = atomicAdd(&one[0], (int)__popcll(m));
          at = __builtin_amdgcn_readfirstlane(at);
          if (need[k]) nl[at + lanes_below(m)] = (unsigned short)v;
        }
      }
      __syncthreads();
      const int np = one[0];
      // a point beyond the margin from j's hull has winding number 0
      auto outside = [&](V3<R> Pv) __attribute__((always_inline)) {
        return outside_by_margin(bx, by, bz, nv, stj.cx, stj.cy, stj.cz, Cj, vsub(Pv, Cj), mj, stj.r);
      };
      Q4<R>* ut = reinterpret_cast<Q4<R>*>(smem + LG.ut);
      if (VPT > 1 && ww == 1) {  // block-uniform: the whole workgroup on one point at a time
        for (int pi = wave; pi < np; pi += W) {  // wave-uniform
          const int v = nl[pi];
          const bool out = outside(lds_v(sx, sy, sz, v));
          if (lane == 0) {
            if (out) wb[v] = R(0);
            else ml[atomicAdd(&one[1], 1)] = (unsigned short)v;  // in any order
          }
          n_wind += !out;
        }
        __syncthreads();
        const int nw = one[1];
        for (int q = 0; q < nw; q++) {  // block-uniform
          const int v = ml[q];
          const double w = winding_part(bx, by, bz, sf, ut, nv, nf, sh, lds_v(sx, sy, sz, v), tid, NT,
                                        []() __attribute__((always_inline)) { __syncthreads(); });
          double* sums = red + (q & 1) * W;
          if (lane == 0) sums[wave] = w;
          __syncthreads();  // the sums are there, the directions read
          if (tid == 0) {
            double tot = sums[0];
            for (int k = 1; k < W; k++) tot += sums[k];
            wb[v] = winding_of<R>(tot);
          }
        }
      } else if (wave < ww) {
        ut += (size_t)wave * nv;
        for (int pi = wave; pi < np; pi += ww) {  // wave-uniform
          const int v = nl[pi];
          const V3<R> Pv = lds_v(sx, sy, sz, v);
          R wv = R(0);
          if (!outside(Pv)) {
            wv = winding_w(bx, by, bz, sf, ut, nv, nf, sh, Pv);
            n_wind++;
          }
          if (lane == 0) wb[v] = wv;
        }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < VPT; k++)
        if (need[k]) touch(k, cj2, wb[tid + k * NT], sh);
    }
    if (passes & 2) {  // block-uniform
      const R L0j = fmax(stj.l0, R(1e-12f));
      const R l0m = fmax(L0i, L0j);
      const bool all_images = pbc && R(2) * (Ri + stj.r + R(2) * l0m) >= R(0.999f) * L;
      if (wave < 2) {  // the first wave lists the candidate's vertices in reach, the second the own ones
        const R rk = (Ri + R(2) * l0m) * R(1.0001f) + R(1e-6f);
        const R r2 = (stj.r + R(2) * l0m) * R(1.0001f) + R(1e-6f);
        int n = 0;
        for (int v0 = 0; v0 < nv; v0 += DPM_WAVE) {
          const int v = v0 + lane;
          bool in = false;
          if (v < nv) {
            if (wave == 0) {
              const V3<R> ds = {bx[v] + sh.x - Ci.x, by[v] + sh.y - Ci.y, bz[v] + sh.z - Ci.z};
              in = all_images || vdot(ds, ds) <= rk * rk;
            } else {
              const V3<R> dp = {sx[v] - stj.cx - sh.x, sy[v] - stj.cy - sh.y, sz[v] - stj.cz - sh.z};
              in = all_images || vdot(dp, dp) <= r2 * r2;
            }
          }
          const unsigned long long m = __ballot(in);
          const int at = n + lanes_below(m);
          if (in) (wave == 0 ? nl : ml)[at] = (unsigned short)v;
          if (wave == 1 && v < nv) sm[v] = in ? (unsigned short)at : (unsigned short)0xffff;
          n += __popcll(m);
        }
        if (lane == 0) one[1 + wave] = n;
      }
      __syncthreads();
      const int nnear = one[1], nmine = one[2];
      if (nnear > 0 && nmine > 0) {  // block-uniform
        // (own vertex, slice of near vertices) per task, slices added in order
        const int S = max(1, min(nnear, kGrpSlices / nmine)), per = (nnear + S - 1) / S;
        Q4<R>* acc = reinterpret_cast<Q4<R>*>(smem + LG.ut);
        for (int i = tid; i < S * nmine; i += NT) {
          const int iv = i % nmine, s = i / nmine;
          acc[i] = pair_sum(ml[iv], s * per, min(nnear, (s + 1) * per), L0j, stj.inv_l0,
                            [&](int m) __attribute__((always_inline)) { return lds_v(bx, by, bz, (int)nl[m]); });
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VPT; k++) {
          const int v = tid + k * NT;
          const int p = v < nv ? (int)sm[v] : 0xffff;
          if (p == 0xffff) continue;
          int cnt_own = 0;
          for (int s = 0; s < S; s++) {
            const Q4<R> q4 = acc[s * nmine + p];
            F[k] = vadd(F[k], V3<R>{q4.x, q4.y, q4.z});
            cnt_own += (int)q4.w;
          }
          if (PROBE && a->p_adh) a->p_adh[base + v] += cnt_own;
        }
      }
    }
  };
  // The candidates of a mask after separate() and a barrier.
  auto take_all = [&](unsigned long long m) __attribute__((always_inline)) {
    n_cand += (unsigned)__popcll(m);
    const int r = ((m >> lane) & 1ull) ? rec[lane] : 0;
    unsigned long long left = __ballot((r & 3) != 0);
    const unsigned long long touching = __ballot((r & 1) != 0);
    const unsigned long long below = (1ull << lane) - 1ull;
    // block-uniform: lists that do not fit, or contact beyond the kept slots
    // (and any contact of a cell of several vertices a thread: the registers of
    // its points cost the 642-vertex step 133 -> 166 us at 4096 cells)
    constexpr bool kTogether = VPT == 1;
    bool each = __ballot(((r & 2) && !(r & 4)) || ((r & 1) && (!kTogether || __popcll(m & below) >= kGrpSlots))) != 0ull;
    // Contact: the points of all touching candidates in one list, the waves
    // taking them in turn; a candidate's vertices come from the L2.  (Taken
    // candidate after candidate, each with its own staging and barriers, a
    // cell with contacts held a step of 256 cells for 24 us against 16.)
    int at[VPT][kGrpSlots];
#pragma unroll
    for (int k = 0; k < VPT; k++)
#pragma unroll
      for (int c = 0; c < kGrpSlots; c++) at[k][c] = -1;
    if (kTogether && touching && !each) {
      unsigned short* points = reinterpret_cast<unsigned short*>(smem + LG.plist);
      R* pw = reinterpret_cast<R*>(smem + LG.pw);
      unsigned long long w = m;
#pragma unroll
      for (int c = 0; c < kGrpSlots; c++) {
        const int b = w ? __ffsll((long long)w) - 1 : 0;
        if (w && ((touching >> b) & 1ull)) {
          const CellStat<R> stj = from_lane(st_l, b);
          const V3<R> sh = shift_to(stj);
          const V3<R> Cj = {stj.cx + sh.x, stj.cy + sh.y, stj.cz + sh.z};
          const R rj = (stj.r + contact_margin(stj.r, stj.em)) * R(1.0001f) + R(1e-6f);
#pragma unroll
          for (int k = 0; k < VPT; k++) {
            const int v = tid + k * NT;
            bool need = false;
            if (v < nv) {
              const V3<R> d = vsub(P[k], Cj);
              need = vdot(d, d) <= rj * rj;
            }
            const unsigned long long mn = __ballot(need);
            if (mn) {
              int p = 0;
              if (lane == 0) p = atomicAdd(&one[3], (int)__popcll(mn));
              p = __builtin_amdgcn_readfirstlane(p) + lanes_below(mn);
              if (need) {
                at[k][c] = p;
                if (p < kGrpPoints) points[p] = (unsigned short)(c << 10 | v);
              }
            }
          }
        }
        w &= w - 1ull;
      }
      __syncthreads();
      const int np = one[3];
      each = np > kGrpPoints;  // block-uniform
      if (!each) {
        if (wave < ww) {
          Q4<R>* ut = reinterpret_cast<Q4<R>*>(smem + LG.acc) + (size_t)wave * nv;
          for (int pi = wave; pi < np; pi += ww) {  // wave-uniform
            const int e = __builtin_amdgcn_readfirstlane((int)points[pi]), c = e >> 10;
            unsigned long long u = m;
            for (int q = 0; q < c; q++) u &= u - 1ull;
            const int b = __ffsll((long long)u) - 1;
            const CellStat<R> stj = from_lane(st_l, b);
            const V3<R> sh = shift_to(stj);
            const V3<R> Cj = {stj.cx + sh.x, stj.cy + sh.y, stj.cz + sh.z};
            const R mj = contact_margin(stj.r, stj.em);
            const size_t bj = (size_t)from_lane(cj_l, b) * nv;
            const V3<R> Pv = lds_v(sx, sy, sz, e & 1023);
            // a point beyond the margin from j's hull has winding number 0
            R wv = R(0);
            if (!outside_by_margin(a->xin + bj, a->yin + bj, a->zin + bj, nv, stj.cx, stj.cy, stj.cz, Cj,
                                   vsub(Pv, Cj), mj, stj.r)) {
              wv = winding_w(a->xin + bj, a->yin + bj, a->zin + bj, sf, ut, nv, nf, sh, Pv);
              n_wind++;
            }
            if (lane == 0) pw[pi] = wv;
          }
        }
      }
      __syncthreads();  // the winding numbers are there, the count is read
      if (tid == 0) one[3] = 0;  // for the next candidates (a barrier ahead of them)
    }
    if (each) {  // block-uniform
      for (; left; left &= left - 1ull) {
        const int b = __ffsll((long long)left) - 1;
        take_one(b, from_lane(r, b) & 3);
      }
      return;
    }
    const R* pw = reinterpret_cast<const R*>(smem + LG.pw);
    Q4<R>* acc = reinterpret_cast<Q4<R>*>(smem + LG.acc);
    auto place_of = [&](int o) __attribute__((always_inline)) {  // lists of the o-th candidate of m
      return smem + LG.slots + (size_t)o * LG.slot;
    };
    while (left) {  // as many candidates as there is room for their partial sums
      int n = 0, lanes[kGrpSlots] = {0, 0, 0, 0}, ends[kGrpSlots] = {0, 0, 0, 0}, total = 0;
#pragma unroll
      for (int c = 0; c < kGrpSlots; c++) {
        if (left) {
          const int b = __ffsll((long long)left) - 1, rb = from_lane(r, b);
          const int tasks = rb & 2 ? ((rb >> 10) & 127) * ((rb >> 17) & 127) : 0;
          if (total + tasks <= kGrpTasks) {
            lanes[c] = b;
            total += tasks;
            n = c + 1;
            left &= left - 1ull;
          }
        }
        ends[c] = total;
      }
      for (int i0 = 0; i0 < total; i0 += NT) {  // uniform: every lane takes part in the shuffles
        const int i = i0 + tid;
        const int c = (i >= ends[0]) + (i >= ends[1]) + (i >= ends[2]);
        const int first = c == 0 ? 0 : c == 1 ? ends[0] : c == 2 ? ends[1] : ends[2];
        const int b = c == 0 ? lanes[0] : c == 1 ? lanes[1] : c == 2 ? lanes[2] : lanes[3];
        const int rb = __shfl(r, b, DPM_WAVE);
        const R L0j = fmax(__shfl(st_l.l0, b, DPM_WAVE), R(1e-12f));
        const double inv_l0j = __shfl(st_l.inv_l0, b, DPM_WAVE);
        if (i < total) {
          const int nnear = (rb >> 3) & 127, nmine = (rb >> 10) & 127, per = rb >> 24;
          // (i - first) / nmine: at most 512 / 64, half away from an integer
          const int s = (int)(((float)(i - first) + 0.5f) * __builtin_amdgcn_rcpf((float)nmine));
          const int iv = i - first - s * nmine;
          const R* qx = reinterpret_cast<const R*>(place_of(__popcll(m & ((1ull << b) - 1ull))));
          const unsigned short* own = reinterpret_cast<const unsigned short*>(qx + 3 * kGrpCap);
          acc[i] = pair_sum(own[iv], s * per, min(nnear, (s + 1) * per), L0j, inv_l0j,
                            [&](int q) __attribute__((always_inline)) { return lds_v(qx, qx + kGrpCap, qx + 2 * kGrpCap, q); });
        }
      }
      __syncthreads();
#pragma unroll
      for (int c = 0; c < kGrpSlots; c++) {
        if (c >= n) break;  // block-uniform
        const int b = lanes[c], rb = from_lane(r, b), nmine = (rb >> 10) & 127, S = (rb >> 17) & 127;
        if (kTogether && (rb & 1)) {  // block-uniform; at[][] by the candidate's slot
          const int cj2 = from_lane(cj_l, b), o = __popcll(m & ((1ull << b) - 1ull));
          const V3<R> sh = shift_to(from_lane(st_l, b));
#pragma unroll
          for (int k = 0; k < VPT; k++) {
            const int p = o == 0 ? at[k][0] : o == 1 ? at[k][1] : o == 2 ? at[k][2] : at[k][3];
            if (p >= 0) touch(k, cj2, pw[p], sh);
          }
        }
        if (!(rb & 2)) continue;
        const Q4<R>* sums = acc + (c > 0 ? ends[c - 1] : 0);
        const unsigned short* place =
            reinterpret_cast<const unsigned short*>(
                reinterpret_cast<const R*>(place_of(__popcll(m & ((1ull << b) - 1ull)))) + 3 * kGrpCap) +
            kGrpCap;
#pragma unroll
        for (int k = 0; k < VPT; k++) {
          const int v = tid + k * NT;
          const int p = v < nv ? (int)place[v] : 0xffff;
          if (p == 0xffff) continue;
          int cnt_own = 0;
          for (int s = 0; s < S; s += 4) {  // four loads in flight, added in order
            Q4<R> q4[4];
#pragma unroll
            for (int j = 0; j < 4; j++) q4[j] = sums[min(s + j, S - 1) * nmine + p];
#pragma unroll
            for (int j = 0; j < 4; j++)
              if (s + j < S) {
                F[k] = vadd(F[k], V3<R>{q4[j].x, q4[j].y, q4[j].z});
                cnt_own += (int)q4[j].w;
              }
          }
          if (PROBE && a->p_adh) a->p_adh[base + v] += cnt_own;
        }
      }
      if (left) __syncthreads();
    }
  };
  if (pairs_on) {  // block-uniform
    int* clist = reinterpret_cast<int*>(smem + LG.clist);
    int* glist = reinterpret_cast<int*>(smem + LG.glist);
    int* plist = reinterpret_cast<int*>(smem + LG.plist);
    int* gath = reinterpret_cast<int*>(smem + LG.gath);
    // candidate source: every cell of the tissue in order, its list, or the
    // cells of the 27 buckets around this cell, sorted by index
    const int* src = listed ? a->nl_idx + (size_t)ci * kNearList : nullptr;
    int nsrc = listed ? nlist : ce - cb;
    if (binned && !ahead) {
      const int nb = a->tbin_nb[t], nbuck = a->tbin_nbuck[t];
      const int* bs = a->bin_start + a->tbin_hoff[t];
      const R wb = L / (R)nb;
      int* gid = gath;       // [31]: distinct buckets
      int* gst = gath + 32;  // [27] bucket starts
      int* gof = gath + 64;  // [28] prefix of bucket sizes
      if (tid < DPM_WAVE) {  // the whole first wave: distinct buckets, their cells' offsets
        int g = 0;
        if (tid < 27) {
          const int gx = bin_coord(Ci.x, L, wb, nb), gy = bin_coord(Ci.y, L, wb, nb), gz = bin_coord(Ci.z, L, wb, nb);
          const int dx = tid % 3 - 1, dy = (tid / 3) % 3 - 1, dz = tid / 9 - 1;
          g = (int)bin_bucket((gx + dx + nb) % nb, (gy + dy + nb) % nb, (gz + dz + nb) % nb, nb, nbuck);
        }
        const int nu = distinct_buckets27(g, bs, gst, gof);
        if (tid == 0) gid[31] = nu;
      }
      __syncthreads();
      const int nu = gid[31], n = gof[nu];
      if (n <= NT) {  // block-uniform; otherwise scan every cell
        if (tid < n) {
          int u = 0;
          while (gof[u + 1] <= tid) u++;
          glist[tid] = a->bin_list[cb + gst[u] + (tid - gof[u])];
        }
        __syncthreads();
        if (tid < n) {  // rank sort (indices are distinct)
          const int v = glist[tid];
          int r = 0;
          for (int u = 0; u < n; u++) r += glist[u] < v;
          clist[r] = v;
        }
        __syncthreads();
        if (tid < n) glist[tid] = clist[tid];
        __syncthreads();
        src = glist;
        nsrc = n;
      }
    }
    if (ahead) nsrc = 0;
    int nnl = 0;  // entries of the list being made
    int c0 = 0, g = 0, ncand = 0;
    unsigned long long m = cmask;
    while (ahead ? cmask != 0 : true) {  // the candidates found ahead, or chunks of 256 cells, 64 candidates at a time
      if (!ahead) {
        while (g >= ncand && c0 < nsrc) {  // the next chunk that has any
          const int k = c0 + tid;
          const int cj = k < nsrc ? (src ? src[k] : cb + k) : ce;
          bool cand = false;
          CellStat<R> stj{};
          if (cj < ce && cj != ci) {
            stj = a->st_in[cj];
            cand = in_reach(stj);
          }
          if (relist) {
            const bool nr = cj < ce && cj != ci && near_list_takes(sti, stj, pbc, L, invL, do_contact, do_adh, *a->nl_skin);
            const int n = block_compact(nr, cj, plist, cnt);
            if (tid < n && nnl + tid < kNearList) a->nl_idx[(size_t)ci * kNearList + nnl + tid] = plist[tid];
            nnl += n;
          }
          ncand = block_compact(cand, cj, clist, cnt);
          g = 0;
          c0 += NT;
        }
        if (g >= ncand) break;
        const int n = min(DPM_WAVE, ncand - g);
        if (lane < n) {
          cj_l = clist[g + lane];
          st_l = a->st_in[cj_l];
        }
        g += n;
        m = n == DPM_WAVE ? ~0ull : (1ull << n) - 1ull;
        separate(m);
        __syncthreads();
      }
      take_all(m);
      if (ahead) break;
      __syncthreads();  // the lists and records are written again next
    }
    if (relist && tid == 0) {
      a->nl_cnt[ci] = nnl <= kNearList ? nnl : -1;
      a->nl_ref[ci] = sti;
    }
  }
  if (a->nl_cnt && ci == cb && tid == 0) a->nl_stale_clear[t] = 0;
  step_args_again<R>(a);

  // ------------------------------------------------------- Euler and stats
  double px = 0.0, py = 0.0, pz = 0.0;
  V3<R> Pn[VPT];
#pragma unroll
  for (int k = 0; k < VPT; k++) {
    const int v = tid + k * NT;
    Pn[k] = P[k];
    if (v >= nv) continue;
    if (a->w_out) a->w_out[base + v] = wsum[k];
    if (a->rec_cell)
      for (int q = npart[k]; q < DPM3D_MAXPART; q++) a->rec_cell[(base + v) * DPM3D_MAXPART + q] = -1;
    if (a->flags & F_WRITE_FORCES) {
      a->fx[base + v] = F[k].x;
      a->fy[base + v] = F[k].y;
      a->fz[base + v] = F[k].z;
    }
    if (a->flags & F_MOVE) {
      if (a->xlo) {
        // x + lo + F dt, the displacement rounded once onto the residual
        R ex, ey, ez;
        Pn[k] = v3(two_sum(P[k].x, fma(F[k].x, a->dt, a->xlo[base + v]), ex),
                   two_sum(P[k].y, fma(F[k].y, a->dt, a->ylo[base + v]), ey),
                   two_sum(P[k].z, fma(F[k].z, a->dt, a->zlo[base + v]), ez));
        a->xlo[base + v] = ex;
        a->ylo[base + v] = ey;
        a->zlo[base + v] = ez;
      } else {
        Pn[k] = v3(fma(F[k].x, a->dt, P[k].x), fma(F[k].y, a->dt, P[k].y), fma(F[k].z, a->dt, P[k].z));
      }
      a->xout[base + v] = Pn[k].x;
      a->yout[base + v] = Pn[k].y;
      a->zout[base + v] = Pn[k].z;
      px += (double)Pn[k].x;
      py += (double)Pn[k].y;
      pz += (double)Pn[k].z;
    }
  }
  if (a->flags & F_MOVE) {  // block-uniform: statistics for the next step (cell_stats)
    px = wave_sum_d(px);
    py = wave_sum_d(py);
    pz = wave_sum_d(pz);
    __syncthreads();  // every read of the step's positions is done
#pragma unroll
    for (int k = 0; k < VPT; k++) {
      const int v = tid + k * NT;
      if (v < nv) {
        sx[v] = Pn[k].x;
        sy[v] = Pn[k].y;
        sz[v] = Pn[k].z;
      }
    }
    if (lane == 0) {
      red[wave] = px;
      red[W + wave] = py;
      red[2 * W + wave] = pz;
    }
    __syncthreads();
    px = py = pz = 0.0;
#pragma unroll
    for (int w = 0; w < W; w++) {
      px += red[w];
      py += red[W + w];
      pz += red[2 * W + w];
    }
    const V3<R> C = {(R)(px / nv), (R)(py / nv), (R)(pz / nv)};
    R rr2 = R(0), e2 = R(0);  // max |d|^2, then one square root (monotonic, correctly rounded)
#pragma unroll
    for (int k = 0; k < VPT; k++)
      if (tid + k * NT < nv) {
        const V3<R> d = vsub(Pn[k], C);
        rr2 = fmax(rr2, vdot(d, d));
      }
    double vol = 0.0;
#pragma unroll
    for (int f = tid; f < nf; f += NT) {
      int i0, i1, i2;
      wface(sf, f, i0, i1, i2);
      const V3<R> P0 = vsub(lds_v(sx, sy, sz, i0), C);
      const V3<R> P1 = vsub(lds_v(sx, sy, sz, i1), C);
      const V3<R> P2 = vsub(lds_v(sx, sy, sz, i2), C);
      vol += (double)vdot(vcross(P0, P1), P2);
      const V3<R> e0 = vsub(P1, P0), e1 = vsub(P2, P1), ee = vsub(P0, P2);
      e2 = fmax(e2, fmax(vdot(e0, e0), fmax(vdot(e1, e1), vdot(ee, ee))));
    }
    rr2 = wave_max_all(rr2);
    e2 = wave_max_all(e2);
    vol = wave_sum_d(vol);
    if (lane == 0) {
      red[3 * W + wave] = vol;
      red[4 * W + wave] = (double)rr2;
      red[5 * W + wave] = (double)e2;
    }
    __syncthreads();
    if (tid == 0) {
      double r2d = 0.0, e2d = 0.0;
      vol = 0.0;
#pragma unroll
      for (int w = 0; w < W; w++) {
        vol += red[3 * W + w];
        r2d = fmax(r2d, red[4 * W + w]);
        e2d = fmax(e2d, red[5 * W + w]);
      }
      // slack of a few ulp so that the culling tests are never tighter than
      // the largest distance a vertex can have from C, or the longest edge
      const R em = sqrt((R)e2d) * R(1.000001f), r = sqrt((R)r2d) * R(1.0000005f) + R(1e-30f);
      a->st_out[ci] = make_cell_stat<R>(C.x, C.y, C.z, r, em, l0i);
      a->vol_out[ci] = fabs(vol / 6.0);
      a->em_out[ci] = em;
      if (nl_on) {
        if (stale > 1) {
          if (ci == cb) a->nl_stale_out[t] = stale - 1;
        } else if (near_list_moved(nl_ref, C, r, em, pbc != 0, L, *a->nl_skin)) {
          a->nl_stale_out[t] = near_list_mark(relist);
        }
      }
    }
  }
  if (a->counters) {
    // per wave, without a workgroup barrier: the wave's contact and winding
    // counts, and the candidates (every thread holds the workgroup's count;
    // wave 0 adds it).  Spread over DPM_COUNTER_SLOTS slots so that
    // workgroups do not serialise on one address; the host sums the slots.
    const unsigned long long any = __ballot(n_contact != 0);
    unsigned c = n_contact;
    if (any)
      for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o, DPM_WAVE);
    if (lane == 0) {
      unsigned long long* slot = a->counters + 4 * ((blockIdx.x * W + wave) % DPM_COUNTER_SLOTS);
      if (blockIdx.x == 0 && wave == 0) atomicAdd(&slot[0], 1ull);
      if (n_wind) atomicAdd(&slot[1], (unsigned long long)n_wind);
      if (c) atomicAdd(&slot[2], (unsigned long long)c);
      if (wave == 0 && n_cand) atomicAdd(&slot[3], (unsigned long long)n_cand);
    }
  }
}

// VPT 1: meshes of at most 256 vertices; VPT 2 (_mid): up to 512, in float; VPT
// 4: up to 1024; _t512: 512 threads (group_threads).  The icospheres of
// subdivision 1 (42 vertices, 80 faces), 2 (162, 320) and 3 (642, 1280) have
// instances with their sizes fixed.  The production instances up to 256
// vertices have the diagnostic outputs compiled out, the _probe ones record
// them.
extern "C" __global__ void __launch_bounds__(256) k3d_step_f32(const Step3D<float>) { k3d_step_body<float, 0, 0, 1, 0, false>(); }
extern "C" __global__ void __launch_bounds__(256) k3d_step_f32_probe(const Step3D<float>) { k3d_step_body<float, 0, 0, 1, 0>(); }
extern "C" __global__ void __launch_bounds__(256, 2) k3d_step_f32_big(const Step3D<float>) { k3d_step_body<float, 0, 0, 4, 0>(); }
extern "C" __global__ void __launch_bounds__(256, 3) k3d_step_f32_mid(const Step3D<float>) { k3d_step_body<float, 0, 0, 2, 0>(); }
extern "C" __global__ void __launch_bounds__(512) k3d_step_f32_t512(const Step3D<float>) { k3d_step_body<float, 0, 0, 1, 0, true, 512>(); }
extern "C" __global__ void __launch_bounds__(512) k3d_step_f64_t512(const Step3D<double>) { k3d_step_body<double, 0, 0, 1, 0, true, 512>(); }
extern "C" __global__ void __launch_bounds__(256, 2) k3d_step_f64(const Step3D<double>) { k3d_step_body<double, 0, 0, 1, 0, false>(); }
extern "C" __global__ void __launch_bounds__(256, 2) k3d_step_f64_probe(const Step3D<double>) { k3d_step_body<double, 0, 0, 1, 0>(); }
extern "C" __global__ void __launch_bounds__(256, 2) k3d_step_f64_big(const Step3D<double>) { k3d_step_body<double, 0, 0, 4, 0>(); }
extern "C" __global__ void __launch_bounds__(256) k3d_step_f32_v42(const Step3D<float>) { k3d_step_body<float, 42, 80, 1, 4, false>(); }
extern "C" __global__ void __launch_bounds__(256, 2) k3d_step_f64_v42(const Step3D<double>) { k3d_step_body<double, 42, 80, 1, 4, false>(); }
extern "C" __global__ void __launch_bounds__(256) k3d_step_f32_v162(const Step3D<float>) { k3d_step_body<float, 162, 320, 1, 4, false>(); }
extern "C" __global__ void __launch_bounds__(256) k3d_step_f32_v162_probe(const Step3D<float>) { k3d_step_body<float, 162, 320, 1, 4>(); }
extern "C" __global__ void __launch_bounds__(256, 2) k3d_step_f64_v162(const Step3D<double>) { k3d_step_body<double, 162, 320, 1, 4>(); }
// Handles with many cells (group_many): registers bounded so that a compute
// unit keeps a cell more, at the cost of a few spills.  us per step, plain |
// bounded: 42 vertices, 1024 cells in contact 54 | 39; 162 vertices, 1024 cells
// in contact 163 | 130, apart 34 | 28, 512 cells apart 21 | 22; 642 vertices,
// 1024 cells apart 63 | 68, 4096 cells 175 | 133; in double, 64 cells 31 | 38,
// 1024 cells 112 | 97.  The general double instance gains nothing (92 vertices,
// 1024 cells in contact 1.2 times slower).
extern "C" __global__ void __launch_bounds__(256, 4) k3d_step_f32_many(const Step3D<float>) { k3d_step_body<float, 0, 0, 1, 0, false>(); }
extern "C" __global__ void __launch_bounds__(256, 4) k3d_step_f32_v42_many(const Step3D<float>) { k3d_step_body<float, 42, 80, 1, 4, false>(); }
extern "C" __global__ void __launch_bounds__(256, 4) k3d_step_f32_v162_many(const Step3D<float>) { k3d_step_body<float, 162, 320, 1, 4, false>(); }
extern "C" __global__ void __launch_bounds__(256) k3d_step_f32_v642(const Step3D<float>) { k3d_step_body<float, 642, 1280, 3, 4>(); }
extern "C" __global__ void __launch_bounds__(256, 3) k3d_step_f32_v642_many(const Step3D<float>) { k3d_step_body<float, 642, 1280, 3, 1>(); }
extern "C" __global__ void __launch_bounds__(256) k3d_step_f64_v642(const Step3D<double>) { k3d_step_body<double, 642, 1280, 3, 1>(); }
extern "C" __global__ void __launch_bounds__(256, 2) k3d_step_f64_v642_many(const Step3D<double>) { k3d_step_body<double, 642, 1280, 3, 1>(); }
