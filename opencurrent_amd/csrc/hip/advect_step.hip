// One step of the scalar transport, and one step of its adjoint, in one
// launch each.
//
// The forward step phi_out = fill(phi + dt * A(u, phi)) was three launches:
// the tendency, the combination (which reads and writes two more grids) and
// the no-corner ghost fill; the adjoint step was two: the transposed stencil
// over the ghost box, then the pass that folds the ghosts' adjoints into the
// cells they derive from.  Here a wave owns a row j (V cells per lane, the
// whole row) and marches along x with its planes in registers; the next
// plane's rows are on their way while one is worked on, k-neighbours come by
// DPP, and what the other launches did happens where the value is:
//   - forward: a boundary cell's thread also stores the face ghosts that
//     derive from its new value (fill rules of faces.h);
//   - adjoint: the ghost layer of lam is zero, so a ghost's adjoint is one
//     product of the cell and the face next to it, and the cell it derives
//     from adds it in bc_adjoint_nocorners' order; ghosts are not stored.
// Same operations in the same order as the separate launches, bit for bit.
// Bound by memory (forward 4 grids read and 1 written, adjoint 8 and 4): at
// 128^3 a step takes 10 us FP32 and 16 FP64 (4.2 and 5.2 TB/s; 21.9 FP32 as
// three launches), an adjoint step 21 and 36 us (4.8 and 5.6 TB/s; 41.9 FP32
// as two).
#include <algorithm>

#include "advect.h"
#include "faces.h"
#include "rows.h"

using namespace ocu_hip;

namespace {

constexpr int NWS = 4;  // rows (waves) per block

// a row's lanes: V consecutive cells each, the row's k = -1 and k = nz values
// in a register beside them (the lane past the row holds k = nz in its first
// cell, or lane 63 takes it as the DPP shift's fill)
template <typename T, int V>
struct RowLanes {
  int k0, kc, gk, nz;
  bool active, g_in_data;
  __device__ RowLanes(int lane, int n) : nz(n) {
    k0 = lane * V;
    active = k0 < n;
    kc = active ? k0 : 0;
    gk = lane == 0 ? -1 : n;
    g_in_data = lane == n / V && n < 64 * V;
  }
  __device__ __forceinline__ Vec<T, V> load(const T *row) const {
    return *reinterpret_cast<const Vec<T, V> *>(row + kc);
  }
  // with the value past the ends
  __device__ __forceinline__ Vec<T, V> load(const T *row, T &g) const {
    Vec<T, V> d = load(row);
    g = row[gk];
    if (g_in_data) d.v[0] = g;
    return d;
  }
};

// tile (row block, chunk of planes) of this block, the XCDs taking
// contiguous runs; false past the last one
__device__ __forceinline__ bool chunk_of(int tiles_j, int ntiles, int &tj, int &ti) {
  const int per = gridDim.x / 8, t = (blockIdx.x % 8) * per + blockIdx.x / 8;
  tj = t % tiles_j;
  ti = t / tiles_j;
  return t < ntiles;
}

template <typename T>
struct StepArgs {
  const T *u, *v, *w, *phi;
  T *out;
  Inv<T> ih;
  T dt;
  Faces f;
  T h[3];
  int64_t xs;
  int ys, nx, ny, nz, scheme, tiles_j, ichunk, ntiles;
};

template <typename T, int V>
__global__ __launch_bounds__(64 * NWS) void k_advect_step_rows(StepArgs<T> A) {
  typedef Vec<T, V> VT;
  int tj, ti;
  if (!chunk_of(A.tiles_j, A.ntiles, tj, ti)) return;
  const int j = tj * NWS + __builtin_amdgcn_readfirstlane(threadIdx.y);
  if (j >= A.ny) return;
  const RowLanes<T, V> L(threadIdx.x, A.nz);
  const int i0 = ti * A.ichunk, i1 = min(A.nx, i0 + A.ichunk);
  const int64_t xs = A.xs, row0 = (int64_t)i0 * xs + (int64_t)j * A.ys;
  const T *ph = A.phi + row0, *u = A.u + row0, *v = A.v + row0, *w = A.w + row0;
  T *out = A.out + row0;
  const int ys = A.ys;
  VT pm = L.load(ph - xs), pc, pn, un, uc = L.load(u);
  T gc, gn, gw, gwn;
  pc = L.load(ph, gc);
  // plane i0's own rows
  VT ym = L.load(ph - ys), yp = L.load(ph + ys), v0 = L.load(v), v1 = L.load(v + ys), w0 = L.load(w, gw);
  pn = L.load(ph + xs, gn);
  un = L.load(u + xs);
  for (int i = i0; i < i1; i++) {
    // the next plane (the last one again at the end of the march)
    const int64_t d = i + 1 < i1 ? xs : 0;
    const VT nym = L.load(ph + d - ys), nyp = L.load(ph + d + ys), nv0 = L.load(v + d), nv1 = L.load(v + d + ys);
    const VT nw0 = L.load(w + d, gwn);
    T gnn;
    const VT pnn = L.load(ph + xs + d, gnn), unn = L.load(u + xs + d);
    const T lo = from_lower(pc.v[V - 1], gc), hi = from_upper(pc.v[0], gc), whi = from_upper(w0.v[0], gw);
    VT r;
#pragma unroll
    for (int e = 0; e < V; e++) {
      const T p = pc.v[e], zm = e > 0 ? pc.v[e - 1] : lo, zp = e < V - 1 ? pc.v[e + 1] : hi;
      const T u_pi = un.v[e], u0 = uc.v[e], v_pj = v1.v[e], vv = v0.v[e], w_pk = e < V - 1 ? w0.v[e + 1] : whi,
              ww = w0.v[e];
      const T du = u_pi * interp(A.scheme, u_pi, p, pn.v[e]) - u0 * interp(A.scheme, u0, pm.v[e], p);
      const T dv = v_pj * interp(A.scheme, v_pj, p, yp.v[e]) - vv * interp(A.scheme, vv, ym.v[e], p);
      const T dw = w_pk * interp(A.scheme, w_pk, p, zp) - ww * interp(A.scheme, ww, zm, p);
      const T t = (-du * A.ih.x) - (dv * A.ih.y) - (dw * A.ih.z);
      r.v[e] = (T)1 * p + A.dt * t;
    }
    if (L.active) {
      *reinterpret_cast<VT *>(out + L.k0) = r;
      // face ghosts whose source this cell is
      auto ghosts = [&](const Face &lo_f, const Face &hi_f, bool first, bool last, T h, int64_t to_lo, int64_t to_hi) {
        auto row = [&](const Face &f, bool neg, int64_t to) {
          VT g;
#pragma unroll
          for (int e = 0; e < V; e++) g.v[e] = xform<T, true>(f, neg, h, r.v[e]);
          *reinterpret_cast<VT *>(out + to + L.k0) = g;
        };
        if (writes(lo_f) && (lo_f.type == OCU_BC_PERIODIC ? last : first)) row(lo_f, true, to_lo);
        if (writes(hi_f) && (hi_f.type == OCU_BC_PERIODIC ? first : last)) row(hi_f, false, to_hi);
      };
      if (j == 0 || j == A.ny - 1)
        ghosts(A.f.yneg, A.f.ypos, j == 0, j == A.ny - 1, A.h[1], (int64_t)(-1 - j) * ys, (int64_t)(A.ny - j) * ys);
      if (i == 0 || i == A.nx - 1)
        ghosts(A.f.xneg, A.f.xpos, i == 0, i == A.nx - 1, A.h[0], (int64_t)(-1 - i) * xs, (int64_t)(A.nx - i) * xs);
      const bool first = L.k0 == 0, last = L.k0 + V == A.nz;
      if (first || last) {
        const Face &zl = A.f.zneg, &zh = A.f.zpos;
        if (writes(zl) && (zl.type == OCU_BC_PERIODIC ? last : first))
          out[-1] = xform<T, true>(zl, true, A.h[2], zl.type == OCU_BC_PERIODIC ? r.v[V - 1] : r.v[0]);
        if (writes(zh) && (zh.type == OCU_BC_PERIODIC ? first : last))
          out[A.nz] = xform<T, true>(zh, false, A.h[2], zh.type == OCU_BC_PERIODIC ? r.v[0] : r.v[V - 1]);
      }
    }
    pm = pc; pc = pn; gc = gn;
    pn = pnn; gn = gnn;
    uc = un; un = unn;
    ym = nym; yp = nyp; v0 = nv0; v1 = nv1; w0 = nw0; gw = gwn;
    ph += d; u += d; v += d; w += d;
    out += xs;
  }
}

template <typename T>
struct AdjArgs {
  const T *u, *v, *w, *phi, *lam;
  T *out, *au, *av, *aw;
  Inv<T> ih;
  T sc;
  T c[6];      // ghost coefficient per face (x high, x low, ...)
  int per[6];  // its source is the opposite end
  int64_t xs;
  int ys, nx, ny, nz, scheme, tiles_j, ichunk, ntiles;
};

template <typename T>
__device__ __forceinline__ T w_low(int scheme, T f) {  // weight of the face's lower cell
  return scheme == OCU_IT_SECOND_ORDER_CENTERED ? (T).5 : f < 0 ? (T)0 : (T)1;
}
template <typename T>
__device__ __forceinline__ T w_high(int scheme, T f) {
  return scheme == OCU_IT_SECOND_ORDER_CENTERED ? (T).5 : f < 0 ? (T)1 : (T)0;
}

template <typename T, int V>
__global__ __launch_bounds__(64 * NWS) void k_advect_adjoint_rows(AdjArgs<T> A) {
  typedef Vec<T, V> VT;
  int tj, ti;
  if (!chunk_of(A.tiles_j, A.ntiles, tj, ti)) return;
  const int j = tj * NWS + __builtin_amdgcn_readfirstlane(threadIdx.y);
  if (j >= A.ny) return;
  const RowLanes<T, V> L(threadIdx.x, A.nz);
  const int i0 = ti * A.ichunk, i1 = min(A.nx, i0 + A.ichunk);
  const int64_t xs = A.xs;
  const int ys = A.ys, nx = A.nx, ny = A.ny, nz = A.nz;
  const int64_t row0 = (int64_t)i0 * xs + (int64_t)j * ys;
  const T *lam = A.lam + row0, *ph = A.phi + row0, *u = A.u + row0, *v = A.v + row0, *w = A.w + row0;
  T *out = A.out + row0, *au = A.au + row0, *av = A.av + row0, *aw = A.aw + row0;
  const T zero = (T)0;
  // the adjoint of the ghost below (above) a cell l across face f
  auto ghost_lo = [&](T ih, T l, T f) { return zero + (zero + (A.sc * (ih * (l - zero)) * f) * w_low(A.scheme, f)); };
  auto ghost_hi = [&](T ih, T l, T f) { return zero + (zero + (A.sc * (ih * (zero - l)) * f) * w_high(A.scheme, f)); };
  const bool ylo = j == 0, yhi = j == ny - 1;
  VT zv;
#pragma unroll
  for (int e = 0; e < V; e++) zv.v[e] = zero;

  VT lm = i0 > 0 ? L.load(lam - xs) : zv, lc = L.load(lam), pm = L.load(ph - xs), uc = L.load(u);
  for (int i = i0; i < i1; i++) {
    VT lp = i < nx - 1 ? L.load(lam + xs) : zv;
    T gp, gw;
    const VT un = L.load(u + xs), pc = L.load(ph, gp), v0 = L.load(v), v1 = L.load(v + ys), w0 = L.load(w, gw);
    const VT lym = ylo ? zv : L.load(lam - ys), lyp = yhi ? zv : L.load(lam + ys), pym = L.load(ph - ys);
    VT a_u = L.load(au), a_v = L.load(av), a_w = L.load(aw);
    // z neighbours; the ghosts of lam are zero
    const T llo = from_lower(lc.v[V - 1], zero), lhi = from_upper(lc.v[0], zero);
    const T plo = from_lower(pc.v[V - 1], gp), whi = from_upper(w0.v[0], gw);
    const bool first = L.k0 == 0, last = L.k0 + V == nz;
    VT r;
#pragma unroll
    for (int e = 0; e < V; e++) {
      const T l = lc.v[e], p = pc.v[e];
      T acc = 0;
      {
        T g = A.sc * (A.ih.x * (l - lm.v[e])), f = uc.v[e];
        acc += (g * f) * w_high(A.scheme, f);
        a_u.v[e] += g * interp(A.scheme, f, pm.v[e], p);
        g = A.sc * (A.ih.x * (lp.v[e] - l));
        f = un.v[e];
        acc += (g * f) * w_low(A.scheme, f);
      }
      {
        T g = A.sc * (A.ih.y * (l - lym.v[e])), f = v0.v[e];
        acc += (g * f) * w_high(A.scheme, f);
        a_v.v[e] += g * interp(A.scheme, f, pym.v[e], p);
        g = A.sc * (A.ih.y * (lyp.v[e] - l));
        f = v1.v[e];
        acc += (g * f) * w_low(A.scheme, f);
      }
      {
        const T lz = e > 0 ? lc.v[e - 1] : llo, lzp = e < V - 1 ? lc.v[e + 1] : (last ? zero : lhi);
        T g = A.sc * (A.ih.z * (l - lz)), f = w0.v[e];
        acc += (g * f) * w_high(A.scheme, f);
        a_w.v[e] += g * interp(A.scheme, f, e > 0 ? pc.v[e - 1] : plo, p);
        g = A.sc * (A.ih.z * (lzp - l));
        f = e < V - 1 ? w0.v[e + 1] : whi;
        acc += (g * f) * w_low(A.scheme, f);
      }
      r.v[e] = l + acc;
    }
    // the ghosts that derive from these cells: x low, x high, y, z
    if (i == (A.per[1] ? nx - 1 : 0)) {
      const VT l = A.per[1] ? L.load(lam - (int64_t)i * xs) : lc, f = L.load(u - (int64_t)i * xs);
#pragma unroll
      for (int e = 0; e < V; e++) r.v[e] += A.c[1] * ghost_lo(A.ih.x, l.v[e], f.v[e]);
    }
    if (i == (A.per[0] ? 0 : nx - 1)) {
      const VT l = A.per[0] ? L.load(lam + (int64_t)(nx - 1 - i) * xs) : lc, f = L.load(u + (int64_t)(nx - i) * xs);
#pragma unroll
      for (int e = 0; e < V; e++) r.v[e] += A.c[0] * ghost_hi(A.ih.x, l.v[e], f.v[e]);
    }
    if (j == (A.per[3] ? ny - 1 : 0)) {
      const VT l = A.per[3] ? L.load(lam - (int64_t)j * ys) : lc, f = L.load(v - (int64_t)j * ys);
#pragma unroll
      for (int e = 0; e < V; e++) r.v[e] += A.c[3] * ghost_lo(A.ih.y, l.v[e], f.v[e]);
    }
    if (j == (A.per[2] ? 0 : ny - 1)) {
      const VT l = A.per[2] ? L.load(lam + (int64_t)(ny - 1 - j) * ys) : lc, f = L.load(v + (int64_t)(ny - j) * ys);
#pragma unroll
      for (int e = 0; e < V; e++) r.v[e] += A.c[2] * ghost_hi(A.ih.y, l.v[e], f.v[e]);
    }
    if (first || last) {
      const bool lo_here = A.per[5] ? last : first, hi_here = A.per[4] ? first : last;
      if (lo_here) {
        T &t = A.per[5] ? r.v[V - 1] : r.v[0];
        t += A.c[5] * ghost_lo(A.ih.z, lam[0], w[0]);
      }
      if (hi_here) {
        T &t = A.per[4] ? r.v[0] : r.v[V - 1];
        t += A.c[4] * ghost_hi(A.ih.z, lam[nz - 1], w[nz]);
      }
    }
    if (L.active) {
      *reinterpret_cast<VT *>(out + L.k0) = r;
      *reinterpret_cast<VT *>(au + L.k0) = a_u;
      *reinterpret_cast<VT *>(av + L.k0) = a_v;
      *reinterpret_cast<VT *>(aw + L.k0) = a_w;
      // the faces past the last cells (their upper cell is a ghost, lam = 0)
      if (i == nx - 1) {
        VT t = L.load(au + xs);
        const VT pn = L.load(ph + xs);
#pragma unroll
        for (int e = 0; e < V; e++)
          t.v[e] += A.sc * (A.ih.x * (zero - lc.v[e])) * interp(A.scheme, un.v[e], pc.v[e], pn.v[e]);
        *reinterpret_cast<VT *>(au + xs + L.k0) = t;
      }
      if (yhi) {
        VT t = L.load(av + ys);
        const VT pn = L.load(ph + ys);
#pragma unroll
        for (int e = 0; e < V; e++)
          t.v[e] += A.sc * (A.ih.y * (zero - lc.v[e])) * interp(A.scheme, v1.v[e], pc.v[e], pn.v[e]);
        *reinterpret_cast<VT *>(av + ys + L.k0) = t;
      }
      if (last)
        aw[nz] += A.sc * (A.ih.z * (zero - lc.v[V - 1])) * interp(A.scheme, w[nz], pc.v[V - 1], ph[nz]);
    }
    lm = lc; lc = lp; uc = un; pm = pc;
    lam += xs; ph += xs; u += xs; v += xs; w += xs; out += xs; au += xs; av += xs; aw += xs;
  }
}

// cells per lane with which the rows of these grids can be walked, or 0: a row
// is one wave's, and its vectors are whole and aligned
int rows_width(int nz, std::initializer_list<const ocu_grid3d *> grids) {
  const int V = nz <= 64 ? 1 : nz <= 128 ? 2 : nz <= 256 ? 4 : 0;
  if (!V || nz % V) return 0;
  for (const ocu_grid3d *g : grids)
    if (!row_aligned(g, V)) return 0;
  return V;
}

// chunks of planes, for about 4096 waves.  The forward march reads a plane
// ahead and loses two planes per chunk (256^3 FP32: 70 us by 16 planes, 93 by
// one); the adjoint reads 8 grids and writes 4 with nothing ahead, so beyond
// two planes a wave's chain of planes costs more than the plane it keeps
// (256^3 FP32: 222 us by 16, 186 by two, 184 by one; 128^3 FP32 21 by any).
void set_chunks(int nx, int ny, int most, int &tiles_j, int &ichunk, int &ntiles) {
  tiles_j = (ny + NWS - 1) / NWS;
  ichunk = std::max(1, std::min({most, nx, (int)((int64_t)nx * ny / 4096)}));
  ntiles = tiles_j * ((nx + ichunk - 1) / ichunk);
}

template <typename T>
T *cell0(const ocu_grid3d *g) {
  return (T *)g->base + g->shift;
}

template <typename T>
void launch_step(int V, const ocu_grid3d *u, const ocu_grid3d *v, const ocu_grid3d *w, const ocu_grid3d *phi,
                 const ocu_grid3d *out, double dt, double hx, double hy, double hz, int scheme, const ocu_bc_set *bc,
                 hipStream_t s) {
  StepArgs<T> A;
  A.u = cell0<T>(u); A.v = cell0<T>(v); A.w = cell0<T>(w); A.phi = cell0<T>(phi);
  A.out = cell0<T>(out);
  A.ih = Inv<T>{(T)(1 / hx), (T)(1 / hy), (T)(1 / hz)};
  A.dt = (T)dt;
  A.f = faces(bc);
  A.h[0] = (T)hx; A.h[1] = (T)hy; A.h[2] = (T)hz;
  A.xs = (int64_t)phi->pny * phi->pnz;
  A.ys = phi->pnz;
  A.nx = phi->nx; A.ny = phi->ny; A.nz = phi->nz;
  A.scheme = scheme;
  set_chunks(A.nx, A.ny, 16, A.tiles_j, A.ichunk, A.ntiles);
  const int nblocks = (A.ntiles + 7) / 8 * 8;
  const dim3 blk(64, NWS);
  if (V == 1) k_advect_step_rows<T, 1><<<nblocks, blk, 0, s>>>(A);
  else if (V == 2) k_advect_step_rows<T, 2><<<nblocks, blk, 0, s>>>(A);
  else k_advect_step_rows<T, 4><<<nblocks, blk, 0, s>>>(A);
}

template <typename T>
void launch_adjoint(int V, const ocu_grid3d *u, const ocu_grid3d *v, const ocu_grid3d *w, const ocu_grid3d *phi,
                    const ocu_grid3d *lam, const ocu_grid3d *out, const ocu_grid3d *au, const ocu_grid3d *av,
                    const ocu_grid3d *aw, double scale, double hx, double hy, double hz, int scheme,
                    const ocu_bc_set *bc, hipStream_t s) {
  AdjArgs<T> A;
  A.u = cell0<T>(u); A.v = cell0<T>(v); A.w = cell0<T>(w); A.phi = cell0<T>(phi); A.lam = cell0<T>(lam);
  A.out = cell0<T>(out); A.au = cell0<T>(au); A.av = cell0<T>(av); A.aw = cell0<T>(aw);
  A.ih = Inv<T>{(T)(1 / hx), (T)(1 / hy), (T)(1 / hz)};
  A.sc = (T)scale;
  const ocu_bc *all[6] = {&bc->xpos, &bc->xneg, &bc->ypos, &bc->yneg, &bc->zpos, &bc->zneg};
  for (int f = 0; f < 6; f++) {
    const int t = all[f]->type;
    A.c[f] = t == OCU_BC_DIRICHELET ? (T)-1 : t == OCU_BC_NONE ? (T)0 : (T)1;
    A.per[f] = t == OCU_BC_PERIODIC;
  }
  A.xs = (int64_t)phi->pny * phi->pnz;
  A.ys = phi->pnz;
  A.nx = phi->nx; A.ny = phi->ny; A.nz = phi->nz;
  A.scheme = scheme;
  set_chunks(A.nx, A.ny, 2, A.tiles_j, A.ichunk, A.ntiles);
  const int nblocks = (A.ntiles + 7) / 8 * 8;
  const dim3 blk(64, NWS);
  if (V == 1) k_advect_adjoint_rows<T, 1><<<nblocks, blk, 0, s>>>(A);
  else if (V == 2) k_advect_adjoint_rows<T, 2><<<nblocks, blk, 0, s>>>(A);
  else k_advect_adjoint_rows<T, 4><<<nblocks, blk, 0, s>>>(A);
}

// the arguments that both entries share, as the separate calls check them
int check_step(const char *what, const ocu_grid3d *u, const ocu_grid3d *v, const ocu_grid3d *w,
               std::initializer_list<const ocu_grid3d *> cells, const ocu_bc_set *bc) {
  OCU_REQUIRE(bc, "%s: null bc", what);
  for (const ocu_grid3d *g : {u, v, w})
    if (int e = check_grid(g, what)) return e;
  for (const ocu_grid3d *g : cells) {
    if (int e = check_grid(g, what)) return e;
    OCU_REQUIRE(layout_match(u, g) && u->dtype == g->dtype && u->dtype != OCU_I32, "%s - layout mismatch", what);
    OCU_REQUIRE(u->nx == g->nx + 1 && u->ny == g->ny && u->nz == g->nz, "%s - u dimensions mismatch", what);
    OCU_REQUIRE(v->nx == g->nx && v->ny == g->ny + 1 && v->nz == g->nz, "%s - v dimensions mismatch", what);
    OCU_REQUIRE(w->nx == g->nx && w->ny == g->ny && w->nz == g->nz + 1, "%s - w dimensions mismatch", what);
    OCU_REQUIRE(g->gx >= 1 && g->gy >= 1 && g->gz >= 1, "%s - must have at least one ghost cell", what);
  }
  OCU_REQUIRE(layout_match(u, v) && layout_match(u, w) && u->dtype == v->dtype && u->dtype == w->dtype,
              "%s - u,v,w layout mismatch", what);
  for (const ocu_bc *b : {&bc->xpos, &bc->xneg, &bc->ypos, &bc->yneg, &bc->zpos, &bc->zneg})
    OCU_REQUIRE(b->type == OCU_BC_NONE || b->type == OCU_BC_PERIODIC || b->type == OCU_BC_DIRICHELET ||
                    b->type == OCU_BC_NEUMANN,
                "%s - invalid boundary condition type %d", what, b->type);
  return OCU_OK;
}

}  // namespace

extern "C" {

int ocu_passive_advect_step(const ocu_grid3d *u, const ocu_grid3d *v, const ocu_grid3d *w, const ocu_grid3d *phi,
                            const ocu_grid3d *phi_out, const ocu_grid3d *dphi, double dt, double hx, double hy,
                            double hz, int scheme, const ocu_bc_set *bc, void *stream) {
  const char *what = "ocu_passive_advect_step";
  if (int e = check_step(what, u, v, w, {phi, phi_out, dphi}, bc)) return e;
  OCU_REQUIRE(scheme == OCU_IT_FIRST_ORDER_UPWIND || scheme == OCU_IT_SECOND_ORDER_CENTERED,
              "%s - invalid interpolation type %d", what, scheme);
  const int nx = phi->nx, ny = phi->ny, nz = phi->nz;
  if ((int64_t)nx * ny * nz == 0) return OCU_OK;
  const int V = phi->base != phi_out->base ? rows_width(nz, {u, v, w, phi, phi_out}) : 0;
  if (!V) {  // in place, or rows the walk does not take
    if (int e = ocu_passive_advect(u, v, w, phi, dphi, nx, ny, nz, hx, hy, hz, scheme, stream)) return e;
    if (int e = ocu_grid_lincomb(phi_out, 1.0, phi, dt, dphi, stream)) return e;
    return ocu_bc_fill_nocorners(phi_out, bc, hx, hy, hz, stream);
  }
  if (phi->dtype == OCU_F64) launch_step<double>(V, u, v, w, phi, phi_out, dt, hx, hy, hz, scheme, bc, S(stream));
  else launch_step<float>(V, u, v, w, phi, phi_out, dt, hx, hy, hz, scheme, bc, S(stream));
  OCU_HIP_LAUNCHED(what);
}

int ocu_passive_advect_adjoint_step(const ocu_grid3d *u, const ocu_grid3d *v, const ocu_grid3d *w,
                                    const ocu_grid3d *phi, const ocu_grid3d *lam, const ocu_grid3d *lam_out,
                                    const ocu_grid3d *adj_u, const ocu_grid3d *adj_v, const ocu_grid3d *adj_w,
                                    double scale, double hx, double hy, double hz, int scheme, const ocu_bc_set *bc,
                                    void *stream) {
  const char *what = "ocu_passive_advect_adjoint_step";
  if (int e = check_step(what, u, v, w, {phi, lam, lam_out}, bc)) return e;
  if (int e = check_step(what, adj_u, adj_v, adj_w, {phi}, bc)) return e;
  OCU_REQUIRE(lam->base != lam_out->base, "%s - lam_out must not alias lam", what);
  OCU_REQUIRE(scheme == OCU_IT_FIRST_ORDER_UPWIND || scheme == OCU_IT_SECOND_ORDER_CENTERED,
              "%s - invalid interpolation type %d", what, scheme);
  const int nx = phi->nx, ny = phi->ny, nz = phi->nz;
  if ((int64_t)nx * ny * nz == 0) return OCU_OK;
  const int V = rows_width(nz, {u, v, w, phi, lam, lam_out, adj_u, adj_v, adj_w});
  if (!V) {
    if (int e = ocu_passive_advect_adjoint(u, v, w, phi, lam, lam_out, adj_u, adj_v, adj_w, scale, nx, ny, nz, hx, hy,
                                           hz, scheme, stream))
      return e;
    return ocu_bc_adjoint_nocorners(lam_out, bc, stream);
  }
  if (phi->dtype == OCU_F64)
    launch_adjoint<double>(V, u, v, w, phi, lam, lam_out, adj_u, adj_v, adj_w, scale, hx, hy, hz, scheme, bc, S(stream));
  else
    launch_adjoint<float>(V, u, v, w, phi, lam, lam_out, adj_u, adj_v, adj_w, scale, hx, hy, hz, scheme, bc, S(stream));
  OCU_HIP_LAUNCHED(what);
}

}  // extern "C"
