// The explicit part of one Eqn_IncompressibleNS3D step in two launches: T's
// interior, then everything else.
//
// The reference's step (eqn_incompressns3d.cu:331-393) runs self-advection,
// three momentum Laplacians, the thermal force, passive advection of T and
// its Laplacian, each writing or updating a tendency grid, then the
// forward-Euler / Adams-Bashforth combinations (linear_combination,
// grid3ddev.cu:283-349) and the no-corner ghost fill of T, then (AB2) copies
// the tendencies to the "last" grids: about 38 grid passes of memory traffic
// per cell.  Here every tendency of a cell is computed in registers (the same
// device functions, in the same order, as the per-operator kernels), combined
// with the old value and written with the new u, v, w and T into a second set
// of buffers (the caller swaps them in afterwards): k_ns_march does T's
// interior, k_ns_shell the other elements of the padded allocation; 4 grids
// read, 4 written (plus, for AB2, the last tendencies read and this step's
// written).  Every element of the new buffers receives exactly what the
// in-place sequence leaves in the old one:
//   - cells the combination covers get old*1 + d*a_dt (+ last*a_ab);
//   - with the reference's whole-allocation combination (allocation waste
//     <= 3%) the other elements get old*1 + 0*a_dt (+ 0*a_ab), the tendency
//     grids being zero outside the cells their operators write;
//   - with the interior-only combination they keep the old value;
//   - T's face ghosts take the no-corner fill of the new interior value
//     they derive from (the interior is written first).
#include "advect.h"
#include "faces.h"

using namespace ocu_hip;

namespace {

template <typename T>
struct NSStep {
  const T *u, *v, *w, *t;       // old values (element 0 of the allocation)
  T *un, *vn, *wn, *tn;         // new values
  T *du, *dv, *dw, *dtt;        // AB2: this step's tendencies (written)
  const T *lu, *lv, *lw, *lt;   // AB2: the last step's tendencies (read)
  Inv<T> ih, ih2;
  T nu, kappa, tcoef, a_dt, a_ab, th[3];
  Faces tf;
  int64_t xs, ys, shift;
  int pre, nx, ny, nz, gx, gy, gz, pnx, pny, pnz;
  int scheme, fper, tper, vaxis, flat, keep, use_last, visc, tdiff;
};

template <typename T>
__device__ __forceinline__ T combine(const NSStep<T> &s, T old, T d, T last) {
  T r = old * (T)1 + d * s.a_dt;
  if (s.use_last) r = r * (T)1 + last * s.a_ab;
  return r;
}

// an element no operator writes: the whole-allocation combination adds
// zero tendencies, the interior one leaves it alone
template <typename T>
__device__ __forceinline__ T untouched(const NSStep<T> &s, int grid, T old) {
  return ((s.flat >> grid) & 1) ? combine(s, old, (T)0, (T)0) : old;
}

// One element (ip, jp, kp) of the padded box (indices from the box corner,
// ghosts included) outside T's interior: the new value of each grid there.
template <typename T>
__device__ __forceinline__ void ns_element(const NSStep<T> &s, int ip, int jp, int kp) {
  const int i = ip - s.gx, j = jp - s.gy, k = kp - s.gz;
  const int64_t e = (int64_t)s.pre + ((int64_t)ip * s.pny + jp) * s.pnz + kp;  // element of the allocation
  const bool ci = i >= 0 && i < s.nx, cj = j >= 0 && j < s.ny, ck = k >= 0 && k < s.nz;
  // the faces past the last cells: advection and the thermal force cover the
  // cell box only
  auto face = [&](const T *old, T *out, T *d, const T *last, int grid, bool in) {
    if (!in) {
      out[e] = untouched(s, grid, old[e]);
      return;
    }
    T t = 0;
    if (s.visc) t = t + s.nu * laplacian_cell(old, e, s.xs, s.ys, s.ih2);
    out[e] = combine(s, old[e], t, s.use_last ? last[e] : (T)0);
    if (s.keep) d[e] = t;
  };
  face(s.u, s.un, s.du, s.lu, 0, i == s.nx && cj && ck);
  face(s.v, s.vn, s.dv, s.lv, 1, ci && j == s.ny && ck);
  face(s.w, s.wn, s.dw, s.lw, 2, ci && cj && k == s.nz);
  // a face ghost of T that the no-corner fill writes takes the fill of its
  // source cell's new value, which k_ns_march has stored
  Face f{OCU_BC_NONE, 0.f, 0.f};
  bool neg = false;
  T h = 0;
  int64_t from = 0;
  auto ghost = [&](const Face &lo, const Face &hi, int c, int n, T hh, int64_t st) {
    neg = c < 0;
    f = neg ? lo : hi;
    h = hh;
    from = (int64_t)(src_index(f, neg, n) - c) * st;
  };
  if ((i == -1 || i == s.nx) && cj && ck) ghost(s.tf.xneg, s.tf.xpos, i, s.nx, s.th[0], s.xs);
  else if (ci && (j == -1 || j == s.ny) && ck) ghost(s.tf.yneg, s.tf.ypos, j, s.ny, s.th[1], s.ys);
  else if (ci && cj && (k == -1 || k == s.nz)) ghost(s.tf.zneg, s.tf.zpos, k, s.nz, s.th[2], 1);
  s.tn[e] = writes(f) ? xform<T, true>(f, neg, h, s.tn[e + from]) : untouched(s, 3, s.t[e]);
}

// the pre-padding before the padded box: untouched elements
template <typename T>
__device__ __forceinline__ void ns_prepad(const NSStep<T> &s, int64_t e) {
  s.un[e] = untouched(s, 0, s.u[e]);
  s.vn[e] = untouched(s, 1, s.v[e]);
  s.wn[e] = untouched(s, 2, s.w[e]);
  s.tn[e] = untouched(s, 3, s.t[e]);
}

// k_ns_march takes T's interior.  Every other element - the u, v and w faces
// at i = nx, j = ny and k = nz, the ghost layers, the padding - goes here, one
// thread each, after the pre-padding: the planes outside the interior's x
// range (count na), then the rows outside its y range (nb), then the row ends
// (nc).  I: the type of the element count (a thread's divisions take longer
// than its copies in 64 bits).  Bound by the row ends: pnz - nz elements of
// each row of eight grids.
template <typename T, typename I>
__global__ __launch_bounds__(256) void k_ns_shell(NSStep<T> s, I na, I nb, I nc) {
  I q = (I)blockIdx.x * 256 + threadIdx.x;
  if (q < (I)s.pre) {
    ns_prepad(s, q);
    return;
  }
  q -= s.pre;
  int ip, jp, kp;
  if (q < na) {
    const I plane = (I)s.pny * s.pnz, pl = q / plane, r = q % plane;
    ip = (int)pl < s.gx ? (int)pl : (int)pl + s.nx;
    jp = (int)(r / s.pnz);
    kp = (int)(r % s.pnz);
  } else if ((q -= na) < nb) {
    const I per = (I)(s.pny - s.ny) * s.pnz, pl = q / per, r = q % per;
    const int rr = (int)(r / s.pnz);
    ip = (int)pl + s.gx;
    jp = rr < s.gy ? rr : rr + s.ny;
    kp = (int)(r % s.pnz);
  } else if ((q -= nb) < nc) {
    const int per = s.pnz - s.nz, t = (int)(q % per);
    const I rowi = q / per;
    ip = (int)(rowi / s.ny) + s.gx;
    jp = (int)(rowi % s.ny) + s.gy;
    kp = t < s.gz ? t : t + s.nz;
  } else {
    return;
  }
  ns_element(s, ip, jp, kp);
}

// ------------------------------------------------------------------------
// T's interior, marching along x
// ------------------------------------------------------------------------
//
// A block owns a tile of MJ rows x 64 cells (j, k) of T's interior and a chunk
// of planes.  A thread keeps its own column's u, v,
// w, T of planes p-2..p+2 in registers and loads those of p+3; off the column
// the cell functions read u at p and p+1, v and w at p-1 and p, and T at p
// (second-order upwind reaches two cells along each axis but stays on it, the
// self-advection velocities one diagonal), so the LDS holds only those planes
// with a halo of R cells in j and k, and one more of each field being
// written: 3 + 3 + 3 + 2.  That leaves room for 16 waves a CU in FP64 where
// planes p-2..p+2 of all four fields left it for 8, and half the LDS reads.
// The step, this kernel and the shell: 512x512x256 FP64 first-order upwind
// 1648 -> 1090 us, 128^3 FP64 second-order upwind 95 -> 73 us, 128^3 FP32 37 ->
// 28 and 55 -> 44 us; the traffic at the copy rate is 830, 26 and 13.
// One barrier per plane orders the accesses: what plane p writes no thread
// reads before plane p + 1.  A place two beyond the box is only ever the far
// sample of second-order upwind, which wraps on a periodic axis: it is loaded
// from where it wraps to, so the cells there are like all others.
constexpr int MTK = 64;
constexpr int MXSH = 20;  // the offsets' x stride is 2^20: no plane comes near it
constexpr int64_t MXS = (int64_t)1 << MXSH;

template <int R, int MJ>
struct Win {
  static constexpr int WK = MTK + 2 * R, WJ = MJ + 2 * R, PL = WJ * WK, HALO = PL - MTK * MJ;
  // slots: u 0..2, v 3..5, w 6..8, T 9..10
  static constexpr int SLOTS = 11;
  static_assert(HALO <= MTK * MJ, "one halo cell per thread at most");
};

// A coordinate of a field's array along an axis of n cells with samples up to
// -1 and top (far2): beyond them it wraps, or (no cell reads it) is the edge.
__device__ __forceinline__ int wrapped(int q, int n, int top, bool per) {
  if (q >= -1 && q <= top) return q;
  return per ? ((q % n) + n) % n : q < 0 ? -1 : top;
}

// One field around a cell: planes p-2..p+2 of its column in registers, the
// cell's place in the LDS planes p-1 (v, w), p and p+1 (u).  Every offset is
// a constant, so one of them remains.
template <typename T>
struct Col {
  T m2, m1, c, p1, p2;
  const T *lm, *l0, *lp;
  __device__ __forceinline__ T operator()(int64_t o) const {
    if (o == 0) return c;
    if (o == MXS) return p1;
    if (o == -MXS) return m1;
    if (o == 2 * MXS) return p2;
    if (o == -2 * MXS) return m2;
    const int di = (int)((o + (MXS >> 1)) >> MXSH), r = (int)(o - ((int64_t)di << MXSH));
    return (di < 0 ? lm : di > 0 ? lp : l0)[r];
  }
};

template <typename T>
struct Tend {
  T du, dv, dw, dt;
};

// the tendencies of interior cell (i, j, k): the sequence of ns_element for a
// cell of T's interior (returned by value, so that they stay in registers)
template <int SCHEME, typename T>
__device__ __forceinline__ Tend<T> ns_tendencies(const NSStep<T> &s, const Col<T> &U, const Col<T> &V, const Col<T> &W,
                                                 const Col<T> &Tt, int64_t ys, int i, int j, int k) {
  constexpr int64_t xs = MXS;
  T du, dv, dw, dt;
  if (SCHEME == OCU_IT_SECOND_ORDER_UPWIND)
    self_advect_up2_at<false, T>(U, V, W, xs, ys, s.ih, i, j, k, s.nx, s.ny, s.nz, s.fper, du, dv, dw);
  else
    self_advect_at<T>(U, V, W, xs, ys, s.ih, SCHEME, du, dv, dw);
  if (s.visc) {
    du = du + s.nu * laplacian_at<T>(U, xs, ys, s.ih2);
    dv = dv + s.nu * laplacian_at<T>(V, xs, ys, s.ih2);
    dw = dw + s.nu * laplacian_at<T>(W, xs, ys, s.ih2);
  }
  if (s.vaxis == 0) du = du + thermal_at<T>(Tt, xs, s.tcoef);
  else if (s.vaxis == 1) dv = dv + thermal_at<T>(Tt, ys, s.tcoef);
  else dw = dw + thermal_at<T>(Tt, (int64_t)1, s.tcoef);
  dt = SCHEME == OCU_IT_SECOND_ORDER_UPWIND
           ? passive_advect_up2_at<false, T>(U, V, W, Tt, xs, ys, s.ih, i, j, k, s.nx, s.ny, s.nz, s.tper)
           : passive_advect_at<T>(U, V, W, Tt, xs, ys, s.ih, SCHEME);
  if (s.tdiff) dt = dt + s.kappa * laplacian_at<T>(Tt, xs, ys, s.ih2);
  return Tend<T>{du, dv, dw, dt};
}

template <typename T, int SCHEME, int R, int MJ>
__global__ __launch_bounds__(MTK *MJ) void k_ns_march(NSStep<T> s, int tiles_k, int tiles_j, int ichunk,
                                                      int ntiles) {
  typedef Win<R, MJ> W;
  extern __shared__ unsigned char ns_smem[];
  T *win = reinterpret_cast<T *>(ns_smem);  // [SLOTS][PL]
  // blocks are dealt round-robin to the 8 XCDs: a contiguous run of tiles
  // per XCD
  const int per = gridDim.x / 8;
  const int logical = (blockIdx.x % 8) * per + (blockIdx.x / 8);
  if (logical >= ntiles) return;  // uniform per block
  const int tk = logical % tiles_k, rem = logical / tiles_k, tj = rem % tiles_j, ti = rem / tiles_j;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * MTK + tx;
  const int k0 = tk * MTK, j0 = tj * MJ, i0 = ti * ichunk, i1 = min(s.nx, i0 + ichunk);
  const int k = k0 + tx, j = j0 + ty;
  const bool mine = k < s.nz && j < s.ny;
  const T *src[4] = {s.u + s.pre, s.v + s.pre, s.w + s.pre, s.t + s.pre};  // corner of the padded box
  const int64_t plane = (int64_t)s.pny * s.pnz;

  // this thread's own place and its halo place in the window, and their
  // elements in a plane of each field's padded box
  const int cell = (ty + R) * W::WK + tx + R;
  auto element = [&](int f, int wj, int wk) {
    const int per_ = f == 3 ? s.tper : s.fper;
    const int jj = wrapped(j0 - R + wj, s.ny, s.ny + (R == 2 && f == 1), R == 2 && (per_ & 2));
    const int kk = wrapped(k0 - R + wk, s.nz, s.nz + (R == 2 && f == 2), R == 2 && (per_ & 4));
    return (unsigned)(jj + s.gy) * (unsigned)s.pnz + (unsigned)(kk + s.gz);
  };
  const bool has_halo = tid < W::HALO;
  int hwj, hwk;  // rows above and below the tile, then the row ends
  {
    constexpr int FULL = 2 * R * W::WK;
    if (tid < FULL) {
      hwj = tid / W::WK, hwk = tid % W::WK;
      if (hwj >= R) hwj += MJ;
    } else {
      const int q = tid - FULL, e = q % (2 * R);
      hwj = R + min(q / (2 * R), MJ - 1), hwk = e < R ? e : e + MTK;
    }
  }
  const int hcell = hwj * W::WK + hwk;
  unsigned own_e[4], halo_e[4];
#pragma unroll
  for (int f = 0; f < 4; f++) own_e[f] = element(f, ty + R, tx + R), halo_e[f] = element(f, hwj, hwk);
  auto at = [&](int f, int q) {
    const int ii = wrapped(q, s.nx, s.nx + (R == 2 && f == 0), R == 2 && ((f == 3 ? s.tper : s.fper) & 1));
    return src[f] + (int64_t)(ii + s.gx) * plane;
  };
  auto slot = [&](int f, int q) { return win + (f * 3 + (f == 3 ? q & 1 : (unsigned)(q + 3) % 3)) * W::PL; };

  T m2[4], m1[4], c0[4], p1[4], p2[4], nx_[4], h[4];
#pragma unroll
  for (int f = 0; f < 4; f++) {
    m2[f] = at(f, i0 - 2)[own_e[f]], m1[f] = at(f, i0 - 1)[own_e[f]], c0[f] = at(f, i0)[own_e[f]];
    p1[f] = at(f, i0 + 1)[own_e[f]], p2[f] = at(f, i0 + 2)[own_e[f]];
  }
  T ha[4] = {}, hb[3] = {};  // halo: u, v, w, T at i0; u at i0 + 1, v and w at i0 - 1
#pragma unroll
  for (int f = 0; f < 4; f++) h[f] = (T)0;
  if (has_halo) {
#pragma unroll
    for (int f = 0; f < 4; f++) {
      ha[f] = at(f, i0)[halo_e[f]];
      if (f < 3) hb[f] = at(f, f == 0 ? i0 + 1 : i0 - 1)[halo_e[f]];
      h[f] = at(f, f == 0 ? i0 + 2 : i0 + 1)[halo_e[f]];
    }
  }
#pragma unroll
  for (int f = 0; f < 4; f++) {
    slot(f, i0)[cell] = c0[f];
    if (f < 3) slot(f, f == 0 ? i0 + 1 : i0 - 1)[cell] = f == 0 ? p1[f] : m1[f];
  }
  if (has_halo) {
#pragma unroll
    for (int f = 0; f < 4; f++) {
      slot(f, i0)[hcell] = ha[f];
      if (f < 3) slot(f, f == 0 ? i0 + 1 : i0 - 1)[hcell] = hb[f];
    }
  }
  __syncthreads();

  for (int p = i0; p < i1; p++) {
    // the planes that p + 1 reads: u at p+2; v, w, T at p+1
#pragma unroll
    for (int f = 0; f < 4; f++) {
      T *dst = slot(f, f == 0 ? p + 2 : p + 1);
      dst[cell] = f == 0 ? p2[f] : p1[f];
      if (has_halo) dst[hcell] = h[f];
    }
    // in flight while plane p is computed
#pragma unroll
    for (int f = 0; f < 4; f++) {
      nx_[f] = at(f, p + 3)[own_e[f]];
      if (has_halo) h[f] = at(f, f == 0 ? p + 3 : p + 2)[halo_e[f]];
    }
    if (mine) {
      const int64_t e = (int64_t)p * s.xs + (int64_t)j * s.ys + k + s.shift;
      auto col = [&](int f) {
        return Col<T>{m2[f], m1[f], c0[f], p1[f], p2[f], slot(f, p - 1) + cell, slot(f, p) + cell, slot(f, p + 1) + cell};
      };
      const Tend<T> d = ns_tendencies<SCHEME, T>(s, col(0), col(1), col(2), col(3), (int64_t)W::WK, p, j, k);
      s.un[e] = combine(s, c0[0], d.du, s.use_last ? s.lu[e] : (T)0);
      s.vn[e] = combine(s, c0[1], d.dv, s.use_last ? s.lv[e] : (T)0);
      s.wn[e] = combine(s, c0[2], d.dw, s.use_last ? s.lw[e] : (T)0);
      s.tn[e] = combine(s, c0[3], d.dt, s.use_last ? s.lt[e] : (T)0);
      if (s.keep) {
        s.du[e] = d.du;
        s.dv[e] = d.dv;
        s.dw[e] = d.dw;
        s.dtt[e] = d.dt;
      }
    }
#pragma unroll
    for (int f = 0; f < 4; f++) m2[f] = m1[f], m1[f] = c0[f], c0[f] = p1[f], p1[f] = p2[f], p2[f] = nx_[f];
    __syncthreads();
  }
}

int check_congruent(const ocu_grid3d *a, const ocu_grid3d *b, const char *what) {
  if (int e = check_grid(b, what)) return e;
  OCU_REQUIRE(layout_match(a, b) && a->dtype == b->dtype && a->gx == b->gx && a->gy == b->gy && a->gz == b->gz &&
                  a->shift == b->shift && a->allocated == b->allocated,
              "%s - grids are not congruent", what);
  return OCU_OK;
}

// the reference's choice in linear_combination (grid3ddev.cu:316): more
// than 3% of the allocation outside the interior -> interior only
bool whole_allocation(const ocu_grid3d *g) {
  const int64_t interior = (int64_t)g->nx * g->ny * g->nz;
  return !((g->allocated - interior) / (float)g->allocated > .03f);
}

template <typename T, int SCHEME, int R, int MJ>
int launch_march(const NSStep<T> &s, hipStream_t stream) {
  const auto kernel = &k_ns_march<T, SCHEME, R, MJ>;
  const int tiles_k = (s.nz + MTK - 1) / MTK, tiles_j = (s.ny + MJ - 1) / MJ;
  const size_t lds = (size_t)Win<R, MJ>::SLOTS * Win<R, MJ>::PL * sizeof(T);
  OCU_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)lds));
  int dev = 0, cus = 256, per = 1;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
    cus = 256;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, MTK * MJ, lds) != hipSuccess || per < 1) per = 1;
  // planes per block: the fewest rounds of resident blocks, each block
  // loading four planes beyond its own
  const int64_t slots = (int64_t)cus * per;
  int ichunk = s.nx;
  int64_t best = INT64_MAX;
  for (int ic = 1;; ic = ic < 8 ? ic + 1 : ic * 2) {
    const int c = min(ic, s.nx);  // the last candidate is the whole extent
    const int64_t nb_ = (int64_t)tiles_k * tiles_j * ((s.nx + c - 1) / c);
    const int64_t cost = ((nb_ + slots - 1) / slots) * (c + 4);
    if (cost < best) best = cost, ichunk = c;
    if (c == s.nx) break;
  }
  const int ntiles = tiles_k * tiles_j * ((s.nx + ichunk - 1) / ichunk);
  const int nblocks = ((ntiles + 7) / 8) * 8;
  kernel<<<nblocks, dim3(MTK, MJ), lds, stream>>>(s, tiles_k, tiles_j, ichunk, ntiles);
  return OCU_OK;
}

template <typename T>
int launch_ns_step(const ocu_grid3d *const *in, const ocu_grid3d *const *out, const ocu_grid3d *const *d,
                   const ocu_grid3d *const *last, const ocu_ns_step_params *p, const ocu_bc_set *tbc,
                   hipStream_t stream) {
  NSStep<T> s;
  const ocu_grid3d *g = in[0];
  s.u = (const T *)in[0]->base, s.v = (const T *)in[1]->base, s.w = (const T *)in[2]->base,
  s.t = (const T *)in[3]->base;
  s.un = (T *)out[0]->base, s.vn = (T *)out[1]->base, s.wn = (T *)out[2]->base, s.tn = (T *)out[3]->base;
  s.keep = p->keep_tendencies != 0, s.use_last = p->use_last != 0;
  s.du = s.keep ? (T *)d[0]->base : nullptr, s.dv = s.keep ? (T *)d[1]->base : nullptr,
  s.dw = s.keep ? (T *)d[2]->base : nullptr, s.dtt = s.keep ? (T *)d[3]->base : nullptr;
  s.lu = s.use_last ? (const T *)last[0]->base : nullptr, s.lv = s.use_last ? (const T *)last[1]->base : nullptr,
  s.lw = s.use_last ? (const T *)last[2]->base : nullptr, s.lt = s.use_last ? (const T *)last[3]->base : nullptr;
  s.ih = Inv<T>{(T)(1 / p->hx), (T)(1 / p->hy), (T)(1 / p->hz)};
  s.ih2 = Inv<T>{(T)(1 / (p->hx * p->hx)), (T)(1 / (p->hy * p->hy)), (T)(1 / (p->hz * p->hz))};
  s.nu = (T)p->viscosity, s.kappa = (T)p->thermal_diffusion, s.tcoef = (T)p->thermal_coef;
  s.a_dt = (T)p->a_dt, s.a_ab = (T)p->a_ab;
  s.th[0] = (T)p->hx, s.th[1] = (T)p->hy, s.th[2] = (T)p->hz;
  s.tf = faces(tbc);
  s.xs = (int64_t)g->pny * g->pnz, s.ys = g->pnz, s.shift = g->shift;
  const int vd = p->vertical_direction;
  s.vaxis = (vd & OCU_DIR_XAXIS_FLAG) ? 0 : (vd & OCU_DIR_YAXIS_FLAG) ? 1 : 2;
  s.pre = (int)(g->shift - ((int64_t)g->gx * g->pny * g->pnz + (int64_t)g->gy * g->pnz + g->gz));
  s.nx = p->nx, s.ny = p->ny, s.nz = p->nz, s.gx = g->gx, s.gy = g->gy, s.gz = g->gz;
  s.pnx = g->pnx, s.pny = g->pny, s.pnz = g->pnz;
  s.scheme = p->advection_scheme, s.fper = p->flow_periodic, s.tper = p->temp_periodic;
  s.flat = 0;
  for (int q = 0; q < 4; q++) s.flat |= whole_allocation(in[q]) << q;
  s.visc = p->viscosity > 0, s.tdiff = p->thermal_diffusion > 0;
  // the interior.  Rows per block: second-order upwind in FP64 needs 174
  // registers, so 8 waves a CU (12 spill: 512x512x256 1.90 ms against 1.95, but
  // 64^3 21.7 us against 19.2); the other schemes' 16 (14: 1.21 ms, 16: 1.09);
  // FP32 has registers for several blocks of 8 a CU (256^3 195 us by 16 rows,
  // 188 by 8)
  constexpr int MJ = sizeof(T) == 8 ? 16 : 8;
  int e;
  if (s.scheme == OCU_IT_SECOND_ORDER_UPWIND) e = launch_march<T, OCU_IT_SECOND_ORDER_UPWIND, 2, 8>(s, stream);
  else if (s.scheme == OCU_IT_SECOND_ORDER_CENTERED)
    e = launch_march<T, OCU_IT_SECOND_ORDER_CENTERED, 1, MJ>(s, stream);
  else e = launch_march<T, OCU_IT_FIRST_ORDER_UPWIND, 1, MJ>(s, stream);
  if (e != OCU_OK) return e;
  OCU_HIP_TRY(hipGetLastError());
  // the shell: everything outside T's interior
  const int64_t na = (int64_t)(s.pnx - s.nx) * s.pny * s.pnz, nb = (int64_t)s.nx * (s.pny - s.ny) * s.pnz,
                nc = (int64_t)s.nx * s.ny * (s.pnz - s.nz);
  const int64_t nshell = s.pre + na + nb + nc;
  const unsigned blocks = (unsigned)((nshell + 255) / 256);
  if (nshell < INT32_MAX - 256)
    k_ns_shell<T, unsigned><<<blocks, 256, 0, stream>>>(s, (unsigned)na, (unsigned)nb, (unsigned)nc);
  else
    k_ns_shell<T, int64_t><<<blocks, 256, 0, stream>>>(s, na, nb, nc);
  return OCU_OK;
}

}  // namespace

extern "C" {

int ocu_ns_step_fused(const ocu_grid3d *u, const ocu_grid3d *v, const ocu_grid3d *w, const ocu_grid3d *temp,
                      const ocu_grid3d *u_new, const ocu_grid3d *v_new, const ocu_grid3d *w_new,
                      const ocu_grid3d *temp_new, const ocu_grid3d *du, const ocu_grid3d *dv, const ocu_grid3d *dw,
                      const ocu_grid3d *dtemp, const ocu_grid3d *last_du, const ocu_grid3d *last_dv,
                      const ocu_grid3d *last_dw, const ocu_grid3d *last_dtemp, const ocu_ns_step_params *p,
                      const ocu_bc_set *temp_bc, void *stream) {
  const char *what = "ocu_ns_step_fused";
  OCU_REQUIRE(p && temp_bc, "%s: null parameters", what);
  const int nx = p->nx, ny = p->ny, nz = p->nz;
  OCU_REQUIRE(u && v && w && temp, "%s: null grid", what);
  if (int e = check_grid(u, what)) return e;
  OCU_REQUIRE(u->nx == nx + 1 && u->ny == ny && u->nz == nz, "%s - u dimensions mismatch", what);
  OCU_REQUIRE(v && v->nx == nx && v->ny == ny + 1 && v->nz == nz, "%s - v dimensions mismatch", what);
  OCU_REQUIRE(w && w->nx == nx && w->ny == ny && w->nz == nz + 1, "%s - w dimensions mismatch", what);
  OCU_REQUIRE(temp && temp->nx == nx && temp->ny == ny && temp->nz == nz, "%s - temperature dimensions mismatch", what);
  OCU_REQUIRE(u->dtype == OCU_F32 || u->dtype == OCU_F64, "%s - dtype", what);
  OCU_REQUIRE(u->gx >= 1 && u->gy >= 1 && u->gz >= 1, "%s - must have at least one ghost cell", what);
  const ocu_grid3d *in[4] = {u, v, w, temp}, *out[4] = {u_new, v_new, w_new, temp_new};
  const ocu_grid3d *d[4] = {du, dv, dw, dtemp}, *last[4] = {last_du, last_dv, last_dw, last_dtemp};
  // all grids share one layout (the congruent MAC layout of init_grids)
  for (int q = 0; q < 4; q++) {
    OCU_REQUIRE(in[q] && out[q], "%s: null grid", what);
    if (int e = check_congruent(u, in[q], what)) return e;
    if (int e = check_congruent(u, out[q], what)) return e;
    OCU_REQUIRE(out[q]->base != in[q]->base, "%s - the new buffers must not alias the old ones", what);
    if (p->keep_tendencies) {
      OCU_REQUIRE(d[q], "%s - keep_tendencies needs the tendency grids", what);
      if (int e = check_congruent(u, d[q], what)) return e;
    }
    if (p->use_last) {
      OCU_REQUIRE(last[q], "%s - use_last needs the last-tendency grids", what);
      if (int e = check_congruent(u, last[q], what)) return e;
    }
    if (p->keep_tendencies && p->use_last)
      OCU_REQUIRE(d[q]->base != last[q]->base, "%s - tendency and last tendency must differ", what);
  }
  OCU_REQUIRE(p->advection_scheme == OCU_IT_FIRST_ORDER_UPWIND || p->advection_scheme == OCU_IT_SECOND_ORDER_CENTERED ||
                  p->advection_scheme == OCU_IT_SECOND_ORDER_UPWIND,
              "%s - invalid interpolation type %d", what, p->advection_scheme);
  OCU_REQUIRE(p->flow_periodic >= 0 && p->flow_periodic <= 7 && p->temp_periodic >= 0 && p->temp_periodic <= 7,
              "%s - invalid periodic axes mask", what);
  const int vd = p->vertical_direction;
  OCU_REQUIRE(vd == OCU_DIR_XPOS || vd == OCU_DIR_XNEG || vd == OCU_DIR_YPOS || vd == OCU_DIR_YNEG ||
                  vd == OCU_DIR_ZPOS || vd == OCU_DIR_ZNEG,
              "%s - bad vertical_direction %d", what, vd);
  const ocu_bc *all[6] = {&temp_bc->xpos, &temp_bc->xneg, &temp_bc->ypos, &temp_bc->yneg, &temp_bc->zpos,
                          &temp_bc->zneg};
  for (auto b : all)
    OCU_REQUIRE(b->type == OCU_BC_NONE || b->type == OCU_BC_PERIODIC || b->type == OCU_BC_DIRICHELET ||
                    b->type == OCU_BC_NEUMANN,
                "%s - invalid temperature boundary condition type %d", what, b->type);
  if ((int64_t)nx * ny * nz == 0) return OCU_OK;
  const int e = u->dtype == OCU_F64 ? launch_ns_step<double>(in, out, d, last, p, temp_bc, S(stream))
                                    : launch_ns_step<float>(in, out, d, last, p, temp_bc, S(stream));
  if (e != OCU_OK) return e;
  OCU_HIP_LAUNCHED(what);
}

}  // extern "C"
