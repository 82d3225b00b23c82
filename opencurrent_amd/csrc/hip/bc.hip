// Ghost-cell fills (ocustorage/grid3dboundary.cu).
//
// apply_3d_boundary_conditions_level1 runs three dependent passes in the
// reference (x, then y over i in [-1,nx], then z over i in [-1,nx] x
// j in [-1,ny]), so edges and corners are produced by the later passes from
// ghosts written by the earlier ones.  Here one launch covers the whole
// first ghost layer: each ghost cell evaluates the same chain of per-axis
// transforms from the interior (or untouched) cell it ultimately derives
// from, with the same operations in the same order, so the values are
// identical and no cell reads a value written by the same launch.
#include <type_traits>

#include "faces.h"

using namespace ocu_hip;

namespace {

template <typename T>
struct L1 {
  DGrid<T> g;
  Faces f;
  T hx, hy, hz;

  // value after the x pass at (i,j,k), j,k interior
  __device__ T vx(int i, int j, int k) const {
    if (i >= 0 && i < g.nx) return g.at(i, j, k);
    bool neg = i < 0;
    const Face &F = neg ? f.xneg : f.xpos;
    if (!writes(F)) return g.at(i, j, k);
    return xform<T, false>(F, neg, hx, g.at(src_index(F, neg, g.nx), j, k));
  }
  // value after the x and y passes at (i,j,k), k interior
  __device__ T vxy(int i, int j, int k) const {
    if (j >= 0 && j < g.ny) return vx(i, j, k);
    bool neg = j < 0;
    const Face &F = neg ? f.yneg : f.ypos;
    if (!writes(F)) return g.at(i, j, k);
    return xform<T, false>(F, neg, hy, vx(i, src_index(F, neg, g.ny), k));
  }
};

// linear thread index -> ghost cell of the first layer:
//   [0, nZ)        z faces, (i,j) in [-1,nx]x[-1,ny], k in {-1, nz}
//   [nZ, nZ+nY)    y faces, i in [-1,nx], k in [0,nz), j in {-1, ny}
//   [.., +nX)      x faces, j in [0,ny), k in [0,nz), i in {-1, nx}
template <typename T>
__global__ void k_bc_level1(L1<T> s, int64_t nZ, int64_t nY, int64_t nX) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int nx = s.g.nx, ny = s.g.ny, nz = s.g.nz;
  if (t < nZ) {
    int64_t per = (int64_t)(nx + 2) * (ny + 2);
    bool neg = t < per;
    int64_t q = neg ? t : t - per;
    int i = (int)(q / (ny + 2)) - 1, j = (int)(q % (ny + 2)) - 1;
    const Face &F = neg ? s.f.zneg : s.f.zpos;
    if (!writes(F)) return;
    int k = neg ? -1 : nz;
    s.g.at(i, j, k) = xform<T, false>(F, neg, s.hz, s.vxy(i, j, src_index(F, neg, nz)));
    return;
  }
  t -= nZ;
  if (t < nY) {
    int64_t per = (int64_t)(nx + 2) * nz;
    bool neg = t < per;
    int64_t q = neg ? t : t - per;
    int i = (int)(q / nz) - 1, k = (int)(q % nz);
    const Face &F = neg ? s.f.yneg : s.f.ypos;
    if (!writes(F)) return;
    int j = neg ? -1 : ny;
    s.g.at(i, j, k) = xform<T, false>(F, neg, s.hy, s.vx(i, src_index(F, neg, ny), k));
    return;
  }
  t -= nY;
  if (t < nX) {
    int64_t per = (int64_t)ny * nz;
    bool neg = t < per;
    int64_t q = neg ? t : t - per;
    int j = (int)(q / nz), k = (int)(q % nz);
    const Face &F = neg ? s.f.xneg : s.f.xpos;
    if (!writes(F)) return;
    int i = neg ? -1 : nx;
    s.g.at(i, j, k) = xform<T, false>(F, neg, s.hx, s.g.at(src_index(F, neg, nx), j, k));
  }
}

// device no-corner fill (grid3dboundary.cu:28-119): faces only, no chains
template <typename T>
__global__ void k_bc_nocorners(DGrid<T> g, Faces f, T hx, T hy, T hz, int64_t nZ, int64_t nY, int64_t nX) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  if (t < nZ) {
    int i = (int)(t / ny), j = (int)(t % ny);
    if (writes(f.zneg)) g.at(i, j, -1) = xform<T, true>(f.zneg, true, hz, g.at(i, j, src_index(f.zneg, true, nz)));
    if (writes(f.zpos)) g.at(i, j, nz) = xform<T, true>(f.zpos, false, hz, g.at(i, j, src_index(f.zpos, false, nz)));
    return;
  }
  t -= nZ;
  if (t < nY) {
    int i = (int)(t / nz), k = (int)(t % nz);
    if (writes(f.yneg)) g.at(i, -1, k) = xform<T, true>(f.yneg, true, hy, g.at(i, src_index(f.yneg, true, ny), k));
    if (writes(f.ypos)) g.at(i, ny, k) = xform<T, true>(f.ypos, false, hy, g.at(i, src_index(f.ypos, false, ny), k));
    return;
  }
  t -= nY;
  if (t < nX) {
    int j = (int)(t / nz), k = (int)(t % nz);
    if (writes(f.xneg)) g.at(-1, j, k) = xform<T, true>(f.xneg, true, hx, g.at(src_index(f.xneg, true, nx), j, k));
    if (writes(f.xpos)) g.at(nx, j, k) = xform<T, true>(f.xpos, false, hx, g.at(src_index(f.xpos, false, nx), j, k));
  }
}

// r = a1*g1 + a2*g2 over the interior with the no-corner fill of r: the thread
// of a boundary cell also stores the ghosts that derive from its value (a
// ghost's source is the cell next to it, or across the domain if periodic).
// A small grid's time is its launches: 101x67x45 in FP32 with the tendency
// before it took 10.2 us as three, 7.9 as two.
template <typename T>
__global__ __launch_bounds__(256) void k_lincomb_nocorners(DGrid<T> r, T a1, DGrid<T> g1, T a2, DGrid<T> g2, Faces f,
                                                           T hx, T hy, T hz) {
  const int k = blockIdx.x * TK + threadIdx.x, j = blockIdx.y * TJ + threadIdx.y, i = blockIdx.z;
  const int nx = r.nx, ny = r.ny, nz = r.nz;
  if (j >= ny || k >= nz) return;
  const int64_t id = r.idx(i, j, k);
  const T x = g1.p[id] * a1 + g2.p[id] * a2;
  r.p[id] = x;
  if (i > 0 && i < nx - 1 && j > 0 && j < ny - 1 && k > 0 && k < nz - 1) return;
  auto ghosts = [&](const Face &lo, const Face &hi, int c, int n, T h, int64_t at_lo, int64_t at_hi) {
    if (writes(lo) && c == src_index(lo, true, n)) r.p[at_lo] = xform<T, true>(lo, true, h, x);
    if (writes(hi) && c == src_index(hi, false, n)) r.p[at_hi] = xform<T, true>(hi, false, h, x);
  };
  ghosts(f.zneg, f.zpos, k, nz, hz, r.idx(i, j, -1), r.idx(i, j, nz));
  ghosts(f.yneg, f.ypos, j, ny, hy, r.idx(i, -1, k), r.idx(i, ny, k));
  ghosts(f.xneg, f.xpos, i, nx, hx, r.idx(-1, j, k), r.idx(nx, j, k));
}

// ---- MAC fill: the reference's three dependent passes (x, y, z) ----

// tangential factor (1.0f - 2.0f * aux) is a float
template <typename T>
__global__ void k_mac_x(DGrid<T> u, DGrid<T> v, DGrid<T> w, Faces f, int nx, int ny, int nz) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  int j = blockIdx.y;
  if (k >= nz || j >= ny) return;
  if (f.xneg.type == OCU_BC_PERIODIC) {
    u.at(-1, j, k) = u.at(nx - 1, j, k);
    v.at(-1, j, k) = v.at(nx - 1, j, k);
    w.at(-1, j, k) = w.at(nx - 1, j, k);
  } else if (f.xneg.type == OCU_BC_FORCED_INFLOW_VARIABLE_SLIP) {
    u.at(-1, j, k) = (T)f.xneg.value;
    u.at(0, j, k) = (T)f.xneg.value;
    float fac = 1.0f - 2.0f * f.xneg.aux;
    v.at(-1, j, k) = v.at(0, j, k) * (T)fac;
    w.at(-1, j, k) = w.at(0, j, k) * (T)fac;
  }
  if (f.xpos.type == OCU_BC_PERIODIC) {
    u.at(nx, j, k) = u.at(0, j, k);
    u.at(nx + 1, j, k) = u.at(1, j, k);
    v.at(nx, j, k) = v.at(0, j, k);
    w.at(nx, j, k) = w.at(0, j, k);
  } else if (f.xpos.type == OCU_BC_FORCED_INFLOW_VARIABLE_SLIP) {
    u.at(nx, j, k) = (T)f.xpos.value;
    u.at(nx + 1, j, k) = (T)f.xpos.value;
    float fac = 1.0f - 2.0f * f.xpos.aux;
    v.at(nx, j, k) = v.at(nx - 1, j, k) * (T)fac;
    w.at(nx, j, k) = w.at(nx - 1, j, k) * (T)fac;
  }
}

template <typename T>
__global__ void k_mac_y(DGrid<T> u, DGrid<T> v, DGrid<T> w, Faces f, int nx, int ny, int nz) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  int i = (int)blockIdx.y - 1;
  if (k >= nz || i > nx) return;
  if (f.yneg.type == OCU_BC_PERIODIC) {
    v.at(i, -1, k) = v.at(i, ny - 1, k);
    u.at(i, -1, k) = u.at(i, ny - 1, k);
    w.at(i, -1, k) = w.at(i, ny - 1, k);
  } else if (f.yneg.type == OCU_BC_FORCED_INFLOW_VARIABLE_SLIP) {
    v.at(i, -1, k) = (T)f.yneg.value;
    v.at(i, 0, k) = (T)f.yneg.value;
    float fac = 1.0f - 2.0f * f.yneg.aux;
    u.at(i, -1, k) = u.at(i, 0, k) * (T)fac;
    w.at(i, -1, k) = w.at(i, 0, k) * (T)fac;
  }
  if (f.ypos.type == OCU_BC_PERIODIC) {
    v.at(i, ny, k) = v.at(i, 0, k);
    v.at(i, ny + 1, k) = v.at(i, 1, k);
    u.at(i, ny, k) = u.at(i, 0, k);
    w.at(i, ny, k) = w.at(i, 0, k);
  } else if (f.ypos.type == OCU_BC_FORCED_INFLOW_VARIABLE_SLIP) {
    v.at(i, ny, k) = (T)f.ypos.value;
    v.at(i, ny + 1, k) = (T)f.ypos.value;
    float fac = 1.0f - 2.0f * f.ypos.aux;
    u.at(i, ny, k) = u.at(i, ny - 1, k) * (T)fac;
    w.at(i, ny, k) = w.at(i, ny - 1, k) * (T)fac;
  }
}

template <typename T>
__global__ void k_mac_z(DGrid<T> u, DGrid<T> v, DGrid<T> w, Faces f, int nx, int ny, int nz) {
  int j = (int)(blockIdx.x * blockDim.x + threadIdx.x) - 1;
  int i = (int)blockIdx.y - 1;
  if (j > ny || i > nx) return;
  if (f.zneg.type == OCU_BC_PERIODIC) {
    w.at(i, j, -1) = w.at(i, j, nz - 1);
    u.at(i, j, -1) = u.at(i, j, nz - 1);
    v.at(i, j, -1) = v.at(i, j, nz - 1);
  } else if (f.zneg.type == OCU_BC_FORCED_INFLOW_VARIABLE_SLIP) {
    w.at(i, j, -1) = (T)f.zneg.value;
    w.at(i, j, 0) = (T)f.zneg.value;
    float fac = 1.0f - 2.0f * f.zneg.aux;
    u.at(i, j, -1) = u.at(i, j, 0) * (T)fac;
    v.at(i, j, -1) = v.at(i, j, 0) * (T)fac;
  }
  if (f.zpos.type == OCU_BC_PERIODIC) {
    w.at(i, j, nz) = w.at(i, j, 0);
    w.at(i, j, nz + 1) = w.at(i, j, 1);
    u.at(i, j, nz) = u.at(i, j, 0);
    v.at(i, j, nz) = v.at(i, j, 0);
  } else if (f.zpos.type == OCU_BC_FORCED_INFLOW_VARIABLE_SLIP) {
    w.at(i, j, nz) = (T)f.zpos.value;
    w.at(i, j, nz + 1) = (T)f.zpos.value;
    float fac = 1.0f - 2.0f * f.zpos.aux;
    u.at(i, j, nz) = u.at(i, j, nz - 1) * (T)fac;
    v.at(i, j, nz) = v.at(i, j, nz - 1) * (T)fac;
  }
}

// The three passes in one launch, where both faces of each axis are periodic
// or both inflow and an axis has two cells or more: a thread computes what its
// places hold after the last pass.  Going back through the passes (z, y, x)
// a place's value is another place's, a multiple of it or a face's value, and
// where that ends no pass writes, so nothing is read that this launch writes;
// places that two passes write get the same value twice.  128^3 FP64 11.1 us as
// three launches, 6.3 as one; 96x64x48 FP32 10.2, 6.5; 512x512x256 FP64 119, 99
// (the z faces' single elements).
template <typename T>
struct MacFill {
  DGrid<T> a[3];         // u, v, w
  int n[3], per[3];      // cells and periodicity of x, y, z
  T lo[3], hi[3];        // inflow faces: normal value
  T flo[3], fhi[3];      // and tangential factor (1 - 2*aux, a float)
};

// array A's value at (i, j, k) after the three passes
template <int A, typename T>
__device__ __forceinline__ T mac_final(const MacFill<T> &m, int i, int j, int k) {
  int c[3] = {i, j, k};
  T f[3] = {(T)1, (T)1, (T)1}, face = 0;
  bool scaled[3] = {false, false, false}, fixed = false;
#pragma unroll
  for (int x = 2; x >= 0; x--) {
    // the places that this pass covers (along the other two axes)
    const bool covers = x == 2   ? i >= -1 && i <= m.n[0] && j >= -1 && j <= m.n[1]
                        : x == 1 ? i >= -1 && i <= m.n[0] && c[2] >= 0 && c[2] < m.n[2]
                                 : c[1] >= 0 && c[1] < m.n[1] && c[2] >= 0 && c[2] < m.n[2];
    if (!covers || fixed) continue;
    const int n = m.n[x];
    if (m.per[x]) {
      c[x] = c[x] < 0 ? c[x] + n : c[x] >= n ? c[x] - n : c[x];
    } else if (x == A) {
      if (c[x] <= 0 || c[x] >= n) {
        fixed = true;
        face = c[x] <= 0 ? m.lo[x] : m.hi[x];
      }
    } else if (c[x] < 0 || c[x] >= n) {
      scaled[x] = true;
      f[x] = c[x] < 0 ? m.flo[x] : m.fhi[x];
      c[x] = c[x] < 0 ? 0 : n - 1;
    }
  }
  T v = fixed ? face : m.a[A].at(c[0], c[1], c[2]);
#pragma unroll
  for (int x = 0; x < 3; x++) v = scaled[x] ? v * f[x] : v;
  return v;
}
// the places of one line of pass X: the normal array A at -1, 0 (inflow), n
// and n+1, the others at -1 and n; every load before the first store
template <int X, typename T>
__device__ __forceinline__ void mac_line(const MacFill<T> &m, int p, int q) {
  constexpr int B = X == 0 ? 1 : 0, C = X == 2 ? 1 : 2;  // the tangential arrays
  const int n = m.n[X];
  auto value = [&](auto arr, int c) {
    constexpr int A = decltype(arr)::value;
    return X == 0 ? mac_final<A, T>(m, c, p, q) : X == 1 ? mac_final<A, T>(m, p, c, q) : mac_final<A, T>(m, p, q, c);
  };
  auto put = [&](int A, int c, T v) {
    const DGrid<T> &g = A == 0 ? m.a[0] : A == 1 ? m.a[1] : m.a[2];
    (X == 0 ? g.at(c, p, q) : X == 1 ? g.at(p, c, q) : g.at(p, q, c)) = v;
  };
  const std::integral_constant<int, X> nx;
  const std::integral_constant<int, B> bx;
  const std::integral_constant<int, C> cx;
  const T n0 = value(nx, -1), n1 = value(nx, n), n2 = value(nx, n + 1);
  const T b0 = value(bx, -1), b1 = value(bx, n), c0 = value(cx, -1), c1 = value(cx, n);
  // (a periodic axis writes no cell 0: its value there is not asked for)
  const T f0 = m.per[X] ? n0 : value(nx, 0);
  put(X, -1, n0);
  if (!m.per[X]) put(X, 0, f0);
  put(X, n, n1);
  put(X, n + 1, n2);
  put(B, -1, b0);
  put(B, n, b1);
  put(C, -1, c0);
  put(C, n, c1);
}

template <typename T>
__global__ __launch_bounds__(256) void k_mac_fill(MacFill<T> m, unsigned nX, unsigned nY, unsigned nZ) {
  unsigned q = blockIdx.x * 256u + threadIdx.x;
  const unsigned ny2 = m.n[1] + 2, nz = m.n[2];
  if (q < nX) mac_line<0, T>(m, (int)(q / nz), (int)(q % nz));                        // j, k inside
  else if ((q -= nX) < nY) mac_line<1, T>(m, (int)(q / nz) - 1, (int)(q % nz));       // i = -1 .. nx, k inside
  else if ((q -= nY) < nZ) mac_line<2, T>(m, (int)(q / ny2) - 1, (int)(q % ny2) - 1);  // i = -1 .. nx, j = -1 .. ny
}

template <typename T>
void launch_mac_fill(const ocu_grid3d *u, const ocu_grid3d *v, const ocu_grid3d *w, const ocu_bc_set *bc, int nx,
                     int ny, int nz, hipStream_t s) {
  MacFill<T> m;
  m.a[0] = dgrid<T>(u); m.a[1] = dgrid<T>(v); m.a[2] = dgrid<T>(w);
  m.n[0] = nx; m.n[1] = ny; m.n[2] = nz;
  const ocu_bc *lo[3] = {&bc->xneg, &bc->yneg, &bc->zneg}, *hi[3] = {&bc->xpos, &bc->ypos, &bc->zpos};
  for (int x = 0; x < 3; x++) {
    m.per[x] = lo[x]->type == OCU_BC_PERIODIC;
    m.lo[x] = (T)lo[x]->value;
    m.hi[x] = (T)hi[x]->value;
    m.flo[x] = (T)(1.0f - 2.0f * lo[x]->aux_value);
    m.fhi[x] = (T)(1.0f - 2.0f * hi[x]->aux_value);
  }
  const unsigned nX = (unsigned)ny * nz, nY = (unsigned)(nx + 2) * nz, nZ = (unsigned)(nx + 2) * (ny + 2);
  k_mac_fill<T><<<(nX + nY + nZ + 255) / 256, 256, 0, s>>>(m, nX, nY, nZ);
}

int check_types(const ocu_bc_set *bc, const int *ok, int nok, const char *what) {
  const ocu_bc *all[6] = {&bc->xpos, &bc->xneg, &bc->ypos, &bc->yneg, &bc->zpos, &bc->zneg};
  for (auto b : all) {
    bool good = false;
    for (int q = 0; q < nok; q++) good |= b->type == ok[q];
    if (!good) {
      set_error("%s - invalid boundary condition types %d, %d, %d, %d, %d, %d", what, bc->xpos.type,
                bc->xneg.type, bc->ypos.type, bc->yneg.type, bc->zpos.type, bc->zneg.type);
      return OCU_ERR_INVALID;
    }
  }
  return OCU_OK;
}

const int kCellTypes[] = {OCU_BC_NONE, OCU_BC_PERIODIC, OCU_BC_DIRICHELET, OCU_BC_NEUMANN};
const int kMacTypes[] = {OCU_BC_NONE, OCU_BC_PERIODIC, OCU_BC_FORCED_INFLOW_VARIABLE_SLIP};

}  // namespace

extern "C" {

int ocu_bc_fill_level1(const ocu_grid3d *g, const ocu_bc_set *bc, double hx, double hy, double hz,
                       void *stream) {
  if (int e = check_grid(g, "apply_3d_boundary_conditions_level1")) return e;
  OCU_REQUIRE(bc, "apply_3d_boundary_conditions_level1: null bc");
  if (int e = check_types(bc, kCellTypes, 4, "apply_3d_boundary_conditions_level1")) return e;
  OCU_REQUIRE(g->gx >= 1 && g->gy >= 1 && g->gz >= 1,
              "apply_3d_boundary_conditions_level1 - must have at least 1 ghost point");
  OCU_REQUIRE(g->dtype != OCU_I32, "apply_3d_boundary_conditions_level1: int grid");
  if (g->nx <= 0 || g->ny <= 0 || g->nz <= 0) return OCU_OK;
  int64_t nZ = 2 * (int64_t)(g->nx + 2) * (g->ny + 2);
  int64_t nY = 2 * (int64_t)(g->nx + 2) * g->nz;
  int64_t nX = 2 * (int64_t)g->ny * g->nz;
  int64_t n = nZ + nY + nX;
  int nb = (int)((n + 255) / 256);
  if (g->dtype == OCU_F64) {
    L1<double> s{dgrid<double>(g), faces(bc), hx, hy, hz};
    k_bc_level1<double><<<nb, 256, 0, S(stream)>>>(s, nZ, nY, nX);
  } else {
    L1<float> s{dgrid<float>(g), faces(bc), (float)hx, (float)hy, (float)hz};
    k_bc_level1<float><<<nb, 256, 0, S(stream)>>>(s, nZ, nY, nX);
  }
  OCU_HIP_LAUNCHED("ocu_bc_fill_level1");
}

int ocu_bc_fill_nocorners(const ocu_grid3d *g, const ocu_bc_set *bc, double hx, double hy, double hz,
                          void *stream) {
  if (int e = check_grid(g, "apply_3d_boundary_conditions_level1_nocorners")) return e;
  OCU_REQUIRE(bc, "apply_3d_boundary_conditions_level1_nocorners: null bc");
  if (int e = check_types(bc, kCellTypes, 4, "apply_3d_boundary_conditions_level1_nocorners")) return e;
  OCU_REQUIRE(g->gx >= 1 && g->gy >= 1 && g->gz >= 1,
              "apply_3d_boundary_conditions_level1_nocorners - must have at least 1 ghost point");
  OCU_REQUIRE(g->dtype != OCU_I32, "apply_3d_boundary_conditions_level1_nocorners: int grid");
  if (g->nx <= 0 || g->ny <= 0 || g->nz <= 0) return OCU_OK;
  int64_t nZ = (int64_t)g->nx * g->ny, nY = (int64_t)g->nx * g->nz, nX = (int64_t)g->ny * g->nz;
  int nb = (int)((nZ + nY + nX + 255) / 256);
  if (g->dtype == OCU_F64)
    k_bc_nocorners<double><<<nb, 256, 0, S(stream)>>>(dgrid<double>(g), faces(bc), hx, hy, hz, nZ, nY, nX);
  else
    k_bc_nocorners<float><<<nb, 256, 0, S(stream)>>>(dgrid<float>(g), faces(bc), (float)hx, (float)hy,
                                                    (float)hz, nZ, nY, nX);
  OCU_HIP_LAUNCHED("ocu_bc_fill_nocorners");
}

int ocu_grid_lincomb_fill(const ocu_grid3d *r, double a1, const ocu_grid3d *g1, double a2, const ocu_grid3d *g2,
                          const ocu_bc_set *bc, double hx, double hy, double hz, void *stream) {
  const char *what = "ocu_grid_lincomb_fill";
  if (int e = check_grid(r, what)) return e;
  if (int e = check_grid(g1, what)) return e;
  if (int e = check_grid(g2, what)) return e;
  OCU_REQUIRE(bc, "%s: null bc", what);
  if (int e = check_types(bc, kCellTypes, 4, what)) return e;
  OCU_REQUIRE(layout_match(r, g1) && layout_match(r, g2), "%s: layout mismatch", what);
  OCU_REQUIRE(r->dtype == g1->dtype && r->dtype == g2->dtype && r->dtype != OCU_I32, "%s: dtype mismatch", what);
  OCU_REQUIRE(r->gx >= 1 && r->gy >= 1 && r->gz >= 1, "%s - must have at least 1 ghost point", what);
  const int64_t interior = (int64_t)r->nx * r->ny * r->nz;
  // where ocu_grid_lincomb works on the whole allocation, its padding and
  // edges take the combination too: two calls
  if (interior == 0 || !((r->allocated - interior) / (float)r->allocated > .03f)) {
    if (int e = ocu_grid_lincomb(r, a1, g1, a2, g2, stream)) return e;
    return ocu_bc_fill_nocorners(r, bc, hx, hy, hz, stream);
  }
  const dim3 grid = stencil_grid(r->nx, r->ny, r->nz);
  if (r->dtype == OCU_F64)
    k_lincomb_nocorners<double><<<grid, stencil_block(), 0, S(stream)>>>(dgrid<double>(r), a1, dgrid<double>(g1), a2,
                                                                         dgrid<double>(g2), faces(bc), hx, hy, hz);
  else
    k_lincomb_nocorners<float><<<grid, stencil_block(), 0, S(stream)>>>(dgrid<float>(r), (float)a1, dgrid<float>(g1),
                                                                        (float)a2, dgrid<float>(g2), faces(bc),
                                                                        (float)hx, (float)hy, (float)hz);
  OCU_HIP_LAUNCHED(what);
}

int ocu_bc_fill_mac_level1(const ocu_grid3d *u, const ocu_grid3d *v, const ocu_grid3d *w,
                           const ocu_bc_set *bc, void *stream) {
  const char *what = "apply_3d_mac_boundary_conditions_level1";
  if (int e = check_grid(u, what)) return e;
  if (int e = check_grid(v, what)) return e;
  if (int e = check_grid(w, what)) return e;
  OCU_REQUIRE(bc, "%s: null bc", what);
  if (int e = check_types(bc, kMacTypes, 3, what)) return e;
  OCU_REQUIRE(layout_match(u, v) && layout_match(u, w), "%s - layout mismatch", what);
  OCU_REQUIRE(u->dtype == v->dtype && u->dtype == w->dtype && u->dtype != OCU_I32, "%s - dtype mismatch", what);
  OCU_REQUIRE(u->gx >= 1 && u->gy >= 1 && u->gz >= 1, "%s - must have at least 1 ghost point", what);
  int nx = u->nx - 1, ny = u->ny, nz = u->nz;
  OCU_REQUIRE(v->nx == nx && v->ny == ny + 1 && v->nz == nz, "%s - v_grid dimension mismatch", what);
  OCU_REQUIRE(w->nx == nx && w->ny == ny && w->nz == nz + 1, "%s - w_grid dimension mismatch", what);
  if (nx <= 0 || ny <= 0 || nz <= 0) return OCU_OK;
  const ocu_bc *lo[3] = {&bc->xneg, &bc->yneg, &bc->zneg}, *hi[3] = {&bc->xpos, &bc->ypos, &bc->zpos};
  bool paired = nx >= 2 && ny >= 2 && nz >= 2 &&
                (int64_t)ny * nz + (int64_t)(nx + 2) * nz + (int64_t)(nx + 2) * (ny + 2) < INT32_MAX;
  for (int x = 0; x < 3; x++) paired &= lo[x]->type == hi[x]->type && lo[x]->type != OCU_BC_NONE;
  if (paired) {
    if (u->dtype == OCU_F64) launch_mac_fill<double>(u, v, w, bc, nx, ny, nz, S(stream));
    else launch_mac_fill<float>(u, v, w, bc, nx, ny, nz, S(stream));
    OCU_HIP_LAUNCHED("ocu_bc_fill_mac_level1");
  }
  Faces f = faces(bc);
  dim3 gx((nz + 63) / 64, ny), gy((nz + 63) / 64, nx + 2), gz((ny + 2 + 63) / 64, nx + 2);
  if (u->dtype == OCU_F64) {
    auto U = dgrid<double>(u), V = dgrid<double>(v), W = dgrid<double>(w);
    k_mac_x<double><<<gx, 64, 0, S(stream)>>>(U, V, W, f, nx, ny, nz);
    k_mac_y<double><<<gy, 64, 0, S(stream)>>>(U, V, W, f, nx, ny, nz);
    k_mac_z<double><<<gz, 64, 0, S(stream)>>>(U, V, W, f, nx, ny, nz);
  } else {
    auto U = dgrid<float>(u), V = dgrid<float>(v), W = dgrid<float>(w);
    k_mac_x<float><<<gx, 64, 0, S(stream)>>>(U, V, W, f, nx, ny, nz);
    k_mac_y<float><<<gy, 64, 0, S(stream)>>>(U, V, W, f, nx, ny, nz);
    k_mac_z<float><<<gz, 64, 0, S(stream)>>>(U, V, W, f, nx, ny, nz);
  }
  OCU_HIP_LAUNCHED("ocu_bc_fill_mac_level1");
}

}  // extern "C"
