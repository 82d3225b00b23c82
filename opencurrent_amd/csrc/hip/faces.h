// The face transforms of the cell-centred ghost fills
// (ocustorage/grid3dboundary.cu): which faces are written, from which cell
// and with which arithmetic.
#pragma once

#include "ocu_hip_common.h"

namespace ocu_hip {

struct Face {
  int type;
  float value;
  float aux;
};
struct Faces {
  Face xpos, xneg, ypos, yneg, zpos, zneg;
};

inline Faces faces(const ocu_bc_set *b) {
  Faces f;
  f.xpos = {b->xpos.type, b->xpos.value, b->xpos.aux_value};
  f.xneg = {b->xneg.type, b->xneg.value, b->xneg.aux_value};
  f.ypos = {b->ypos.type, b->ypos.value, b->ypos.aux_value};
  f.yneg = {b->yneg.type, b->yneg.value, b->yneg.aux_value};
  f.zpos = {b->zpos.type, b->zpos.value, b->zpos.aux_value};
  f.zneg = {b->zneg.type, b->zneg.value, b->zneg.aux_value};
  return f;
}

__device__ __forceinline__ bool writes(const Face &f) {
  return f.type == OCU_BC_PERIODIC || f.type == OCU_BC_DIRICHELET || f.type == OCU_BC_NEUMANN;
}

// value of the ghost on face f from the interior value a it derives from.
// Level-1 Dirichlet: `-phi + 2 * bc.value` (2*value in float,
// grid3dboundary.cu:250); no-corner Dirichlet: `-phi + 2.0 * (T)value`
// (double, :44).  Neumann: phi -/+ h*value in T.
template <typename T, bool DBL_DIRICHLET>
__device__ __forceinline__ T xform(const Face &f, bool neg, T h, T a) {
  if (f.type == OCU_BC_DIRICHELET) {
    if (DBL_DIRICHLET) return (T)(-(double)a + 2.0 * (double)(T)f.value);
    return -a + (T)(2 * f.value);
  }
  if (f.type == OCU_BC_NEUMANN) return neg ? a - h * (T)f.value : a + h * (T)f.value;
  return a;  // periodic: the source index already wrapped
}

// interior source index along one axis for the ghost at c (c == -1 or n)
__device__ __forceinline__ int src_index(const Face &f, bool neg, int n) {
  if (f.type == OCU_BC_PERIODIC) return neg ? n - 1 : 0;
  return neg ? 0 : n - 1;
}

}  // namespace ocu_hip
