// dcl_reinit.hpp -- device helpers shared by the two reinitialisations
// (reinit.hip: the fast marching in the reference's order; reinit_sweep.hip:
// the parallel sweeps): window indexing.
#pragma once

#include "dcl_common.hpp"

namespace dcl {

__device__ __forceinline__ int64_t ri_index(const KWin& w, int d3, int x, int y, int z) {
  return ((int64_t)(d3 ? z - w.pz : 0) * w.ny + (y - w.py)) * w.nx + (x - w.px);
}

__device__ __forceinline__ bool ri_inside(const KWin& w, int d3, int x, int y, int z) {
  return x >= w.px && x < w.px + w.nx && y >= w.py && y < w.py + w.ny && (!d3 || (z >= w.pz && z < w.pz + w.nz));
}

}  // namespace dcl
