// exact_common.h -- pieces shared by the kernels that reproduce the
// reference's patch arithmetic (k_exact.hip, k_qr.hip): the patch sets, the
// sample points and the sign of get_reflector.
#ifndef SPRGPU_EXACT_COMMON_H
#define SPRGPU_EXACT_COMMON_H

#include "device.h"
#include "spr_math.h"

namespace sprg {

__device__ __forceinline__ double sgn(double x) { return (x < 0) ? -1 : 1; }

__device__ __forceinline__ int64_t node_of(const MeshView& m, int32_t t, int n)
{
  return n < 4 ? (int64_t)m.tv[4 * (int64_t)t + n]
               : m.nv + (int64_t)m.te[6 * (int64_t)t + (n - 4)];
}

// The initial tet set of patch p: getAdjacent(vertex | edge, 3).
__device__ __forceinline__ void patch_set(const FitArgs& a, int64_t p,
                                          const int32_t** set, int* ns)
{
  const MeshView& m = a.m;
  if (p < m.nv) {
    *set = m.v2t + m.v2t_off[p];
    *ns = m.v2t_off[p + 1] - m.v2t_off[p];
  } else {
    int64_t e = p - m.nv;
    *set = m.e2t + m.e2t_off[e];
    *ns = m.e2t_off[e + 1] - m.e2t_off[e];
  }
}

// MODE: FIT_REGULAR walks items[bucket] (patch ids), FIT_EXPANDED walks
// xitems[bucket] (expanded-set ids), FIT_MIXED walks items[bucket] holding
// either (bit 31 set: an expanded-set id) -- the fast forms' refits.
enum { FIT_REGULAR = 0, FIT_EXPANDED = 1, FIT_MIXED = 2 };

template <int MODE>
__device__ __forceinline__ const int32_t* fit_list(const FitArgs& a, int bucket, int* nitems)
{
  constexpr bool EXP = MODE == FIT_EXPANDED;
  *nitems = a.L.count[(EXP ? NBUCKET : 0) + bucket];
  return EXP ? a.L.xitems[bucket] : a.L.items[bucket];
}

// A list entry's patch and tet set.
template <int MODE>
__device__ __forceinline__ void fit_item(const FitArgs& a, int32_t entry, int64_t* p, const int32_t** set, int* ns)
{
  if (MODE == FIT_EXPANDED || (MODE == FIT_MIXED && entry < 0)) {
    const int32_t it = entry & 0x7fffffff;
    *p = a.L.x_patch[it];
    *set = a.L.x_set + a.L.x_off[it];
    *ns = a.L.x_len[it];
  } else {
    *p = entry;
    patch_set(a, *p, set, ns);
  }
}

}  // namespace sprg

#endif
