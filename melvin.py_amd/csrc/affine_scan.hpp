// Scans of first-order recurrences v_j = a_j v_{j-1} + b_j (complex v and b,
// real a, FP64) over the lanes of a wavefront, for the tridiagonal solves.
// Each lane holds the affine map of its chunk; the scan composes them.
//
// The exchange between lanes is DPP (row shifts inside 16 lanes, then the
// four rows' totals through readlane), which is ordinary VALU work: a
// shuffle of a double goes through the LDS pipe twice and each of a scan's
// six dependent steps would wait for it.
#pragma once
#include <hip/hip_runtime.h>

namespace mlv {

// v -> a v + (x + i y)
struct Affine {
  double a, x, y;
};
// the map `in` followed by the map `out`
__device__ __forceinline__ Affine aff_after(const Affine& out, const Affine& in) {
  return {out.a * in.a, fma(out.a, in.x, out.x), fma(out.a, in.y, out.y)};
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v, double ident) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(ident), __double2loint(v), CTRL, 0xf,
                                             0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(ident), __double2hiint(v), CTRL, 0xf,
                                             0xf, false);
  return __hiloint2double(hi, lo);
}
// Lanes without a source inside their row of 16 get the identity map.
template <int CTRL>
__device__ __forceinline__ Affine dpp_aff(const Affine& m) {
  return {dpp_f64<CTRL>(m.a, 1.0), dpp_f64<CTRL>(m.x, 0.0), dpp_f64<CTRL>(m.y, 0.0)};
}
__device__ __forceinline__ double lane_f64(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Exclusive scan: the composition of the maps of the lanes before this one
// (BACK: after it, from lane 63 down), and the whole wavefront's in `total`
// (the same for every lane).
template <bool BACK>
__device__ __forceinline__ Affine wave_affine_scan(Affine m, Affine& total) {
  constexpr int SH = BACK ? 0x100 : 0x110;  // row_shl : row_shr
  m = aff_after(m, dpp_aff<SH + 1>(m));
  m = aff_after(m, dpp_aff<SH + 2>(m));
  m = aff_after(m, dpp_aff<SH + 4>(m));
  m = aff_after(m, dpp_aff<SH + 8>(m));
  const Affine e = dpp_aff<SH + 1>(m);
  const int row = (threadIdx.x & 63) >> 4;
  Affine p = {1.0, 0.0, 0.0}, pre = p;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = BACK ? 3 - i : i;
    const int src = BACK ? 16 * r : 16 * r + 15;
    if (row == r) pre = p;
    p = aff_after(Affine{lane_f64(m.a, src), lane_f64(m.x, src), lane_f64(m.y, src)}, p);
  }
  total = p;
  return aff_after(e, pre);
}

}  // namespace mlv
