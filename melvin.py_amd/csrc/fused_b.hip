// Fused step, z-pass kernel B; the bodies are in fused_zpass.hpp.
#include "fused_zpass.hpp"

namespace mlv {

// The register pass (double precision).
template <typename T, int V>
__global__ void __launch_bounds__(64 * z_waves(V))
    k_stepZ(const JobDev<T>* __restrict__ jobs, const int* __restrict__ pref, int njobs,
            int stage, int flags, const cx<T>* __restrict__ tw) {
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int lb = xcd_logical(pref[njobs]);
  if (lb < 0) return;
  const int j = find_job(pref, njobs, lb);
  const JobDev<T>& J = jobs[j];
  const int local = lb - pref[j];
  switch (J.lognz) {
#define X(L)                                                                \
  case L:                                                                   \
    if constexpr (z_reg_fits<T>(L, V))                                      \
      stepZ_body<T, L, V>(J, J.st[stage], local, flags, tw, lds);           \
    break;
    X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10)
#undef X
    default:
      break;
  }
}

// The LDS-staged pass.  Single precision is held to 128 VGPRs: four
// wavefronts per SIMD, as many as the four blocks per CU its LDS allows at
// 1024 points.  Double precision has the extents up to 1024 in a kernel of
// their own (LO): the larger ones' 32 points per thread take 178 VGPRs, which
// leave two of the three blocks per CU that MHD's LDS allows there (4 x 1024^2
// 81 us a launch, 65 in the kernel of its own).
template <typename T, int V, int SPLIT, int PLAN, int LO>
__global__ void __launch_bounds__(kNT)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 1)))
    k_stepB(const JobDev<T>* __restrict__ jobs, const int* __restrict__ pref, int njobs,
            int stage, int flags, const cx<T>* __restrict__ tw) {
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int lb = xcd_logical(pref[njobs]);
  if (lb < 0) return;
  roleB<T, V, SPLIT, PLAN, LO>(jobs, pref, njobs, lb, stage, flags, tw, lds);
}

// --------------------------------------------------------------------------
// Launchers
// --------------------------------------------------------------------------
template <typename T, int V>
static void launchZ(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                    const cx<T>* tw, hipStream_t s) {
  const ZLaunch& z = bl.z[bl.planB];
  MLV_SET_LDS_ONCE((k_stepZ<T, V>), z.lds[V]);
  hipLaunchKernelGGL((k_stepZ<T, V>), dim3(xcd_grid(z.n[stage][V])), dim3(64 * z_waves(V)),
                     z.lds[V], s, jobs, (const int*)z.pref[stage][V], bl.njobs, stage, flags, tw);
}

template <typename T, int V, int SPLIT, int PLAN, int LO>
static void launchB_lo(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                       const cx<T>* tw, hipStream_t s) {
  const ZLaunch& b = bl.zsweep[bl.planB];
  MLV_SET_LDS_ONCE((k_stepB<T, V, SPLIT, PLAN, LO>), b.lds[V]);
  hipLaunchKernelGGL((k_stepB<T, V, SPLIT, PLAN, LO>), dim3(xcd_grid(b.n[stage][V])), dim3(kNT),
                     b.lds[V], s, jobs, (const int*)b.pref[stage][V], bl.njobs, stage, flags, tw);
}

template <typename T, int V, int SPLIT, int PLAN>
static void launchB_plan(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                         const cx<T>* tw, hipStream_t s) {
  if constexpr (sizeof(T) == 8 && z_staged_lo<T>(V, PLAN))
    if (bl.lognz_max <= kZLo)
      return launchB_lo<T, V, SPLIT, PLAN, kZLo>(jobs, bl, stage, flags, tw, s);
  launchB_lo<T, V, SPLIT, PLAN, 12>(jobs, bl, stage, flags, tw, s);
}

template <typename T, int V>
static void launchB(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                    const cx<T>* tw, hipStream_t s) {
  if constexpr (sizeof(T) == 8)
    if (bl.z[bl.planB].n[stage][V]) launchZ<T, V>(jobs, bl, stage, flags, tw, s);
  if (bl.zsweep[bl.planB].n[stage][V] == 0) return;
  const bool two = bl.planB == kPlanTwoSweep;
  if constexpr (sizeof(T) == 4) {
    if (fixed_logn(bl.lognz_all)) return launch_zpass_fixed(V, jobs, bl, stage, flags, tw, s);
    if (bl.split) {  // some job carries mean profiles
      two ? launchB_plan<T, V, 1, kPlanTwoSweep>(jobs, bl, stage, flags, tw, s)
          : launchB_plan<T, V, 1, kPlanSplit>(jobs, bl, stage, flags, tw, s);
      return;
    }
  }
  two ? launchB_plan<T, V, 0, kPlanTwoSweep>(jobs, bl, stage, flags, tw, s)
      : launchB_plan<T, V, 0, kPlanSplit>(jobs, bl, stage, flags, tw, s);
}

template <typename T>
void launch_zpass(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                  const cx<T>* tw, hipStream_t s) {
  launchB<T, BV_VORT1>(jobs, bl, stage, flags, tw, s);
  launchB<T, BV_VORT2>(jobs, bl, stage, flags, tw, s);
  launchB<T, BV_VORT3>(jobs, bl, stage, flags, tw, s);
  launchB<T, BV_MHD1>(jobs, bl, stage, flags, tw, s);
  launchB<T, BV_MHD2>(jobs, bl, stage, flags, tw, s);
}

template <typename T, int V>
static void prepareB(const BatchLaunch& bl) {
  for (int p = 0; p < 2; ++p) {
    const size_t zl = bl.z[p].lds[V], bs = bl.zsweep[p].lds[V];
    if constexpr (sizeof(T) == 8)
      if (zl) MLV_SET_LDS_ONCE((k_stepZ<T, V>), zl);
    if (!bs) continue;
    if constexpr (sizeof(T) == 8) {
      if (bl.lognz_max <= kZLo) {
        if constexpr (z_staged_lo<T>(V, kPlanSplit))
          MLV_SET_LDS_ONCE((k_stepB<T, V, 0, kPlanSplit, kZLo>), bs);
        MLV_SET_LDS_ONCE((k_stepB<T, V, 0, kPlanTwoSweep, kZLo>), bs);
        continue;
      }
    } else {
      MLV_SET_LDS_ONCE((k_stepB<T, V, 1, kPlanSplit, 12>), bs);
      MLV_SET_LDS_ONCE((k_stepB<T, V, 1, kPlanTwoSweep, 12>), bs);
    }
    MLV_SET_LDS_ONCE((k_stepB<T, V, 0, kPlanSplit, 12>), bs);
    MLV_SET_LDS_ONCE((k_stepB<T, V, 0, kPlanTwoSweep, 12>), bs);
  }
}

template <typename T>
void prepare_zpass(const BatchLaunch& bl) {
  prepareB<T, BV_VORT1>(bl);
  prepareB<T, BV_VORT2>(bl);
  prepareB<T, BV_VORT3>(bl);
  prepareB<T, BV_MHD1>(bl);
  prepareB<T, BV_MHD2>(bl);
  if constexpr (sizeof(T) == 4)
    if (fixed_logn(bl.lognz_all)) prepare_zpass_fixed(bl);
}

template void launch_zpass<float>(const JobDev<float>*, const BatchLaunch&, int, int,
                                  const cx<float>*, hipStream_t);
template void launch_zpass<double>(const JobDev<double>*, const BatchLaunch&, int, int,
                                   const cx<double>*, hipStream_t);
template void prepare_zpass<float>(const BatchLaunch&);
template void prepare_zpass<double>(const BatchLaunch&);

}  // namespace mlv
