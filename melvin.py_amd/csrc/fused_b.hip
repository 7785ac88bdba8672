// Fused step, z-pass kernel B; the bodies are in fused_zpass.hpp.
#include "fused_zpass.hpp"

namespace mlv {

// The register pass (double precision).  LO: the largest z extent (log2) of
// the launch's jobs that this kernel is compiled for: 2048 points take 32 per
// thread and would set every size's registers.
template <typename T, int V, int LO>
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
    if constexpr (L <= LO && z_reg_fits<T>(L, V))                                            \
      stepZ_body<T, L, V>(J, J.st[stage], local, flags, tw, lds);           \
    break;
    X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11)
#undef X
    default:
      break;
  }
}

// The LDS-staged pass.  Single precision is held to 128 VGPRs: four
// wavefronts per SIMD, as many as the four blocks per CU its LDS allows at
// 1024 points.
template <typename T, int V, int SPLIT, int PLAN>
__global__ void __launch_bounds__(kNT)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 1)))
    k_stepB(const JobDev<T>* __restrict__ jobs, const int* __restrict__ pref, int njobs,
            int stage, int flags, const cx<T>* __restrict__ tw) {
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int lb = xcd_logical(pref[njobs]);
  if (lb < 0) return;
  roleB<T, V, SPLIT, PLAN>(jobs, pref, njobs, lb, stage, flags, tw, lds);
}

// --------------------------------------------------------------------------
// Launchers
// --------------------------------------------------------------------------
template <typename T, int V, int LO>
static void launchZ(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                    const cx<T>* tw, hipStream_t s) {
  const ZLaunch& z = bl.z[bl.planB];
  MLV_SET_LDS_ONCE((k_stepZ<T, V, LO>), z.lds[V]);
  hipLaunchKernelGGL((k_stepZ<T, V, LO>), dim3(xcd_grid(z.n[stage][V])), dim3(64 * z_waves(V)),
                     z.lds[V], s, jobs, (const int*)z.pref[stage][V], bl.njobs, stage, flags, tw);
}

template <typename T, int V, int SPLIT, int PLAN>
static void launchB_plan(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                         const cx<T>* tw, hipStream_t s) {
  const ZLaunch& b = bl.zsweep[bl.planB];
  MLV_SET_LDS_ONCE((k_stepB<T, V, SPLIT, PLAN>), b.lds[V]);
  hipLaunchKernelGGL((k_stepB<T, V, SPLIT, PLAN>), dim3(xcd_grid(b.n[stage][V])), dim3(kNT),
                     b.lds[V], s, jobs, (const int*)b.pref[stage][V], bl.njobs, stage, flags, tw);
}

template <typename T, int V>
static void launchB(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                    const cx<T>* tw, hipStream_t s) {
  const bool swept = bl.zsweep[bl.planB].n[stage][V] != 0;
  if constexpr (sizeof(T) == 8) {
    if (bl.z[bl.planB].n[stage][V]) {
      if (bl.lognz_max <= kZLo)
        launchZ<T, V, kZLo>(jobs, bl, stage, flags, tw, s);
      else
        launchZ<T, V, 11>(jobs, bl, stage, flags, tw, s);
    }
    if (swept) launchB_plan<T, V, 0, kPlanTwoSweep>(jobs, bl, stage, flags, tw, s);
  } else {
    if (!swept) return;
    if (fixed_logn(bl.lognz_all)) return launch_zpass_fixed(V, jobs, bl, stage, flags, tw, s);
    const bool two = bl.planB == kPlanTwoSweep;
    if (bl.split)  // some job carries mean profiles
      two ? launchB_plan<T, V, 1, kPlanTwoSweep>(jobs, bl, stage, flags, tw, s)
          : launchB_plan<T, V, 1, kPlanSplit>(jobs, bl, stage, flags, tw, s);
    else
      two ? launchB_plan<T, V, 0, kPlanTwoSweep>(jobs, bl, stage, flags, tw, s)
          : launchB_plan<T, V, 0, kPlanSplit>(jobs, bl, stage, flags, tw, s);
  }
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
    if constexpr (sizeof(T) == 8) {
      if (zl && bl.lognz_max <= kZLo) MLV_SET_LDS_ONCE((k_stepZ<T, V, kZLo>), zl);
      if (zl && bl.lognz_max > kZLo) MLV_SET_LDS_ONCE((k_stepZ<T, V, 11>), zl);
      if (bs) MLV_SET_LDS_ONCE((k_stepB<T, V, 0, kPlanTwoSweep>), bs);
    } else if (bs) {
      MLV_SET_LDS_ONCE((k_stepB<T, V, 0, kPlanSplit>), bs);
      MLV_SET_LDS_ONCE((k_stepB<T, V, 0, kPlanTwoSweep>), bs);
      MLV_SET_LDS_ONCE((k_stepB<T, V, 1, kPlanSplit>), bs);
      MLV_SET_LDS_ONCE((k_stepB<T, V, 1, kPlanTwoSweep>), bs);
    }
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
