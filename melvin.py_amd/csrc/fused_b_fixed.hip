// Fused step, single precision's z-pass kernel B compiled for one z size at a
// time (2^9 .. 2^11 points): a batch whose jobs all share that size launches these, whose
// register allocation is their own instead of the largest over every size
// the generic kernel (fused_b.hip) handles.  The body is in fused_zpass.hpp.
#include "fused_zpass.hpp"

namespace mlv {

using T = float;

template <int V, int SPLIT, int PLAN, int LOGN>
__global__ void __launch_bounds__(kNT)
    __attribute__((amdgpu_waves_per_eu(4)))
    k_stepB_fixed(const JobDev<T>* __restrict__ jobs, const int* __restrict__ pref, int njobs,
                  int stage, int flags, const cx<T>* __restrict__ tw) {
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int lb = xcd_logical(pref[njobs]);
  if (lb < 0) return;
  roleB_fixed<T, V, SPLIT, PLAN, LOGN>(jobs, pref, njobs, lb, stage, flags, tw, lds);
}

template <int V, int SPLIT, int PLAN, int LOGN>
static void launch_one(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                       const cx<T>* tw, hipStream_t s) {
  const ZLaunch& z = bl.zsweep[bl.planB];
  MLV_SET_LDS_ONCE((k_stepB_fixed<V, SPLIT, PLAN, LOGN>), z.lds[V]);
  hipLaunchKernelGGL((k_stepB_fixed<V, SPLIT, PLAN, LOGN>), dim3(xcd_grid(z.n[stage][V])),
                     dim3(kNT), z.lds[V], s, jobs, (const int*)z.pref[stage][V], bl.njobs, stage,
                     flags, tw);
}

template <int V, int SPLIT, int PLAN>
static void launch_logn(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                        const cx<T>* tw, hipStream_t s) {
  switch (bl.lognz_all) {
    case 9:
      launch_one<V, SPLIT, PLAN, 9>(jobs, bl, stage, flags, tw, s);
      break;
    case 10:
      launch_one<V, SPLIT, PLAN, 10>(jobs, bl, stage, flags, tw, s);
      break;
    case 11:
      launch_one<V, SPLIT, PLAN, 11>(jobs, bl, stage, flags, tw, s);
      break;
    default:
      break;
  }
}

template <int V>
static void launch_v(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                     const cx<T>* tw, hipStream_t s) {
  // single precision with mean profiles: SPLIT = 1 (as in fused_b.hip)
  const bool split = bl.split;
  if (bl.planB == kPlanTwoSweep) {
    if (split)
      launch_logn<V, 1, kPlanTwoSweep>(jobs, bl, stage, flags, tw, s);
    else
      launch_logn<V, 0, kPlanTwoSweep>(jobs, bl, stage, flags, tw, s);
  } else {
    if (split)
      launch_logn<V, 1, kPlanSplit>(jobs, bl, stage, flags, tw, s);
    else
      launch_logn<V, 0, kPlanSplit>(jobs, bl, stage, flags, tw, s);
  }
}

void launch_zpass_fixed(int v, const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                        const cx<T>* tw, hipStream_t s) {
  switch (v) {
    case BV_VORT1:
      launch_v<BV_VORT1>(jobs, bl, stage, flags, tw, s);
      break;
    case BV_VORT2:
      launch_v<BV_VORT2>(jobs, bl, stage, flags, tw, s);
      break;
    case BV_VORT3:
      launch_v<BV_VORT3>(jobs, bl, stage, flags, tw, s);
      break;
    case BV_MHD1:
      launch_v<BV_MHD1>(jobs, bl, stage, flags, tw, s);
      break;
    case BV_MHD2:
      launch_v<BV_MHD2>(jobs, bl, stage, flags, tw, s);
      break;
    default:
      break;
  }
}

template <int V, int L>
static void prepare_vl(const BatchLaunch& bl) {
  MLV_SET_LDS_ONCE((k_stepB_fixed<V, 0, kPlanSplit, L>), bl.zsweep[0].lds[V]);
  MLV_SET_LDS_ONCE((k_stepB_fixed<V, 0, kPlanTwoSweep, L>), bl.zsweep[0].lds[V]);
  MLV_SET_LDS_ONCE((k_stepB_fixed<V, 1, kPlanSplit, L>), bl.zsweep[0].lds[V]);
  MLV_SET_LDS_ONCE((k_stepB_fixed<V, 1, kPlanTwoSweep, L>), bl.zsweep[0].lds[V]);
}

template <int V>
static void prepare_v(const BatchLaunch& bl) {
  if (!bl.zsweep[0].lds[V]) return;
  if (bl.lognz_all == 9) prepare_vl<V, 9>(bl);
  if (bl.lognz_all == 10) prepare_vl<V, 10>(bl);
  if (bl.lognz_all == 11) prepare_vl<V, 11>(bl);
}

void prepare_zpass_fixed(const BatchLaunch& bl) {
  prepare_v<BV_VORT1>(bl);
  prepare_v<BV_VORT2>(bl);
  prepare_v<BV_VORT3>(bl);
  prepare_v<BV_MHD1>(bl);
  prepare_v<BV_MHD2>(bl);
}

}  // namespace mlv
