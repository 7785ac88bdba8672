// Fused step, update kernel C, the dt setter and the device CFL /
// diagnostics kernel; the update body is in fused_update.hpp.
#include "fused_update.hpp"

namespace mlv {

// Single precision is held to 128 VGPRs (four wavefronts per SIMD).
template <typename T, int NT, int LO>
__global__ void __launch_bounds__(NT)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 1)))
    k_stepC(const JobDev<T>* __restrict__ jobs, JobDev<T>* clock, const int* __restrict__ pref,
            int njobs, int stage, int step, const cx<T>* __restrict__ tw) {
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int lb = xcd_logical(pref[njobs]);
  if (lb < 0) return;
  roleC<T, NT, LO>(jobs, clock, pref, njobs, lb, stage, step, tw, lds);
}

// Shape 2, for a batch whose jobs all have 2^LOGN points along x.
template <int LOGN>
__global__ void __launch_bounds__(64 * kGroupCols) __attribute__((amdgpu_waves_per_eu(4)))
    k_stepC_group(const JobDev<float>* __restrict__ jobs, JobDev<float>* clock,
                  const int* __restrict__ pref, int njobs, int stage, int step,
                  const cx<float>* __restrict__ tw) {
  extern __shared__ char smem_raw[];
  cx<float>* lds = reinterpret_cast<cx<float>*>(smem_raw);
  const int lb = xcd_logical(pref[njobs]);
  if (lb < 0) return;
  roleC_group<float, LOGN>(jobs, clock, pref, njobs, lb, stage, step, tw, lds);
}

template <typename T>
__global__ void k_set_dt(JobDev<T>* jobs, int j, double dt) {
  if (threadIdx.x == 0 && blockIdx.x == 0) jobs[j].dt = dt;
}

// One block per job, after a step whose z pass wrote diagnostics partials:
// tracker record and CFL rule (diag_apply).  The first advected scalar
// exists in vorticity and DDC jobs of two or more fields.
template <typename T>
__global__ void __launch_bounds__(kNT) k_diag(JobDev<T>* jobs, double cutoff, int cadence) {
  JobDev<T>& J = jobs[blockIdx.x];
  // loops has been advanced by this step's update kernel: the step was this
  // job's check loop when the count before it was a multiple of cadence
  if ((J.loops - 1) % cadence != 0) return;
  double dt = J.dt;
  const bool flux = J.problem != MLV_PROB_MHD && J.nfield >= 2;
  if (diag_apply<kNT>(J.diag, J.nbB, J.dx, J.dz, (double)J.nx * (double)J.nz, flux, cutoff, J.t,
                      J.loops, dt))
    J.dt = dt;
}


// --------------------------------------------------------------------------
// Launchers
// --------------------------------------------------------------------------
template <typename T, int NT, int LO>
static void launchC_lo(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int step,
                       const cx<T>* tw, hipStream_t s) {
  MLV_SET_LDS_ONCE((k_stepC<T, NT, LO>), bl.ldsC);
  hipLaunchKernelGGL((k_stepC<T, NT, LO>), dim3(xcd_grid(bl.nC[stage])), dim3(NT), bl.ldsC, s, jobs,
                     const_cast<JobDev<T>*>(jobs), (const int*)bl.prefC[stage], bl.njobs, stage,
                     step, tw);
}

template <typename T, int NT>
static void launchC(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int step,
                    const cx<T>* tw, hipStream_t s) {
  const int lo = xp_lo<T>(bl.lognx_max);
  if (lo == kXpLo) return launchC_lo<T, NT, kXpLo>(jobs, bl, stage, step, tw, s);
  if constexpr (xp_fits<T>(11, NT)) {  // (no smaller block holds a column)
    if constexpr (sizeof(T) == 8)
      if (lo == 11) return launchC_lo<T, NT, 11>(jobs, bl, stage, step, tw, s);
    launchC_lo<T, NT, 12>(jobs, bl, stage, step, tw, s);
  }
}

template <int LOGN>
static void launchC_group(const JobDev<float>* jobs, const BatchLaunch& bl, int stage, int step,
                          const cx<float>* tw, hipStream_t s) {
  MLV_SET_LDS_ONCE((k_stepC_group<LOGN>), bl.ldsC);
  hipLaunchKernelGGL((k_stepC_group<LOGN>), dim3(xcd_grid(bl.nC[stage])), dim3(64 * kGroupCols),
                     bl.ldsC, s, jobs, const_cast<JobDev<float>*>(jobs),
                     (const int*)bl.prefC[stage], bl.njobs, stage, step, tw);
}

template <typename T>
void launch_update(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int step,
                   const cx<T>* tw, hipStream_t s) {
  if (bl.nC[stage] == 0) return;
  if constexpr (sizeof(T) == 4) {
    if (bl.wideC == 2 && bl.lognx_all == 9) return launchC_group<9>(jobs, bl, stage, step, tw, s);
    if (bl.wideC == 2 && bl.lognx_all == 10) return launchC_group<10>(jobs, bl, stage, step, tw, s);
  }
  switch (bl.ntC[bl.wideC]) {
    case 64: return launchC<T, 64>(jobs, bl, stage, step, tw, s);
    case 128: return launchC<T, 128>(jobs, bl, stage, step, tw, s);
    case 256: return launchC<T, 256>(jobs, bl, stage, step, tw, s);
    default: return launchC<T, 512>(jobs, bl, stage, step, tw, s);
  }
}

template <typename T, int NT>
static void prepareC(const BatchLaunch& bl, size_t lds) {
  const int lo = xp_lo<T>(bl.lognx_max);
  if (lo == kXpLo) MLV_SET_LDS_ONCE((k_stepC<T, NT, kXpLo>), lds);
  if constexpr (xp_fits<T>(11, NT)) {
    if constexpr (sizeof(T) == 8)
      if (lo == 11) MLV_SET_LDS_ONCE((k_stepC<T, NT, 11>), lds);
    if (lo == 12) MLV_SET_LDS_ONCE((k_stepC<T, NT, 12>), lds);
  }
}

template <typename T>
void prepare_update(const BatchLaunch& bl) {
  for (int c = 0; c < 3; ++c) {
    if (!bl.okC[c]) continue;
    const size_t lds = bl.ldsCp[c];
    if constexpr (sizeof(T) == 4) {
      if (c == 2 && group_shape(bl.lognx_all)) {
        if (bl.lognx_all == 9) MLV_SET_LDS_ONCE((k_stepC_group<9>), lds);
        if (bl.lognx_all == 10) MLV_SET_LDS_ONCE((k_stepC_group<10>), lds);
        continue;
      }
    }
    if (bl.ntC[c] == 64) prepareC<T, 64>(bl, lds);
    if (bl.ntC[c] == 128) prepareC<T, 128>(bl, lds);
    if (bl.ntC[c] == 256) prepareC<T, 256>(bl, lds);
    if (bl.ntC[c] == 512) prepareC<T, 512>(bl, lds);
  }
}

template <typename T>
hipError_t fused_set_dt(JobDev<T>* jobs, int job, double dt, hipStream_t s) {
  hipLaunchKernelGGL(k_set_dt<T>, dim3(1), dim3(64), 0, s, jobs, job, dt);
  return hipGetLastError();
}

template <typename T>
hipError_t fused_diag(JobDev<T>* jobs, int njobs, double cutoff, int cadence, hipStream_t s) {
  hipLaunchKernelGGL(k_diag<T>, dim3(njobs), dim3(kNT), 0, s, jobs, cutoff, cadence);
  return hipGetLastError();
}

template void launch_update<float>(const JobDev<float>*, const BatchLaunch&, int, int,
                                   const cx<float>*, hipStream_t);
template void launch_update<double>(const JobDev<double>*, const BatchLaunch&, int, int,
                                    const cx<double>*, hipStream_t);
template void prepare_update<float>(const BatchLaunch&);
template void prepare_update<double>(const BatchLaunch&);
template hipError_t fused_diag<float>(JobDev<float>*, int, double, int, hipStream_t);
template hipError_t fused_diag<double>(JobDev<double>*, int, double, int, hipStream_t);
template hipError_t fused_set_dt<float>(JobDev<float>*, int, double, hipStream_t);
template hipError_t fused_set_dt<double>(JobDev<double>*, int, double, hipStream_t);

}  // namespace mlv
