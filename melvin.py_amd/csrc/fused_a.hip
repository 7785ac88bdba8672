// Fused step, x-inverse kernel A (spectral prologue + inverse x pass, and the
// single-precision x-mean profiles); the bodies are in fused_xinv.hpp.
#include "fused_xinv.hpp"

namespace mlv {

// Logical blocks [0, nA) are kernel A's, then kMeanCh / 2 per job for the
// mean profiles.
template <typename T, int NT, int LO, bool MIXED>
__global__ void __launch_bounds__(NT)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 1)))
    k_stepA(const JobDev<T>* __restrict__ jobs, const int* __restrict__ pref, int njobs, int nA,
            int nM, int stage, int step, const cx<T>* __restrict__ tw) {
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  int lb = xcd_logical(nA + nM);
  if (lb < 0) return;
  if (sizeof(T) == 4 && lb >= nA) {
    lb -= nA;
    const JobDev<T>& J = jobs[lb / (kMeanCh / 2)];
    if (stage >= J.nstage || !J.split) return;
    const int pair = lb % (kMeanCh / 2), par = (J.par0 + step) & 1;
    switch (J.lognz) {
#define X(L)                                                               \
  case L:                                                                  \
    if constexpr (mean_fits(L, NT))                                        \
      stepM_body<T, L, NT>(J, J.st[stage], pair, par, tw, lds);            \
    break;
      X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)
#undef X
      default:
        break;
    }
    return;
  }
  const int j = find_job(pref, njobs, lb);
  const JobDev<T>& J = jobs[j];
  const int local = lb - pref[j], par = (J.par0 + step) & 1;
  switch (J.lognx) {
#define X(L)                                                               \
  case L:                                                                  \
    if constexpr (L <= LO && xp_fits<T>(L, NT) && (!MIXED || xmix_nt(L) == NT))           \
      stepA_body<T, L, NT, MIXED>(J, J.st[stage], local, par, tw, lds);    \
    break;
    X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)
#undef X
    default:
      break;
  }
}

// --------------------------------------------------------------------------
// Launchers
// --------------------------------------------------------------------------
template <typename T, int NT, int LO, bool MIXED>
static void launchA_lo(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int step,
                    const cx<T>* tw, hipStream_t s) {
  const int nA = bl.nA[stage], nM = sizeof(T) == 4 && bl.split ? bl.njobs * (kMeanCh / 2) : 0;
  MLV_SET_LDS_ONCE((k_stepA<T, NT, LO, MIXED>), bl.ldsA);
  hipLaunchKernelGGL((k_stepA<T, NT, LO, MIXED>), dim3(xcd_grid(nA + nM)), dim3(NT), bl.ldsA, s, jobs,
                     (const int*)bl.prefA[stage], bl.njobs, nA, nM, stage, step, tw);
}

template <typename T, int NT, bool MIXED>
static void launchA(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int step,
                    const cx<T>* tw, hipStream_t s) {
  const int lo = xp_lo<T>(bl.lognx_max);
  if (lo == kXpLo) return launchA_lo<T, NT, kXpLo, MIXED>(jobs, bl, stage, step, tw, s);
  if constexpr (!MIXED && xp_fits<T>(11, NT)) {  // (no smaller block holds a column)
    if constexpr (sizeof(T) == 8)
      if (lo == 11) return launchA_lo<T, NT, 11, MIXED>(jobs, bl, stage, step, tw, s);
    launchA_lo<T, NT, 12, MIXED>(jobs, bl, stage, step, tw, s);
  }
}

template <typename T>
void launch_xinv(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int step,
                 const cx<T>* tw, hipStream_t s) {
  if (bl.nA[stage] == 0) return;
  const int nt = bl.ntA[bl.shapeA];
  if constexpr (sizeof(T) == 4) {
    if (bl.shapeA == 2) return launchA<T, 1024, true>(jobs, bl, stage, step, tw, s);
  }
  switch (nt) {
    case 64: return launchA<T, 64, false>(jobs, bl, stage, step, tw, s);
    case 128: return launchA<T, 128, false>(jobs, bl, stage, step, tw, s);
    case 256: return launchA<T, 256, false>(jobs, bl, stage, step, tw, s);
    default: return launchA<T, 512, false>(jobs, bl, stage, step, tw, s);
  }
}

template <typename T, int NT>
static void prepareA(const BatchLaunch& bl, size_t lds) {
  const int lo = xp_lo<T>(bl.lognx_max);
  if (lo == kXpLo) MLV_SET_LDS_ONCE((k_stepA<T, NT, kXpLo, false>), lds);
  if constexpr (xp_fits<T>(11, NT)) {
    if constexpr (sizeof(T) == 8)
      if (lo == 11) MLV_SET_LDS_ONCE((k_stepA<T, NT, 11, false>), lds);
    if (lo == 12) MLV_SET_LDS_ONCE((k_stepA<T, NT, 12, false>), lds);
  }
}

template <typename T>
void prepare_xinv(const BatchLaunch& bl) {
  for (int a = 0; a < 3; ++a) {
    if (!bl.okA[a]) continue;
    const size_t lds = bl.ldsAp[a];
    if constexpr (sizeof(T) == 4) {
      if (a == 2) {
        MLV_SET_LDS_ONCE((k_stepA<T, 1024, kXpLo, true>), lds);
        continue;
      }
    }
    if (bl.ntA[a] == 64) prepareA<T, 64>(bl, lds);
    if (bl.ntA[a] == 128) prepareA<T, 128>(bl, lds);
    if (bl.ntA[a] == 256) prepareA<T, 256>(bl, lds);
    if (bl.ntA[a] == 512) prepareA<T, 512>(bl, lds);
  }
}

template void launch_xinv<float>(const JobDev<float>*, const BatchLaunch&, int, int,
                                 const cx<float>*, hipStream_t);
template void launch_xinv<double>(const JobDev<double>*, const BatchLaunch&, int, int,
                                  const cx<double>*, hipStream_t);
template void prepare_xinv<float>(const BatchLaunch&);
template void prepare_xinv<double>(const BatchLaunch&);

}  // namespace mlv
