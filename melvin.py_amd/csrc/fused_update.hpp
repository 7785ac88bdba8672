// Device body of the fused step's update kernel C (forward x pass, FD
// operator, sources, Adams-Bashforth + semi-implicit update), launched by
// fused_c.hip in its generic and size-specialised forms.
#pragma once
#include "fused.hpp"
#include "diag_dev.hpp"
#include "grid.hpp"

namespace mlv {
// --------------------------------------------------------------------------
// Kernel C: forward x pass, FD operator, sources, AB + semi-implicit update
// --------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T modk(const cx<T>* __restrict__ tw, int k, int logn, int order,
                                  double h) {
  const T s1 = tsin<T>(tw, k, logn);
  if (order == 2) return s1 / (T)h;
  const T s2 = tsin<T>(tw, 2 * k, logn);
  return fma1(T(8), s1, -s2) / (T)(6.0 * h);
}

// NT threads per block, TC = NT / TPS columns of one equation, consecutive
// threads on consecutive columns: a load of Px / Pz covers whole groups of
// their kz-grouped layout, and the x = t + m TPS that a thread holds after
// the transform are the rows it updates, so the result never goes back
// through LDS (it did, twice, when a wavefront's columns were transformed in
// LDS and updated from it).
// What bounds it: at 16 x 1024^2 FP32 (two fields, AB4) its 597 MB, 145 us =
// 4.1 TB/s of the 5.2 a copy reaches (shape 2, below: 138); on small grids the
// chain of one block: 256^2 FP64 14.1 -> 6.8 us, 4 x 512^2 FP32 20.2 -> 9.4,
// 1024^2 FP64 20.5 -> 18.6.  512-thread blocks, whose Px / Pz runs are twice
// as long, measured 4 us more at 16 x 1024^2 and 38.7 against 30.3 us on a
// mixed batch of double diffusion: more, shorter blocks hide each other's
// barriers.
//
// GROUP (shape 2: single precision, batches of one x size of 512 or 1024
// points): blocks of a whole column group, 64 threads a column, one wavefront
// per column from the transform on.  The group's rows are loaded and
// differenced as above, pass through LDS to their columns' wavefronts and,
// transformed with the same radices, through LDS again, to be updated row by
// row: 512 bytes of each array at a time, four rows of a thread in flight
// where its registers would hold two.  What bounds it: the launch's memory
// traffic, once it is large: 64 x 1024^2 with a scalar 496 us (4.8 TB/s of its
// 2.39 GB, where a copy reaches 5.2) against 527 in blocks of two columns,
// which touch each group's lines four times over (46.5 million requests at the
// L2 against 26.1, for the same misses), and 16 of them 138 against 145.  Below
// two and a half blocks per CU the chain of one block is longer: 1024^2 16.9
// against 12.0.
template <typename T, int LOGN, int NT, bool GROUP = false>
__device__ __forceinline__ void stepC_body(const JobDev<T>& J, const StageDev& S, int local, int cur,
                                           int par, const cx<T>* __restrict__ tw, cx<T>* lds) {
#pragma clang fp contract(off)  // fused operations are spelled out (fma1)
  constexpr int N = 1 << LOGN, LOGE = GROUP ? group_loge(LOGN) : xp_loge<T>(LOGN);
  constexpr int E = 1 << LOGE, TPS = N / E, TC = NT / TPS;
  static_assert(!GROUP || (TPS == 64 && TC == kGroupCols), "a wavefront per column of a group");
  constexpr int nn = xp_nn(N), rows = 2 * nn + 1;
  const int nm = J.nm;
  const size_t chs = work_chs(N, nm);
  const size_t ssz = (size_t)rows * nm;
  const int ntile = (nm + TC - 1) / TC;
  const int eqi = local / ntile, tile = local % ntile;
  const int field = S.eq_field[eqi];
  const int c = threadIdx.x % TC, t = rf_thread<TPS>(threadIdx.x / TC);
  int col = tile * TC + c;
  const bool cok = col < nm;
  const cx<T>* __restrict__ pxc = glb(J.work) + (size_t)pchan(J.pbase, eqi, 0) * chs;
  const cx<T>* __restrict__ pzc = glb(J.work) + (size_t)pchan(J.pbase, eqi, 1) * chs;
  // One transform per column: the periodic x difference acts on the
  // intermediate rows (it commutes with the z transform) and the z
  // difference is its modified wavenumber, so
  //   D = F_x[ FDx(Px) + i sz(kz) Pz ].
  const int order = J.fd_order;
  const T ihx = order == 2 ? (T)(1.0 / (2.0 * J.dx)) : (T)(1.0 / (3.0 * J.dx));
  const uint32_t p0 = (uint32_t)pidx(0, cok ? col : 0, N) * sizeof(cx<T>);
  cx<T> v[E], zv[E];
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const uint32_t o = p0 + (uint32_t)(t + m * TPS) * (kPGroup * sizeof(cx<T>));
    v[m] = at32(pxc, o);
    zv[m] = at32(pzc, o);
  }
  const T szc = modk<T>(tw, cok ? col : 0, J.lognz, order, J.dz);
  // a column's elements in LDS, beside the other columns' or (GROUP) apart
  constexpr int SD = GROUP ? 1 : TC;
  cx<T>* __restrict__ slot = lds + (GROUP ? c * group_len(LOGN) : c);
#pragma unroll
  for (int m = 0; m < E; ++m) slot[rf_pad<LOGE>(t, m * TPS) * SD] = v[m];
  rf_sync<NT>();
#pragma unroll
  for (int m = 0; m < E; ++m) {
    auto at = [&](int d) { return slot[rf_near<LOGN, LOGE>(t, m, d) * SD]; };
    const cx<T> a1 = at(1), b1 = at(-1);
    cx<T> d;
    if (order == 2) {
      d = mk<T>((a1.x - b1.x) * ihx, (a1.y - b1.y) * ihx);
    } else {
      const cx<T> a2 = at(2), b2 = at(-2);
      d = mk<T>(fma1(T(0.25), b2.x - a2.x, T(2) * (a1.x - b1.x)) * ihx,
                fma1(T(0.25), b2.y - a2.y, T(2) * (a1.y - b1.y)) * ihx);
    }
    v[m] = mk<T>(fma1(-szc, zv[m].y, d.x), fma1(szc, zv[m].x, d.y));
  }
  rf_sync<NT>();
  const int lane = threadIdx.x & 63;
  if constexpr (GROUP) {
#pragma unroll
    for (int m = 0; m < E; ++m) slot[rf_pad<LOGE>(t, m * TPS)] = v[m];
    rf_sync<NT>();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    col = tile * TC + wv;
    if (col >= nm) return;
    slot = lds + wv * group_len(LOGN);
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = slot[rf_pad<LOGE>(lane, m * TPS)];
    rf_sync<64>();
    rf_fft<T, LOGN, LOGE, -1, 1, 64, xp_loge<T>(LOGN)>(v, slot, lane, tw);
    rf_sync<64>();
#pragma unroll
    for (int m = 0; m < E; ++m)
      if (xp_any(m, TPS, N)) slot[rf_pad<LOGE>(lane, m * TPS)] = v[m];
    rf_sync<64>();
  } else {
    rf_fft<T, LOGN, LOGE, -1, TC, NT>(v, slot, t, tw);
    if (!cok) return;
  }

  const int q = J.q;
  const double dt = J.dt, alpha = J.alpha;
  const double c1 = (1 - alpha) * dt, c2 = alpha * dt;
  const double hab = q == 2 ? dt / 2 : dt / 24;
  const double coeff = J.coeff[field];
  const T scale = (T)J.scale;
  const cx<T>* __restrict__ sin_ = glb(J.state[par][field]);
  cx<T>* __restrict__ sout = glb(J.state[par ^ 1][field]);
  cx<T>* __restrict__ hist = glb(J.hist[field]);
  const bool ddc = J.problem == MLV_PROB_DDC;
  const cx<T>* __restrict__ se1 = ddc ? glb(J.state[par][field == 0 ? 1 : 0]) : nullptr;
  const cx<T>* __restrict__ se2 = ddc && field == 0 ? glb(J.state[par][2]) : nullptr;
  uint32_t* __restrict__ carry = sizeof(T) == 4 ? glb(J.comp[field]) : nullptr;
  const cx<T>* __restrict__ hist1 = hist + (size_t)((cur + q - 1) % q) * ssz;
  const cx<T>* __restrict__ hist2 = hist + (size_t)((cur + q - 2) % q) * ssz;
  const cx<T>* __restrict__ hist3 = hist + (size_t)((cur + q - 3) % q) * ssz;
  cx<T>* __restrict__ histc = hist + (size_t)cur * ssz;
  const float fcoeff = (float)coeff, ffx2 = (float)J.fx2, ffz2 = (float)J.fz2;
  const float fdt = (float)dt, fc2 = (float)c2;
  const uint32_t cbase = (uint32_t)col * rows;
  // rows updated U at a time, their loads issued before any is used (single
  // precision: all of them at once spill, 176 against 150 us at 16 x 1024^2)
  constexpr int U = E >= 16 && sizeof(T) == 4 && !GROUP ? 2 : 4;
  // row groups: the points a thread holds, or runs of 64 rows
  constexpr int G = GROUP ? (rows + 63) / 64 : E;
  auto any = [](int m) { return GROUP || xp_any(m, TPS, N); };
  auto row_of = [&](int m) {
    if constexpr (GROUP) return lane + 64 * m < rows ? lane + 64 * m : -1;
    else return xp_row(t + m * TPS, N);
  };
#pragma unroll(GROUP ? 1 : E)
  for (int m0 = 0; m0 < G; m0 += U) {
    // (a group's loads stay behind the group before: hoisted, they spill)
    if constexpr (sizeof(T) == 4) __builtin_amdgcn_sched_barrier(0);
    cx<T> vv[U], h1[U], h2[U], h3[U], e1[U], e2[U];
    uint32_t lo[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!any(m0 + u)) continue;
      const int r = row_of(m0 + u);
      if (r < 0) continue;
      const uint32_t o = (cbase + r) * (uint32_t)sizeof(cx<T>);
      vv[u] = at32(sin_, o);
      h1[u] = at32(hist1, o);
      if (q == 4) {
        h2[u] = at32(hist2, o);
        h3[u] = at32(hist3, o);
      }
      if (carry) lo[u] = at32(carry, (cbase + r) * 4u);
      if (se1) e1[u] = at32(se1, o);
      if (se2) e2[u] = at32(se2, o);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!any(m0 + u)) continue;
      const int r = row_of(m0 + u);
      if (r < 0) continue;
      const int n = r <= nn ? r : r - rows, m = col;
      const uint32_t o = (cbase + r) * (uint32_t)sizeof(cx<T>);
      cx<T> D;
      if constexpr (GROUP)
        D = slot[rf_pad<LOGE>(r <= nn ? r : r + N - rows)];
      else
        D = v[m0 + u];
      cx<T> rhs = mk<T>(D.x * scale, D.y * scale);
      if (ddc) {
        const double Pr = J.param[0], R0 = J.param[1];
        if (field == 0) {
          const T y = (T)(J.fx * n);
          const cx<T> t = e1[u], sv = e2[u];
          const T pr = (T)Pr;
          rhs = mk<T>(fma1(-pr, y * sv.y, rhs.x), fma1(pr, y * sv.x, rhs.y));
          rhs = mk<T>(fma1(pr, y * t.y, rhs.x), fma1(-pr, y * t.x, rhs.y));
        } else {
          double lap = fma1(J.fx2, (double)(n * n), J.fz2 * (double)(m * m));
          if (r == 0 && m == 0) lap = 1.0;
          const T rl = (T)(1.0 / lap);
          const cx<T> w = e1[u];
          const cx<T> ps = mk<T>(-w.x * rl, -w.y * rl);
          const T y = (T)(J.fx * n);
          cx<T> uz = mk<T>(-(y * ps.y), y * ps.x);
          if (field == 2) {
            const T ir0 = (T)(1.0 / R0);
            uz = mk<T>(uz.x * ir0, uz.y * ir0);
          }
          rhs = csub<T>(rhs, uz);
        }
      }
      at32(histc, o) = rhs;
      T abx, aby;
      if (q == 2) {
        abx = fma1(T(3), rhs.x, -h1[u].x);
        aby = fma1(T(3), rhs.y, -h1[u].y);
      } else {
        abx = fma1(T(-9), h3[u].x, fma1(T(37), h2[u].x, fma1(T(55), rhs.x, T(-59) * h1[u].x)));
        aby = fma1(T(-9), h3[u].y, fma1(T(37), h2[u].y, fma1(T(55), rhs.y, T(-59) * h1[u].y)));
      }
      const cx<T> v = vv[u];
      cx<T> nv;
      const bool masked = ddc && field != 0 && m == 0;
      if constexpr (sizeof(T) == 8) {
        // (1 + (1-a) dt L) v + AB, divided by (1 - a dt L)  (Integrator.py:58-63)
        const double lin = coeff * fma1(J.fx2, (double)(n * n), J.fz2 * (double)(m * m));
        const T num = (T)fma1(c1, lin, 1.0);
        const T rden = (T)(1.0 / fma1(-c2, lin, 1.0));
        nv = mk<T>(fma1(num, v.x, (T)hab * abx) * rden, fma1(num, v.y, (T)hab * aby) * rden);
      } else {
        // The same update written as an increment, v + (dt L v + AB)/(1 - a dt L),
        // so the rounding falls on the small change, not on (1 + (1-a) dt L);
        // the factors therefore only need single precision.  With a carry
        // array the addition is Kahan-compensated: increments below half an
        // ulp of v are kept instead of being dropped every step.
        const float lin = fcoeff * fma1(ffx2, (float)(n * n), ffz2 * (float)(m * m));
        const T a = fdt * lin;
        const T rden = __builtin_amdgcn_rcpf(fma1(-fc2, lin, 1.0f));
        const T ix = fma1(a, v.x, (T)hab * abx) * rden, iy = fma1(a, v.y, (T)hab * aby) * rden;
        if (carry) {
          const float2 l = bf2_load(lo[u]);
          const T yx = ix - (T)l.x, yy = iy - (T)l.y;
          const T tx = v.x + yx, ty = v.y + yy;
          at32(carry, (cbase + r) * 4u) = masked ? 0u : bf2_pack((float)((tx - v.x) - yx), (float)((ty - v.y) - yy));
          nv = mk<T>(tx, ty);
        } else {
          nv = mk<T>(v.x + ix, v.y + iy);
        }
      }
      if (masked) nv = czero<T>();
      at32(sout, o) = nv;
    }
  }
}

// Kernel C's work for logical block lb of a launch over the job table's
// update blocks (prefix array pref).  The block of local index 0 of a job
// advances the job's device-side t and loop count after its last stage
// (Simulation.py:199-209), through `clock` -- the same table, as a plain
// pointer: the launch reads those two fields through neither pointer, so
// the read-only, non-aliased `jobs` stays valid for every field it reads.
// LO: the largest size (log2) of the launch's jobs this kernel is compiled for.
template <typename T, int NT, int LO>
__device__ __forceinline__ void roleC(const JobDev<T>* __restrict__ jobs, JobDev<T>* clock,
                                      const int* __restrict__ pref, int njobs, int lb, int stage,
                                      int step, const cx<T>* __restrict__ tw, cx<T>* lds) {
  const int j = find_job(pref, njobs, lb);
  const JobDev<T>& J = jobs[j];
  const int local = lb - pref[j];
  const int par = (J.par0 + step) & 1;
  const int cur = ring(J.curr0, step, J.q);
  if (stage == J.nstage - 1 && local == 0 && threadIdx.x == 0) {
    clock[j].t = clock[j].t + J.dt;
    clock[j].loops = clock[j].loops + 1;
  }
  switch (J.lognx) {
#define X(L)                                                            \
  case L:                                                               \
    if constexpr (L <= LO && xp_fits<T>(L, NT))                              \
      stepC_body<T, L, NT>(J, J.st[stage], local, cur, par, tw, lds);   \
    break;
    X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)
#undef X
    default:
      break;
  }
}

// Shape 2's work for logical block lb, in a batch of 2^LOGN points along x.
template <typename T, int LOGN>
__device__ __forceinline__ void roleC_group(const JobDev<T>* __restrict__ jobs, JobDev<T>* clock,
                                            const int* __restrict__ pref, int njobs, int lb,
                                            int stage, int step, const cx<T>* __restrict__ tw,
                                            cx<T>* lds) {
  const int j = find_job(pref, njobs, lb);
  const JobDev<T>& J = jobs[j];
  const int local = lb - pref[j];
  if (stage == J.nstage - 1 && local == 0 && threadIdx.x == 0) {
    clock[j].t = clock[j].t + J.dt;
    clock[j].loops = clock[j].loops + 1;
  }
  stepC_body<T, LOGN, 64 * kGroupCols, true>(J, J.st[stage], local, ring(J.curr0, step, J.q),
                                             (J.par0 + step) & 1, tw, lds);
}

}  // namespace mlv
