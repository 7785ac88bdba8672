// Fused Fourier-x / FD-z step kernels over a job table (see fdz.hpp).
#include <math.h>

#include "affine_scan.hpp"
#include "diag_dev.hpp"
#include "fdz.hpp"
#include "grid.hpp"

namespace mlv {

template <typename T>
__device__ __forceinline__ double2 d2(cx<T> v) {
  return make_double2((double)v.x, (double)v.y);
}
template <typename T>
__device__ __forceinline__ cx<T> t2(double2 v) {
  return mk<T>((T)v.x, (T)v.y);
}

// --------------------------------------------------------------------------
// Tridiagonal solve of one row by its WPR wavefronts, FP64.
//
// The system has identity first and last rows and constant interior bands
// (lower = upper = lo).  fc holds, for the thread's element i -- element t K
// + i of the row -- (cp, 1/den) of the Thomas factorisation, read by
// row_factors from the chunk-major tables (entry i * LR + t, LR = 64 WPR
// threads per row).
//   forward   d_j = (r_j - lower_j d_{j-1}) / den_j
//   backward  x_j = d_j - cp_j x_{j+1},  x_{nz-1} = d_{nz-1}
// Each recurrence is an affine map per element; a thread composes the maps
// of its chunk, a scan composes them across the lanes (affine_scan.hpp: DPP;
// with shuffles the row kernel took 21.4 us at 1024x513 FP32 predictor-
// corrector, 20.1 now; eight such jobs 77.9, now 75.9) and, through tot,
// across the wavefronts, and the thread then replays its chunk from the value
// entering it.  buf holds the right-hand side on entry and the solution on
// exit.
// --------------------------------------------------------------------------
template <int WPR>
__device__ __forceinline__ void row_sync() {
  if constexpr (WPR == 1)
    wave_sync();
  else
    __syncthreads();  // a block holds exactly one row
}

template <int KT, int WPR>
__device__ __forceinline__ void row_factors(double2 (&fc)[KT], gptr<const double2> fac, int K,
                                            int t) {
#pragma unroll
  for (int i = 0; i < KT; ++i) {
    fc[i] = make_double2(0.0, 1.0);
    if (i < K) fc[i] = fac[i * (64 * WPR) + t];
  }
}

// The value entering a thread's chunk: the wavefronts' maps before its own,
// then the lanes' before its own (BACK: after it).
template <int WPR, bool BACK>
__device__ __forceinline__ double2 row_scan(const Affine& m, Affine* __restrict__ tot, int t) {
  Affine all;
  const Affine e = wave_affine_scan<BACK>(m, all);
  double px = 0.0, py = 0.0;
  if constexpr (WPR > 1) {
    const int wv = t >> 6;
    if ((t & 63) == 0) tot[wv] = all;
    __syncthreads();
    auto step = [&](int w) {
      px = fma(tot[w].a, px, tot[w].x);
      py = fma(tot[w].a, py, tot[w].y);
    };
    if constexpr (BACK)
      for (int w = WPR - 1; w > wv; --w) step(w);
    else
      for (int w = 0; w < wv; ++w) step(w);
  }
  return make_double2(fma(e.a, px, e.x), fma(e.a, py, e.y));
}

template <int KT, int WPR>
__device__ __forceinline__ void row_tridiag(double2* __restrict__ buf, const double2 (&fc)[KT],
                                            double lo, int nz, int K, int t,
                                            Affine* __restrict__ tot) {
  const int j0 = t * K;
  double2 d[KT];
  Affine m = {1.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < KT; ++i) {
    const int j = j0 + i;
    d[i] = make_double2(0.0, 0.0);
    if (i < K && j < nz) {
      d[i] = buf[j];
      const double l = (j == 0 || j == nz - 1) ? 0.0 : lo;
      m = aff_after(Affine{-l * fc[i].y, d[i].x * fc[i].y, d[i].y * fc[i].y}, m);
    }
  }
  double2 p = row_scan<WPR, false>(m, tot, t);
  m = {1.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < KT; ++i) {
    const int j = j0 + i;
    if (i < K && j < nz) {
      const double l = (j == 0 || j == nz - 1) ? 0.0 : lo;
      p.x = d[i].x = (d[i].x - l * p.x) * fc[i].y;
      p.y = d[i].y = (d[i].y - l * p.y) * fc[i].y;
    }
  }
#pragma unroll
  for (int i = KT - 1; i >= 0; --i)
    if (i < K && j0 + i < nz) m = aff_after(Affine{-fc[i].x, d[i].x, d[i].y}, m);
  p = row_scan<WPR, true>(m, tot + WPR, t);
#pragma unroll
  for (int i = KT - 1; i >= 0; --i) {
    const int j = j0 + i;
    if (i < K && j < nz) {
      p.x = d[i].x - fc[i].x * p.x;
      p.y = d[i].y - fc[i].x * p.y;
      buf[j] = p;
    }
  }
}

// First z difference of the row in buf at j (pddz, SpatialDifferentiator.py:
// 91-104, 159-185): zero on the end points the stencil does not reach.
__device__ __forceinline__ double2 ddz_row(const double2* __restrict__ b, int j, int nz, int order,
                                           double ih) {
  if (order == 2) {
    if (j < 1 || j > nz - 2) return make_double2(0.0, 0.0);
    return make_double2((b[j + 1].x - b[j - 1].x) * ih, (b[j + 1].y - b[j - 1].y) * ih);
  }
  if (j < 2 || j > nz - 3) return make_double2(0.0, 0.0);
  return make_double2(
      (-0.25 * b[j + 2].x + 2.0 * b[j + 1].x - 2.0 * b[j - 1].x + 0.25 * b[j - 2].x) * ih,
      (-0.25 * b[j + 2].y + 2.0 * b[j + 1].y - 2.0 * b[j - 1].y + 0.25 * b[j - 2].y) * ih);
}

// Second z difference (pd2dz2, SpatialDifferentiator.py:106-128).
__device__ __forceinline__ double2 d2dz2_row(const double2* __restrict__ b, int j, int nz,
                                             int order, double idz2) {
  if (order == 2) {
    if (j < 1 || j > nz - 2) return make_double2(0.0, 0.0);
    return make_double2((b[j + 1].x - 2.0 * b[j].x + b[j - 1].x) * idz2,
                        (b[j + 1].y - 2.0 * b[j].y + b[j - 1].y) * idz2);
  }
  if (j < 2 || j > nz - 3) return make_double2(0.0, 0.0);
  const double c1 = -1.0 / 12, c2 = 4.0 / 3, c3 = -5.0 / 2;
  return make_double2(
      (c1 * b[j + 2].x + c2 * b[j + 1].x + c3 * b[j].x + c2 * b[j - 1].x + c1 * b[j - 2].x) * idz2,
      (c1 * b[j + 2].y + c2 * b[j + 1].y + c3 * b[j].y + c2 * b[j - 1].y + c1 * b[j - 2].y) * idz2);
}

// --------------------------------------------------------------------------
// Row kernel body: mode n, field f (0 omega, 1 T), by the row's WPR
// wavefronts (thread t of 64 WPR).  Element-wise work uses the coalesced
// layout j = t + 64 WPR i.  The row owns two LDS rows of FP64 complex
// values: buf (operands with neighbours, and the tridiagonal solves) and
// vrow (the state v_n the update starts from).
// --------------------------------------------------------------------------
template <typename T, int KT, int WPR>
__device__ __forceinline__ void fdz_row(const FdzJob<T>& J, int stage, int n, int f, int step,
                                        double2* __restrict__ buf, double2* __restrict__ vrow,
                                        int t, Affine* __restrict__ tot,
                                        const double2* __restrict__ tw64) {
  constexpr int LR = 64 * WPR;  // threads per row
  const int Z = J.nz, K = J.K;
  const int par = (J.par0 + step) & 1;
  const size_t row = (size_t)n * Z;
  const int order = J.fd_order;
  const int kw = order == 2 ? 1 : 2;  // width of the wall band
  const double dz = J.dz;
  const double ih = order == 2 ? 1.0 / (2.0 * dz) : 1.0 / (3.0 * dz);
  if (stage != FDZ_PROLOGUE) {
    const int q = J.q;
    const int cur = ring(J.curr0, step, q);
    const bool expl = J.scheme == MLV_FDZ_EXPLICIT;
    const int ws = stage == FDZ_CORR ? (cur + 1) % q : cur;  // ring slot written
    const int s1 = (ws + q - 1) % q, s2 = (ws + q - 2) % q, s3 = (ws + q - 3) % q;
    const size_t ssz = (size_t)J.nn * Z;
    cx<T>* __restrict__ hist = glb(J.hist[f]);
    const cx<T>* __restrict__ qx = glb(J.qw[2 * f]) + row;
    const cx<T>* __restrict__ qz = glb(J.qw[2 * f + 1]) + row;
    const cx<T>* __restrict__ vin = glb(J.state[par][f]) + row;
    const cx<T>* __restrict__ cin = J.comp[f] ? glb(J.comp[f]) + row : nullptr;
    const cx<T>* __restrict__ tsrc = glb(stage == FDZ_CORR ? J.star[1] : J.state[par][1]) + row;
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int j = t + LR * i;
      if (i < K && j < Z) {
        buf[j] = d2<T>(qz[j]);
        double2 v = d2<T>(vin[j]);
        if (cin) {
          const double2 c = d2<T>(cin[j]);
          v.x -= c.x;
          v.y -= c.y;
        }
        vrow[j] = v;
      }
    }
    double sx;  // modified wavenumber of the x difference, sin(2 pi n / nx) from the table
    {
      const int sh = LOG_NMAX - J.lognx;
      const double s1x = -tw64[n << sh].y;
      sx = order == 2 ? s1x / J.dx : (8.0 * s1x + tw64[(2 * n) << sh].y) / (6.0 * J.dx);
    }
    row_sync<WPR>();
    // -Pr Ra i (2 pi n / lx) T  (rayleigh_benard_convection.py:101-104)
    const double buoy = f == 0 ? J.Pr * J.Ra * (J.fx * (double)n) : 0.0;
    const double coeff = f == 0 ? J.Pr : 1.0;
    const double k2 = J.fx2 * (double)n * (double)n;  // -(2 pi n / lx)^2
    const double idz2 = 1.0 / (dz * dz);
    const double dt = J.dt;
    double2 inc[KT];
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int j = t + LR * i;
      inc[i] = make_double2(0.0, 0.0);
      if (i < K && j < Z) {
        const size_t e = row + j;
        // issue the global loads first
        const double2 a = d2<T>(qx[j]);
        const double2 t = f == 0 ? d2<T>(tsrc[j]) : make_double2(0.0, 0.0);
        const double2 h1 = d2<T>(hist[(size_t)s1 * ssz + e]);
        double2 h2 = make_double2(0.0, 0.0), h3 = make_double2(0.0, 0.0);
        if (q == 4) {
          h2 = d2<T>(hist[(size_t)s2 * ssz + e]);
          h3 = d2<T>(hist[(size_t)s3 * ssz + e]);
        }
        // advection N = -(i sx Qx + Dz Qz), buoyancy
        const double2 dd = ddz_row(buf, j, Z, order, ih);
        double2 h0 = make_double2(sx * a.y - dd.x, -(sx * a.x) - dd.y);
        h0.x += buoy * t.y;
        h0.y -= buoy * t.x;
        const double2 v = vrow[j];
        double2 lv = make_double2(0.0, 0.0);
        if (expl) {
          // diffusion added into the stored RHS (Integrator.py:53-56):
          // coeff * (sd2dx2 + pd2dz2) v
          const double2 dzz = d2dz2_row(vrow, j, Z, order, idz2);
          h0.x += coeff * (k2 * v.x + dzz.x);
          h0.y += coeff * (k2 * v.y + dzz.y);
        } else if (j > 0 && j < Z - 1) {
          // L v = -kx^2 v + second-order D2z v on interior points, 0 on walls
          lv = make_double2(k2 * v.x + (vrow[j + 1].x - 2.0 * v.x + vrow[j - 1].x) * idz2,
                            k2 * v.y + (vrow[j + 1].y - 2.0 * v.y + vrow[j - 1].y) * idz2);
        }
        hist[(size_t)ws * ssz + e] = t2<T>(h0);
        double2 E;
        if (stage == FDZ_CORR) {  // Adams-Moulton (Integrator.py:20-33)
          if (q == 2) {
            E = make_double2(dt / 2 * (h0.x + h1.x), dt / 2 * (h0.y + h1.y));
          } else {
            E = make_double2(dt / 24 * (9 * h0.x + 19 * h1.x - 5 * h2.x + h3.x),
                             dt / 24 * (9 * h0.y + 19 * h1.y - 5 * h2.y + h3.y));
          }
        } else {  // Adams-Bashforth (Integrator.py:5-18)
          if (q == 2) {
            E = make_double2(dt / 2 * (3 * h0.x - h1.x), dt / 2 * (3 * h0.y - h1.y));
          } else {
            E = make_double2(dt / 24 * (55 * h0.x - 59 * h1.x + 37 * h2.x - 9 * h3.x),
                             dt / 24 * (55 * h0.y - 59 * h1.y + 37 * h2.y - 9 * h3.y));
          }
        }
        inc[i] = expl ? E : make_double2(dt * coeff * lv.x + E.x, dt * coeff * lv.y + E.y);
      }
    }
    row_sync<WPR>();
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int j = t + LR * i;
      if (i < K && j < Z) buf[j] = inc[i];
    }
    if (!expl) {
      // increment form of the theta scheme:
      //   (I - a dt c L) delta = dt c L v + E,  v_new = v + delta
      double2 fd[KT];
      row_factors<KT, WPR>(fd, glb(J.fac[1 + f]) + (size_t)n * K * LR, K, t);
      row_sync<WPR>();
      row_tridiag<KT, WPR>(buf, fd, J.lo[1 + f], Z, K, t, tot);
    }
    row_sync<WPR>();
    // new state and wall writes (rayleigh_benard_convection.py:113-142);
    // buf[j] becomes -omega_new for the Poisson solve (same thread, same j)
    cx<T>* __restrict__ out = glb(stage == FDZ_PRED ? J.star[f] : J.state[par ^ 1][f]) + row;
    cx<T>* __restrict__ cout = (stage != FDZ_PRED && J.comp[f]) ? glb(J.comp[f]) + row : nullptr;
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int j = t + LR * i;
      if (i < K && j < Z) {
        const double2 dl = buf[j], v0 = vrow[j];
        double2 v = make_double2(v0.x + dl.x, v0.y + dl.y);
        bool wall;
        if (f == 0) {
          wall = n == 0 || j < kw || j >= Z - kw;
          if (wall) v = make_double2(0.0, 0.0);
        } else {
          wall = j < kw || j >= Z - kw;
          if (wall) v = make_double2((j < kw && n == 0) ? 1.0 : 0.0, 0.0);
        }
        const cx<T> hi = t2<T>(v);
        out[j] = hi;
        if (cout) {
          // value = hi - residual, with the residual rounded once
          cout[j] = wall ? czero<T>() : mk<T>((T)((double)hi.x - v.x), (T)((double)hi.y - v.y));
        }
        // the Poisson solve sees the value the next evaluation reads
        const double2 wv = (cout || sizeof(T) == 8) ? v : d2<T>(hi);
        buf[j] = make_double2(-wv.x, -wv.y);
      }
    }
  } else {
    const cx<T>* __restrict__ vin = glb(J.state[par][0]) + row;
    const cx<T>* __restrict__ cin = J.comp[0] ? glb(J.comp[0]) + row : nullptr;
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int j = t + LR * i;
      if (i < K && j < Z) {
        double2 w = d2<T>(vin[j]);
        if (cin) {
          const double2 c = d2<T>(cin[j]);
          w.x -= c.x;
          w.y -= c.y;
        }
        buf[j] = make_double2(-w.x, -w.y);
      }
    }
  }
  if (f != 0) return;
  // psi = solve(-omega) (utility.py:65, LaplacianSolver.py:70-78),
  // ux_s = -pddz(psi), uz_s = i kx psi (utility.py:66-79)
  double2 fp[KT];
  row_factors<KT, WPR>(fp, glb(J.fac[0]) + (size_t)n * K * LR, K, t);
  row_sync<WPR>();
  row_tridiag<KT, WPR>(buf, fp, J.lo[0], Z, K, t, tot + 2 * WPR);
  row_sync<WPR>();
  const int vs = stage == FDZ_PRED ? 2 : (stage == FDZ_PROLOGUE ? par : par ^ 1);
  cx<T>* __restrict__ ux = glb(J.vel[vs][0]) + row;
  cx<T>* __restrict__ uz = glb(J.vel[vs][1]) + row;
  cx<T>* __restrict__ ps = vs < 2 && J.psi[vs] ? glb(J.psi[vs]) + row : nullptr;
  const double kx = J.fx * (double)n;
#pragma unroll
  for (int i = 0; i < KT; ++i) {
    const int j = t + LR * i;
    if (i < K && j < Z) {
      const double2 p = buf[j];
      const double2 dd = ddz_row(buf, j, Z, order, ih);
      ux[j] = t2<T>(make_double2(-dd.x, -dd.y));
      uz[j] = t2<T>(make_double2(-(kx * p.y), kx * p.x));
      if (ps) ps[j] = (n == 0 || j < kw || j >= Z - kw) ? czero<T>() : t2<T>(p);
    }
  }
}

// Blocks of 128 threads: two rows of one wavefront, or one row of two.  One
// launch runs every job's rows, each wavefront taking the branch of its job's
// variant (fdz_row_var).  (A launch per variant left a batch of ragged sizes
// with up to five launches that each filled a fraction of the chip: six FP64
// jobs of nz 33 to 257 took 39.6 us of row kernels per step, 14.4 in one
// launch.  The kernel holds 124 VGPRs: reading all operands and factors up
// front costs 149 and a wavefront per SIMD, 81.8 against 75.9 us for eight jobs
// of 1024x513, with no gain for one.)
// VAR >= 0: a batch of one variant runs the kernel compiled for it alone, whose
// 68 to 98 VGPRs leave room for a wavefront or three more per SIMD (us per
// launch, all variants' kernel and its own: 100 FP32 jobs of 256x129 47.6 and
// 42.5, 16 of 2048x17 31.9 and 25.3, 64 of 256x257 96 and 85).
template <typename T, int VAR>
__global__ void __launch_bounds__(kFdzRowThreads)
    k_fdz_rows(const FdzJob<T>* __restrict__ jobs, FdzJob<T>* clock, const int* __restrict__ pref,
               int njobs, int phase, int step, const double2* __restrict__ tw64) {
  extern __shared__ char smem_raw[];
  __shared__ Affine tot[2 * 2 * 2];  // two solves, two directions, two wavefronts
  const int lb = xcd_logical(pref[njobs]);
  if (lb < 0) return;
  const int jb = find_job(pref, njobs, lb);
  const FdzJob<T>& J = jobs[jb];
  const int wpr = VAR >= 0 ? kFdzRowWpr[VAR < 0 ? 0 : VAR] : J.wpr, lr = 64 * wpr;
  const int rib = threadIdx.x / lr, t = threadIdx.x % lr;  // row in block, thread in row
  const int lw = (lb - pref[jb]) * fdz_rows_per_block(wpr) + rib;
  int stage, nwf;
  if (phase < 0) {
    stage = FDZ_PROLOGUE;
    nwf = 1;
  } else {
    stage = J.scheme == MLV_FDZ_PC ? (phase == 0 ? FDZ_PRED : FDZ_CORR) : FDZ_MAIN;
    nwf = 2;
  }
  if (phase == (J.scheme == MLV_FDZ_PC ? 1 : 0) && lb == pref[jb] && threadIdx.x == 0) {
    // t += dt after each loop (Simulation.py:199-209), through `clock` (the
    // same table as a plain pointer); this launch reads these two fields
    // through neither pointer
    clock[jb].t = clock[jb].t + J.dt;
    clock[jb].loops = clock[jb].loops + 1;
  }
  // (uniform over a block when wpr > 1: the block is one row)
  if (lw >= nwf * J.nn) return;
  const int n = lw / nwf, f = lw % nwf, zstride = J.nz | 1;
  double2* buf = reinterpret_cast<double2*>(smem_raw) + (size_t)(2 * rib) * zstride;
  double2* vrow = buf + zstride;
#define MLV_ROW(KT, WPR) fdz_row<T, KT, WPR>(J, stage, n, f, step, buf, vrow, t, tot, tw64)
  if constexpr (VAR >= 0) {
    MLV_ROW(kFdzRowKt[VAR], kFdzRowWpr[VAR]);
  } else if (wpr == 1) {
    if (J.K <= 1)
      MLV_ROW(1, 1);
    else if (J.K <= 2)
      MLV_ROW(2, 1);
    else
      MLV_ROW(4, 1);
  } else {
    if (J.K <= 4)
      MLV_ROW(4, 2);
    else
      MLV_ROW(6, 2);
  }
#undef MLV_ROW
}

// --------------------------------------------------------------------------
// Column kernel: PB pairs of adjacent z columns per block, the NT threads in
// four groups, one per field (ux, uz, omega, T).
//
// Two real sequences share one complex transform (a + i b).  The rounding
// of a transform is relative to the whole complex sequence, so the pair
// must hold values of similar size: omega is ~Ra times T once convection
// starts, and packing omega with T would bury T under omega's rounding.
// Each transform therefore pairs the same field at two adjacent z columns.
//
// A group transforms its field of the block's pairs in registers
// (fft_reg.hpp), leaves the values in LDS, forms one product and transforms
// that back: group 0 ux T', 1 uz T', 2 ux omega, 3 uz omega.  At up to 1024
// points a transform is one wavefront's, so the two block barriers around the
// exchange of the values are the only ones.  Consecutive threads take
// consecutive pairs, so a load covers PB pairs of a row; each mode is loaded
// once and goes through LDS to its points k and N - k (loaded at both points
// it would be twice as many scattered 16-byte reads).
// What bounds it: one chain of loads, two transforms and stores per block, at
// one block per CU for one 1024x513 job.  Per launch, against columns staged
// and transformed in LDS: 1024x513 FP32 20.4 -> 17.4 us, FP64 25.4 -> 21.7,
// 512x257 FP32 14.7 -> 9.0, 256x129 FP64 14.2 -> 8.8, 2048x600 FP64 60.5 ->
// 49.6; eight 1024x513 FP32 jobs 64.8 -> 55.9 (1.6 TB/s).  Three wavefronts
// per SIMD in single precision at up to 1024 points: a bound of four costs
// 66.9 instead of 64.6 us a step there.
// --------------------------------------------------------------------------
// Hides where p comes from, so that what is read through it again is read
// again: the compiler would keep the first transform's twiddles and the
// velocities' spectra (56 and 24 registers in single precision) to the end of
// the kernel, and spill them.
template <typename P>
__device__ __forceinline__ void opaque(P& p) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(p));
#endif
}

template <typename T>
struct ColPair {
  cx<T> a, b;  // two adjacent columns (aligned as one element only)
};

template <typename T, int LOGN, int NT>
__device__ __forceinline__ void fdz_cols_body(const FdzJob<T>& J, int local, int phase, int flags,
                                              int step, const cx<T>* tw, cx<T>* lds,
                                              T* __restrict__ tmean) {
#pragma clang fp contract(off)
  constexpr int N = 1 << LOGN, LOGE = fdz_loge(LOGN), E = 1 << LOGE, TPS = N / E;
  constexpr int GT = NT / 4, PB = GT / TPS;  // threads of a group, pairs of a block
  constexpr int REG = rf_len(LOGN, LOGE) * PB;
  constexpr int nn = (N - 1) / 3, KI = (nn + TPS - 1) / TPS;
  // synchronises a group's transforms: a wavefront's own, or the block's
  constexpr int ST = GT <= 64 ? 64 : NT;
  const int Z = J.nz;
  const int par = (J.par0 + step) & 1;
  const bool corr = J.scheme == MLV_FDZ_PC && phase == 1;
  const int vs = corr ? 2 : par;
  const int f = __builtin_amdgcn_readfirstlane(threadIdx.x / GT);
  const int g = threadIdx.x % GT, sub = g % PB, t = rf_thread<TPS>(g / PB);
  const int c0 = 2 * (local * PB + sub);  // the pair's first column
  const bool live = c0 < Z, two = c0 + 1 < Z;
  auto region = [&](int fld, int sb) { return lds + fld * REG + sb; };
  cx<T>* __restrict__ mine = region(f, sub);
  // The x mean of T, Tm(z) = Re T[kx=0], is O(1) (the conductive profile)
  // while the rest is small: transforming T whole in single precision would
  // spread Tm's rounding over every mode.  Tm is constant along x, so
  // F_x(u Tm) = Tm F_x(u) exactly; the transforms carry T - Tm and the
  // Tm u_s term is added per mode after the forward transform.
  const gptr<const cx<T>> tsrc = glb(corr ? J.star[1] : J.state[par][1]);
  gptr<const cx<T>> src =
      f < 2 ? glb(J.vel[vs][f]) : (f == 3 ? tsrc : glb(corr ? J.star[0] : J.state[par][0]));
  for (int c = threadIdx.x; c < 2 * PB; c += NT)
    if (2 * local * PB + c < Z) tmean[c] = tsrc[2 * local * PB + c].x;
  // A pair is one load of two elements; the last column of an odd row comes
  // with the one before it, and idle lanes read the row's first two.
  const int ld = !live ? 0 : (two ? c0 : c0 - 1);
  cx<T> ka[KI], kb[KI];
  auto load = [&] {
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const int k = t + i * TPS;
      const auto p = *reinterpret_cast<gptr<const ColPair<T>>>(src + (k < nn ? k : 0) * Z + ld);
      ka[i] = two ? p.a : p.b;
      kb[i] = p.b;
      // irfft ignores the imaginary part of the kx = 0 term
      if (k == 0) ka[i].y = kb[i].y = T(0);
    }
  };
  load();
#pragma unroll
  for (int i = 0; i < KI; ++i) {
    const int k = t + i * TPS;
    if (!live || (f == 3 && k == 0)) ka[i] = czero<T>();  // (T without its x mean)
    if (!two || (f == 3 && k == 0)) kb[i] = czero<T>();
    if (k == 0) {
      mine[0] = mk<T>(ka[i].x, kb[i].x);
    } else if (k < nn) {
      mine[rf_pad<LOGE>(t, i * TPS) * PB] = mk<T>(ka[i].x - kb[i].y, ka[i].y + kb[i].x);
      mine[rf_mirror<LOGN, LOGE>(t, i) * PB] = mk<T>(ka[i].x + kb[i].y, kb[i].x - ka[i].y);
    }
  }
  rf_sync<ST>();
  cx<T> v[E];
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int x = t + m * TPS;
    v[m] = czero<T>();
    if (x < nn || x > N - nn) v[m] = mine[rf_pad<LOGE>(t, m * TPS) * PB];
  }
  rf_sync<ST>();
  rf_fft<T, LOGN, LOGE, +1, PB, ST>(v, mine, t, tw);
  rf_sync<ST>();
#pragma unroll
  for (int m = 0; m < E; ++m) mine[rf_pad<LOGE>(t, m * TPS) * PB] = v[m];
  __syncthreads();
  const bool wp = (flags & kFdzWritePhys) && !corr;
  const bool dg = (flags & kFdzDiag) && !corr && J.loops % (flags >> kFdzDiagShift) == 0;
  if (wp || dg) {
    T mux = -INFINITY, muz = -INFINITY;  // NaN-propagating maxima, as np.max
    double ke = 0.0, ens = 0.0, flux = 0.0;
    for (int e = threadIdx.x; e < PB * N; e += NT) {
      const int sb = e % PB, x = e / PB, ca = 2 * (local * PB + sb), at = rf_pad<LOGE>(x) * PB;
      if (ca >= Z) continue;
      cx<T> q[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) q[c] = region(c, sb)[at];
      // real parts: the pair's first column, imaginary parts: its second
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        if (ca + r >= Z) continue;
        auto val = [&](int c) { return r ? q[c].y : q[c].x; };
        const T vx = val(0), vz = val(1), w = val(2), tt = val(3) + tmean[2 * sb + r];
        if (dg) {
          mux = nan_max(mux, vx);
          muz = nan_max(muz, vz);
          ke += (double)vz * (double)vz + (double)vx * (double)vx;
          ens += (double)w * (double)w;
          flux += (double)tt * (double)vz;
        }
        if (wp) {
          const size_t o = (size_t)x * Z + ca + r;
          const gptr<T> p0 = glb(J.phys[0]), p1 = glb(J.phys[1]), p2 = glb(J.phys[2]),
                        p3 = glb(J.phys[3]);
          if (p0) p0[o] = vx;
          if (p1) p1[o] = vz;
          if (p2) p2[o] = w;
          if (p3) p3[o] = tt;
        }
      }
    }
    if (dg)
      block_diag<NT>((double)mux, (double)muz, ke, ens, flux,
                     glb(J.diag) + (size_t)kDiagPart * local);
  }
  // the product: own value times T' (velocities), or ux / uz times omega
  {
    const cx<T>* __restrict__ pa = region(f == 3 ? 1 : 0, sub);
    const cx<T>* __restrict__ pb = region(f < 2 ? 3 : 2, sub);
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const int at = rf_pad<LOGE>(t, m * TPS) * PB;
      const cx<T> b = pb[at];
      cx<T> a = v[m];
      if (f >= 2) a = pa[at];
      v[m] = mk<T>(a.x * b.x, a.y * b.y);
    }
  }
  // every value is read before any transform writes over it
  __syncthreads();
  opaque(tw);
  rf_fft<T, LOGN, LOGE, -1, PB, ST>(v, mine, t, tw);
  rf_sync<ST>();
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int x = t + m * TPS;
    if (x < nn || x > N - nn) mine[rf_pad<LOGE>(t, m * TPS) * PB] = v[m];
  }
  rf_sync<ST>();
  if (f < 2) {
    opaque(src);
    load();
  }
  // group 0 Qx_T, 1 Qz_T, 2 Qx_omega, 3 Qz_omega
  const gptr<cx<T>> dst = glb(J.qw[f ^ 2]);
  const T hs = (T)(0.5 / (double)N);
  const T tm0 = tmean[2 * sub], tm1 = tmean[2 * sub + 1];
#pragma unroll
  for (int i = 0; i < KI; ++i) {
    const int k = t + i * TPS;
    if (!live || k >= nn) continue;
    // (y + conj ym) / 2 is the first column's spectrum, (y - conj ym) / 2i
    // the second's
    const cx<T> y = mine[rf_pad<LOGE>(t, i * TPS) * PB],
                ym = mine[rf_mirror<LOGN, LOGE>(t, i) * PB];
    ColPair<T> p;
    p.a = mk<T>(hs * (y.x + ym.x), hs * (y.y - ym.y));
    p.b = mk<T>(hs * (y.y + ym.y), hs * (ym.x - y.x));
    if (f < 2) {
      p.a = mk<T>(fma1(tm0, ka[i].x, p.a.x), fma1(tm0, ka[i].y, p.a.y));
      p.b = mk<T>(fma1(tm1, kb[i].x, p.b.x), fma1(tm1, kb[i].y, p.b.y));
    }
    if (two)
      *reinterpret_cast<gptr<ColPair<T>>>(dst + k * Z + c0) = p;
    else
      dst[k * Z + c0] = p.a;
  }
}

// NT = 512 runs the jobs of 2048 points, whose transforms take two
// wavefronts each, 256 all others (a job's blocks are in one of the two
// launches' prefix arrays).
template <typename T, int NT>
__global__ void __launch_bounds__(NT)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? (NT == 256 ? 3 : 4) : 2)))
    k_fdz_cols(const FdzJob<T>* __restrict__ jobs, const int* __restrict__ pref, int njobs,
               int phase, int flags, int step, const cx<T>* __restrict__ tw) {
  extern __shared__ char smem_raw[];
  __shared__ T tmean[2 * 64];  // two columns of at most 64 pairs
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int lb = xcd_logical(pref[njobs]);
  if (lb < 0) return;
  const int jb = find_job(pref, njobs, lb);
  const FdzJob<T>& J = jobs[jb];
  const int local = lb - pref[jb];
  switch (J.lognx) {
#define X(L)                                                                   \
  case L:                                                                      \
    if constexpr (fdz_col_threads(L) == NT)                                    \
      fdz_cols_body<T, L, NT>(J, local, phase, flags, step, tw, lds, tmean);   \
    break;
    X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11)
#undef X
    default:
      break;
  }
}

// Thomas factors of one job's operator for mode n, by lr = 64 wpr threads
// (FP64), in the row kernel's layout.
//   which = 0: Poisson, interior bands [1/dz^2, -(kx^2 + 2/dz^2), 1/dz^2]
//              (LaplacianSolver.py:21-52)
//   which > 0: theta diffusion, [-a/dz^2, 1 + a (kx^2 + 2/dz^2), -a/dz^2]
// First and last rows (and the padding up to lr K) are identity rows.  The
// table is chunk-major (entry i * lr + t is element t K + i): thread t
// computes its chunk [t K, t K + K) and stores entry i of it with the
// other threads' entries i, so each store instruction writes consecutive
// entries.  The interior recurrence cp_j = lo / (dg - lo cp_{j-1}) has
// constant coefficients: a thread runs it from the first row up to its
// chunk, stopping once it maps a value to itself in floating point (every
// later factor is then that value; diffusion gets there within a few dozen
// rows), and then through its chunk -- the same operations in the same
// order as a single sequential pass, so the table is bit-identical to one.
__device__ void fdz_factor_row(double2* __restrict__ fac, int n, int nz, int K, int lr,
                               double fxabs, double dz, int which, double a, int t) {
  gptr<double2> F = glb(fac) + (size_t)n * K * lr;
  const double k = (double)n * fxabs;
  const double k2 = k * k;
  const double idz2 = 1.0 / (dz * dz);
  double lo, dg;
  if (which == 0) {
    lo = idz2;
    dg = -(k2 + 2.0 / (dz * dz));
  } else {
    lo = -a * idz2;
    dg = 1.0 + a * (k2 + 2.0 / (dz * dz));
  }
  const int j0 = t * K;
  // factors of element j - 1 before element j (row 0: cp = 0)
  double cp = 0.0, rp = 0.0;
  for (int j = 1; j < j0 && j < nz - 1; ++j) {
    const double rd = 1.0 / (dg - lo * cp);
    const double c = lo * rd;
    const bool fixed = c == cp && rd == rp;
    cp = c;
    rp = rd;
    if (fixed) break;
  }
  for (int i = 0; i < K; ++i) {
    const int j = j0 + i;
    double2 v = make_double2(0.0, 1.0);  // identity rows and padding
    if (j >= 1 && j < nz - 1) {
      const double rd = 1.0 / (dg - lo * cp);
      const double c = lo * rd;
      cp = c;
      rp = rd;
      v = make_double2(c, rd);
    }
    F[i * lr + t] = v;
  }
}

// Grid: one block of lr threads per mode.
__global__ void __launch_bounds__(128) k_fdz_factors(double2* __restrict__ fac, int nn, int nz,
                                                     int K, int lr, double fxabs, double dz,
                                                     int which, double a) {
  if ((int)blockIdx.x < nn && (int)threadIdx.x < lr)
    fdz_factor_row(fac, blockIdx.x, nz, K, lr, fxabs, dz, which, a, threadIdx.x);
}

// One block per job: tracker record and CFL rule (diag_apply) from the
// column kernel's partials; a changed dt also moves the theta operators'
// interior bands and flags the job for k_fdz_refactor.
template <typename T>
__global__ void __launch_bounds__(kNT) k_fdz_diag(FdzJob<T>* jobs, double cutoff, int cadence) {
  FdzJob<T>& J = jobs[blockIdx.x];
  // loops has been advanced by this step's last row kernel
  if ((J.loops - 1) % cadence != 0) {
    if (threadIdx.x == 0) J.refactor = 0;
    return;
  }
  double dt = J.dt;
  const bool changed = diag_apply<kNT>(J.diag, J.nbC, J.dx, J.dz, (double)J.nx * (double)J.nz,
                                       true, cutoff, J.t, J.loops, dt);
  if (threadIdx.x == 0) {
    J.refactor = changed ? 1 : 0;
    if (changed) {
      const double idz2 = 1.0 / (J.dz * J.dz);
      J.dt = dt;
      J.lo[1] = -(J.alpha * dt * J.Pr) * idz2;
      J.lo[2] = -(J.alpha * dt * 1.0) * idz2;
    }
  }
}

// Theta tables of the jobs whose dt the last CFL update changed: grid
// (modes, jobs, 2 operators) of 128-thread blocks, 64 wpr of them used.
template <typename T>
__global__ void __launch_bounds__(128) k_fdz_refactor(const FdzJob<T>* __restrict__ jobs) {
  const FdzJob<T>& J = jobs[blockIdx.y];
  if (!J.refactor || J.scheme == MLV_FDZ_EXPLICIT || (int)threadIdx.x >= 64 * J.wpr) return;
  const int n = blockIdx.x;
  if (n >= J.nn) return;
  const int which = 1 + (int)blockIdx.z;
  const double a = J.alpha * J.dt * (which == 1 ? J.Pr : 1.0);
  fdz_factor_row(J.fac[which], n, J.nz, J.K, 64 * J.wpr, J.fx, J.dz, which, a, threadIdx.x);
}

template <typename T>
__global__ void k_fdz_set_dt(FdzJob<T>* jobs, int j, double dt, double lo_w, double lo_t) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    jobs[j].dt = dt;
    jobs[j].lo[1] = lo_w;
    jobs[j].lo[2] = lo_t;
  }
}

// --------------------------------------------------------------------------
// Host side
// --------------------------------------------------------------------------
template <typename T, int VAR>
static void launch_rows_var(const FdzJob<T>* jobs, const FdzLaunch& fl, int phase, int step,
                            hipStream_t s) {
  const int p = phase < 0 ? 2 : phase;
  MLV_SET_LDS_ONCE((k_fdz_rows<T, VAR>), fl.ldsrow);
  hipLaunchKernelGGL((k_fdz_rows<T, VAR>), dim3(xcd_grid(fl.nrow[p])), dim3(kFdzRowThreads),
                     fl.ldsrow, s, jobs, const_cast<FdzJob<T>*>(jobs), (const int*)fl.prefrow[p],
                     fl.njobs, phase, step, fl.tw64);
}

#define MLV_ROW_VARS(X) X(-1) X(0) X(1) X(2) X(3)

template <typename T>
static void launch_rows(const FdzJob<T>* jobs, const FdzLaunch& fl, int phase, int step,
                        hipStream_t s) {
  if (fl.nrow[phase < 0 ? 2 : phase] <= 0) return;
  switch (fl.rowvar) {
#define X(V) \
  case V: return launch_rows_var<T, V>(jobs, fl, phase, step, s);
    MLV_ROW_VARS(X)
#undef X
    default: break;
  }
}

// Column blocks of the jobs whose blocks have NT threads.
template <typename T, int NT>
static void launch_cols(const FdzJob<T>* jobs, const FdzLaunch& fl, int phase, int flags, int step,
                        const cx<T>* tw, hipStream_t s) {
  constexpr int w = NT >> 9;
  if (fl.ncol[w][phase] <= 0) return;
  MLV_SET_LDS_ONCE((k_fdz_cols<T, NT>), fl.ldscol[w]);
  hipLaunchKernelGGL((k_fdz_cols<T, NT>), dim3(xcd_grid(fl.ncol[w][phase])), dim3(NT),
                     fl.ldscol[w], s, jobs, (const int*)fl.prefcol[w][phase], fl.njobs, phase,
                     flags, step, tw);
}

template <typename T>
hipError_t fdz_phase(const FdzJob<T>* jobs, const FdzLaunch& fl, int phase, int flags, int step,
                     const cx<T>* tw, hipStream_t s, hipEvent_t* ev) {
  if (ev) (void)hipEventRecord(ev[0], s);
  launch_cols<T, 256>(jobs, fl, phase, flags, step, tw, s);
  launch_cols<T, 512>(jobs, fl, phase, flags, step, tw, s);
  if (ev) (void)hipEventRecord(ev[1], s);
  launch_rows<T>(jobs, fl, phase, step, s);
  if (ev) (void)hipEventRecord(ev[2], s);
  return hipGetLastError();
}

template <typename T>
hipError_t fdz_prologue(const FdzJob<T>* jobs, const FdzLaunch& fl, int step, hipStream_t s) {
  launch_rows<T>(jobs, fl, -1, step, s);
  return hipGetLastError();
}

hipError_t fdz_factors(double2* fac, int nn, int nz, int K, int wpr, double fxabs, double dz,
                       int which, double a, hipStream_t s) {
  hipLaunchKernelGGL(k_fdz_factors, dim3(nn), dim3(64 * wpr), 0, s, fac, nn, nz, K, 64 * wpr,
                     fxabs, dz, which, a);
  return hipGetLastError();
}

template <typename T>
hipError_t fdz_set_dt(FdzJob<T>* jobs, int job, double dt, double lo_w, double lo_t,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_fdz_set_dt<T>, dim3(1), dim3(64), 0, s, jobs, job, dt, lo_w, lo_t);
  return hipGetLastError();
}

template <typename T>
hipError_t fdz_diag(FdzJob<T>* jobs, int njobs, int max_nn, double cutoff, int cadence,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_fdz_diag<T>, dim3(njobs), dim3(kNT), 0, s, jobs, cutoff, cadence);
  hipLaunchKernelGGL(k_fdz_refactor<T>, dim3(max_nn, njobs, 2), dim3(kFdzRowThreads), 0, s,
                     (const FdzJob<T>*)jobs);
  return hipGetLastError();
}

template <typename T>
hipError_t fdz_prepare(const FdzLaunch& fl) {
  if (fl.ldscol[0]) MLV_SET_LDS_ONCE((k_fdz_cols<T, 256>), fl.ldscol[0]);
  if (fl.ldscol[1]) MLV_SET_LDS_ONCE((k_fdz_cols<T, 512>), fl.ldscol[1]);
  switch (fl.rowvar) {
#define X(V)                                             \
  case V:                                                \
    MLV_SET_LDS_ONCE((k_fdz_rows<T, V>), fl.ldsrow);     \
    break;
    MLV_ROW_VARS(X)
#undef X
    default: break;
  }
  return hipGetLastError();
}

template hipError_t fdz_phase<float>(const FdzJob<float>*, const FdzLaunch&, int, int, int,
                                     const cx<float>*, hipStream_t, hipEvent_t*);
template hipError_t fdz_phase<double>(const FdzJob<double>*, const FdzLaunch&, int, int, int,
                                      const cx<double>*, hipStream_t, hipEvent_t*);
template hipError_t fdz_prologue<float>(const FdzJob<float>*, const FdzLaunch&, int, hipStream_t);
template hipError_t fdz_prologue<double>(const FdzJob<double>*, const FdzLaunch&, int, hipStream_t);
template hipError_t fdz_set_dt<float>(FdzJob<float>*, int, double, double, double, hipStream_t);
template hipError_t fdz_set_dt<double>(FdzJob<double>*, int, double, double, double, hipStream_t);
template hipError_t fdz_diag<float>(FdzJob<float>*, int, int, double, int, hipStream_t);
template hipError_t fdz_diag<double>(FdzJob<double>*, int, int, double, int, hipStream_t);
template hipError_t fdz_prepare<float>(const FdzLaunch&);
template hipError_t fdz_prepare<double>(const FdzLaunch&);

}  // namespace mlv
