// Per-mode tridiagonal solve of the FD-z Poisson problem
// (LaplacianSolver.py:21-56, 70-78): for every x mode n the constant matrix
// with diagonal -((2*pi*n/lx)^2 + 2/dz^2), off-diagonals 1/dz^2 and identity
// wall rows, by Thomas's elimination with host-precomputed factors:
//   d_j = (r_j - l_j d_{j-1}) * (1/den_j),   x_j = d_j - c_j x_{j+1}.
// FP64 throughout; the state type only changes the load and store.
#include "affine_scan.hpp"
#include "common.hpp"
#include "grid.hpp"
#include "ops.hpp"

namespace mlv {

// One block per mode: thread t owns the K <= KT consecutive elements
// [t K, t K + K).  Both recurrences are affine maps per element; a thread
// composes its chunk's, a scan over the lanes (affine_scan.hpp) and over the
// wavefronts' totals gives the value entering the chunk, and the thread
// replays the chunk from it.  The row passes through LDS so that global
// loads and stores are contiguous; the factors are stored chunk-major
// (entry i NT + t of a row is element t K + i, see thomas_layout).
// What bounds it: the serial chain of a row.  One thread per mode (the
// serial kernel below) waits on a memory round trip per element, 330 us at
// 341 modes of 513 points in FP64; 6.5 us here (1.7 TB/s of its 11 MB).
// With uz, also i kx psi (the velocity of utility.py:66-79), whose separate
// pass cost 2.4 us.
template <typename T, int NT>
__global__ void __launch_bounds__(NT) k_thomas(const cx<T>* __restrict__ rhs,
                                               cx<T>* __restrict__ out, cx<T>* __restrict__ uz,
                                               const double2* __restrict__ fac, double lower,
                                               double sign, double fx, int nz, int K) {
  constexpr int KT = kThomasKT, NW = NT / 64;
  extern __shared__ char smem_raw[];
  double2* row = reinterpret_cast<double2*>(smem_raw);
  __shared__ Affine tot[2][NW];
  const int n = blockIdx.x, t = threadIdx.x, wv = t >> 6;
  const size_t base = (size_t)n * nz;
  const double2* __restrict__ f = fac + (size_t)n * NT * K + t;
  double2 fc[KT], d[KT];
#pragma unroll
  for (int i = 0; i < KT; ++i)
    if (i < K) fc[i] = f[i * NT];
  {
    cx<T> r[KT];
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int j = t + i * NT;
      if (j < nz) r[i] = rhs[base + j];
    }
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int j = t + i * NT;
      if (j < nz) row[j] = make_double2(sign * (double)r[i].x, sign * (double)r[i].y);
    }
  }
  __syncthreads();
  const int j0 = t * K;
  Affine m = {1.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < KT; ++i) {
    const int j = j0 + i;
    const bool ok = i < K && j < nz;
    d[i] = ok ? row[j] : make_double2(0.0, 0.0);
    if (ok) {
      const double l = (j == 0 || j == nz - 1) ? 0.0 : lower;
      m = aff_after(Affine{-l * fc[i].y, d[i].x * fc[i].y, d[i].y * fc[i].y}, m);
    }
  }
  Affine all;
  Affine e = wave_affine_scan<false>(m, all);
  if (NW > 1) {
    if ((t & 63) == 0) tot[0][wv] = all;
    __syncthreads();
  }
  double px = 0.0, py = 0.0;  // the value entering the wavefront, then the chunk
  if constexpr (NW > 1)
    for (int w = 0; w < wv; ++w) {
      px = fma(tot[0][w].a, px, tot[0][w].x);
      py = fma(tot[0][w].a, py, tot[0][w].y);
    }
  px = fma(e.a, px, e.x);
  py = fma(e.a, py, e.y);
  m = {1.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < KT; ++i) {
    const int j = j0 + i;
    if (i < K && j < nz) {
      const double l = (j == 0 || j == nz - 1) ? 0.0 : lower;
      px = d[i].x = (d[i].x - l * px) * fc[i].y;
      py = d[i].y = (d[i].y - l * py) * fc[i].y;
    }
  }
#pragma unroll
  for (int i = KT - 1; i >= 0; --i)
    if (i < K && j0 + i < nz) m = aff_after(Affine{-fc[i].x, d[i].x, d[i].y}, m);
  e = wave_affine_scan<true>(m, all);
  if (NW > 1) {
    if ((t & 63) == 0) tot[1][wv] = all;
    __syncthreads();
  }
  px = py = 0.0;
  if constexpr (NW > 1)
    for (int w = NW - 1; w > wv; --w) {
      px = fma(tot[1][w].a, px, tot[1][w].x);
      py = fma(tot[1][w].a, py, tot[1][w].y);
    }
  px = fma(e.a, px, e.x);
  py = fma(e.a, py, e.y);
#pragma unroll
  for (int i = KT - 1; i >= 0; --i) {
    const int j = j0 + i;
    if (i < K && j < nz) {
      px = d[i].x - fc[i].x * px;
      py = d[i].y - fc[i].x * py;
      row[j] = make_double2(px, py);
    }
  }
  __syncthreads();
  const T y = (T)(fx * n);
#pragma unroll
  for (int i = 0; i < KT; ++i) {
    const int j = t + i * NT;
    if (j < nz) {
      const double2 v = row[j];
      const cx<T> p = mk<T>((T)v.x, (T)v.y);
      out[base + j] = p;
      if (uz) uz[base + j] = mk<T>(-(y * p.y), y * p.x);
    }
  }
}

// Rows longer than a block's threads hold (thomas_layout): one thread per
// mode sweeps its row; factors row-major.  uz is not formed here: the store
// lengthens each step of the sweep (64 x 5000 FP64 1881 -> 1954 us), a pass of
// its own is short beside it.
template <typename T>
__global__ void __launch_bounds__(64) k_thomas_serial(const cx<T>* __restrict__ rhs,
                                                      cx<T>* __restrict__ out,
                                                      double2* __restrict__ dwork,
                                                      const double2* __restrict__ fac,
                                                      double lower, double sign, int nn, int nz) {
  const int n = blockIdx.x * 64 + threadIdx.x;
  if (n >= nn) return;
  const size_t row = (size_t)n * nz;
  double2 d = make_double2(0.0, 0.0);
  for (int j = 0; j < nz; ++j) {
    const cx<T> r = rhs[row + j];
    const double l = (j == 0 || j == nz - 1) ? 0.0 : lower;
    const double s = fac[row + j].y;
    d = make_double2((sign * (double)r.x - l * d.x) * s, (sign * (double)r.y - l * d.y) * s);
    dwork[row + j] = d;
  }
  double2 x = make_double2(0.0, 0.0);
  for (int j = nz - 1; j >= 0; --j) {
    const double c = fac[row + j].x;
    const double2 dj = dwork[row + j];
    x = make_double2(dj.x - c * x.x, dj.y - c * x.y);
    out[row + j] = mk<T>((T)x.x, (T)x.y);
  }
}

template <typename T, int NT>
static void launch_nt(const void* rhs, void* out, void* uz, const double2* fac, double lower,
                      double sign, double fx, int nn, int nz, int K, hipStream_t s) {
  // (rows near 4096 points take over 64 KB with the wavefronts' totals)
  const size_t lds = (size_t)nz * sizeof(double2);
  MLV_SET_LDS_ONCE((&k_thomas<T, NT>), lds);
  hipLaunchKernelGGL((k_thomas<T, NT>), dim3(nn), dim3(NT), lds, s, (const cx<T>*)rhs, (cx<T>*)out,
                     (cx<T>*)uz, fac, lower, sign, fx, nz, K);
}

template <typename T>
hipError_t launch_thomas(const void* rhs, void* out, void* uz, void* dwork, const double2* fac,
                         double lower, double sign, double fx, int nn, int nz, hipStream_t s) {
  int nt, K;
  thomas_layout(nz, &nt, &K);
  switch (nt) {
    case 64: launch_nt<T, 64>(rhs, out, uz, fac, lower, sign, fx, nn, nz, K, s); break;
    case 128: launch_nt<T, 128>(rhs, out, uz, fac, lower, sign, fx, nn, nz, K, s); break;
    case 256: launch_nt<T, 256>(rhs, out, uz, fac, lower, sign, fx, nn, nz, K, s); break;
    case 512: launch_nt<T, 512>(rhs, out, uz, fac, lower, sign, fx, nn, nz, K, s); break;
    case 1024: launch_nt<T, 1024>(rhs, out, uz, fac, lower, sign, fx, nn, nz, K, s); break;
    default:
      hipLaunchKernelGGL(k_thomas_serial<T>, dim3((nn + 63) / 64), dim3(64), 0, s,
                         (const cx<T>*)rhs, (cx<T>*)out, (double2*)dwork, fac, lower, sign, nn, nz);
  }
  return hipGetLastError();
}

template hipError_t launch_thomas<float>(const void*, void*, void*, void*, const double2*, double,
                                         double, double, int, int, hipStream_t);
template hipError_t launch_thomas<double>(const void*, void*, void*, void*, const double2*, double,
                                          double, double, int, int, hipStream_t);

}  // namespace mlv
