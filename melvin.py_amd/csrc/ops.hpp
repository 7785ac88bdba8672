// Host-side launchers and enums of the element-wise operator kernels.
#pragma once
#include <hip/hip_runtime.h>
#include "common.hpp"
#include "../../include/melvin_hip.h"

namespace mlv {

// internal spectral kind: out += d2/dx2(in) (FD-z snabla2)
constexpr int kSpecAddD2dx2 = 100;

// real: bit 0 / bit 1 make the x / z first-derivative factor real (sine and
// cosine bases) instead of i times the factor (complex exponentials)
template <typename T>
hipError_t launch_spec(const void* in, void* out, int rows, int cols, int nn, int fully, int kind,
                       double fx, double fz, double fx2, double fz2, hipStream_t s,
                       int real = 0);
// Batched dense complex matrix-vector products, out[b, k] = sum_j M[k, j] in[b, j]
// (M row-major K x J); the input may be real, the output reduced to its real
// part.  Strides in elements.
template <typename T>
hipError_t launch_dense(const void* M, int K, int J, int batch, const void* in, int in_cplx,
                        long long in_sb, long long in_sj, void* out, int out_real,
                        long long out_sb, long long out_sk, hipStream_t s);
template <typename T>
hipError_t launch_update(void* var, void* hist, const void* lin, size_t n, int q, int curr,
                         int scheme, double c1, double c2, double h, hipStream_t s);
template <typename T>
hipError_t launch_fd(const void* in, void* out, int rows, int cols, int comp, int kind, int order,
                     int periodic, double h, hipStream_t s);
template <typename T>
hipError_t launch_flux(const void* ux, const void* uz, const void* f, void* out, int nx, int nz,
                       int order, int xper, int zper, double dx, double dz, hipStream_t s);
// Blocks of the first reduction stage at most (one (sum, compensation) pair
// of partials each); the partials buffer holds 2 * kRedBlocks doubles.
constexpr int kRedBlocks = 1024;
template <typename T>
hipError_t launch_reduce(const void* a, const void* b, size_t n, int op, double scale,
                         double* part, double* out, hipStream_t s);
size_t reduce_partials_bytes();
template <typename T>
hipError_t launch_combine(const void* hist, void* out, size_t n, int q, int curr, int moulton,
                          double h, hipStream_t s);
template <typename T>
hipError_t launch_velocity(const void* w, void* psi, void* ux, void* uz, int rows, int cols, int nn,
                           double fx, double fz, double fx2, double fz2, hipStream_t s);
// Tridiagonal Poisson solve per x mode: out = solve(sign rhs) and, with uz
// (rows of a block, nt > 0, only), uz = i fx n out.  fac holds (cp_j, 1/den_j) per element, rows of K nt
// entries in the chunk-major layout of thomas_layout(nz) -- entry i nt + t is
// element t K + i, padding (0, 1) -- or row-major where nt = 0 (dwork then
// holds (nn, nz) complex128).
template <typename T>
hipError_t launch_thomas(const void* rhs, void* out, void* uz, void* dwork, const double2* fac,
                         double lower, double sign, double fx, int nn, int nz, hipStream_t s);
// Threads per row and elements per thread of the solve: the fewest threads
// that hold the row at kThomasKT elements each (about as many wavefronts as
// the modes of one plan leave the chip room for), 0 threads for rows beyond
// 1024 threads' reach, which one thread per mode sweeps.
constexpr int kThomasKT = 4;
inline void thomas_layout(int nz, int* nt, int* K) {
  int n = 64;
  while (n <= 1024 && n * kThomasKT < nz) n *= 2;
  *nt = n <= 1024 ? n : 0;
  *K = n <= 1024 ? (nz + n - 1) / n : 0;
}

}  // namespace mlv
