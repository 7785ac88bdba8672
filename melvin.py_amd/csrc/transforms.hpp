// Host-side launchers for the spectral transform kernels.
#pragma once
#include <hip/hip_runtime.h>
#include "fft.hpp"
#include "fft_reg.hpp"

namespace mlv {

// Threads per block of the fused steps' FFT-carrying kernels.
constexpr int kNT = 256;

// The operator-level transforms' split (fft_reg.hpp): log2 of the points per
// thread, 8 up to 1024 points and 16 above.  At 4096 a block of four columns
// would pass 1024 threads with 8; at 2048 they measure no better (us per
// launch, 16 and 8: 2048 x 1024 FP32 inverse 8.6 and 8.6, forward 7.8 and 7.8,
// 2048^2 FP64 14.6 and 15.3, 11.8 and 13.0; 4096 columns FP32 22.2 and 25.0).
__host__ __device__ constexpr int tr_loge(int logn) { return logn >= 11 ? 4 : 3; }
// LDS of `slots` transforms of 2^logn points.
template <typename T>
constexpr size_t tr_lds_bytes(int logn, int slots) {
  return (size_t)slots * rf_len(logn, tr_loge(logn)) * sizeof(cx<T>);
}
// Columns per block of the x passes at least: `least`, or as many as fill a
// wavefront.
__host__ __device__ constexpr int tr_cols(int logn, int least) {
  const int fill = 64 >> (logn - tr_loge(logn));
  return fill > least ? fill : least;
}
// The most LDS a transform along x / z of a plan takes.
template <typename T>
inline size_t tr_lds_max(int logn) {
  return tr_lds_bytes<T>(logn, tr_cols(logn, sizeof(T) == 4 ? 4 : 2));
}

// A list of up to two arrays that one launch transforms.
struct Two {
  const void* in[2];
  void* out[2];
  int n;
};
// psi = solve(-w), ux = -d(psi)/dz, uz = d(psi)/dx as the x pass's input.
struct VelArgs {
  const void* w;
  void *psi, *ux, *uz;  // spectra written
  double fx, fz, fx2, fz2;
};
// pddx(ux f) + pddz(uz f) as a forward transform's input
// (Variable.py:125-127).
struct FluxArgs {
  const void *ux, *uz, *f;
  int order, zper;
  double dx, dz;
};

// The 2-D transforms' intermediate (between the x and the z pass) holds x
// rows in pairs interleaved by kz where `pairs` is set: element (x, k) at
// (x / 2) 2 nm + 2 k + x % 2 of an (nx, nm) array; otherwise (and for a
// transform along z alone) it is row-major.
//
// nrow: rows of the x-pass spectrum (default 2 nn + 1, the compact layout;
// nx for a full spectrum, rows in FFT order); scale multiplies the input
// of launch_xinv and the outputs of the c2r passes.
template <typename T>
hipError_t launch_xinv(int logn, const void* in, void* out, int nn, int nm, const void* tw,
                       hipStream_t s, int nrow = -1, double scale = 1.0);
// ux and uz intermediates (out, and out + nx nm) of a vorticity spectrum.
template <typename T>
hipError_t launch_xinv_vel(int logn, const VelArgs& a, void* out, int nn, int nm, const void* tw,
                           hipStream_t s);
template <typename T>
hipError_t launch_xfwd(int logn, const void* in, void* out, int nn, int nm, double scale,
                       const void* tw, hipStream_t s, int nrow = -1);
template <typename T>
hipError_t launch_zc2r(int logn, const Two& a, int nx, int nm, const void* tw, hipStream_t s,
                       double scale = 1.0, bool pairs = true);
template <typename T>
hipError_t launch_zr2c(int logn, const void* in, void* out, int nx, int nm, const void* tw,
                       hipStream_t s, bool pairs = true);
template <typename T>
hipError_t launch_zr2c_flux(int logn, const FluxArgs& a, void* out, int nx, int nm, const void* tw,
                            hipStream_t s);
template <typename T>
hipError_t launch_xc2r_cols(int logn, const Two& a, int nn, int nz, const void* tw, hipStream_t s,
                            double scale = 1.0);
template <typename T>
hipError_t launch_xr2c_cols(int logn, const void* in, void* out, int nn, int nz, double scale,
                            const void* tw, hipStream_t s);
template <typename T>
hipError_t launch_xr2c_cols_flux(int logn, const FluxArgs& a, void* out, int nn, int nz,
                                 double scale, const void* tw, hipStream_t s);

}  // namespace mlv
