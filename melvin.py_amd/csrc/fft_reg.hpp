// Power-of-two FFT held in registers, with LDS as the exchange between
// passes only.
//
// E = 2^LOGE points per thread, TPS = N / E threads per transform; thread t
// holds the points t + m TPS, m < E, on entry and on exit, so a kernel loads
// its first pass straight from global memory and stores its last pass
// straight to it.  Between two passes the points go once through LDS.  The
// LDS engine in fft.hpp stages the input and the output there as well (two
// more trips) and holds 16 or 32 points per thread; here a transform spreads
// over two to four times as many threads, every global load of a thread is
// in flight at once, and a pass is a shorter chain, which is what one small
// or single transform waits for.
//
// Stockham autosort, decimation in time: pass p of radix R on sub-transforms
// of length Ns (the product of the earlier radices) takes the butterfly
// j = t + i TPS (i < E / R) from the points j + r N / R -- registers
// i + r E / R -- and leaves its outputs at (j - j % Ns) R + j % Ns + r Ns.
// In the last pass those are the points j + r N / R again.  The twiddles are
// the (Ns, R)-keyed tables of fft.hpp.
#pragma once
#include "fft.hpp"

namespace mlv {

// Passes, and the radix (log2) and sub-transform length (log2) of pass p:
// as few passes as the largest radix 2^logm allows, the larger radices
// first.  The radices alone decide a transform's rounding: two splits with
// the same logm give the same bits.
__host__ __device__ constexpr int rf_passes(int logn, int logm) { return (logn + logm - 1) / logm; }
__host__ __device__ constexpr int rf_logr(int logn, int logm, int p) {
  const int np = rf_passes(logn, logm);
  return logn / np + (p < logn % np ? 1 : 0);
}
__host__ __device__ constexpr int rf_logns(int logn, int logm, int p) {
  int s = 0;
  for (int i = 0; i < p; ++i) s += rf_logr(logn, logm, i);
  return s;
}
// LDS position of point i: one spare element every E, so the first
// exchange's writes (E consecutive points per thread) step by E + 1.
template <int LOGE>
__host__ __device__ constexpr int rf_pad(int i) {
  return i + (i >> LOGE);
}
// Position of point t + d, d a constant once unrolled.  A multiple of E moves
// the position by a constant, which becomes the access's immediate offset;
// as rf_pad(t + d) the compiler keeps a register per point (the 1024-point
// FP32 column pass of the FD-z step: 171 VGPRs, 126 so).
template <int LOGE>
__host__ __device__ constexpr int rf_pad(int t, int d) {
  return d % (1 << LOGE) == 0 ? rf_pad<LOGE>(t) + rf_pad<LOGE>(d) : rf_pad<LOGE>(t + d);
}
// Position of point -(t + m TPS) mod N, the mirror of a thread's point m.
template <int LOGN, int LOGE>
__host__ __device__ constexpr int rf_mirror(int t, int m) {
  constexpr int N = 1 << LOGN, TPS = N >> LOGE;
  return m == 0 && t == 0 ? 0 : rf_pad<LOGE>(TPS - t, N - (m + 1) * TPS);
}
// Position of the neighbour at distance |d| <= 2 of a thread's point m,
// periodic.
template <int LOGN, int LOGE>
__host__ __device__ constexpr int rf_near(int t, int m, int d) {
  constexpr int N = 1 << LOGN, TPS = N >> LOGE;
  const bool inside = m * TPS >= 2 && (m + 1) * TPS + 2 <= N;
  return inside ? rf_pad<LOGE>(t + d, m * TPS) : rf_pad<LOGE>((t + m * TPS + d) & (N - 1));
}
__host__ __device__ constexpr int rf_len(int logn, int loge) {
  return (1 << logn) + ((1 << logn) >> loge);
}

// A transform's thread among TPS, from its index.  Spelled out as 0 where it
// is the only one: with the index only known to be 0 from its range, the
// compiler drops n from the test "n == 0 and column 0" of a row n = t - 1 (the
// x inverse at 8 points: its assembly tests the column alone).
template <int TPS>
__device__ __forceinline__ int rf_thread(int t) {
  return TPS == 1 ? 0 : t;
}

// Synchronisation of the threads that share LDS: a block of one wavefront
// needs no barrier.
template <int NT>
__device__ __forceinline__ void rf_sync() {
  if constexpr (NT <= 64)
    wave_sync();
  else
    __syncthreads();
}

// DIR = -1 forward, +1 inverse, unnormalised.  lds is the transform's own
// region (element stride STRIDE: interleaved transforms pass lds + slot), t
// the thread in the transform, NT the threads that synchronise together.
// Before the call nobody still reads or writes the region; after it the last
// reads of the region may be pending (rf_sync before writing it again).
// IMM: positions at constant distances (two-argument rf_pad).
template <typename T, int LOGN, int LOGE, int DIR, int STRIDE, int NT,
          int LOGM = (LOGE < 4 ? LOGE : 4), bool IMM = true, int PASS = 0>
__device__ __forceinline__ void rf_fft(cx<T> (&v)[1 << LOGE], cx<T>* __restrict__ lds, int t,
                                       const cx<T>* __restrict__ tw) {
  constexpr int N = 1 << LOGN, E = 1 << LOGE, TPS = N / E;
  static_assert(LOGM <= LOGE && LOGM <= 4, "a butterfly is one thread's, radix 16 at most");
  constexpr int LOGR = rf_logr(LOGN, LOGM, PASS), R = 1 << LOGR;
  constexpr int LOGNS = rf_logns(LOGN, LOGM, PASS), NS = 1 << LOGNS;
  constexpr int B = E / R;  // butterflies per thread
  constexpr bool LAST = PASS == rf_passes(LOGN, LOGM) - 1;
  auto at = [](int i, int d) { return IMM ? rf_pad<LOGE>(i, d) : rf_pad<LOGE>(i + d); };
  cx<T> u[B][R];
#pragma unroll
  for (int i = 0; i < B; ++i) {
#pragma unroll
    for (int r = 0; r < R; ++r) u[i][r] = v[i + r * B];
    if constexpr (PASS > 0) {
      const int jm = (t + i * TPS) & (NS - 1);
      const cx<T>* __restrict__ w = tw + fft_keyed_table(LOGNS, LOGR) + jm;
#pragma unroll
      for (int r = 1; r < R; ++r) {
        cx<T> wr = w[(r - 1) * NS];
        if (DIR > 0) wr.y = -wr.y;
        u[i][r] = cmul<T>(u[i][r], wr);
      }
    }
    Dft<R, DIR, T>::run(u[i]);
  }
  if constexpr (LAST) {
#pragma unroll
    for (int i = 0; i < B; ++i)
#pragma unroll
      for (int r = 0; r < R; ++r) v[i + r * B] = u[i][r];
  } else {
    if constexpr (PASS > 0) rf_sync<NT>();  // the previous exchange's reads
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const int j = t + i * TPS;
      const int jm = j & (NS - 1);
      const int base = (j - jm) * R + jm;
#pragma unroll
      for (int r = 0; r < R; ++r) lds[at(base, r * NS) * STRIDE] = u[i][r];
    }
    rf_sync<NT>();
#pragma unroll
    for (int m = 0; m < E; ++m) v[m] = lds[at(t, m * TPS) * STRIDE];
    rf_fft<T, LOGN, LOGE, DIR, STRIDE, NT, LOGM, IMM, PASS + 1>(v, lds, t, tw);
  }
}

}  // namespace mlv
