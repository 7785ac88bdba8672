// Device bodies of the fused step's x-inverse kernel A (spectral prologue +
// inverse x pass) and, in the same launch, of its x-mean profiles
// (single precision).
#pragma once
#include "fused.hpp"
#include "diag_dev.hpp"
#include "grid.hpp"

namespace mlv {
// --------------------------------------------------------------------------
// Kernel A: spectral prologue + inverse x pass, NT threads per block, TC =
// NT / TPS columns: consecutive threads take consecutive columns, so that a
// store covers whole row pairs of the interleaved channel layout, and a
// load's lanes still read runs of 64 / TC consecutive rows of each column.
// What bounds it: at 16 x 1024^2 FP32 the 300 MB it moves, 70 us with the mean
// profiles (70 + 7.7 in a launch of their own before); on small grids the
// chain of one block: 256^2 FP64 8.0 -> 4.3 us, 1024^2 FP64 15.6 -> 12.5,
// 4 x 512^2 FP32 11.9 + 6.5 -> 9.4.
// --------------------------------------------------------------------------
// The spectral value of channel op at mode (n, m) from the field's f; ps
// receives psi = solve(-f) (utility.py:65, LaplacianSolver.py:64-66) where
// the op derives from it.
template <typename T>
__device__ __forceinline__ cx<T> xinv_value(int op, cx<T> f, int n, int m, const JobDev<T>& J,
                                            cx<T>& ps) {
#pragma clang fp contract(off)
  if (op == XOP_ID) return f;
  T rl, yz, yx;
  if constexpr (sizeof(T) == 8) {
    double lap = fma1(J.fx2, (double)(n * n), J.fz2 * (double)(m * m));
    if (n == 0 && m == 0) lap = 1.0;
    rl = 1.0 / lap;
    yz = J.fz * m;
    yx = J.fx * n;
  } else {
    // single precision: the symbol and its reciprocal in FP32 (hardware
    // reciprocal, 1 ulp) instead of an FP64 division
    float lap = fma1((float)J.fx2, (float)(n * n), (float)J.fz2 * (float)(m * m));
    if (n == 0 && m == 0) lap = 1.0f;
    rl = __builtin_amdgcn_rcpf(lap);
    yz = (float)J.fz * (float)m;
    yx = (float)J.fx * (float)n;
  }
  ps = mk<T>(-f.x * rl, -f.y * rl);
  // ux = -d(psi)/dz, uz = d(psi)/dx
  return op == XOP_UX ? mk<T>(yz * ps.y, -(yz * ps.x)) : mk<T>(-(yx * ps.y), yx * ps.x);
}

// MIXED (block shape 2): a block holds kMixCols columns of every op of the
// stage -- slot s is op s % nA of column c0 + s / nA -- so that the ops
// derived from one field read its columns once between them, where one op
// per block reads each column once per op; otherwise a block holds TC
// columns of one op, ops outermost, so that consecutive blocks write
// neighbouring tiles of one channel.
template <typename T, int LOGN, int NT, bool MIXED>
__device__ __forceinline__ void stepA_body(const JobDev<T>& J, const StageDev& S, int local,
                                           int par, const cx<T>* __restrict__ tw, cx<T>* lds) {
  constexpr int N = 1 << LOGN, LOGE = xp_loge<T>(LOGN), E = 1 << LOGE, TPS = N / E;
  constexpr int TC = NT / TPS;
  constexpr int nn = xp_nn(N), rows = 2 * nn + 1;
  const int nm = J.nm;
  const int c = threadIdx.x % TC, t = rf_thread<TPS>(threadIdx.x / TC);
  int opi, col;
  bool ok;
  if constexpr (MIXED) {
    opi = c % S.nA;
    col = local * kMixCols + c / S.nA;
    ok = c < kMixCols * S.nA && col < nm;
  } else {
    const int ntile = (nm + TC - 1) / TC;
    opi = local / ntile;
    col = (local % ntile) * TC + c;
    ok = col < nm;
  }
  const XinvOp op = S.a[opi];
  const cx<T>* __restrict__ src = glb(J.state[op.from_new ? (par ^ 1) : par][op.src]);
  cx<T>* __restrict__ dst = glb(J.work) + (size_t)op.ch * work_chs(N, nm);
  cx<T>* __restrict__ psi_out = (op.op == XOP_UX && op.src == 0 && !op.from_new) ? glb(J.psi) : nullptr;
  const uint32_t base = (uint32_t)(ok ? col : 0) * rows;
  cx<T> v[E];
#pragma unroll
  for (int m = 0; m < E; ++m) {
    v[m] = czero<T>();
    if (!xp_any(m, TPS, N)) continue;
    const int r = xp_row(t + m * TPS, N);
    if (ok && r >= 0) v[m] = at32(src, (base + r) * (uint32_t)sizeof(cx<T>));
  }
#pragma unroll
  for (int m = 0; m < E; ++m) {
    if (!xp_any(m, TPS, N)) continue;
    const int r = xp_row(t + m * TPS, N);
    if (ok && r >= 0) {
      cx<T> ps;
      v[m] = xinv_value<T>(op.op, v[m], r <= nn ? r : r - rows, col, J, ps);
      if (psi_out) at32(psi_out, (base + r) * (uint32_t)sizeof(cx<T>)) = ps;
      // single precision: the channel's x mean (its kx = 0 row) is carried
      // by the mean profiles, so the transforms see only the fluctuation and
      // round relative to it
      if (sizeof(T) == 4 && J.split && r == 0) v[m] = czero<T>();
    }
  }
  rf_fft<T, LOGN, LOGE, +1, TC, NT>(v, lds + c, t, tw);
  if (ok) {
#pragma unroll
    for (int m = 0; m < E; ++m)
      at32(dst, (uint32_t)(xrow_base(t + m * TPS, nm) + col * kXil) * (uint32_t)sizeof(cx<T>)) = v[m];
  }
}

// --------------------------------------------------------------------------
// Mean profiles (single precision): the x mean of each channel an x-inverse
// op of the stage writes, as a function of z -- the z c2r of the channel's
// kx = 0 coefficients -- into J.mean[op.ch * nz + n], one block per pair of
// ops.  Kernel A leaves the kx = 0 row out of the channels, so kernel B's
// products are formed from mean + fluctuation with the mean-times-mean part
// left out: its x difference is zero, and in z it vanishes because uz and bz
// have no x mean.  Without the split, an O(1) x-independent profile (a shear
// layer, a current sheet) puts FP32 rounding of its own size into products
// whose x differences should cancel exactly.
// The blocks read the same state as kernel A's and nothing reads both
// before kernel B, so they run in kernel A's launch: one of their own was 6
// to 8 us per stage of a chain that fills a fraction of the chip.
// --------------------------------------------------------------------------
template <typename T, int LOGN, int NT>
__device__ __forceinline__ void stepM_body(const JobDev<T>& J, const StageDev& S, int pair,
                                           int par, const cx<T>* __restrict__ tw, cx<T>* lds) {
  constexpr int N = 1 << LOGN;
  // eight points per thread, or as many as let the block hold the transform
  constexpr int LOGE = mean_loge(LOGN, NT), E = 1 << LOGE, TPS = N / E;
  const int o0 = 2 * pair;
  if (o0 >= S.nA) return;
  const bool hb = o0 + 1 < S.nA;
  const XinvOp oa = S.a[o0], ob = S.a[hb ? o0 + 1 : o0];
  constexpr int nm = xp_nn(N);
  const int rows = J.rows;
  const cx<T>* __restrict__ fa = glb(J.state[oa.from_new ? (par ^ 1) : par][oa.src]);
  const cx<T>* __restrict__ fb = glb(J.state[ob.from_new ? (par ^ 1) : par][ob.src]);
  // (threads beyond one transform's repeat it)
  const int t = threadIdx.x % TPS;
  cx<T> v[E];
#pragma unroll
  for (int m = 0; m < E; ++m) {
    const int x = t + m * TPS;
    const int k = 2 * x <= N ? x : N - x;
    v[m] = czero<T>();
    if (k < nm) {
      cx<T> ps;
      const cx<T> a = xinv_value<T>(oa.op, fa[(size_t)k * rows], 0, k, J, ps);
      const cx<T> b = hb ? xinv_value<T>(ob.op, fb[(size_t)k * rows], 0, k, J, ps) : czero<T>();
      v[m] = k == 0 ? mk<T>(a.x, b.x)
                    : (x == k ? mk<T>(a.x - b.y, a.y + b.x) : mk<T>(a.x + b.y, b.x - a.y));
    }
  }
  // (constant distances here cost the 16 x 1024^2 step 1375 us against 1358)
  rf_fft<T, LOGN, LOGE, +1, 1, NT, 3, false>(v, lds, t, tw);
  if ((int)threadIdx.x < TPS) {
    T* __restrict__ ma = glb(J.mean) + (size_t)oa.ch * N;
    T* __restrict__ mb = glb(J.mean) + (size_t)ob.ch * N;
#pragma unroll
    for (int m = 0; m < E; ++m) {
      ma[t + m * TPS] = v[m].x;
      if (hb) mb[t + m * TPS] = v[m].y;
    }
  }
}

}  // namespace mlv
