// Operator-level spectral transforms (the SpectralTransformer mirror).
//
// Fully spectral 2-D, spectral (2nn+1, nm) <-> physical (nx, nz):
//   to_physical = k_xinv   (x pass: zero-pad rows to nx, inverse c2c along x)
//                 k_zc2r   (z pass: Hermitian-extend nm columns, inverse along z)
//   to_spectral = k_zr2c   (z pass: forward along z, keep kz < nm)
//                 k_xfwd   (x pass: forward along x, keep |kx| <= nn, scale)
// The intermediate between the passes is the only workspace.  Zero padding
// and truncation never touch memory.
//
// Fourier-x / FD-z, spectral (nn, nz) <-> physical (nx, nz):
//   k_xc2r_cols / k_xr2c_cols: one pass over z-column pairs along x.
//
// Real transforms pack two real sequences into one complex transform
// (rows x, x+1 for the z pass; columns z, z+1 for the FD-z x pass).  As in
// numpy's c2r, the imaginary parts of each sequence's DC bin and, when the
// input holds it, its Nyquist bin are ignored.
//
// The same kernels give numpy.fft's rfft / irfft / rfft2 / irfft2 (full
// half-spectra, unnormalised forward, 1/n inverse): nm = nz/2 + 1 or
// nn = nx/2 + 1 bins, and the x passes over all nx rows (nrow = nx).
//
// What bounds them: a plan's arrays are a few MB and stay in the caches, so
// a pass is the chain of one block -- its loads, the transform's exchanges,
// its stores -- times the blocks a CU gets.  Each transform is therefore
// spread over N/8 (N/16 from 2048 points) threads with every load in flight
// at once and only the exchanges between passes in LDS (fft_reg.hpp), and a
// block holds few transforms, so that even 256^2 spreads over the chip.
// Measured against the LDS-staged blocks of 16 or 32 points per thread used
// before (us per launch): 1024^2 FP64 x inverse 13.9 -> 7.2, z c2r 10.6 ->
// 5.7, x forward 13.3 -> 5.4, z r2c behind a separate flux pass 14.1 + 10.0
// -> 12.5; 256^2 FP64 10.0 -> 3.7, 8.5 -> 3.6, 9.1 -> 3.8, 11.0 + 4.0 -> 5.1;
// 2048x1024 FP32 21.3 -> 10.0, 10.6 -> 6.4, 20.3 -> 7.5, 12.7 -> 7.9.
#include "transforms.hpp"
#include "grid.hpp"

namespace mlv {

// --------------------------------------------------------------------------
// x passes: TC columns per block, consecutive threads on consecutive columns
// --------------------------------------------------------------------------
template <int LOGN, int TC>
struct XShape {
  static constexpr int N = 1 << LOGN, LOGE = tr_loge(LOGN), E = 1 << LOGE, TPS = N / E;
  static constexpr int C = tr_cols(LOGN, TC), NT = C * TPS;
};

// rows of a compact (nrow < N) or full spectrum <-> x, -1 for a zero row
__device__ __forceinline__ int x_row(int x, int N, int nn, int nrow) {
  return x <= nn ? x : (x >= N - nn ? x - N + nrow : -1);
}
__device__ __forceinline__ size_t pair_at(int x, int k, int nm) {
  return (size_t)(x >> 1) * (2 * (size_t)nm) + 2 * (size_t)k + (x & 1);
}

template <typename T, int LOGN, int TC>
__global__ void __launch_bounds__((XShape<LOGN, TC>::NT))
    k_xinv(const cx<T>* __restrict__ in, cx<T>* __restrict__ out, int nn, int nrow, int nm, T scale,
           const cx<T>* __restrict__ tw, int ntile) {
  using S = XShape<LOGN, TC>;
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int tile = xcd_logical(ntile);
  if (tile < 0) return;
  const int c = threadIdx.x % S::C, t = rf_thread<S::TPS>(threadIdx.x / S::C);
  const int col = tile * S::C + c;
  cx<T> v[S::E];
#pragma unroll
  for (int m = 0; m < S::E; ++m) {
    const int r = x_row(t + m * S::TPS, S::N, nn, nrow);
    v[m] = (col < nm && r >= 0) ? in[(size_t)r * nm + col] : czero<T>();
  }
#pragma unroll
  for (int m = 0; m < S::E; ++m) v[m] = cscale<T>(v[m], scale);
  rf_fft<T, LOGN, S::LOGE, +1, S::C, S::NT>(v, lds + c, t, tw);
  if (col < nm) {
#pragma unroll
    for (int m = 0; m < S::E; ++m) out[pair_at(t + m * S::TPS, col, nm)] = v[m];
  }
}

// The velocity's x pass from the vorticity (utility.py:62-79 with
// LaplacianSolver.py:58-68): blockIdx.y = 0 writes psi and the ux spectrum
// and transforms ux, 1 writes the uz spectrum and transforms uz.  Separate
// passes would read w, psi, ux and uz again and take three more launches.
template <typename T, int LOGN, int TC>
__global__ void __launch_bounds__((XShape<LOGN, TC>::NT))
    k_xinv_vel(const cx<T>* __restrict__ w, cx<T>* __restrict__ psi, cx<T>* __restrict__ ux,
               cx<T>* __restrict__ uz, cx<T>* __restrict__ out, int nn, int nm, double fx,
               double fz, double fx2, double fz2, const cx<T>* __restrict__ tw, int ntile) {
  // the operators round as the reference's expressions do
#pragma clang fp contract(off)
  using S = XShape<LOGN, TC>;
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int tile = xcd_logical(ntile);
  if (tile < 0) return;
  const int c = threadIdx.x % S::C, t = rf_thread<S::TPS>(threadIdx.x / S::C);
  const int col = tile * S::C + c, rows = 2 * nn + 1;
  const bool isz = blockIdx.y != 0;
  cx<T> v[S::E];
#pragma unroll
  for (int m = 0; m < S::E; ++m) {
    const int r = x_row(t + m * S::TPS, S::N, nn, rows);
    v[m] = (col < nm && r >= 0) ? w[(size_t)r * nm + col] : czero<T>();
  }
#pragma unroll
  for (int m = 0; m < S::E; ++m) {
    const int r = x_row(t + m * S::TPS, S::N, nn, rows);
    if (col < nm && r >= 0) {
      const size_t e = (size_t)r * nm + col;
      const int n = r <= nn ? r : r - rows;
      double lap = fx2 * (double)(n * n) + fz2 * (double)(col * col);
      if (r == 0 && col == 0) lap = 1.0;
      const double rl = 1.0 / lap;
      const cx<T> p = mk<T>((T)(-(double)v[m].x * rl), (T)(-(double)v[m].y * rl));
      if (isz) {
        const T y = (T)(fx * n);
        v[m] = mk<T>(-(y * p.y), y * p.x);
        uz[e] = v[m];
      } else {
        const T y = (T)(fz * col);
        v[m] = mk<T>(y * p.y, -(y * p.x));
        psi[e] = p;
        ux[e] = v[m];
      }
    }
  }
  rf_fft<T, LOGN, S::LOGE, +1, S::C, S::NT>(v, lds + c, t, tw);
  if (col < nm) {
    cx<T>* __restrict__ o = out + (isz ? (size_t)S::N * nm : 0);
#pragma unroll
    for (int m = 0; m < S::E; ++m) o[pair_at(t + m * S::TPS, col, nm)] = v[m];
  }
}

template <typename T, int LOGN, int TC>
__global__ void __launch_bounds__((XShape<LOGN, TC>::NT))
    k_xfwd(const cx<T>* __restrict__ in, cx<T>* __restrict__ out, int nn, int nrow, int nm, T scale,
           const cx<T>* __restrict__ tw, int ntile) {
  using S = XShape<LOGN, TC>;
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int tile = xcd_logical(ntile);
  if (tile < 0) return;
  const int c = threadIdx.x % S::C, t = rf_thread<S::TPS>(threadIdx.x / S::C);
  const int col = tile * S::C + c;
  cx<T> v[S::E];
#pragma unroll
  for (int m = 0; m < S::E; ++m)
    v[m] = col < nm ? in[pair_at(t + m * S::TPS, col, nm)] : czero<T>();
  rf_fft<T, LOGN, S::LOGE, -1, S::C, S::NT>(v, lds + c, t, tw);
#pragma unroll
  for (int m = 0; m < S::E; ++m) {
    // (a full spectrum's Nyquist row is x = nn: x_row takes the first case)
    const int r = x_row(t + m * S::TPS, S::N, nn, nrow);
    if (col < nm && r >= 0) out[(size_t)r * nm + col] = cscale<T>(v[m], scale);
  }
}

// --------------------------------------------------------------------------
// z passes: TPS threads per row pair
// --------------------------------------------------------------------------
template <int LOGN>
struct ZShape {
  static constexpr int N = 1 << LOGN, LOGE = tr_loge(LOGN), E = 1 << LOGE, TPS = N / E;
  static constexpr int SL = TPS >= 64 ? 1 : 64 / TPS, NT = SL * TPS;
  static constexpr int LDSN = rf_len(LOGN, LOGE);
  // LDS elements a row pair: the transform's, or (STAGED) its coefficients,
  // at most N + 2, or its points, padded
  static constexpr int slot(bool staged) { return staged && N + 2 > LDSN ? N + 2 : LDSN; }
};
// Launches of many rows of at most 32 points (STAGED) pass them through LDS
// on their way in and out: a wavefront holds 32 to 128 of them, and with each
// thread loading its own row's points a load touches as many lines as it has
// lanes.  Below this many rows the two more trips cost more than the lines
// (us per launch, direct and staged, FP64 c2r, then FP32 r2c: 2^16 rows of 8
// points 5.1 and 5.3, 5.0 and 4.2; of 16 7.3 and 6.6, 6.4 and 5.1; of 32 10.2
// and 9.8, 6.5 and 6.2; 2^19 rows of 8 points 38 and 14, 21 and 8; 2^14 rows
// 3.4 and 4.8, 3.3 and 3.8).
constexpr int kStagedRows = 65536;
template <int LOGN>
static bool staged_rows(int rows) {
  return LOGN <= 5 && rows >= kStagedRows;
}

// Position in LDS of the point n of row r of pair sl, rows of 2^LOGN points:
// one spare element a pair, so that lanes on consecutive pairs differ in bank.
template <int LOGN>
__device__ __forceinline__ int pts_at(int sl, int r, int n) {
  return sl * (2 << LOGN) + sl + (r << LOGN) + n;
}
// A block's run of `n` elements, at most MOST, between memory and LDS (PAD:
// with the spare element after every 2^PAD), all of a thread's loads in
// flight at once.
template <int MOST, int NT, int PAD, typename V>
__device__ __forceinline__ void run_load(const V* __restrict__ p, V* __restrict__ lds, int n) {
  constexpr int IT = (MOST + NT - 1) / NT;
  V v[IT];
  // (unconditional, clamped: predicated element by element they are waited
  // for one by one)
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int e = threadIdx.x + i * NT;
    v[i] = p[e < n ? e : 0];
  }
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int e = threadIdx.x + i * NT;
    if (e < n) lds[PAD > 0 ? e + (e >> PAD) : e] = v[i];
  }
}
template <int MOST, int NT, int PAD, typename V>
__device__ __forceinline__ void run_store(V* __restrict__ p, const V* __restrict__ lds, int n) {
#pragma unroll
  for (int i = 0; i < (MOST + NT - 1) / NT; ++i) {
    const int e = threadIdx.x + i * NT;
    if (e < n) p[e] = lds[PAD > 0 ? e + (e >> PAD) : e];
  }
}

// The packed spectrum a + i b at x of two real sequences whose coefficients
// k < nk are at(k, a, b); zero beyond.
template <typename T, typename F>
__device__ __forceinline__ cx<T> herm_at(int x, int N, int nk, F at) {
  const int k = 2 * x <= N ? x : N - x;
  if (k >= nk) return czero<T>();
  cx<T> a, b;
  at(k, a, b);
  if (k == 0 || 2 * k == N) return mk<T>(a.x, b.x);
  return x == k ? mk<T>(a.x - b.y, a.y + b.x) : mk<T>(a.x + b.y, b.x - a.y);
}

template <typename T, int LOGN, bool PAIRS, bool STAGED>
__global__ void __launch_bounds__((ZShape<LOGN>::NT))
    k_zc2r(const cx<T>* __restrict__ in0, const cx<T>* __restrict__ in1, T* __restrict__ out0,
           T* __restrict__ out1, int nx, int nm, T scale, const cx<T>* __restrict__ tw) {
  using S = ZShape<LOGN>;
  extern __shared__ char smem_raw[];
  const int sl = threadIdx.x / S::TPS, t = threadIdx.x % S::TPS;
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw) + sl * S::LDSN;
  const cx<T>* __restrict__ in = blockIdx.y ? in1 : in0;
  T* __restrict__ out = blockIdx.y ? out1 : out0;
  const int x0 = 2 * blockIdx.x * S::SL, xa = x0 + 2 * sl, xb = xa + 1;
  const bool live = xa < nx, two = xb < nx;
  const int nrow = min(2 * S::SL, nx - x0);
  cx<T> v[S::E];
  static_assert(!(PAIRS && STAGED), "rows in order");
  if constexpr (STAGED) {
    cx<T>* run = reinterpret_cast<cx<T>*>(smem_raw);
    run_load<S::SL * (S::N + 2), S::NT, 0>(in + (size_t)x0 * nm, run, nrow * nm);
    rf_sync<S::NT>();
#pragma unroll
    for (int m = 0; m < S::E; ++m)
      v[m] = herm_at<T>(t + m * S::TPS, S::N, live ? nm : 0, [&](int k, cx<T>& a, cx<T>& b) {
        a = run[2 * sl * nm + k];
        b = two ? run[(2 * sl + 1) * nm + k] : czero<T>();
      });
    rf_sync<S::NT>();
  } else {
    // (each coefficient is read for k and for N - k; the second read hits L1)
#pragma unroll
    for (int m = 0; m < S::E; ++m)
      v[m] = herm_at<T>(t + m * S::TPS, S::N, live ? nm : 0, [&](int k, cx<T>& a, cx<T>& b) {
        if constexpr (PAIRS) {
          const cx<T>* __restrict__ p = in + pair_at(xa, k, nm);
          a = p[0];
          b = p[1];
        } else {
          a = in[(size_t)xa * nm + k];
          b = two ? in[(size_t)xb * nm + k] : czero<T>();
        }
      });
  }
  rf_fft<T, LOGN, S::LOGE, +1, 1, S::NT>(v, lds, t, tw);
  if constexpr (STAGED) {
    T* pts = reinterpret_cast<T*>(smem_raw);
    rf_sync<S::NT>();
#pragma unroll
    for (int m = 0; m < S::E; ++m) {
      pts[pts_at<LOGN>(sl, 0, t + m * S::TPS)] = v[m].x * scale;
      pts[pts_at<LOGN>(sl, 1, t + m * S::TPS)] = v[m].y * scale;
    }
    rf_sync<S::NT>();
    run_store<2 * S::SL * S::N, S::NT, LOGN + 1>(out + (size_t)x0 * S::N, pts, nrow * S::N);
  } else if (live) {
#pragma unroll
    for (int m = 0; m < S::E; ++m) {
      const int n = t + m * S::TPS;
      out[(size_t)xa * S::N + n] = v[m].x * scale;
      if (two) out[(size_t)xb * S::N + n] = v[m].y * scale;
    }
  }
}

// A forward transform's real input, as pairs of sequences: an array, or the
// flux divergence pddx(ux f) + pddz(uz f) of three formed where it is used,
// so that it is neither written nor read back (a pass of its own took 10 us
// at 1024^2 FP64).  A source fills v[m] with the two sequences' values at
// t + m TPS of the transform's axis ("own"); p and p + 1 are the sequences'
// positions on the other axis ("cross"), element (p, i) at p sp + i si.
template <typename T>
struct PlainSrc {
  static constexpr bool PLAIN = true;
  const T* __restrict__ f;
  size_t sp, si;
  template <int LOGN, int LOGE, int STRIDE, int NT>
  __device__ __forceinline__ void load(cx<T> (&v)[1 << LOGE], cx<T>*, int t, int p, bool live,
                                       bool two) const {
    constexpr int E = 1 << LOGE, TPS = (1 << LOGN) / E;
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const T* __restrict__ q = f + (size_t)p * sp + (size_t)(t + m * TPS) * si;
      v[m] = mk<T>(live ? q[0] : T(0), two ? q[sp] : T(0));
    }
  }
};
// uc / uo: the velocity along the cross / own axis.  The cross difference
// reads the sequences beside the pair (ORDER + 2 of f and uc per pair, where
// a point by itself reads 2 ORDER + 2); the own difference's products pass
// to the neighbouring threads through the transform's LDS.  The own axis is
// periodic; the cross axis wraps or (per = 0) has no difference within
// ORDER / 2 of its ends.
template <typename T, int ORDER>
struct FluxSrc {
  static constexpr bool PLAIN = false;
  const T *__restrict__ uc, *__restrict__ uo, *__restrict__ f;
  size_t sp, si;
  int nc, per;
  T ihc, iho;  // 1 / (2 h) (order 2) or 1 / (3 h) of each axis
  __device__ __forceinline__ static T diff(T m2, T m1, T p1, T p2) {
    if constexpr (ORDER == 2) return p1 - m1;
    return T(-0.25) * p2 + T(2) * p1 - T(2) * m1 + T(0.25) * m2;
  }
  template <int LOGN, int LOGE, int STRIDE, int NT>
  __device__ __forceinline__ void load(cx<T> (&v)[1 << LOGE], cx<T>* __restrict__ lds, int t,
                                       int p, bool live, bool two) const {
    constexpr int N = 1 << LOGN, E = 1 << LOGE, TPS = N / E, W = ORDER / 2, NR = 2 + 2 * W;
    constexpr int MB = ORDER == 2 ? 4 : 2;  // points whose loads are in flight together
    size_t at[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      int q = p + r - W;
      if (per)
        q = q < 0 ? q + nc : (q >= nc ? q - nc : q);
      else
        q = min(max(q, 0), nc - 1);
      at[r] = (live ? (size_t)q : 0) * sp;
    }
    const bool ina = per || (p >= W && p <= nc - 1 - W);
    const bool inb = per || (p + 1 >= W && p + 1 <= nc - 1 - W);
    cx<T> g[E];
#pragma unroll
    for (int m0 = 0; m0 < E; m0 += MB) {
      T fv[MB][NR], cv[MB][NR], ov[MB][2];
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const size_t i = (size_t)(t + (m0 + m) * TPS) * si;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          fv[m][r] = f[at[r] + i];
          cv[m][r] = uc[at[r] + i];
        }
        ov[m][0] = uo[at[W] + i];
        ov[m][1] = uo[at[W + 1] + i];
      }
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        T q[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) q[r] = cv[m][r] * fv[m][r];
        const T da = diff(q[0], q[W - 1], q[W + 1], q[2 * W]);
        const T db = diff(q[1], q[W], q[W + 2], q[2 * W + 1]);
        g[m0 + m] = mk<T>(ina ? da * ihc : T(0), inb ? db * ihc : T(0));
        lds[rf_pad<LOGE>(t, (m0 + m) * TPS) * STRIDE] =
            mk<T>(ov[m][0] * fv[m][W], ov[m][1] * fv[m][W + 1]);
      }
    }
    rf_sync<NT>();
#pragma unroll
    for (int m = 0; m < E; ++m) {
      auto own = [&](int d) { return lds[rf_near<LOGN, LOGE>(t, m, d) * STRIDE]; };
      const cx<T> m1 = own(-1), p1 = own(1);
      cx<T> m2 = m1, p2 = p1;
      if constexpr (ORDER == 4) {
        m2 = own(-2);
        p2 = own(2);
      }
      v[m] = mk<T>(live ? g[m].x + diff(m2.x, m1.x, p1.x, p2.x) * iho : T(0),
                   two ? g[m].y + diff(m2.y, m1.y, p1.y, p2.y) * iho : T(0));
    }
    rf_sync<NT>();
  }
};

template <typename T, int LOGN, bool PAIRS, bool STAGED, typename Src>
__global__ void __launch_bounds__((ZShape<LOGN>::NT))
    k_zr2c(Src src, cx<T>* __restrict__ out, int nx, int nm, const cx<T>* __restrict__ tw) {
  using S = ZShape<LOGN>;
  extern __shared__ char smem_raw[];
  const int sl = threadIdx.x / S::TPS, t = threadIdx.x % S::TPS;
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw) + sl * S::LDSN;
  const int x0 = 2 * blockIdx.x * S::SL, xa = x0 + 2 * sl, xb = xa + 1;
  const bool live = xa < nx, two = xb < nx;
  const int nrow = min(2 * S::SL, nx - x0);
  cx<T> v[S::E];
  if constexpr (STAGED) {
    T* pts = reinterpret_cast<T*>(smem_raw);
    run_load<2 * S::SL * S::N, S::NT, LOGN + 1>(src.f + (size_t)x0 * S::N, pts, nrow * S::N);
    rf_sync<S::NT>();
#pragma unroll
    for (int m = 0; m < S::E; ++m)
      v[m] = mk<T>(live ? pts[pts_at<LOGN>(sl, 0, t + m * S::TPS)] : T(0),
                   two ? pts[pts_at<LOGN>(sl, 1, t + m * S::TPS)] : T(0));
    rf_sync<S::NT>();
  } else {
    src.template load<LOGN, S::LOGE, 1, S::NT>(v, lds, t, xa, live, two);
  }
  rf_fft<T, LOGN, S::LOGE, -1, 1, S::NT>(v, lds, t, tw);
  rf_sync<S::NT>();
#pragma unroll
  for (int m = 0; m < S::E; ++m) lds[rf_pad<S::LOGE>(t, m * S::TPS)] = v[m];
  rf_sync<S::NT>();
  // coefficients k <= N / 2 of both rows (a half-spectrum ends at N / 2)
  cx<T> va[S::E / 2 + 1], vb[S::E / 2 + 1];
#pragma unroll
  for (int m = 0; m <= S::E / 2; ++m) {
    const int k = t + m * S::TPS;
    if (live && k < nm) {
      const cx<T> y = lds[rf_pad<S::LOGE>(t, m * S::TPS)];
      const cx<T> ym = lds[rf_mirror<LOGN, S::LOGE>(t, m)];
      va[m] = mk<T>(T(0.5) * (y.x + ym.x), T(0.5) * (y.y - ym.y));
      vb[m] = mk<T>(T(0.5) * (y.y + ym.y), T(0.5) * (ym.x - y.x));
      if constexpr (STAGED) continue;
      if constexpr (PAIRS) {
        cx<T>* __restrict__ p = out + pair_at(xa, k, nm);
        p[0] = va[m];
        p[1] = vb[m];
      } else {
        out[(size_t)xa * nm + k] = va[m];
        if (two) out[(size_t)xb * nm + k] = vb[m];
      }
    }
  }
  if constexpr (STAGED) {
    cx<T>* run = reinterpret_cast<cx<T>*>(smem_raw);
    rf_sync<S::NT>();
#pragma unroll
    for (int m = 0; m <= S::E / 2; ++m) {
      const int k = t + m * S::TPS;
      if (live && k < nm) {
        run[2 * sl * nm + k] = va[m];
        if (two) run[(2 * sl + 1) * nm + k] = vb[m];
      }
    }
    rf_sync<S::NT>();
    run_store<S::SL * (S::N + 2), S::NT, 0>(out + (size_t)x0 * nm, run, nrow * nm);
  }
}

// --------------------------------------------------------------------------
// FD-z x transforms: spectral (nn, nz) <-> physical (nx, nz), TC pairs of
// columns per block, consecutive threads on consecutive pairs
// --------------------------------------------------------------------------
template <typename T, int LOGN, int TC>
__global__ void __launch_bounds__((XShape<LOGN, TC>::NT))
    k_xc2r_cols(const cx<T>* __restrict__ in0, const cx<T>* __restrict__ in1, T* __restrict__ out0,
                T* __restrict__ out1, int nn, int nz, T scale, const cx<T>* __restrict__ tw,
                int ntile) {
  using S = XShape<LOGN, TC>;
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int tile = xcd_logical(ntile);
  if (tile < 0) return;
  const cx<T>* __restrict__ in = blockIdx.y ? in1 : in0;
  T* __restrict__ out = blockIdx.y ? out1 : out0;
  const int c = threadIdx.x % S::C, t = rf_thread<S::TPS>(threadIdx.x / S::C);
  const int za = 2 * (tile * S::C + c);
  const bool live = za < nz, two = za + 1 < nz;
  cx<T> v[S::E];
#pragma unroll
  for (int m = 0; m < S::E; ++m)
    v[m] = herm_at<T>(t + m * S::TPS, S::N, live ? nn : 0, [&](int k, cx<T>& a, cx<T>& b) {
      a = in[(size_t)k * nz + za];
      b = two ? in[(size_t)k * nz + za + 1] : czero<T>();
    });
  rf_fft<T, LOGN, S::LOGE, +1, S::C, S::NT>(v, lds + c, t, tw);
  if (live) {
#pragma unroll
    for (int m = 0; m < S::E; ++m) {
      const size_t o = (size_t)(t + m * S::TPS) * nz + za;
      out[o] = v[m].x * scale;
      if (two) out[o + 1] = v[m].y * scale;
    }
  }
}

template <typename T, int LOGN, int TC, typename Src>
__global__ void __launch_bounds__((XShape<LOGN, TC>::NT))
    k_xr2c_cols(Src src, cx<T>* __restrict__ out, int nn, int nz, T scale,
                const cx<T>* __restrict__ tw, int ntile) {
  using S = XShape<LOGN, TC>;
  extern __shared__ char smem_raw[];
  cx<T>* lds = reinterpret_cast<cx<T>*>(smem_raw);
  const int tile = xcd_logical(ntile);
  if (tile < 0) return;
  const int c = threadIdx.x % S::C, t = rf_thread<S::TPS>(threadIdx.x / S::C);
  const int za = 2 * (tile * S::C + c);
  const bool live = za < nz, two = za + 1 < nz;
  cx<T> v[S::E];
  src.template load<LOGN, S::LOGE, S::C, S::NT>(v, lds + c, t, za, live, two);
  rf_fft<T, LOGN, S::LOGE, -1, S::C, S::NT>(v, lds + c, t, tw);
  rf_sync<S::NT>();
#pragma unroll
  for (int m = 0; m < S::E; ++m) lds[rf_pad<S::LOGE>(t, m * S::TPS) * S::C + c] = v[m];
  rf_sync<S::NT>();
#pragma unroll
  for (int m = 0; m <= S::E / 2; ++m) {
    const int k = t + m * S::TPS;
    if (live && k < nn) {
      const cx<T> y = lds[rf_pad<S::LOGE>(t, m * S::TPS) * S::C + c];
      const cx<T> ym = lds[rf_mirror<LOGN, S::LOGE>(t, m) * S::C + c];
      const T h = T(0.5);
      const size_t o = (size_t)k * nz + za;
      out[o] = cscale<T>(mk<T>(h * (y.x + ym.x), h * (y.y - ym.y)), scale);
      if (two) out[o + 1] = cscale<T>(mk<T>(h * (y.y + ym.y), h * (ym.x - y.x)), scale);
    }
  }
}

// --------------------------------------------------------------------------
// Host launchers
// --------------------------------------------------------------------------
#define MLV_LOGN_CASES(X) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)

// Switch over the transform length; X(L) launches the kernel compiled for it.
#define MLV_BY_LOGN(logn)            \
  switch (logn) {                    \
    MLV_LOGN_CASES(X)                \
    default:                         \
      return hipErrorInvalidValue;   \
  }                                  \
  return hipGetLastError()

// Columns (or column pairs) per block of an x pass of `n` of them: two, or
// four once that still leaves a block per CU: the rows of a tile are then
// read in runs of twice the length (FP64 inverse of 256 x 16384 reals 20.7 us a
// call with two, 15.2 with four, 1024 x 4096 20.3 and 16.7).  Double precision
// takes four up to 1024 points, beyond which they pass the LDS or the
// registers, and not where it forms a flux, whose operands spill.
template <typename T, bool FLUX>
constexpr bool four_cols(int logn) {
  return sizeof(T) == 4 || (logn <= 10 && !FLUX);
}

#define MLV_COLS(L, n, KERN, ...)                                                                 \
  do {                                                                                            \
    if constexpr (four_cols<T, flux>(L)) {                                                        \
      if ((n) >= 4 * 256) {                                                                       \
        using S = XShape<L, 4>;                                                                   \
        const size_t lds = tr_lds_bytes<T>(L, S::C);                                              \
        const int nt = ((n) + S::C - 1) / S::C;                                                   \
        MLV_SET_LDS_ONCE((KERN(L, 4)), lds);                                                      \
        hipLaunchKernelGGL((KERN(L, 4)), dim3(xcd_grid(nt), ny), dim3(S::NT), lds, s, __VA_ARGS__, nt); \
        break;                                                                                    \
      }                                                                                           \
    }                                                                                             \
    {                                                                                             \
      using S = XShape<L, 2>;                                                                     \
      const size_t lds = tr_lds_bytes<T>(L, S::C);                                                \
      const int nt = ((n) + S::C - 1) / S::C;                                                     \
      MLV_SET_LDS_ONCE((KERN(L, 2)), lds);                                                        \
      hipLaunchKernelGGL((KERN(L, 2)), dim3(xcd_grid(nt), ny), dim3(S::NT), lds, s, __VA_ARGS__, nt); \
    }                                                                                             \
  } while (0)

#define MLV_ROWS(L, STAGED, KERN, ...)                                                            \
  do {                                                                                            \
    using S = ZShape<L>;                                                                          \
    const size_t lds = (size_t)S::SL * S::slot(STAGED) * sizeof(cx<T>);                           \
    const int nb = ((nx + 1) / 2 + S::SL - 1) / S::SL;                                            \
    MLV_SET_LDS_ONCE((KERN(L)), lds);                                                             \
    hipLaunchKernelGGL((KERN(L)), dim3(nb, ny), dim3(S::NT), lds, s, __VA_ARGS__);                \
  } while (0)

template <typename T>
hipError_t launch_xinv(int logn, const void* in, void* out, int nn, int nm, const void* tw,
                       hipStream_t s, int nrow, double scale) {
  if (nrow < 0) nrow = 2 * nn + 1;
  constexpr bool flux = false;
  const int ny = 1;
#define KX(L, C) k_xinv<T, L, C>
#define X(L)                                                                                \
  case L:                                                                                   \
    MLV_COLS(L, nm, KX, (const cx<T>*)in, (cx<T>*)out, nn, nrow, nm, (T)scale,              \
             (const cx<T>*)tw);                                                             \
    break;
  MLV_BY_LOGN(logn);
#undef X
#undef KX
}

template <typename T>
hipError_t launch_xinv_vel(int logn, const VelArgs& a, void* out, int nn, int nm, const void* tw,
                           hipStream_t s) {
  constexpr bool flux = false;
  const int ny = 2;
#define KX(L, C) k_xinv_vel<T, L, C>
#define X(L)                                                                                \
  case L:                                                                                   \
    MLV_COLS(L, nm, KX, (const cx<T>*)a.w, (cx<T>*)a.psi, (cx<T>*)a.ux, (cx<T>*)a.uz,       \
             (cx<T>*)out, nn, nm, a.fx, a.fz, a.fx2, a.fz2, (const cx<T>*)tw);              \
    break;
  MLV_BY_LOGN(logn);
#undef X
#undef KX
}

template <typename T>
hipError_t launch_xfwd(int logn, const void* in, void* out, int nn, int nm, double scale,
                       const void* tw, hipStream_t s, int nrow) {
  if (nrow < 0) nrow = 2 * nn + 1;
  constexpr bool flux = false;
  const int ny = 1;
#define KX(L, C) k_xfwd<T, L, C>
#define X(L)                                                                                \
  case L:                                                                                   \
    MLV_COLS(L, nm, KX, (const cx<T>*)in, (cx<T>*)out, nn, nrow, nm, (T)scale,              \
             (const cx<T>*)tw);                                                             \
    break;
  MLV_BY_LOGN(logn);
#undef X
#undef KX
}

template <typename T>
hipError_t launch_zc2r(int logn, const Two& a, int nx, int nm, const void* tw, hipStream_t s,
                       double scale, bool pairs) {
  const int ny = a.n;
  const cx<T>*i0 = (const cx<T>*)a.in[0], *i1 = (const cx<T>*)a.in[1];
  T *o0 = (T*)a.out[0], *o1 = (T*)a.out[1];
#define KP(L) k_zc2r<T, L, true, false>
#define KR(L) k_zc2r<T, L, false, false>
#define KS(L) k_zc2r<T, (L <= 5 ? L : 3), false, true>
#define X(L)                                                                                \
  case L:                                                                                   \
    if (pairs)                                                                              \
      MLV_ROWS(L, false, KP, i0, i1, o0, o1, nx, nm, (T)scale, (const cx<T>*)tw);           \
    else if (staged_rows<L>(nx))                                                            \
      MLV_ROWS(L, true, KS, i0, i1, o0, o1, nx, nm, (T)scale, (const cx<T>*)tw);            \
    else                                                                                    \
      MLV_ROWS(L, false, KR, i0, i1, o0, o1, nx, nm, (T)scale, (const cx<T>*)tw);           \
    break;
  MLV_BY_LOGN(logn);
#undef X
#undef KP
#undef KR
#undef KS
}

template <typename T, bool PAIRS, typename Src>
static hipError_t zr2c_src(int logn, const Src& src, void* out, int nx, int nm, const void* tw,
                           hipStream_t s) {
  const int ny = 1;
#define KR(L) k_zr2c<T, L, PAIRS, false, Src>
#define KS(L) k_zr2c<T, (L <= 5 ? L : 3), false, true, PlainSrc<T>>
#define X(L)                                                                                \
  case L:                                                                                   \
    if constexpr (!PAIRS) {                                                                 \
      if (staged_rows<L>(nx)) {                                                             \
        MLV_ROWS(L, true, KS, src, (cx<T>*)out, nx, nm, (const cx<T>*)tw);                  \
        break;                                                                              \
      }                                                                                     \
    }                                                                                       \
    MLV_ROWS(L, false, KR, src, (cx<T>*)out, nx, nm, (const cx<T>*)tw);                     \
    break;
  MLV_BY_LOGN(logn);
#undef X
#undef KR
#undef KS
}

// The flux source of a z pass (own axis z) or of an FD-z x pass (own axis x).
template <typename T, int ORDER>
static FluxSrc<T, ORDER> flux_src(const FluxArgs& a, int nx, int nz, bool own_z) {
  const double k = ORDER == 2 ? 2.0 : 3.0;
  const T ihx = (T)(1.0 / (k * a.dx)), ihz = (T)(1.0 / (k * a.dz));
  const T *ux = (const T*)a.ux, *uz = (const T*)a.uz, *f = (const T*)a.f;
  if (own_z) return {ux, uz, f, (size_t)nz, 1, nx, 1, ihx, ihz};
  return {uz, ux, f, 1, (size_t)nz, nz, a.zper, ihz, ihx};
}

template <typename T>
hipError_t launch_zr2c(int logn, const void* in, void* out, int nx, int nm, const void* tw,
                       hipStream_t s, bool pairs) {
  const PlainSrc<T> src = {(const T*)in, (size_t)1 << logn, 1};
  return pairs ? zr2c_src<T, true>(logn, src, out, nx, nm, tw, s)
               : zr2c_src<T, false>(logn, src, out, nx, nm, tw, s);
}

template <typename T>
hipError_t launch_zr2c_flux(int logn, const FluxArgs& a, void* out, int nx, int nm, const void* tw,
                            hipStream_t s) {
  return a.order == 2 ? zr2c_src<T, true>(logn, flux_src<T, 2>(a, nx, 1 << logn, true), out, nx, nm, tw, s)
                      : zr2c_src<T, true>(logn, flux_src<T, 4>(a, nx, 1 << logn, true), out, nx, nm, tw, s);
}

template <typename T>
hipError_t launch_xc2r_cols(int logn, const Two& a, int nn, int nz, const void* tw, hipStream_t s,
                            double scale) {
  constexpr bool flux = false;
  const int ny = a.n, np = (nz + 1) / 2;
#define KX(L, C) k_xc2r_cols<T, L, C>
#define X(L)                                                                                \
  case L:                                                                                   \
    MLV_COLS(L, np, KX, (const cx<T>*)a.in[0], (const cx<T>*)a.in[1], (T*)a.out[0],         \
             (T*)a.out[1], nn, nz, (T)scale, (const cx<T>*)tw);                             \
    break;
  MLV_BY_LOGN(logn);
#undef X
#undef KX
}

template <typename T, typename Src>
static hipError_t xr2c_src(int logn, const Src& src, void* out, int nn, int nz, double scale,
                           const void* tw, hipStream_t s) {
  constexpr bool flux = !Src::PLAIN;
  const int ny = 1, np = (nz + 1) / 2;
#define KX(L, C) k_xr2c_cols<T, L, C, Src>
#define X(L)                                                                                \
  case L:                                                                                   \
    MLV_COLS(L, np, KX, src, (cx<T>*)out, nn, nz, (T)scale, (const cx<T>*)tw);              \
    break;
  MLV_BY_LOGN(logn);
#undef X
#undef KX
}

template <typename T>
hipError_t launch_xr2c_cols(int logn, const void* in, void* out, int nn, int nz, double scale,
                            const void* tw, hipStream_t s) {
  return xr2c_src<T>(logn, PlainSrc<T>{(const T*)in, 1, (size_t)nz}, out, nn, nz, scale, tw, s);
}

template <typename T>
hipError_t launch_xr2c_cols_flux(int logn, const FluxArgs& a, void* out, int nn, int nz,
                                 double scale, const void* tw, hipStream_t s) {
  return a.order == 2
             ? xr2c_src<T>(logn, flux_src<T, 2>(a, 1 << logn, nz, false), out, nn, nz, scale, tw, s)
             : xr2c_src<T>(logn, flux_src<T, 4>(a, 1 << logn, nz, false), out, nn, nz, scale, tw, s);
}

#define MLV_INST(T)                                                                               \
  template hipError_t launch_xinv<T>(int, const void*, void*, int, int, const void*, hipStream_t, \
                                     int, double);                                                \
  template hipError_t launch_xinv_vel<T>(int, const VelArgs&, void*, int, int, const void*,       \
                                         hipStream_t);                                            \
  template hipError_t launch_xfwd<T>(int, const void*, void*, int, int, double, const void*,      \
                                     hipStream_t, int);                                           \
  template hipError_t launch_zc2r<T>(int, const Two&, int, int, const void*, hipStream_t, double, \
                                     bool);                                                       \
  template hipError_t launch_zr2c<T>(int, const void*, void*, int, int, const void*, hipStream_t, \
                                     bool);                                                       \
  template hipError_t launch_zr2c_flux<T>(int, const FluxArgs&, void*, int, int, const void*,     \
                                          hipStream_t);                                           \
  template hipError_t launch_xc2r_cols<T>(int, const Two&, int, int, const void*, hipStream_t,    \
                                          double);                                                \
  template hipError_t launch_xr2c_cols<T>(int, const void*, void*, int, int, double, const void*, \
                                          hipStream_t);                                           \
  template hipError_t launch_xr2c_cols_flux<T>(int, const FluxArgs&, void*, int, int, double,     \
                                               const void*, hipStream_t);
MLV_INST(float)
MLV_INST(double)

}  // namespace mlv
