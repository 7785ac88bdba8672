// Device bodies of the fused step's z-pass kernel B (c2r of the channel
// rows, physical products, r2c of the products), launched by fused_b.hip.
#pragma once
#include "fused.hpp"
#include "diag_dev.hpp"
#include "grid.hpp"

namespace mlv {
// --------------------------------------------------------------------------
// Kernel B: z pass, c2r of the channels, products, r2c of the products.
//
// A row pair's channels pack both rows into one complex sequence each, and
// so do its products: output (e, k) holds row a's u_k f_e in the real and
// row b's in the imaginary part.  One wavefront transforms one channel of a
// pair (of 64 / TPS pairs where a row takes fewer threads) in registers
// (fft_reg.hpp), leaves its values in LDS, forms one product with the value
// that it holds itself and one that it reads, and transforms that back: the
// two block barriers are around the exchange, and every transform's own
// exchanges stay inside the wavefront.
// Double precision's z pass: what bounds it is the chain of one pair at small
// sizes (256^2 9.8 -> 5.8 us) and its traffic above (1024^2 19.3 -> 19.0 us,
// 45 MB).
// --------------------------------------------------------------------------
// Two consecutive elements (16 bytes in single precision, one load).
template <typename T>
__device__ __forceinline__ void load_two(const cx<T>* __restrict__ p, cx<T>& a, cx<T>& b) {
  if constexpr (sizeof(T) == 4) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    a = mk<T>(v.x, v.y);
    b = mk<T>(v.z, v.w);
  } else {
    a = p[0];
    b = p[1];
  }
}

// Running diagnostics partials of a z-pass thread.
template <typename T>
struct BDiag {
  T mux = -INFINITY, muz = -INFINITY;  // NaN-propagating maxima, as np.max
  double ke = 0.0, ens = 0.0, flux = 0.0;
};

// A job's partials of the blocks beyond its count (the two plans split a
// grid into different numbers of blocks) hold no points; the last block
// writes them.
template <int NT>
__device__ __forceinline__ void neutral_parts(double* part, int local, int count, int all) {
  if (local != count - 1) return;
  for (int i = count + (int)threadIdx.x; i < all; i += NT) {
    double* p = part + (size_t)kDiagPart * i;
    p[0] = p[1] = -INFINITY;
    for (int q = 2; q < kDiagPart; ++q) p[q] = 0.0;
  }
}

// The output a wavefront forms and the channels it multiplies: its own (or,
// for a wavefront without one, `first`) and `second`.  MHD's outputs take
// two more (-(u f) + b g).
struct ZOut {
  int e, k;           // equation, 0 for Px / 1 for Pz; e < 0: none
  int first, second;  // channels
};
template <int V>
__device__ __forceinline__ constexpr ZOut z_out(int ch) {
  if constexpr (V == BV_VORT1) {  // f, ux, uz
    if (ch == 1) return {0, 0, 1, 0};
    if (ch == 2) return {0, 1, 2, 0};
  } else if constexpr (V == BV_VORT2) {  // f0, f1, ux, uz
    if (ch == 0) return {0, 0, 0, 2};
    if (ch == 1) return {1, 1, 1, 3};
    if (ch == 2) return {1, 0, 2, 1};
    if (ch == 3) return {0, 1, 3, 0};
  } else if constexpr (V == BV_VORT3) {  // f0, f1, f2, ux, uz
    if (ch == 0) return {0, 0, 0, 3};
    if (ch == 1) return {1, 1, 1, 4};
    if (ch == 2) return {2, 0, 2, 3};
    if (ch == 3) return {1, 0, 3, 1};
    if (ch == 4) return {0, 1, 4, 0};
    if (ch == 5) return {2, 1, 4, 2};
  } else {  // w, j, ux, uz, bx, bz
    const int f = V == BV_MHD1 ? 0 : 1;
    if (ch == 2) return {0, 0, 2, f};
    if (ch == 3) return {0, 1, 3, f};
  }
  return {-1, 0, 0, 0};
}

template <typename T, int LOGN, int V>
__device__ __forceinline__ void stepZ_body(const JobDev<T>& J, const StageDev& S, int local,
                                           int flags, const cx<T>* __restrict__ tw, cx<T>* lds) {
#pragma clang fp contract(off)
  using Pg = BProg<V>;
  constexpr int NIN = Pg::NIN, NW = z_waves(V), NT = 64 * NW;
  constexpr int N = 1 << LOGN, TPS = z_tps(LOGN), E = N / TPS, PB = 64 / TPS;
  constexpr int LOGE = z_loge(LOGN), LDSN = rf_len(LOGN, LOGE), nm = xp_nn(N);
  const int nx = J.nx;
  const uint32_t chs = (uint32_t)work_chs(nx, nm);
  const int ch = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, sub = lane / TPS, t = rf_thread<TPS>(lane % TPS);
  const int x0 = 2 * (local * PB + sub);
  const bool live = x0 < nx;
  auto region = [&](int c, int sb) { return lds + (c * PB + sb) * LDSN; };
  cx<T>* __restrict__ mine = region(ch, sub);
  cx<T>* __restrict__ work = glb(J.work);
  // the wavefront's product
  const ZOut o = z_out<V>(ch);
  const bool out = o.e >= 0;
  constexpr bool mhd = V == BV_MHD1 || V == BV_MHD2;
  const int cb = 4 + o.k, cg = V == BV_MHD1 ? 1 : 0;  // MHD's second pair
  cx<T> v[E];
  if (ch < NIN) {
    const uint32_t base = ((uint32_t)ch * chs + (uint32_t)xrow_base(live ? x0 : 0, nm)) * (uint32_t)sizeof(cx<T>);
    // a wavefront issuing its loads goes ahead of other blocks' arithmetic
    __builtin_amdgcn_s_setprio(1);
    cx<T> a[E], b[E];
#pragma unroll
    for (int m = 0; m < E; ++m) {
      a[m] = b[m] = czero<T>();
      if (!z_any(m, TPS, N)) continue;
      const int x = t + m * TPS, k = 2 * x <= N ? x : N - x;
      if (k < nm) load_two<T>(&at32(work, base + (uint32_t)k * (2 * (uint32_t)sizeof(cx<T>))), a[m], b[m]);
    }
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const int x = t + m * TPS;
      v[m] = 2 * x <= N ? mk<T>(a[m].x - b[m].y, a[m].y + b[m].x)
                        : mk<T>(a[m].x + b[m].y, b[m].x - a[m].y);
      if (m == 0 && t == 0) v[m] = mk<T>(a[m].x, b[m].x);
    }
    rf_fft<T, LOGN, LOGE, +1, 1, 64>(v, mine, t, tw);
    rf_sync<64>();
#pragma unroll
    for (int m = 0; m < E; ++m) mine[rf_pad<LOGE>(t, m * TPS)] = v[m];
  }
  __syncthreads();
  // this job's check loop (J.loops counts the loops before this one)
  const bool diag = (flags & kDiag) && J.loops % (flags >> kDiagShift) == 0;
  if (diag || (flags & kWritePhys)) {
    BDiag<T> d;
    for (int i = threadIdx.x; i < PB * N; i += NT) {
      const int sb = i / N, n = i % N, xa = 2 * (local * PB + sb);
      if (xa >= nx) continue;
      cx<T> q[NIN];
#pragma unroll
      for (int c = 0; c < NIN; ++c) {
        q[c] = region(c, sb)[rf_pad<LOGE>(n)];
      }
      if (diag) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          auto val = [&](int c) { return r ? q[c].y : q[c].x; };
          const double ux = (double)val(Pg::UX), uz = (double)val(Pg::UZ), w = (double)val(0);
          d.mux = nan_max(d.mux, val(Pg::UX));
          d.muz = nan_max(d.muz, val(Pg::UZ));
          d.ke += uz * uz + ux * ux;
          d.ens += w * w;
          if constexpr (Pg::FLUX >= 0) d.flux += (double)val(Pg::FLUX) * uz;
        }
      }
      if (flags & kWritePhys) {
#pragma unroll
        for (int c = 0; c < NIN; ++c)
#pragma unroll
          for (int p = 0; p < kMaxPhys; ++p)
            if (S.phys_ch[p] == c) {
              T* __restrict__ o = glb(J.phys[p]) + (size_t)xa * N + n;
              o[0] = q[c].x;
              o[N] = q[c].y;
            }
      }
    }
    if (diag) {
      double* part = glb(J.diag);
      block_diag<NT>((double)d.mux, (double)d.muz, d.ke, d.ens, d.flux,
                     part + (size_t)kDiagPart * local);
      neutral_parts<NT>(part, local, (nx + 2 * PB - 1) / (2 * PB), J.nbB);
    }
  }
  if (out) {
    const cx<T>* __restrict__ sec = region(o.second, sub);
    const cx<T>* __restrict__ fst = region(o.first, sub);
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const int i = rf_pad<LOGE>(t, m * TPS);
      const cx<T> a = o.first == ch ? v[m] : fst[i], b = sec[i];
      const T px = a.x * b.x, py = a.y * b.y;
      if constexpr (mhd) {
        const cx<T> c = region(cb, sub)[i], g = region(cg, sub)[i];
        v[m] = mk<T>(fma1(c.x, g.x, -px), fma1(c.y, g.y, -py));
      } else {
        v[m] = mk<T>(-px, -py);
      }
    }
  }
  // every value is read before any transform writes over it
  __syncthreads();
  if (!out) return;
  rf_fft<T, LOGN, LOGE, -1, 1, 64>(v, mine, t, tw);
  rf_sync<64>();
#pragma unroll
  for (int m = 0; m < E; ++m)
    if (z_any(m, TPS, N)) mine[rf_pad<LOGE>(t, m * TPS)] = v[m];
  rf_sync<64>();
  const uint32_t obase = ((uint32_t)pchan(NIN, o.e, o.k) * chs + (uint32_t)x0 * kPGroup) * (uint32_t)sizeof(cx<T>);
#pragma unroll
  for (int m = 0; m <= E / 2; ++m) {
    if (m * TPS >= nm) continue;
    const int k = t + m * TPS;
    if (live && k < nm) {
      const cx<T> y = mine[rf_pad<LOGE>(t, m * TPS)], ym = mine[rf_mirror<LOGN, LOGE>(t, m)];
      const uint32_t at = obase + (uint32_t)pidx(0, k, nx) * (uint32_t)sizeof(cx<T>);
      at32(work, at) = mk<T>(T(0.5) * (y.x + ym.x), T(0.5) * (y.y - ym.y));
      at32(work, at + kPGroup * (uint32_t)sizeof(cx<T>)) = mk<T>(T(0.5) * (y.y + ym.y), T(0.5) * (ym.x - y.x));
    }
  }
}

// --------------------------------------------------------------------------
// The LDS-staged z pass: channel rows staged in LDS, 16 or 32 points per
// thread.  Single precision runs it at every size (its blocks hold more
// rows and its products, between two fused passes, cost no LDS trip of their
// own: 106 against 120 us at 16 x 1024^2 with the register pass, 12 against 15
// on tearing at 4 x 512^2, 43 against 58 on a mixed batch of double
// diffusion), double precision the two-sweep plan and the sizes that
// z_reg_fits leaves out.
// --------------------------------------------------------------------------
// SPLIT (single precision): jobs with split carry mean profiles (kernel M)
// and mean-free channels; a batch without such jobs runs SPLIT = 0.
// Shapes of a z-pass block of program V at 2^LOGN points with P points per
// thread: RB rows, each of NIN input channels (packed two real sequences
// per LDS slot) and NEQ product slots.
template <typename T, int LOGN, int V, int P>
struct BShape {
  using Pg = BProg<V>;
  static constexpr int NIN = Pg::NIN, NEQ = Pg::NEQ;
  static constexpr int N = 1 << LOGN;
  static constexpr int SL = fft_slots<LOGN, kNT, P>();
  static constexpr int LDSN = fft_ldsn(N);
  static constexpr int RB = brows(NIN, NEQ, SL);
  static constexpr int NW = kNT / 64;
  static constexpr int KIT = ((N - 1) / 3 + 63) / 64;  // bound on ceil(nm / 64)
  // Row-pair slots (an even number of rows): slot s holds channel s % NIN of
  // the rows x0 + 2 (s / NIN) and x0 + 2 (s / NIN) + 1, which the
  // interleaved channel layout stores side by side, so one load of two
  // elements per k fills both halves of the slot and every load instruction
  // uses whole cache lines.  Otherwise consecutive sequences share a slot.
  static constexpr bool PAIR = RB % 2 == 0 && kXil == 2;
  static constexpr int SLN = PAIR ? NIN * (RB / 2) : (RB * NIN + 1) / 2;  // input slots
  static constexpr int WPS = SLN >= NW ? 1 : NW / SLN;  // wavefronts per input slot
  // slot, and half (0 real, 1 imaginary part), of sequence q = row * NIN +
  // channel
  static constexpr int slot_of(int q) { return PAIR ? (q / NIN / 2) * NIN + q % NIN : q / 2; }
  static constexpr int half_of(int q) { return PAIR ? (q / NIN) % 2 : q % 2; }
  // slots in use for a block of nrows rows (even when PAIR: RB is even and
  // the grid sizes are powers of two)
  __device__ __forceinline__ static int nslots(int nrows) {
    return PAIR ? NIN * (nrows / 2) : (nrows * NIN + 1) / 2;
  }
  static constexpr int NO = RB * NEQ;                  // product slots
  static constexpr int WPO = NO >= NW ? 1 : NW / NO;   // wavefronts per product slot
  static_assert(SLN <= bslots_used(NIN, NEQ, SL) && NO <= bslots_used(NIN, NEQ, SL),
                "the launch's LDS holds the slots in use");
};

// Load phase: the block's input channel rows into the LDS slots, two real
// sequences per slot packed as one Hermitian spectrum (zero-padded from nm
// to N/2).  One wavefront per slot (WPS per slot when the block has fewer
// slots than wavefronts, splitting its k range): lane l handles k = l + 64 i,
// so no index needs a division by the runtime row length nm.
template <typename T, typename Sh>
__device__ __forceinline__ void bload(const cx<T>* __restrict__ work, size_t chs, int nm, int x0,
                                      int nseq, int nslot, cx<T>* lds) {
  constexpr int N = Sh::N, NIN = Sh::NIN, KIT = Sh::KIT, WPS = Sh::WPS, NW = Sh::NW;
  constexpr int KB = KIT < 6 ? KIT : 6;
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int ssub = wv % WPS;
  for (int s = wv / WPS; s < nslot; s += NW / WPS) {
    cx<T>* z = lds + s * Sh::LDSN;
    const cx<T>* __restrict__ pa;
    const cx<T>* __restrict__ pb = nullptr;
    if constexpr (Sh::PAIR) {
      // channel s % NIN, rows x0 + 2 (s / NIN) + {0, 1}: element k of the
      // pair at 2k and 2k + 1
      pa = work + (size_t)(s % NIN) * chs + xrow_base(x0 + 2 * (s / NIN), nm);
    } else {
      const int qa = 2 * s, qb = qa + 1;
      pa = work + (size_t)(qa % NIN) * chs + xrow_base(x0 + qa / NIN, nm);
      if (qb < nseq) pb = work + (size_t)(qb % NIN) * chs + xrow_base(x0 + qb / NIN, nm);
    }
    // loads of up to KB iterations in flight before any is used
#pragma unroll 1
    for (int i0 = ssub * KB; i0 < KIT; i0 += WPS * KB) {
      cx<T> av[KB], bv[KB];
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int k = lane + 64 * (i0 + i);
        if constexpr (Sh::PAIR) {
          if (k < nm) {
            load_two<T>(pa + (size_t)k * kXil, av[i], bv[i]);
          } else {
            av[i] = czero<T>();
            bv[i] = czero<T>();
          }
        } else {
          av[i] = k < nm ? pa[(size_t)k * kXil] : czero<T>();
          bv[i] = (pb && k < nm) ? pb[(size_t)k * kXil] : czero<T>();
        }
      }
#pragma unroll
      for (int i = 0; i < KB; ++i) {
        const int k = lane + 64 * (i0 + i);
        if (k < nm) {
          const cx<T> a = av[i], b = bv[i];
          if (k == 0) {
            z[0] = mk<T>(a.x, b.x);
          } else {
            z[fft_pad(k)] = mk<T>(a.x - b.y, a.y + b.x);
            z[fft_pad(N - k)] = mk<T>(a.x + b.y, b.x - a.y);
          }
        }
      }
    }
    for (int k = nm + lane + 64 * ssub; k <= N - nm; k += 64 * WPS) z[fft_pad(k)] = czero<T>();
  }
}

// The physical work at one point n of the block's rows, v[q] the value of
// sequence q = row * NIN + channel (a fluctuation when kSplit): the
// diagnostics partials, the physical outputs, and each row's products into
// px / pz[row * NEQ + e].
template <typename T, typename Sh>
__device__ __forceinline__ void bpoint(const JobDev<T>& J, const StageDev& S, bool kSplit,
                                       bool diag, int flags, int x0, int nrows, int nseq, int n,
                                       const T* v, BDiag<T>& d, T* px, T* pz) {
  using Pg = typename Sh::Pg;
  constexpr int NIN = Sh::NIN, NEQ = Sh::NEQ, RB = Sh::RB, N = Sh::N;
  T mv[NIN];
#pragma unroll
  for (int q = 0; q < NIN; ++q)
    mv[q] = (kSplit && !Pg::zero_mean(q)) ? glb(J.mean)[(size_t)q * N + n] : T(0);
  // the whole value of sequence q (row q / NIN, channel q % NIN)
  auto whole = [&](int q) { return kSplit ? mv[q % NIN] + v[q] : v[q]; };
  if (diag) {
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      if (r < nrows) {
        const T ux = whole(r * NIN + Pg::UX), uz = whole(r * NIN + Pg::UZ);
        d.mux = nan_max(d.mux, ux);
        d.muz = nan_max(d.muz, uz);
        d.ke += (double)uz * (double)uz + (double)ux * (double)ux;
        const double w = (double)whole(r * NIN);
        d.ens += w * w;
        if constexpr (Pg::FLUX >= 0) d.flux += (double)whole(r * NIN + Pg::FLUX) * (double)uz;
      }
    }
  }
  if (flags & kWritePhys) {
#pragma unroll
    for (int q = 0; q < RB * NIN; ++q) {
      if (q < nseq) {
#pragma unroll
        for (int i = 0; i < kMaxPhys; ++i)
          if (S.phys_ch[i] == q % NIN) glb(J.phys[i])[(size_t)(x0 + q / NIN) * N + n] = whole(q);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    if (kSplit)
      Pg::template products_split<T>(mv, &v[r * NIN], &px[r * NEQ], &pz[r * NEQ]);
    else
      Pg::template products<T>(&v[r * NIN], &px[r * NEQ], &pz[r * NEQ]);
  }
}

// Output phase: the kz < nm coefficients of each product row, split from
// the packed (Px + i Pz) spectrum, into the Px / Pz channels (pidx layout).
// A work item is (equation, row pair, four kz groups); its lanes take row
// (lane >> 3) & 1 of the pair, group (lane >> 4) of the four and kz % 8 =
// lane & 7, so each 16 lanes store one group of both rows -- one whole line
// per channel.  Every product slot must be complete for the whole block.
template <typename T, typename Sh>
__device__ __forceinline__ void bstore(cx<T>* __restrict__ work, size_t chs, int nm, int nx,
                                       int x0, int nrows, const cx<T>* lds) {
  constexpr int N = Sh::N, NIN = Sh::NIN, NEQ = Sh::NEQ, RB = Sh::RB, NW = Sh::NW;
  static_assert(kPGroup == 8, "lane mapping: 8 kz per group");
  constexpr int NPAIR = (RB + 1) / 2;
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r2 = (lane >> 3) & 1, gsub = lane >> 4, kk = lane & 7;
  const int nquad = (nm + 4 * kPGroup - 1) / (4 * kPGroup);
  const int nitem = NEQ * NPAIR * nquad;
  for (int it = wv; it < nitem; it += NW) {
    const int eq = it % NEQ, rest = it / NEQ;
    const int pr = rest % NPAIR, quad = rest / NPAIR;
    const int r = 2 * pr + r2;
    const int k = (quad * 4 + gsub) * kPGroup + kk;
    if (r < nrows && k < nm) {
      const cx<T>* z = lds + (r * NEQ + eq) * Sh::LDSN;
      const cx<T> y = z[fft_pad(k)];
      const cx<T> ym = z[fft_pad((N - k) & (N - 1))];
      const size_t at = pidx(x0 + r, k, nx);
      work[(size_t)pchan(NIN, eq, 0) * chs + at] = mk<T>(T(0.5) * (y.x + ym.x), T(0.5) * (y.y - ym.y));
      work[(size_t)pchan(NIN, eq, 1) * chs + at] = mk<T>(T(0.5) * (y.y + ym.y), T(0.5) * (ym.x - y.x));
    }
  }
}

// Generic z pass: load, inverse transforms, products point by point through
// the LDS, forward transforms, store.
template <typename T, int LOGN, int V, int SPLIT>
__device__ __forceinline__ void stepB_body(const JobDev<T>& J, const StageDev& S, int local,
                                           int flags, const cx<T>* __restrict__ tw, cx<T>* lds) {
  using Pg = BProg<V>;
  constexpr int P = bpoints<T>(LOGN, Pg::NIN, Pg::NEQ);
  using Sh = BShape<T, LOGN, V, P>;
  constexpr int NIN = Sh::NIN, NEQ = Sh::NEQ, N = Sh::N, LDSN = Sh::LDSN, RB = Sh::RB;
  if constexpr (!bfits(NIN, NEQ, Sh::SL)) {
    return;  // rejected on the host
  } else {
    const int nx = J.nx, nm = J.nm;
    const size_t chs = work_chs(nx, nm);
    const int x0 = local * RB;
    const int nrows = min(RB, nx - x0);
    const int nseq = nrows * NIN;
    const int nslot = Sh::nslots(nrows);
    // slot s is loaded by wavefront s and transformed by the same
    // wavefront: no workgroup barrier before the inverse transform
    constexpr bool WL_IN = fft_tps<N, P>() == 64 && Sh::WPS == 1 && Sh::SL == Sh::NW;
    // a wavefront issuing its loads goes ahead of other blocks' arithmetic
    __builtin_amdgcn_s_setprio(1);
    bload<T, Sh>(glb(J.work), chs, nm, x0, nseq, nslot, lds);
    __builtin_amdgcn_s_setprio(0);
    if constexpr (WL_IN)
      wave_sync();
    else
      __syncthreads();
    fft_lds<T, LOGN, +1, kNT, P>(lds, nslot, tw);
    // this job's check loop (J.loops counts the loops before this one)
    const bool diag = (flags & kDiag) && J.loops % (flags >> kDiagShift) == 0;
    BDiag<T> d;
    // single precision: the channels are fluctuations about their x means,
    // whose z profiles kernel M wrote
    const bool kSplit = SPLIT && J.split;
    for (int n = threadIdx.x; n < N; n += kNT) {
      T v[RB * NIN];
#pragma unroll
      for (int q = 0; q < RB * NIN; ++q) {
        if (q < nseq) {
          const cx<T> z = lds[Sh::slot_of(q) * LDSN + fft_pad(n)];
          v[q] = Sh::half_of(q) ? z.y : z.x;
        } else {
          v[q] = T(0);
        }
      }
      T px[RB * NEQ], pz[RB * NEQ];
      bpoint<T, Sh>(J, S, kSplit, diag, flags, x0, nrows, nseq, n, v, d, px, pz);
#pragma unroll
      for (int o = 0; o < RB * NEQ; ++o)
        if (o < nrows * NEQ) lds[o * LDSN + fft_pad(n)] = mk<T>(px[o], pz[o]);
    }
    if (diag) {
      double* part = glb(J.diag);
      block_diag<kNT>((double)d.mux, (double)d.muz, d.ke, d.ens, d.flux,
                      part + (size_t)kDiagPart * local);
      neutral_parts<kNT>(part, local, (nx + RB - 1) / RB, J.nbB);
    }
    __syncthreads();
    fft_lds<T, LOGN, -1, kNT, P, true>(lds, nrows * NEQ, tw);
    bstore<T, Sh>(glb(J.work), chs, nm, nx, x0, nrows, lds);
  }
}

// z pass with the physical products between two fused passes, for
// N = 512, 1024, 2048 at 16 points per thread (256 threads, 4096 / N slots).
// The inverse transforms run the standard plan 16, 16, R (R = N / 256); its
// last pass (Ns = 256) gives thread t the butterfly t of every slot, whose
// outputs are the points t + 256 r, r < R.  The forward transforms run the
// remainder-first plan R, 16, 16, whose first pass (Ns = 1) takes exactly
// those points.  So thread t reads the last inverse pass's inputs, finishes
// the inverse, forms every row's products at its R points, and does the
// first forward pass in registers: the products never make an LDS round
// trip of their own, and the twiddles of the last inverse pass, which
// depend only on t, are loaded once for all slots.
template <typename T, int LOGN, int V, int SPLIT>
__device__ __forceinline__ void stepB_split(const JobDev<T>& J, const StageDev& S, int local,
                                            int flags, const cx<T>* __restrict__ tw, cx<T>* lds) {
  constexpr int P = 16;
  using Sh = BShape<T, LOGN, V, P>;
  constexpr int NIN = Sh::NIN, NEQ = Sh::NEQ, N = Sh::N, LDSN = Sh::LDSN, RB = Sh::RB;
  constexpr int LOGR = LOGN - 8, R = 1 << LOGR, NSL = 256;
  static_assert(LOGR >= 1 && LOGR <= 3 && kNT == NSL, "split pass shape");
  static_assert(fft_pass_logr(LOGN, 8) == LOGR, "standard plan ends with radix N/256");
  const int nx = J.nx, nm = J.nm;
  const size_t chs = work_chs(nx, nm);
  const int x0 = local * RB;
  const int nrows = min(RB, nx - x0);
  const int nseq = nrows * NIN;
  const int nslot = Sh::nslots(nrows);
  constexpr bool WL_IN = fft_tps<N, P>() == 64 && Sh::WPS == 1 && Sh::SL == Sh::NW;
  // a wavefront issuing its loads goes ahead of other blocks' arithmetic
  __builtin_amdgcn_s_setprio(1);
  bload<T, Sh>(glb(J.work), chs, nm, x0, nseq, nslot, lds);
  __builtin_amdgcn_s_setprio(0);
  if constexpr (WL_IN)
    wave_sync();
  else
    __syncthreads();
  // inverse: the two radix-16 passes
  fft_pass<T, LOGN, 4, 0, +1, kNT, P>(lds, nslot, tw);
  fft_pass<T, LOGN, 4, 4, +1, kNT, P>(lds, nslot, tw);
  __syncthreads();
  // the last inverse pass: butterfly j of every slot
  const int j = threadIdx.x;
  cx<T> w[R];
  {
    const cx<T>* t = tw + fft_pass_table(LOGN, 8) + j;
#pragma unroll
    for (int r = 1; r < R; ++r) {
      w[r] = t[(r - 1) * NSL];
      w[r].y = -w[r].y;  // inverse
    }
  }
  T val[R][2 * Sh::SLN];  // val[r][q]: sequence q at the point j + 256 r
#pragma unroll
  for (int s = 0; s < Sh::SLN; ++s) {
    cx<T> v[R];
    if (s < nslot) {
      const cx<T>* p = lds + s * LDSN + fft_pad(j);
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = p[r * (NSL + NSL / 16)];
#pragma unroll
      for (int r = 1; r < R; ++r) v[r] = cmul<T>(v[r], w[r]);
      Dft<R, +1, T>::run(v);
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = czero<T>();
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      val[r][2 * s] = v[r].x;
      val[r][2 * s + 1] = v[r].y;
    }
  }
  const bool diag = (flags & kDiag) && J.loops % (flags >> kDiagShift) == 0;
  BDiag<T> d;
  const bool kSplit = SPLIT && J.split;
  cx<T> pr[Sh::NO][R];  // product slot o = row * NEQ + e at the point j + 256 r
#pragma unroll
  for (int r = 0; r < R; ++r) {
    T v[RB * NIN];
#pragma unroll
    for (int q = 0; q < RB * NIN; ++q)
      v[q] = q < nseq ? val[r][2 * Sh::slot_of(q) + Sh::half_of(q)] : T(0);
    T px[Sh::NO], pz[Sh::NO];
    bpoint<T, Sh>(J, S, kSplit, diag, flags, x0, nrows, nseq, j + NSL * r, v, d, px, pz);
#pragma unroll
    for (int o = 0; o < Sh::NO; ++o) pr[o][r] = mk<T>(px[o], pz[o]);
  }
  if (diag) block_diag<kNT>((double)d.mux, (double)d.muz, d.ke, d.ens, d.flux,
                            glb(J.diag) + (size_t)kDiagPart * local);
  // every thread has read its inputs before any product slot is written
  // over them
  __syncthreads();
  // the first forward pass (radix R, Ns = 1): outputs at R j + r
#pragma unroll
  for (int o = 0; o < Sh::NO; ++o) {
    if (o < nrows * NEQ) {
      Dft<R, -1, T>::run(pr[o]);
      cx<T>* p = lds + o * LDSN;
#pragma unroll
      for (int r = 0; r < R; ++r) p[fft_pad(R * j + r)] = pr[o][r];
    }
  }
  __syncthreads();
  // the remaining forward passes: radix 16 at Ns = R and Ns = 16 R
  fft_pass<T, LOGN, 4, LOGR, -1, kNT, P, true>(lds, nrows * NEQ, tw);
  fft_pass<T, LOGN, 4, LOGR + 4, -1, kNT, P, true>(lds, nrows * NEQ, tw);
  __syncthreads();
  bstore<T, Sh>(glb(J.work), chs, nm, nx, x0, nrows, lds);
}

template <typename T, int LOGN, int V>
__host__ __device__ constexpr bool bsplit_ok() {
  static_assert(fft_slots<LOGN, kNT, 16>() == ((kNT * 16) >> LOGN), "slots at 16 points");
  return bsplit_fits<T>(LOGN, V);
}

// Kernel B's work for logical block lb of a launch over the job table's
// z-pass blocks of program V (prefix array pref), in plan PLAN.  LO: the
// largest z extent (log2) of the launch's jobs it is compiled for.
template <typename T, int V, int SPLIT, int PLAN, int LO>
__device__ __forceinline__ void roleB(const JobDev<T>* __restrict__ jobs, const int* __restrict__ pref,
                                      int njobs, int lb, int stage, int flags,
                                      const cx<T>* __restrict__ tw, cx<T>* lds) {
  const int j = find_job(pref, njobs, lb);
  const JobDev<T>& J = jobs[j];
  const int local = lb - pref[j];
  switch (J.lognz) {
#define X(L)                                                          \
  case L:                                                             \
    if constexpr (L > LO || (sizeof(T) == 8 && (L < 9 || (PLAN == kPlanSplit && z_reg_fits<T>(L, V))))) \
      break; /* the register pass's */                                \
    else if constexpr (PLAN == kPlanSplit && bsplit_ok<T, L, V>())    \
      stepB_split<T, L, V, SPLIT>(J, J.st[stage], local, flags, tw, lds); \
    else                                                              \
      stepB_body<T, L, V, SPLIT>(J, J.st[stage], local, flags, tw, lds);  \
    break;
    X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)
#undef X
    default:
      break;
  }
}

// Kernel B's work for a batch whose jobs all have 2^LOGN points along z.
template <typename T, int V, int SPLIT, int PLAN, int LOGN>
__device__ __forceinline__ void roleB_fixed(const JobDev<T>* __restrict__ jobs,
                                            const int* __restrict__ pref, int njobs, int lb,
                                            int stage, int flags, const cx<T>* __restrict__ tw,
                                            cx<T>* lds) {
  const int j = find_job(pref, njobs, lb);
  const JobDev<T>& J = jobs[j];
  const int local = lb - pref[j];
  if constexpr (PLAN == kPlanSplit && bsplit_ok<T, LOGN, V>())
    stepB_split<T, LOGN, V, SPLIT>(J, J.st[stage], local, flags, tw, lds);
  else
    stepB_body<T, LOGN, V, SPLIT>(J, J.st[stage], local, flags, tw, lds);
}

}  // namespace mlv
