// Fused fully-spectral timestep over a table of jobs (simulations).
//
// One stage of a step is three kernels:
//   A  x pass inverse: per output channel, a spectral prologue on a state
//      field (identity, or velocity from the streamfunction psi = -f/lap),
//      zero-pad |kx| <= nn to nx, inverse FFT along x -> channel (nx, nm).
//   B  z pass per row block: c2r of every channel row, physical products
//      (the flux terms sign * u * f of each equation), r2c of the products,
//      keep kz < nm -> Px_e, Pz_e channels (nx, nm).  Optionally writes the
//      physical rows of the input channels (for CFL and diagnostics).
//   C  x pass forward per equation: FFT along x of Px_e and Pz_e, keep
//      |kx| <= nn, apply the periodic finite-difference operator as its
//      exact modified wavenumber, add the equation's spectral source terms,
//      store the RHS into the Adams-Bashforth ring, and apply the
//      semi-implicit update, writing the new state to the other buffer of
//      a ping-pong pair.
//
// The periodic central difference of a periodic grid function is a
// circulant operator, so on the DFT grid it is exactly multiplication by
// i*sin(k*h)/h (order 2) or i*(8 sin(k h) - sin(2 k h))/(6 h) (order 4).
// Applying it after the forward transform is therefore the same discrete
// operator as the reference's physical-space stencil followed by rfft2
// (Variable.py:125-127, SpatialDifferentiator.py:76-104,130-185), without
// a halo exchange between rows.
#pragma once
#include <hip/hip_runtime.h>
#include "../../include/melvin_hip.h"
#include "diag.hpp"
#include "transforms.hpp"

namespace mlv {

constexpr int kMaxFields = 4;
constexpr int kMaxChan = 8;   // input channels of the z pass
constexpr int kMaxEq = 3;
constexpr int kMaxA = 8;
constexpr int kMaxPhys = 8;

enum XinvOpKind : int { XOP_ID = 0, XOP_UX = 1, XOP_UZ = 2 };

struct XinvOp {
  int src;       // field index
  int op;        // XinvOpKind
  int ch;        // destination channel
  int from_new;  // read the field from the freshly written state buffer
};

// z-pass variants (compile-time product programs)
enum BVariant : int { BV_VORT1 = 0, BV_VORT2 = 1, BV_VORT3 = 2, BV_MHD1 = 3, BV_MHD2 = 4, BV_COUNT = 5 };

struct StageDev {
  int nA;
  XinvOp a[kMaxA];
  int bvar;      // BVariant
  int neq;       // equations updated by kernel C
  int eq_field[kMaxEq];
  int phys_ch[kMaxPhys];  // z-pass input index written to phys[i] (-1 = none)
};

template <typename T>
struct JobDev {
  int problem, nstage;
  int nx, nz, lognx, lognz, nn, nm, rows;
  int q, curr0, par0, fd_order;
  int pbase;                 // first workspace channel of the Px/Pz outputs
  double fx, fz, fx2, fz2;   // 2*pi/L and -(2*pi)^2/L^2, as the reference forms them
  double dx, dz, scale;      // grid spacings, 1/(nx*nz)
  double alpha, dt;
  double coeff[kMaxFields];  // diffusion coefficient of each field's equation
  double param[4];           // problem parameters (DDC: Pr, R0)
  int nfield;
  cx<T>* state[2][kMaxFields];
  cx<T>* hist[kMaxFields];
  // single precision, optional: the Kahan residual of the state (value =
  // state - residual) as bfloat16 (re, im) pairs packed in 32 bits; it only
  // has to resolve a fraction of one FP32 ulp, so 8 bits of it suffice
  uint32_t* comp[kMaxFields];
  cx<T>* work;
  // single precision with split = 1: each z-pass input channel's x mean as
  // a function of z (kMeanCh rows of nz values, in the workspace after the
  // channels); the x passes then carry only the fluctuations
  int split;
  T* mean;
  cx<T>* psi;
  T* phys[kMaxPhys];
  StageDev st[2];
  // device-side time keeping and diagnostics (see k_diag): the update kernel
  // advances t and loops every step; diag holds the z pass's per-block
  // partials (kDiagPart doubles per block, nbB blocks), then the record
  // count, the CFL breach flag and the series of kDiagRec-double records
  double t;
  long long loops;
  int nbB;
  double* diag;
};

// bfloat16 pair <-> float2 (round to nearest even; the residuals are finite)
__device__ __forceinline__ float2 bf2_load(uint32_t v) {
  return make_float2(__uint_as_float(v << 16), __uint_as_float(v & 0xffff0000u));
}
__device__ __forceinline__ uint32_t bf16_bits(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ uint32_t bf2_pack(float re, float im) {
  return bf16_bits(re) | (bf16_bits(im) << 16);
}

// a*b without its mean-times-mean part: (am + af)(bm + bf) - am bm, with
// means m and fluctuations f (single-precision mean split, see kernel M)
template <typename T>
__device__ __forceinline__ T bil(T am, T af, T bm, T bf) {
  return fma1(am + af, bf, af * bm);
}

// Per-variant channel/product description used by kernel B.  products()
// takes whole values; products_split() takes the x means m and the
// fluctuations f of the channels and leaves out the mean-times-mean part.
template <int V> struct BProg;
template <int NF> struct BVortProg {
  static constexpr int NIN = NF + 2;  // fields, ux, uz
  static constexpr int NEQ = NF;
  static constexpr int UX = NF, UZ = NF + 1;  // velocity channels
  static constexpr int FLUX = NF >= 2 ? 1 : -1;  // scalar whose flux f*uz is tracked
  // channels whose x mean is zero (d/dx of a potential)
  static constexpr bool zero_mean(int q) { return q == UZ; }
  template <typename T>
  __device__ __forceinline__ static void products(const T* v, T* px, T* pz) {
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      px[e] = -(v[NF] * v[e]);
      pz[e] = -(v[NF + 1] * v[e]);
    }
  }
  template <typename T>
  __device__ __forceinline__ static void products_split(const T* m, const T* f, T* px, T* pz) {
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      px[e] = -bil(m[NF], f[NF], m[e], f[e]);
      pz[e] = -bil(m[NF + 1], f[NF + 1], m[e], f[e]);
    }
  }
};
template <> struct BProg<BV_VORT1> : BVortProg<1> {};
template <> struct BProg<BV_VORT2> : BVortProg<2> {};
template <> struct BProg<BV_VORT3> : BVortProg<3> {};
// MHD channels: 0 w, 1 j, 2 ux, 3 uz, 4 bx, 5 bz
template <> struct BProg<BV_MHD1> {
  static constexpr int NIN = 6;
  static constexpr int UX = 2, UZ = 3;
  static constexpr int FLUX = -1;
  static constexpr bool zero_mean(int q) { return q == 3 || q == 5; }  // uz, bz
  static constexpr int NEQ = 1;
  template <typename T>
  __device__ __forceinline__ static void products(const T* v, T* px, T* pz) {
    px[0] = -(v[2] * v[0]) + v[4] * v[1];
    pz[0] = -(v[3] * v[0]) + v[5] * v[1];
  }
  template <typename T>
  __device__ __forceinline__ static void products_split(const T* m, const T* f, T* px, T* pz) {
    px[0] = -bil(m[2], f[2], m[0], f[0]) + bil(m[4], f[4], m[1], f[1]);
    pz[0] = -bil(m[3], f[3], m[0], f[0]) + bil(m[5], f[5], m[1], f[1]);
  }
};
template <> struct BProg<BV_MHD2> {
  static constexpr int NIN = 6;
  static constexpr int UX = 2, UZ = 3;
  static constexpr int FLUX = -1;
  static constexpr bool zero_mean(int q) { return q == 3 || q == 5; }  // uz, bz
  static constexpr int NEQ = 1;
  template <typename T>
  __device__ __forceinline__ static void products(const T* v, T* px, T* pz) {
    px[0] = -(v[2] * v[1]) + v[4] * v[0];
    pz[0] = -(v[3] * v[1]) + v[5] * v[0];
  }
  template <typename T>
  __device__ __forceinline__ static void products_split(const T* m, const T* f, T* px, T* pz) {
    px[0] = -bil(m[2], f[2], m[1], f[1]) + bil(m[4], f[4], m[0], f[0]);
    pz[0] = -bil(m[3], f[3], m[1], f[1]) + bil(m[5], f[5], m[0], f[0]);
  }
};

// The x passes (kernels A and C) hold 2^xp_loge points of a column per
// thread (fft_reg.hpp): 8, and above 1024 points 16 (FP64 at 4096 points 32)
// where that keeps a block of several columns within its threads.  Sixteen
// at 1024 points in single precision leave the update two rows' loads in
// flight per thread instead of four: 180 against 154 us per launch at 16 x
// 1024^2.  The count depends on the precision and the size alone, so a job
// computes the same bits in any batch and block shape.
template <typename T>
__host__ __device__ constexpr int xp_loge(int logn) {
  return sizeof(T) == 4 ? (logn >= 11 ? 4 : 3) : (logn >= 12 ? 5 : logn >= 11 ? 4 : 3);
}
template <typename T>
__host__ __device__ constexpr int xp_tps(int logn) {
  return 1 << (logn - xp_loge<T>(logn));
}
// Columns per block of nt threads, and the LDS they take.
template <typename T>
__host__ __device__ constexpr int xp_cols(int logn, int nt) {
  return nt / xp_tps<T>(logn);
}
template <typename T>
__host__ __device__ constexpr size_t xp_lds_bytes(int logn, int nt) {
  return (size_t)xp_cols<T>(logn, nt) * rf_len(logn, xp_loge<T>(logn)) * sizeof(cx<T>);
}
constexpr size_t kLdsMax = 160 * 1024;
template <typename T>
__host__ __device__ constexpr bool xp_fits(int logn, int nt) {
  return xp_cols<T>(logn, nt) >= 1 && xp_lds_bytes<T>(logn, nt) <= kLdsMax;
}
// The compact spectrum's row of x among n points, -1 for a truncated mode:
// nn = (n - 1) / 3 follows from n, so most rows' cases are decided when a
// size's body is compiled.
__host__ __device__ constexpr int xp_nn(int n) { return (n - 1) / 3; }
__device__ __forceinline__ constexpr int xp_row(int x, int n) {
  return x <= xp_nn(n) ? x : (x >= n - xp_nn(n) ? x - n + 2 * xp_nn(n) + 1 : -1);
}
// Whether thread t's point t + m tps (0 <= t < tps) can be kept for some t.
__host__ __device__ constexpr bool xp_any(int m, int tps, int n) {
  return m * tps <= xp_nn(n) || (m + 1) * tps - 1 >= n - xp_nn(n);
}
// Points per thread (log2) of a mean profile's transform in a block of nt
// threads, and whether it fits.
__host__ __device__ constexpr int mean_loge(int logn, int nt) {
  int e = 3;
  while ((1 << (logn - e)) > nt) ++e;
  return e;
}
__host__ __device__ constexpr bool mean_fits(int logn, int nt) {
  return mean_loge(logn, nt) <= 4;
}
inline size_t mean_lds_bytes(int logn, int nt) {
  return (size_t)rf_len(logn, mean_loge(logn, nt)) * sizeof(cx<float>);
}

// Kernel A's block shapes (BatchLaunch::shapeA): 0, of at most 512 threads in
// single and 256 in double precision; 1, half of shape 0's; 2, mixed tiles
// (stepA_body's MIXED), single precision at 2^9 and 2^10 points with xmix_nt
// threads, when kMixCols columns of every op of any stage fit the block.
// Kernel C's tile shapes (BatchLaunch::wideC): 0 (narrow) of at most 256
// threads; 1 (wide) of 512; 2, single precision in a batch of one x size, whole
// column groups (group_shape; at 2^11 points shape 1's blocks).
// "At most": a batch whose blocks would leave the chip idle takes smaller
// ones (fill_threads in capi.cpp).
constexpr int kMixCols = 2;
__host__ __device__ constexpr int xmix_nt(int logn) {
  return logn == 9 || logn == 10 ? 1024 : 0;
}
inline bool xmix_fits(int logn, int max_nA) {
  return xmix_nt(logn) > 0 && kMixCols * max_nA <= xp_cols<float>(logn, xmix_nt(logn));
}

// Rows per z-pass block: as many as fit the LDS slots, at most 8.
__host__ __device__ constexpr int brows(int nin, int neq, int slots) {
  int best = 1;
  for (int r = 1; r <= 8; ++r) {
    const int need_in = (r * nin + 1) / 2;
    const int need_out = r * neq;
    const int need = need_in > need_out ? need_in : need_out;
    if (need <= slots) best = r;
  }
  return best;
}
__host__ __device__ constexpr bool bfits(int nin, int neq, int slots) {
  return ((nin + 1) / 2 <= slots) && (neq <= slots);
}
// Points per thread of the LDS-staged z pass of a program with nin inputs and
// neq equations: 16 up to N = 1024, which leaves more blocks and a smaller
// register file, and at N = 2048 when the program fits the two slots that
// leaves; otherwise 32.
template <typename T>
__host__ __device__ constexpr int bpoints(int logn, int nin, int neq) {
  return (logn <= 10 || (logn == 11 && bfits(nin, neq, (kNT * 16) >> 11))) ? 16 : 32;
}
__host__ __device__ constexpr int bvar_nin(int v) { return v <= BV_VORT3 ? v + 3 : 6; }
__host__ __device__ constexpr int bvar_neq(int v) { return v <= BV_VORT3 ? v + 1 : 1; }

// Sizes with a choice of z-pass plan: 2^9..2^11 points when the program runs
// at 16 points per thread and fits the slots of the two-sweep pass.
template <typename T>
__host__ __device__ constexpr bool bsplit_fits(int logn, int v) {
  return logn >= 9 && logn <= 11 && bpoints<T>(logn, bvar_nin(v), bvar_neq(v)) == 16 &&
         bfits(bvar_nin(v), bvar_neq(v), (kNT * 16) >> logn);
}
// Plans of the z pass (BatchLaunch::planB).  kPlanTwoSweep runs the sizes
// that bsplit_fits names on the LDS-staged pass in 16,16,R passes both ways,
// the products in a sweep of their own.  kPlanSplit runs them on the register
// pass (stepZ_body) where z_reg_fits, else with the products between the last
// inverse and the first forward pass.
constexpr int kPlanSplit = 0, kPlanTwoSweep = 1;

// The register z pass: 2^logn points over z_tps threads (a wavefront, or
// part of one: 8 points per thread up to 512, 16 at 1024), one wavefront per
// input channel or output, whichever are more.
__host__ __device__ constexpr int z_tps(int logn) { return logn >= 9 ? 64 : 1 << (logn - 3); }
__host__ __device__ constexpr int z_loge(int logn) { return logn >= 9 ? logn - 6 : 3; }
__host__ __device__ constexpr int z_waves(int v) {
  const int in = bvar_nin(v), out = 2 * bvar_neq(v);
  return in > out ? in : out;
}
__host__ __device__ constexpr int z_rows(int logn) { return 2 * (64 / z_tps(logn)); }
template <typename T>
__host__ __device__ constexpr size_t z_lds_bytes(int logn, int v) {
  return (size_t)z_waves(v) * (64 / z_tps(logn)) * rf_len(logn, z_loge(logn)) * sizeof(cx<T>);
}
// Sizes the register pass takes, in double precision: up to 1024 points, 512
// for three fields and for MHD, four of whose six wavefronts have no product
// to transform back.  Above, it loses to the split pass (us per launch,
// register and split: vortex 2048^2 62 and 52, 4 of them 234 and 227, with a
// scalar 81 and 70; MHD 1024^2 24.2 and 23.2, 4 of them 77 and 65; three
// fields 1024^2 29.5 and 29.3, 4 of them 95 and 85; MHD 4 x 512^2 21 and 22,
// vortex 1024^2 16 and 17, three fields 512^2 13 and 15).  The kernel's
// registers are its largest size's: without 1024 points three fields' other
// sizes gain too (32 x 512^2 196 -> 160, 128 x 256^2 204 -> 160).
template <typename T>
__host__ __device__ constexpr bool z_reg_fits(int logn, int v) {
  return sizeof(T) == 8 && logn <= (v >= BV_VORT3 ? 9 : 10);
}
// The LDS-staged pass of double precision is compiled for z extents up to
// 2^kZLo and for all.
constexpr int kZLo = 10;
// Whether program v has a size up to 2^kZLo on that pass under a plan.
template <typename T>
__host__ __device__ constexpr bool z_staged_lo(int v, int plan) {
  return plan == kPlanTwoSweep || !z_reg_fits<T>(kZLo, v);
}
// Whether register m of a thread holds a kept coefficient or its mirror.
__host__ __device__ constexpr bool z_any(int m, int tps, int n) {
  return m * tps < xp_nn(n) || (m + 1) * tps - 1 > n - xp_nn(n);
}
// workspace channel of equation e's Px (k=0) / Pz (k=1) output; the
// z-pass inputs occupy channels [0, base)
__host__ __device__ constexpr int pchan(int base, int e, int k) { return base + 2 * e + k; }

// Layout of the z-pass input channels (kernel A writes them, kernel B reads
// them): x rows in groups of kXil, interleaved by kz, so that one of A's
// column tiles stores runs of kXil x TC elements rather than TC.  Element
// (x, k) of a channel is at xrow_base(x, nm) + kXil k.  Groups of two beat
// four: A's runs are 64 bytes instead of 128 (+10 us at 64 x 1024^2), but a
// z-pass block reads both rows of each group (-32 us).
constexpr int kXil = 2;
__host__ __device__ constexpr size_t xrow_base(int x, int nm) {
  return (size_t)(x / kXil) * (kXil * (size_t)nm) + (size_t)(x % kXil);
}

// LDS slots a z-pass block of `slots` available slots touches: its input
// slots (a row pair's channel per slot when the row count is even, as
// BShape lays them out) or its product slots, whichever is more.  The
// launch sizes the LDS to these alone, so a slot the block never uses does
// not cost blocks per CU (3 of 4 slots for a one-field vortex at 1024 z
// points: 5 blocks per CU instead of 4).
__host__ __device__ constexpr int bslots_used(int nin, int neq, int slots) {
  const int rb = brows(nin, neq, slots);
  const int in = (rb % 2 == 0 && kXil == 2) ? nin * (rb / 2) : (rb * nin + 1) / 2;
  const int out = rb * neq;
  return in > out ? in : out;
}

// Layout of the Px / Pz channels (kernel B writes them, kernel C reads
// them): kz in groups of kPGroup, each group x-major, so element (x, k) is
// at pidx(x, k, nx).  A column tile of kernel C (kPGroup columns, or half
// that) is then one contiguous run, and a z-pass block, which holds a row
// pair, stores each group of both rows as one whole 128-byte line (single
// precision).  Row-major rows cost the update kernel 64-byte runs at a
// stride of a row.
constexpr int kPGroup = 8;
__host__ __device__ constexpr size_t pidx(int x, int k, int nx) {
  return (size_t)(k / kPGroup) * ((size_t)nx * kPGroup) + (size_t)x * kPGroup + (size_t)(k % kPGroup);
}
// Kernel C's shape 2 (stepC_body's GROUP): a group's columns per block, and a
// column's points per thread (log2) and LDS elements.
constexpr int kGroupCols = kPGroup;
constexpr int kGroupPad = 4;  // spare elements a column: the eight differ in bank
__host__ __device__ constexpr int group_loge(int logn) { return logn - 6; }
__host__ __device__ constexpr int group_len(int logn) {
  return rf_len(logn, group_loge(logn)) + kGroupPad;
}
// Sizes it is compiled for: 64 threads a column, and the transform's radices
// (xp_loge) at most its points per thread.
__host__ __device__ constexpr bool group_shape(int logn) { return logn == 9 || logn == 10; }

// Elements per workspace channel: (nx, nm), nm rounded up to whole groups.
__host__ __device__ constexpr size_t work_chs(int nx, int nm) {
  return (size_t)nx * (size_t)((nm + kPGroup - 1) / kPGroup * kPGroup);
}

// Rows of the mean-profile area (the most z-pass input channels).
constexpr int kMeanCh = 6;
// Workspace of a job, in complex elements: the z-pass inputs and the Px/Pz
// outputs, (nin + 2 neq) channels of work_chs, then the mean profiles.
inline size_t fused_work_elems(int nin, int neq, int nx, int nz) {
  const int nm = (nz - 1) / 3;
  return (size_t)(nin + 2 * neq) * work_chs(nx, nm) + (size_t)(kMeanCh / 2) * nz;
}

// A z-pass launch's blocks, LDS and device prefix arrays by stage and program.
struct ZLaunch {
  int n[2][BV_COUNT];
  size_t lds[BV_COUNT];
  int* pref[2][BV_COUNT];
};

struct BatchLaunch {
  int njobs;
  int split;                           // some job carries mean profiles
  int shapeA;                          // block shape of kernel A
  int planB;                           // plan of kernel B (kPlanSplit / kPlanTwoSweep)
  int wideC;                           // tile shape of kernel C
  int nA[2], nC[2];                    // total blocks per launch
  size_t ldsA, ldsC;
  int* prefA[2];                       // device prefix arrays (njobs + 1)
  int* prefC[2];
  // by plan: the jobs on the register z pass, and those on the LDS-staged pass
  ZLaunch z[2], zsweep[2];
  // the shapes of kernels A and C (index = shape): whether every job takes
  // it, threads per block, blocks, LDS and prefix arrays; nA / ldsA / prefA
  // and nC / ldsC / prefC above are the selected one's
  int okA[3], ntA[3], nAp[3][2];
  size_t ldsAp[3];
  int* prefAp[3][2];
  int okC[3], ntC[3], nCp[3][2];
  size_t ldsCp[3];
  int* prefCp[3][2];
  // whether some job's z pass takes the split-pass plan under kPlanSplit
  int splitB;
  // log2 of the x / z size shared by every job, -1 when they differ: a single-
  // precision batch of one z size launches z-pass kernels compiled for that
  // size alone (fixed_logn), whose registers are their own rather than the
  // largest over every size the generic kernels handle
  int lognx_all, lognz_all;
  int lognx_max, lognz_max;            // the largest sizes (log2)
};

// Kernels A and C are compiled for x sizes up to 2^kXpLo and for all, in
// double precision also for up to 2^11: the larger sizes' points per thread
// would set every size's registers.  (2048^2 FP64 in kernel C compiled for 4096
// points, 402 registers, one wavefront per SIMD: 39.7 us a launch, with a
// scalar 76 and 4 of them 293; compiled for 2048, 243 registers: 30.0, 64 and
// 240.)
constexpr int kXpLo = 10;
template <typename T>
constexpr int xp_lo(int logn) {
  return logn <= kXpLo ? kXpLo : (sizeof(T) == 8 && logn == 11 ? 11 : 12);
}

// One-size batches that take kernel C's shape 2, kernel A's mixed tiles and
// single precision's z-pass kernels of one size.
__host__ __device__ constexpr bool fixed_logn(int logn) { return logn >= 9 && logn <= 11; }

// Select kernel A's block shape.
inline void select_a_shape(BatchLaunch& bl, int shape) {
  bl.shapeA = shape;
  bl.ldsA = bl.ldsAp[shape];
  for (int s = 0; s < 2; ++s) {
    bl.nA[s] = bl.nAp[shape][s];
    bl.prefA[s] = bl.prefAp[shape][s];
  }
}

// Select kernel C's tile shape.
inline void select_c_policy(BatchLaunch& bl, int shape) {
  bl.wideC = shape;
  bl.ldsC = bl.ldsCp[shape];
  for (int s = 0; s < 2; ++s) {
    bl.nC[s] = bl.nCp[shape][s];
    bl.prefC[s] = bl.prefCp[shape][s];
  }
}

// `step` is the batch's step count modulo 4 (a multiple of both ring
// lengths and of the ping-pong period), so a captured sequence of 4k steps
// replays correctly.
template <typename T>
hipError_t fused_stage(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                       int step, const cx<T>* tw, hipStream_t s, hipEvent_t* ev = nullptr);
template <typename T>
hipError_t fused_set_dt(JobDev<T>* jobs, int job, double dt, hipStream_t s);
// flags of a stage's z pass: physical outputs, diagnostics partials; with
// kDiag the CFL cadence sits in the bits from kDiagShift up, and a job
// writes partials on the loops whose count before the loop is a multiple of
// it (the reference's ticker fires after loops 1, 1 + cadence, ...)
constexpr int kWritePhys = 1, kDiag = 2, kDiagShift = 8;
// After a step whose z pass ran with kDiag: for each job whose check loop
// it was, reduce its partials, append a tracker record, and apply the CFL
// rule to its dt.
template <typename T>
hipError_t fused_diag(JobDev<T>* jobs, int njobs, double cutoff, int cadence, hipStream_t s);
template <typename T>
hipError_t fused_prepare(const BatchLaunch& bl);

// Launchers and one-time LDS set-up of the three kernel families (one
// translation unit each: fused_a.hip, fused_b.hip, fused_c.hip).
template <typename T>
void launch_xinv(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int step,
                 const cx<T>* tw, hipStream_t s);
template <typename T>
void launch_zpass(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int flags,
                  const cx<T>* tw, hipStream_t s);
template <typename T>
void launch_update(const JobDev<T>* jobs, const BatchLaunch& bl, int stage, int step,
                   const cx<T>* tw, hipStream_t s);
template <typename T>
void prepare_xinv(const BatchLaunch& bl);
template <typename T>
void prepare_zpass(const BatchLaunch& bl);
template <typename T>
void prepare_update(const BatchLaunch& bl);

// Single precision's z pass of program v for a batch of one z size
// (fixed_logn), compiled in its own translation unit (fused_b_fixed.hip).
void launch_zpass_fixed(int v, const JobDev<float>* jobs, const BatchLaunch& bl, int stage,
                        int flags, const cx<float>* tw, hipStream_t s);
void prepare_zpass_fixed(const BatchLaunch& bl);

}  // namespace mlv
