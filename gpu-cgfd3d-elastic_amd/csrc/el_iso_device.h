// el_iso_device.h -- device-side building blocks of the gfx950 el_iso path:
// storage conversion, MacCormack/DRP operator constants, the padded HBM
// layout and the by-value argument blocks of the stage kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>
#include <cstdint>
#include <type_traits>

namespace cgfd {

constexpr int kNG = 3;    // ghost points per side (src/forward/fd_t.cu:64-66)
constexpr int kNC = 9;    // wavefield components
enum Cmp { VX = 0, VY, VZ, TXX, TYY, TZZ, TYZ, TXZ, TXY };
enum Met { JAC = 0, XIX, XIY, XIZ, ETX, ETY, ETZ, ZTX, ZTY, ZTZ, NMET };
// RK modes of a stage kernel.  The classical RK4 step is evaluated from the
// stage values U1..U3 (U_{i+1} = W^n + a_i dt K_i):
//   S0:   U1 = W + a0 dt K0                      (input W^n)
//   S12:  U2 = W + a1 dt K1, U3 = W + a2 dt K2   (input U1 / U2, W^n read at the point)
//   S1Q:  S12's U2, and Q = W + (U1 - W) / 2 + (U2 - W)
//   S3Q:  W^{n+1} = Q + w3 (U3 - Q) + b3 dt K3   (input U3; written over Q)
//   S3:   W^{n+1} = W + w1 (U1 - W) + w2 (U2 - W) + w3 (U3 - W) + b3 dt K3
//         (input U3; written over U1)
// with w_i = b_{i-1} / a_{i-1} = 1/3, 2/3, 1/3, which equals
// W + dt (b0 K0 + b1 K1 + b2 K2 + b3 K3); Q's weights are w1 / (1 - w3) = 1/2 and
// w2 / (1 - w3) = 1.  FP32 and FP64 storage run S0, S1Q, S12, S3Q: Q carries W, U1
// and U2 into the last stage in one level, 108 instead of 117 level words per
// point and step, and S3Q reads 9 words at the point where S3 reads 27 (per
// step, before and after: 400x400x200 Cartesian FP32 5.46 -> 4.96 ms, 64 shots
// of 100x100x60 12.3 -> 10.7 ms, 128x128x96 curvilinear FP64 1.51 -> 1.26 ms).
// Q is stored near W, not near (1 - w3) W, and everything added to it is an
// increment: its rounding reaches W^{n+1} with 1 - w3 = 2/3, the weight that
// U2's has in S3, and a field with no rates keeps its bits (error against 64
// bits, Q scaled by (1 - w3) -> this: 400x400x200 1.3 -> 1.1e-7 after 24 FP32
// steps, 100x100x60 2.7 -> 2.3e-7 after 40, 128x128x96 5.7 -> 5.4e-16 after 24 in
// FP64; S3 1.3e-7, 2.2e-7).  16-bit storage runs S0, S12, S12, S3, so that the sum
// is formed in FP32 from the stored levels and never stored in 16 bits.
// MODE_RHS writes the right-hand side alone (the per-stage operator).
enum Mode { MODE_RHS = 0, MODE_S0 = 1, MODE_S12 = 2, MODE_S3 = 3, MODE_S1Q = 4, MODE_S3Q = 5 };

// What the nine metric components of a grid need per point.
//   MET_ALL:   nine arrays
//   MET_CONST: nothing; xi_x, eta_y, zeta_z are constants and the others zero
//              (Cartesian grid)
//   MET_VERT:  zeta_x, zeta_y, zeta_z; xi_x and eta_y are constants and the other
//              xi, eta terms zero (grid lines in x and y evenly spaced and
//              vertical lines in z: every grid over topography that moves points
//              up and down only)
//   MET_REF:   as MET_CONST, with the products of the zero terms still taken
//              (16-bit storage, see the autotuner)
enum MetClass { MET_ALL = 0, MET_CONST = 1, MET_VERT = 2, MET_REF = 3 };

// ---- storage traits ---------------------------------------------------------
template <typename TS> struct St;
// ld/st: ordinary accesses; ld_nt/st_nt: non-temporal (streamed once, kept
// out of the way of the wavefield planes that the stencil re-reads from L2)
// raw / ld_raw / cvt: the loaded bits kept unconverted (a prefetch buffer
// converts where the value is used, one plane later)
template <> struct St<float> {
  static constexpr bool scaled = false;
  using raw = float;
  __device__ __forceinline__ static raw ld_raw(const float *p) { return *p; }
  __device__ __forceinline__ static raw ld_raw_nt(const float *p) { return __builtin_nontemporal_load(p); }
  __device__ __forceinline__ static float cvt(raw r) { return r; }
  __device__ __forceinline__ static float ld(const float *p) { return *p; }
  __device__ __forceinline__ static void st(float *p, float v) { *p = v; }
  __device__ __forceinline__ static float ld_nt(const float *p) { return __builtin_nontemporal_load(p); }
  __device__ __forceinline__ static void st_nt(float *p, float v) { __builtin_nontemporal_store(v, p); }
};
template <> struct St<double> {
  static constexpr bool scaled = false;
  using raw = double;
  __device__ __forceinline__ static raw ld_raw(const double *p) { return *p; }
  __device__ __forceinline__ static raw ld_raw_nt(const double *p) { return __builtin_nontemporal_load(p); }
  __device__ __forceinline__ static double cvt(raw r) { return r; }
  __device__ __forceinline__ static double ld(const double *p) { return *p; }
  __device__ __forceinline__ static void st(double *p, double v) { *p = v; }
  __device__ __forceinline__ static double ld_nt(const double *p) { return __builtin_nontemporal_load(p); }
  __device__ __forceinline__ static void st_nt(double *p, double v) { __builtin_nontemporal_store(v, p); }
};
template <> struct St<__half> {
  static constexpr bool scaled = true;
  using raw = unsigned short;
  __device__ __forceinline__ static raw ld_raw(const __half *p) { return *reinterpret_cast<const unsigned short *>(p); }
  __device__ __forceinline__ static raw ld_raw_nt(const __half *p) {
    return __builtin_nontemporal_load(reinterpret_cast<const unsigned short *>(p));
  }
  __device__ __forceinline__ static float cvt(raw r) { return __half2float(__ushort_as_half(r)); }
  __device__ __forceinline__ static float ld(const __half *p) { return __half2float(*p); }
  __device__ __forceinline__ static void st(__half *p, float v) { *p = __float2half(v); }
  __device__ __forceinline__ static float ld_nt(const __half *p) {
    const unsigned short u = __builtin_nontemporal_load(reinterpret_cast<const unsigned short *>(p));
    return __half2float(__ushort_as_half(u));
  }
  __device__ __forceinline__ static void st_nt(__half *p, float v) {
    __builtin_nontemporal_store(__half_as_ushort(__float2half(v)), reinterpret_cast<unsigned short *>(p));
  }
};
template <> struct St<__hip_bfloat16> {
  static constexpr bool scaled = true;
  using raw = unsigned short;
  __device__ __forceinline__ static raw ld_raw(const __hip_bfloat16 *p) {
    return *reinterpret_cast<const unsigned short *>(p);
  }
  __device__ __forceinline__ static raw ld_raw_nt(const __hip_bfloat16 *p) {
    return __builtin_nontemporal_load(reinterpret_cast<const unsigned short *>(p));
  }
  // bfloat16 is the upper half of a float
  __device__ __forceinline__ static float cvt(raw r) { return __uint_as_float((unsigned)r << 16); }
  __device__ __forceinline__ static float ld(const __hip_bfloat16 *p) { return __bfloat162float(*p); }
  __device__ __forceinline__ static void st(__hip_bfloat16 *p, float v) { *p = __float2bfloat16(v); }
  __device__ __forceinline__ static float ld_nt(const __hip_bfloat16 *p) {
    // bfloat16 is the upper half of a float
    const unsigned short u = __builtin_nontemporal_load(reinterpret_cast<const unsigned short *>(p));
    return __uint_as_float((unsigned)u << 16);
  }
  __device__ __forceinline__ static void st_nt(__hip_bfloat16 *p, float v) {
    const __hip_bfloat16 b = __float2bfloat16(v);
    unsigned short u;
    __builtin_memcpy(&u, &b, 2);
    __builtin_nontemporal_store(u, reinterpret_cast<unsigned short *>(p));
  }
};

// non-temporal load of a model coefficient
template <typename T> __device__ __forceinline__ T ld_nt(const T &r) { return __builtin_nontemporal_load(&r); }

// Load/store through a uniform base pointer and a 32-bit byte offset: the
// compiler then addresses with a scalar base plus one 32-bit VGPR offset
// (valid while a component stays below 4 GiB).
template <typename T> __device__ __forceinline__ const T &at_b(const T *base, unsigned byte_off) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + byte_off);
}
template <typename T> __device__ __forceinline__ T &at_b(T *base, unsigned byte_off) {
  return *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + byte_off);
}

// ---- the RK combinations (see Mode), one evaluation order for every kernel ----
// S3: partial = w1 (U1 - W) + w2 (U2 - W); W^{n+1} = W + ((partial + w3 (U3 - W)) + b3 dt K3)
template <typename TC> __device__ __forceinline__ TC rk_partial(const TC *w, TC y0, TC u1, TC u2) {
  return w[0] * (u1 - y0) + w[1] * (u2 - y0);
}
template <typename TC> __device__ __forceinline__ TC rk_final(TC y0, TC partial, TC w3, TC u3, TC cbh) {
  return y0 + ((partial + w3 * (u3 - y0)) + cbh);
}
// S1Q and S3Q spell their roundings out: which product of a sum the compiler
// fuses would otherwise differ between the sweep's variants, and at a wave front
// the stages cancel, which made it 4e-6 of a seismogram instead of 1e-10.
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
// S1Q: Q from W, U1 and U2's increment d2 = a1 dt K1 (the increment itself:
// U2's rounding then stays out of Q).  The weights b_i in FP32 lie 3e-8 above
// their fractions, all four alike, which S3 and the per-stage sums of the
// reference carry as a clock that much fast; w[1] = w1 / (1 - w3) / (1/2) - 1 = 4.5e-8
// lends it to K0 and K1 (without it the DRP coefficients' own -6e-8 stands out: 3.0
// against 2.4e-7 of the 100x100x60 explosion after 40 steps).  s + e is the
// exact sum of y0 and t, so Q is rounded once.
template <typename TC>
__device__ __forceinline__ void rk_sum(const TC *w, TC y0, TC u1, TC ca, TC h, TC &u2, TC &q) {
#pragma clang fp contract(off)
  const TC d2 = ca * h;
  u2 = y0 + d2;
  const TC t = fma_t(TC(0.5), u1 - y0, d2);
  const TC s = y0 + t, b = s - y0, e = (y0 - (s - b)) + (t - b);
  q = s + fma_t(w[1], t, e);
}
// S3Q: the 1e-8 by which an FP32 w3 misses 1/3 multiplies U3 - Q, an increment
template <typename TC> __device__ __forceinline__ TC rk_end(const TC *w, TC q, TC u3, TC cb, TC h) {
#pragma clang fp contract(off)
  return q + fma_t(w[2], u3 - q, cb * h);
}

// ---- operator constants (src/forward/fd_t.cu:76-148) ----------------------
// DIR 0 = backward {-3,-2,-1,0,1}, DIR 1 = forward {-1,0,1,2,3}.
template <typename TC, int DIR> struct Drp;
template <typename TC> struct Drp<TC, 0> {
  static constexpr int lo = -3;
  __device__ __forceinline__ static TC c(int n) {
    return n == 0 ? TC(-0.041686285) : n == 1 ? TC(0.333411808) : n == 2 ? TC(-1.250117713)
         : n == 3 ? TC(0.666745142) : TC(0.291647047);
  }
};
template <typename TC> struct Drp<TC, 1> {
  static constexpr int lo = -1;
  __device__ __forceinline__ static TC c(int n) {
    return n == 0 ? TC(-0.291647047) : n == 1 ? TC(-0.666745142) : n == 2 ? TC(1.250117713)
         : n == 3 ? TC(-0.333411808) : TC(0.041686285);
  }
};

// ---- padded HBM layout --------------------------------------------------------
// Physical point (i,j,k), 0-based, lives at (k+3)*pz + (j+3)*px + (i+xa) within a
// component; xa >= 3 aligns i = 0 to 128 bytes, px is the padded row pitch.
struct Layout {
  int ni, nj, nk;
  int xa;
  long px, pz, cs;
  __host__ __device__ __forceinline__ long off(int i, int j, int k) const {
    return (long)(k + kNG) * pz + (long)(j + kNG) * px + (long)(i + xa);
  }
};

// ---- kernel argument blocks ------------------------------------------------------
template <typename TS, typename TM> struct FaceArgs {
  int on, dim;
  int i1, i2, j1, j2, k1, k2;   // physical inclusive box
  int bi, bj;                   // box extents along i and j
  long fsize;                   // points in the box
  long shot_stride;             // elements between shots of this face's buffer
  const TM *A, *B, *D;          // nlay+1 profile values
  // shot-0 level bases, component stride fsize: stage input, W^n, output,
  // the last stage's level (see StageArgs) and U2 (read by S3)
  TS *a_in, *a_pre, *a_out, *a_end, *a_u2;
};

// boxes one per-point launch may cover (the boundary shell splits into at most 26)
constexpr int kMaxBox = 26;

// storage types whose stage kernels add sources from the step's table
template <typename TS> constexpr bool kBoxedSrc = !St<TS>::scaled;

// Bounding box (physical) of one shot's source points; ni = 0: none.  The shot's
// rates of a step are [4 stages][9][nk][nj][ni] from element off of the table.
struct SrcBox {
  int i0, j0, k0, ni, nj, nk;
  long off;
  __host__ __device__ __forceinline__ int vol() const { return ni * nj * nk; }
};

template <typename TS, typename TM> struct StageArgs {
  Layout L;
  const TM *met;   // NMET components, stride L.cs
  const TM *med;   // lam, mu, 1/rho, stride L.cs
  const TM *mat;   // 18 components [c][j][i] on the physical top plane
  int free_top;
  int met_class;   // MetClass of the uploaded metric (sweeps)
  int surf_class;  // the same for the free-surface rows
  TM cmet[9];      // xi_x..zeta_z where the class makes them constant (the zero ones exactly 0)
  FaceArgs<TS, TM> f[6];
  // shot-0 level bases: stage input, W^n, output, the last stage's level (S1Q
  // writes Q, S3Q reads Q and S3 reads U1 there; both write W^{n+1} over it)
  // and U2 (S3)
  TS *w_in, *w_pre, *w_out, *w_end, *w_u2;
  long shot_stride;
  int mode;
  TM ca, cb;      // a_i dt and b_i dt of the stage
  TM rk_w[3];     // w1, w2, w3 of the last stage's combination (S1Q, S3Q: see rk_sum)
  float sc[kNC], isc[kNC];  // storage scale (value = stored*sc) and its inverse
  int nbox;
  int box[kMaxBox][6];      // i1,i2,j1,j2,k1,k2 inclusive, physical
  long box_end[kMaxBox];    // cumulative point counts
  const int *shot_active;   // per-shot 0/1, or null
  // Source rates of this step and stage over each shot's box, added to the
  // right-hand side where it is formed (null: sources come from k_source, and
  // always with 16-bit storage, whose outputs are rounded before the source).
  const SrcBox *sbox;       // [nshots]
  const TM *src_v;          // the table (SrcBox::off)
  int istage;
};

// Source contributions grouped by grid point (CSR), all shots of a session: the
// points of shots with a box first.
template <typename TS, typename TM> struct SrcArgs {
  Layout L;
  int npt, npt_box;         // points; those of shots with a box
  int p0;                   // first point k_source takes
  const int *pt_shot;       // [npt]
  const long *pt_off;       // [npt] layout offset
  const int *pt_beg;        // [npt+1] into contributions
  const int *ct_src;        // [nct] global source id
  const TM *ct_coef;        // [nct]
  const int *s_itb, *s_ite; // [nsrc_total]
  const long *s_tab;        // [nsrc_total] offset of the source's (it,stage) table
  const int *s_kind;        // [nsrc_total] bit0 force, bit1 moment
  const TM *F;              // [3][ntab]
  const TM *M;              // [6][ntab]
  long ntab;
  const TM *met;            // for jac
  const TM *med;            // for 1/rho
  TS *w_out, *w_end;   // stage output (S0..S2) / Q (S1Q), W^{n+1} (S3, S3Q) of each shot
  long shot_stride;
  int mode, istage;
  TM ca, cb;
  const int *clock;         // current global step
  const int *shot_start;    // per-shot start step
  const int *shot_active;
  int only_shot;            // >= 0: inject this shot only, at step fixed_it
  int fixed_it;
  float isc[kNC];
  const int *pt_cell;       // [npt_box] cell in the shot's box
  const SrcBox *sbox;       // [nshots]
  TM *src_v;                // rates of a step tabulated by k_step_head (SrcBox::off), or null
};

template <typename TS, typename TC> struct RecvArgs {
  int nrec;                 // receivers over all shots
  const int *r_shot;
  const long *r_off;        // [nrec][8] layout offsets
  const TC *r_frac;         // [nrec][3]
  const long *r_out;        // [nrec] offset of the receiver's [9][pitch] block in seismo
  const int *r_nt;          // [nrec] samples kept
  int ring;                 // 0: pitch nt, sample it in column it; > 0: pitch ring, column it % ring
  TC *seismo;
  const TS *w_pre;
  long shot_stride, cs;
  const int *clock;
  const int *shot_start;
  const int *shot_active;
  float sc[kNC];
};

}  // namespace cgfd
