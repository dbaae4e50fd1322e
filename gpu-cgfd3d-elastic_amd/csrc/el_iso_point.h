// el_iso_point.h -- the stage update of one grid point (inner, free-surface and
// PML forms with the fused RK update), and the tile form of the free-surface
// rows that shares it.
#pragma once
#include "el_iso_device.h"
#include "el_iso_launch.h"
#include "el_iso_pml.h"

namespace cgfd {

template <int DIR, typename TC, typename F>
__device__ __forceinline__ TC drp5(F f, long s) {
  constexpr int lo = Drp<TC, DIR>::lo;
  return Drp<TC, DIR>::c(0) * f((lo + 0) * s) + Drp<TC, DIR>::c(1) * f((lo + 1) * s) +
         Drp<TC, DIR>::c(2) * f((lo + 2) * s) + Drp<TC, DIR>::c(3) * f((lo + 3) * s) +
         Drp<TC, DIR>::c(4) * f((lo + 4) * s);
}

// RK update of the wavefield at one point from its right-hand side h (MODE:
// the RK mode, a compile-time constant, so each mode's loads are
// unconditional and issue together)
template <int MODE, typename TS, typename TC>
__device__ __forceinline__ void rk_store(const StageArgs<TS, TC> &a, long so, int o, const TC *h) {
  const long cs = a.L.cs;
  const unsigned qb = (unsigned)o * (unsigned)sizeof(TS);
#pragma unroll
  for (int c = 0; c < kNC; c++) {
    TS *wout = a.w_out + so + c * cs, *wend = a.w_end + so + c * cs;
    const TS *wpre = a.w_pre + so + c * cs, *wu2 = a.w_u2 + so + c * cs;
    const TS *win = a.w_in + so + c * cs;
    const TC sc = St<TS>::scaled ? (TC)a.sc[c] : TC(1);
    const TC is = St<TS>::scaled ? (TC)a.isc[c] : TC(1);
    if constexpr (MODE == MODE_RHS) {
      St<TS>::st(&at_b(wout, qb), h[c] * is);
    } else if constexpr (MODE == MODE_S0) {
      const TC v = (TC)St<TS>::ld(&at_b(win, qb)) * sc;
      St<TS>::st(&at_b(wout, qb), (v + a.ca * h[c]) * is);
    } else if constexpr (MODE == MODE_S12) {
      const TC pre = (TC)St<TS>::ld(&at_b(wpre, qb)) * sc;
      St<TS>::st(&at_b(wout, qb), (pre + a.ca * h[c]) * is);
    } else if constexpr (MODE == MODE_S1Q) {
      const TC pre = (TC)St<TS>::ld(&at_b(wpre, qb)) * sc, u1 = (TC)St<TS>::ld(&at_b(win, qb)) * sc;
      TC u2, q;
      rk_sum(a.rk_w, pre, u1, a.ca, h[c], u2, q);
      St<TS>::st(&at_b(wout, qb), u2 * is);
      St<TS>::st(&at_b(wend, qb), q * is);
    } else if constexpr (MODE == MODE_S3Q) {
      const TC q = (TC)St<TS>::ld(&at_b(wend, qb)) * sc, u3 = (TC)St<TS>::ld(&at_b(win, qb)) * sc;
      St<TS>::st(&at_b(wend, qb), rk_end(a.rk_w, q, u3, a.cb, h[c]) * is);
    } else {
      const TC pre = (TC)St<TS>::ld(&at_b(wpre, qb)) * sc;
      const TC u3 = (TC)St<TS>::ld(&at_b(win, qb)) * sc;
      const TC part = rk_partial(a.rk_w, pre, (TC)St<TS>::ld(&at_b(wend, qb)) * sc, (TC)St<TS>::ld(&at_b(wu2, qb)) * sc);
      St<TS>::st(&at_b(wend, qb), rk_final(pre, part, a.rk_w[2], u3, a.cb * h[c]) * is);
    }
  }
}

// The stage update of one point.  acc.d(axis, c) gives the x and y derivatives
// of component c.  SURF: every point of the call lies on one free-surface row,
// acc.vx / acc.vy hold the conservative traction vectors at the x / y taps, and
// tder says whether the stress derivatives are needed (inner momentum form, PML
// faces).  MET: the metric components that are constant or zero (MetClass) are
// neither loaded nor multiplied.
template <int DX, int DY, int DZ, int MODE, bool SURF, int MET, typename TS, typename TC, typename ACC>
__device__ __forceinline__ void point_update(const StageArgs<TS, TC> &a, int shot, int i, int j, int k, bool tder,
                                             const ACC &acc) {
  const Layout &L = a.L;
  // element offsets inside one component stay below 2^31: 32-bit offsets from
  // uniform component bases let the compiler use scalar-base addressing
  const int o = (int)L.off(i, j, k);
  const long so = (long)shot * a.shot_stride;
  const TS *win = a.w_in + so;
  const long cs = L.cs;
  auto W = [&](int c, long d) -> TC {
    return (TC)St<TS>::ld(&at_b(win + c * cs, (unsigned)(o + (int)d) * (unsigned)sizeof(TS)));
  };
  auto S = [&](int c) -> TC { return St<TS>::scaled ? (TC)a.sc[c] : TC(1); };

  const bool top = a.free_top != 0;
  const int ktop = L.nk - 1;
  constexpr int zlast = (DZ == 0) ? 1 : 3;
  const bool image = top && k >= ktop - zlast;
  TC Dx[kNC], Dy[kNC], Dz[kNC];
#pragma unroll
  for (int c = 0; c < kNC; c++) {
    auto f = [&](long d) { return W(c, d); };
    Dx[c] = Dy[c] = Dz[c] = TC(0);
    if (!SURF || c < 3 || tder) {
      Dx[c] = acc.d(std::integral_constant<int, 0>{}, c);
      Dy[c] = acc.d(std::integral_constant<int, 1>{}, c);
    }
    if (!SURF || !image || c < 3) {
      Dz[c] = drp5<DZ, TC>(f, L.pz);
      if (St<TS>::scaled) Dz[c] *= S(c);
    }
  }
  const TC *met = a.met;
  auto Mt = [&](int m, long d) -> TC {
    return at_b(met + m * cs, (unsigned)(o + (int)d) * (unsigned)sizeof(TC));
  };
  constexpr bool ALL = MET == MET_ALL, CST = MET == MET_CONST;
  const TC xix = ALL ? Mt(XIX, 0) : a.cmet[0], xiy = ALL ? Mt(XIY, 0) : TC(0), xiz = ALL ? Mt(XIZ, 0) : TC(0);
  const TC etx = ALL ? Mt(ETX, 0) : TC(0), ety = ALL ? Mt(ETY, 0) : a.cmet[4], etz = ALL ? Mt(ETZ, 0) : TC(0);
  const TC ztx = CST ? TC(0) : Mt(ZTX, 0), zty = CST ? TC(0) : Mt(ZTY, 0), ztz = CST ? a.cmet[8] : Mt(ZTZ, 0);
  const unsigned ob = (unsigned)o * (unsigned)sizeof(TC);
  const TC lam = at_b(a.med, ob), mu = at_b(a.med + cs, ob), slw = at_b(a.med + 2 * cs, ob);
  // lam + 2.0*mu: the double-promoted sum of the reference rounds to the same
  // float as the float sum whenever lam and 2mu are within 2^29 of each other.
  const TC lam2mu = lam + TC(2) * mu;

  TC h[kNC];
  if (image) {
    // traction image: conservative form with the odd extension of J*zeta.T
    constexpr int zlo = (DZ == 0) ? -3 : -1;
    const int n_free = ktop - k - zlo;
    const TC slwjac = slw / Mt(JAC, 0);
    constexpr int T1[3] = {TXX, TXY, TXZ}, T2[3] = {TXY, TYY, TYZ}, T3[3] = {TXZ, TYZ, TZZ};
#pragma unroll
    for (int cc = 0; cc < 3; cc++) {
      auto vec = [&](long d, int e1, int e2, int e3) -> TC {
        if constexpr (CST) return Mt(JAC, d) * (ztz * (W(T3[cc], d) * S(T3[cc])));  // along z only, see SurfAcc
        return Mt(JAC, d) * (Mt(e1, d) * (W(T1[cc], d) * S(T1[cc])) + Mt(e2, d) * (W(T2[cc], d) * S(T2[cc])) +
                             Mt(e3, d) * (W(T3[cc], d) * S(T3[cc])));
      };
      constexpr int xlo = (DX == 0) ? -3 : -1, ylo = (DY == 0) ? -3 : -1;
      TC DxTx = TC(0), DyTy = TC(0), DzTz = TC(0);
#pragma unroll
      for (int n = 0; n < 5; n++) {
        if constexpr (SURF) {
          DxTx += Drp<TC, DX>::c(n) * acc.vx(cc, n);
          DyTy += Drp<TC, DY>::c(n) * acc.vy(cc, n);
        } else {
          DxTx += Drp<TC, DX>::c(n) * vec((long)(xlo + n), XIX, XIY, XIZ);
          DyTy += Drp<TC, DY>::c(n) * vec((long)(ylo + n) * L.px, ETX, ETY, ETZ);
        }
      }
#pragma unroll
      for (int n = 0; n < 5; n++) {
        TC v;
        if (n < n_free) v = vec((long)(zlo + n) * L.pz, ZTX, ZTY, ZTZ);
        else if (n == n_free) v = TC(0);
        else v = -vec((long)(zlo + n - 2 * (n - n_free)) * L.pz, ZTX, ZTY, ZTZ);
        DzTz += Drp<TC, DZ>::c(n) * v;
      }
      h[VX + cc] = (DxTx + DyTy + DzTz) * slwjac;
    }
  } else if constexpr (!ALL) {
    // here and in the stresses below the roundings are spelled out: the rows ride
    // with the sweep or have a launch of their own, and the compiler fuses other
    // products of a sum in one kernel than in the other
#pragma clang fp contract(off)
    constexpr int T1[3] = {TXX, TXY, TXZ}, T2[3] = {TXY, TYY, TYZ}, T3[3] = {TXZ, TYZ, TZZ};
#pragma unroll
    for (int c = 0; c < 3; c++) {
      TC s = fma_t(xix, Dx[T1[c]], fma_t(ety, Dy[T2[c]], ztz * Dz[T3[c]]));
      if constexpr (!CST) s = fma_t(ztx, Dz[T1[c]], fma_t(zty, Dz[T2[c]], s));
      h[c] = slw * s;
    }
  } else {
    h[VX] = slw * (xix * Dx[TXX] + xiy * Dx[TXY] + xiz * Dx[TXZ] + etx * Dy[TXX] + ety * Dy[TXY] + etz * Dy[TXZ] +
                   ztx * Dz[TXX] + zty * Dz[TXY] + ztz * Dz[TXZ]);
    h[VY] = slw * (xix * Dx[TXY] + xiy * Dx[TYY] + xiz * Dx[TYZ] + etx * Dy[TXY] + ety * Dy[TYY] + etz * Dy[TYZ] +
                   ztx * Dz[TXY] + zty * Dz[TYY] + ztz * Dz[TYZ]);
    h[VZ] = slw * (xix * Dx[TXZ] + xiy * Dx[TYZ] + xiz * Dx[TZZ] + etx * Dy[TXZ] + ety * Dy[TYZ] + etz * Dy[TZZ] +
                   ztx * Dz[TXZ] + zty * Dz[TYZ] + ztz * Dz[TZZ]);
  }

  TC DzVx = Dz[VX], DzVy = Dz[VY], DzVz = Dz[VZ];
  if (top && k >= ktop - 2) {
    const int n = ktop - k;
    if (n == 0) {
      const long pl = (long)L.ni * L.nj, q = (long)j * L.ni + i;
      const TC *A = a.mat + q, *B = a.mat + 9 * pl + q;
      DzVx = A[0] * Dx[VX] + A[pl] * Dx[VY] + A[2 * pl] * Dx[VZ] + B[0] * Dy[VX] + B[pl] * Dy[VY] + B[2 * pl] * Dy[VZ];
      DzVy = A[3 * pl] * Dx[VX] + A[4 * pl] * Dx[VY] + A[5 * pl] * Dx[VZ] + B[3 * pl] * Dy[VX] + B[4 * pl] * Dy[VY] +
             B[5 * pl] * Dy[VZ];
      DzVz = A[6 * pl] * Dx[VX] + A[7 * pl] * Dx[VY] + A[8 * pl] * Dx[VZ] + B[6 * pl] * Dy[VX] + B[7 * pl] * Dy[VY] +
             B[8 * pl] * Dy[VZ];
    } else if (n == 1) {
      // 2nd-order op, layer 1 (fd_t.cu:82-85, 103-106)
      const long z = L.pz;
      if (DZ == 0) {
        DzVx = -W(VX, -z) + W(VX, 0); DzVy = -W(VY, -z) + W(VY, 0); DzVz = -W(VZ, -z) + W(VZ, 0);
      } else {
        DzVx = -W(VX, 0) + W(VX, z); DzVy = -W(VY, 0) + W(VY, z); DzVz = -W(VZ, 0) + W(VZ, z);
      }
      DzVx *= S(VX); DzVy *= S(VY); DzVz *= S(VZ);
    } else {
      // 4th-order op, layer 2 (fd_t.cu:86-89, 107-110)
      const long z = L.pz;
      const TC c0 = (DZ == 0) ? TC(1.0 / 6.0) : TC(-7.0 / 6.0);
      const TC c1 = (DZ == 0) ? TC(-8.0 / 6.0) : TC(8.0 / 6.0);
      const TC c2 = (DZ == 0) ? TC(7.0 / 6.0) : TC(-1.0 / 6.0);
      const long s0 = (DZ == 0) ? -2 * z : 0, s1 = (DZ == 0) ? -z : z, s2 = (DZ == 0) ? 0 : 2 * z;
      DzVx = (c0 * W(VX, s0) + c1 * W(VX, s1) + c2 * W(VX, s2)) * S(VX);
      DzVy = (c0 * W(VY, s0) + c1 * W(VY, s1) + c2 * W(VY, s2)) * S(VY);
      DzVz = (c0 * W(VZ, s0) + c1 * W(VZ, s1) + c2 * W(VZ, s2)) * S(VZ);
    }
  }
  if constexpr (!ALL) {
#pragma clang fp contract(off)
    const TC DzV[3] = {DzVx, DzVy, DzVz};
    // s + dV_c / dx_b
    auto add = [&](TC s, int c, int b) -> TC {
      s = b == 0 ? fma_t(xix, Dx[c], s) : b == 1 ? fma_t(ety, Dy[c], s) : fma_t(ztz, DzV[c], s);
      if constexpr (!CST) {
        if (b < 2) s = fma_t(b == 0 ? ztx : zty, DzV[c], s);
      }
      return s;
    };
    const TC g0 = add(TC(0), 0, 0), g1 = add(TC(0), 1, 1), g2 = ztz * DzV[2];
    h[TXX] = fma_t(lam2mu, g0, lam * add(g2, 1, 1));
    h[TYY] = fma_t(lam2mu, g1, lam * add(g2, 0, 0));
    h[TZZ] = fma_t(lam2mu, g2, lam * add(g1, 0, 0));
    h[TXY] = mu * add(add(TC(0), 1, 0), 0, 1);
    h[TXZ] = mu * add(add(TC(0), 2, 0), 0, 2);
    h[TYZ] = mu * add(add(TC(0), 2, 1), 1, 2);
  } else {
    h[TXX] = lam2mu * (xix * Dx[VX] + etx * Dy[VX] + ztx * DzVx) +
             lam * (xiy * Dx[VY] + ety * Dy[VY] + zty * DzVy + xiz * Dx[VZ] + etz * Dy[VZ] + ztz * DzVz);
    h[TYY] = lam2mu * (xiy * Dx[VY] + ety * Dy[VY] + zty * DzVy) +
             lam * (xix * Dx[VX] + etx * Dy[VX] + ztx * DzVx + xiz * Dx[VZ] + etz * Dy[VZ] + ztz * DzVz);
    h[TZZ] = lam2mu * (xiz * Dx[VZ] + etz * Dy[VZ] + ztz * DzVz) +
             lam * (xix * Dx[VX] + etx * Dy[VX] + ztx * DzVx + xiy * Dx[VY] + ety * Dy[VY] + zty * DzVy);
    h[TXY] = mu * (xiy * Dx[VX] + xix * Dx[VY] + ety * Dy[VX] + etx * Dy[VY] + zty * DzVx + ztx * DzVy);
    h[TXZ] = mu * (xiz * Dx[VX] + xix * Dx[VZ] + etz * Dy[VX] + etx * Dy[VZ] + ztz * DzVx + ztx * DzVz);
    h[TYZ] = mu * (xiz * Dx[VY] + xiy * Dx[VZ] + etz * Dy[VY] + ety * Dy[VZ] + ztz * DzVy + zty * DzVz);
  }

  // ---- CFS-PML faces, in the reference's face order ----
  pml_apply<MODE, TS, TC>(a, shot, i, j, k, Dx, Dy, Dz, xix, xiy, xiz, etx, ety, etz, ztx, zty, ztz, lam, mu, lam2mu,
                          slw, h);
  if constexpr (kBoxedSrc<TS> && MODE != MODE_RHS)
    if (a.sbox) src_add<TS, TC>(a, shot, i, j, k, h);

  rk_store<MODE, TS, TC>(a, so, o, h);
}

// ---- free-surface rows ----
// A workgroup updates one 32x8 tile of one of the 4 rows.  The wavefield, and on
// the rows of the traction image the x and y traction vectors J e.T, are staged
// in LDS once with their halos; a point then reads 90 LDS values where the
// per-point form made 135 loads for its derivatives and 315 more for the image
// (J, three metric terms and three stresses at each of its 45 taps; what is left
// of them are the taps along z).  The rows are latency-bound either way: one row per workgroup instead of
// a march over the four keeps four times as many in flight, which small grids
// need (64x64 columns: 64 workgroups), for z taps that hit the L2.
constexpr int kSurfX = 32, kSurfY = 8, kSurfComp = kNC + 6;
constexpr int kSurfLds = kSurfComp * (kSurfY + 4) * (kSurfX + 4);

template <int DX, int DY, typename TC> struct SurfAcc {
  static constexpr int LW = kSurfX + 4, LH = kSurfY + 4;
  static constexpr int HXL = DX == 0 ? 3 : 1, HYL = DY == 0 ? 3 : 1;
  const TC *lds;
  int lx, ly;
  __device__ __forceinline__ TC at(int c, int row, int col) const { return lds[(c * LH + row) * LW + col]; }
  __device__ __forceinline__ TC d(std::integral_constant<int, 0>, int c) const {
    return drp5<DX, TC>([&](long n) { return at(c, ly + HYL, lx + HXL + (int)n); }, 1);
  }
  __device__ __forceinline__ TC d(std::integral_constant<int, 1>, int c) const {
    return drp5<DY, TC>([&](long n) { return at(c, ly + HYL + (int)n, lx + HXL); }, 1);
  }
  __device__ __forceinline__ TC vx(int cc, int n) const { return at(kNC + cc, ly + HYL, lx + n); }
  __device__ __forceinline__ TC vy(int cc, int n) const { return at(kNC + 3 + cc, ly + n, lx + HXL); }
};

template <int DX, int DY, int DZ, int MODE, int MET, typename TS, typename TC>
__device__ __forceinline__ void surface_tile(const StageArgs<TS, TC> &a, int shot, int tx, int ty, int k, TC *lds) {
  using Acc = SurfAcc<DX, DY, TC>;
  constexpr int LW = Acc::LW, LH = Acc::LH, HXL = Acc::HXL, HYL = Acc::HYL;
  const Layout &L = a.L;
  const int tid = threadIdx.x, lx = tid % kSurfX, ly = tid / kSurfX;
  const int i0 = tx * kSurfX, j0 = ty * kSurfY;
  const int i = i0 + lx, j = j0 + ly;
  const int ktop = L.nk - 1;
  const bool image = k >= ktop - (DZ == 0 ? 1 : 3);
  bool tder = !image;
#pragma unroll
  for (int f = 0; f < 4; f++) {
    const FaceArgs<TS, TC> &F = a.f[f];
    if (F.on && F.i1 < i0 + kSurfX && F.i2 >= i0 && F.j1 < j0 + kSurfY && F.j2 >= j0) tder = true;
  }
  const TS *win = a.w_in + (long)shot * a.shot_stride;
  // stage the point (pi, pj), clamped to the grid and its ghosts, at LDS cell:
  // wavefield, x vectors (vx) and y vectors (vy)
  auto stage = [&](int pi, int pj, int cell, bool vx, bool vy) {
    pi = pi <= L.ni + 2 ? pi : L.ni + 2;
    pj = pj <= L.nj + 2 ? pj : L.nj + 2;
    const unsigned o = (unsigned)L.off(pi, pj, k);
    auto Mt = [&](int m) -> TC { return at_b(a.met + m * L.cs, o * (unsigned)sizeof(TC)); };
    TC w[kNC];
#pragma unroll
    for (int c = 0; c < kNC; c++) {
      w[c] = (TC)St<TS>::ld(&at_b(win + c * L.cs, o * (unsigned)sizeof(TS)));
      if (St<TS>::scaled) w[c] *= (TC)a.sc[c];
    }
    TC J = TC(0), ex[3], ey[3];
    if (image) {
      J = Mt(JAC);
#pragma unroll
      for (int q = 0; q < 3; q++) {
        if constexpr (MET == MET_ALL) {
          ex[q] = vx ? Mt(XIX + q) : TC(0);
          ey[q] = vy ? Mt(ETX + q) : TC(0);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kNC; c++)
      if (c < 3 || tder) lds[c * (LH * LW) + cell] = w[c];
    if (image) {
      constexpr int T1[3] = {TXX, TXY, TXZ}, T2[3] = {TXY, TYY, TYZ}, T3[3] = {TXZ, TYZ, TZZ};
#pragma unroll
      for (int cc = 0; cc < 3; cc++) {
        if constexpr (MET != MET_ALL) {
          if (vx) lds[(kNC + cc) * (LH * LW) + cell] = J * (a.cmet[0] * w[T1[cc]]);
          if (vy) lds[(kNC + 3 + cc) * (LH * LW) + cell] = J * (a.cmet[4] * w[T2[cc]]);
          continue;
        }
        if (vx) lds[(kNC + cc) * (LH * LW) + cell] = J * (ex[0] * w[T1[cc]] + ex[1] * w[T2[cc]] + ex[2] * w[T3[cc]]);
        if (vy) lds[(kNC + 3 + cc) * (LH * LW) + cell] = J * (ey[0] * w[T1[cc]] + ey[1] * w[T2[cc]] + ey[2] * w[T3[cc]]);
      }
    }
  };
  stage(i, j, (ly + HYL) * LW + lx + HXL, true, true);
  if (tid < 4 * kSurfX) {  // y halo: 4 rows of the tile's columns
    const int hrow = tid / kSurfX, row = hrow < HYL ? hrow : kSurfY + hrow;
    stage(i0 + lx, j0 - HYL + row, row * LW + lx + HXL, false, true);
  } else if (tid < 4 * kSurfX + 4 * kSurfY) {  // x halo: 4 columns of the tile's rows
    const int q = tid - 4 * kSurfX, hcol = q % 4, row = q / 4, col = hcol < HXL ? hcol : kSurfX + hcol;
    stage(i0 - HXL + col, j0 + row, (row + HYL) * LW + col, true, false);
  }
  __syncthreads();
  if (i < L.ni && j < L.nj) point_update<DX, DY, DZ, MODE, true, MET>(a, shot, i, j, k, tder, Acc{lds, lx, ly});
}

}  // namespace cgfd
