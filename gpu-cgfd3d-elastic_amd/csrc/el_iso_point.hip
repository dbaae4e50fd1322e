// el_iso_point.hip -- per-point stage kernel of the el_iso RK4 path.
//
// One thread updates one grid point of one shot: 27 one-sided DRP
// derivatives, the momentum/Hooke right-hand side (inner form, or the
// traction-image / vlow forms on the free-surface rows), the CFS-PML ADE
// corrections of every face box containing the point, then the fused RK
// update of the wavefield and of the PML memory (stage-value form, see Mode
// in el_iso_device.h).  It covers any list of boxes: the PML slabs in the shell
// split and the whole domain in the plain method.  Next to a sweep the
// free-surface rows go to k_surface, the tile form of the same update.
//
// Semantics follow, in order, sv_curv_col_el_iso_rhs_inner_gpu
// (src/forward/sv_curv_col_el_iso_gpu.cu:291-452),
// sv_curv_col_el_iso_rhs_timg_z2_gpu (src/forward/sv_curv_col_el_gpu.cu:19-221),
// sv_curv_col_el_iso_rhs_vlow_z2_gpu (sv_curv_col_el_iso_gpu.cu:462-603),
// sv_curv_col_el_iso_rhs_cfspml_gpu (sv_curv_col_el_iso_gpu.cu:680-1147) and the
// RK axpys wav_update / wav_update_end (src/forward/wav_t.cu:362-378) as driven by
// drv_rk_curv_col.cu:339-491.
#include "el_iso_point.h"

namespace cgfd {

// the point of a box list that global thread gid maps to; false past the end
template <typename TS, typename TC>
__device__ __forceinline__ bool box_point(const StageArgs<TS, TC> &a, long gid, int &i, int &j, int &k) {
  int b = 0;
  while (b < a.nbox && gid >= a.box_end[b]) b++;
  if (b >= a.nbox) return false;
  const long loc = gid - (b ? a.box_end[b - 1] : 0);
  const int bx = a.box[b][1] - a.box[b][0] + 1, by = a.box[b][3] - a.box[b][2] + 1;
  i = a.box[b][0] + (int)(loc % bx);
  const long t = loc / bx;
  j = a.box[b][2] + (int)(t % by);
  k = a.box[b][4] + (int)(t / by);
  return true;
}

// derivatives straight from the level in memory
template <int DX, int DY, typename TS, typename TC> struct MemAcc {
  const StageArgs<TS, TC> &a;
  const TS *win;
  int o;
  template <int AXIS> __device__ __forceinline__ TC d(std::integral_constant<int, AXIS>, int c) const {
    auto f = [&](long n) -> TC {
      return (TC)St<TS>::ld(&at_b(win + c * a.L.cs, (unsigned)(o + (int)n) * (unsigned)sizeof(TS)));
    };
    TC v = drp5<AXIS == 0 ? DX : DY, TC>(f, AXIS == 0 ? 1 : a.L.px);
    if (St<TS>::scaled) v *= (TC)a.sc[c];
    return v;
  }
};

template <int DX, int DY, int DZ, int MODE, typename TS, typename TC>
__global__ __launch_bounds__(256) void k_point(StageArgs<TS, TC> a) {
  const int shot = blockIdx.y;
  if (a.shot_active && !a.shot_active[shot]) return;
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int i, j, k;
  if (!box_point(a, gid, i, j, k)) return;
  const MemAcc<DX, DY, TS, TC> acc{a, a.w_in + (long)shot * a.shot_stride, (int)a.L.off(i, j, k)};
  point_update<DX, DY, DZ, MODE, false, MET_ALL>(a, shot, i, j, k, true, acc);
}

// The 4 free-surface rows (surface_tile); workgroups as in the sweep: each XCD
// takes a contiguous eighth of a shot's tiles.
template <int DX, int DY, int DZ, int MODE, int MET, typename TS, typename TC>
__global__ __launch_bounds__(256, 2) void k_surface(StageArgs<TS, TC> a, int ntx, int nty) {
  __shared__ TC lds[kSurfLds];
  const int per_shot = ntx * nty * 4, part = (per_shot + 7) / 8;
  const int xcd = blockIdx.x % 8, m = blockIdx.x / 8;
  const int shot = m / part, q = xcd * part + (m - shot * part);
  if (q >= per_shot || (a.shot_active && !a.shot_active[shot])) return;
  surface_tile<DX, DY, DZ, MODE, MET>(a, shot, q % ntx, q / ntx % nty, a.L.nk - 4 + q / (ntx * nty), lds);
}

// ---- sources (sv_curv_col_el_iso_rhs_src_gpu, sv_curv_col_el_gpu.cu:227-301) ----
// Rates (dU/dt) that the shot's sources give grid point p at stage istage of
// step it, contributions summed in source order; false where none acts.
template <typename TS, typename TC>
__device__ __forceinline__ bool src_rate(const SrcArgs<TS, TC> &a, int p, int it, int istage, TC *v) {
  const long o = a.pt_off[p];
  const TC jac = a.met[JAC * a.L.cs + o], slw = a.med[2 * a.L.cs + o];
#pragma unroll
  for (int c = 0; c < kNC; c++) v[c] = TC(0);
  bool any = false;
  for (int q = a.pt_beg[p]; q < a.pt_beg[p + 1]; q++) {
    const int s = a.ct_src[q];
    if (it < a.s_itb[s] || it > a.s_ite[s]) continue;
    any = true;
    const long ist = a.s_tab[s] + (long)(it - a.s_itb[s]) * 4 + istage;
    const TC coef = a.ct_coef[q];
    if (a.s_kind[s] & 1) {
      const TC V = coef * slw / jac;
      v[VX] += a.F[ist] * V;
      v[VY] += a.F[a.ntab + ist] * V;
      v[VZ] += a.F[2 * a.ntab + ist] * V;
    }
    if (a.s_kind[s] & 2) {
      const TC rjac = coef / jac;
      v[TXX] += -a.M[ist] * rjac;
      v[TYY] += -a.M[a.ntab + ist] * rjac;
      v[TZZ] += -a.M[2 * a.ntab + ist] * rjac;
      v[TYZ] += -a.M[3 * a.ntab + ist] * rjac;
      v[TXZ] += -a.M[4 * a.ntab + ist] * rjac;
      v[TXY] += -a.M[5 * a.ntab + ist] * rjac;
    }
  }
  return any;
}

// One thread per distinct grid point; the rates, from the step's table where
// there is one (10.8 -> 8.7 us on a single moment source: the contributions
// are a chain of dependent loads), are applied to the RK outputs of this stage.  Serves 16-bit storage,
// the bare right-hand side and shots whose sources spread too far for a box (see
// k_step_head).
template <typename TS, typename TC>
__global__ __launch_bounds__(256) void k_source(SrcArgs<TS, TC> a) {
  const int p = a.p0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= a.npt) return;
  const int shot = a.pt_shot[p];
  if (a.only_shot >= 0 && shot != a.only_shot) return;
  if (a.only_shot < 0 && !a.shot_active[shot]) return;
  const int it = a.only_shot >= 0 ? a.fixed_it : *a.clock - a.shot_start[shot];
  const long o = a.pt_off[p];
  const long cs = a.L.cs;
  TC v[kNC];
  if (a.src_v && p < a.npt_box) {
    const int vol = a.sbox[shot].vol();
    const TC *r = a.src_v + a.sbox[shot].off + a.istage * kNC * vol + a.pt_cell[p];
#pragma unroll
    for (int c = 0; c < kNC; c++) v[c] = r[c * vol];
  } else if (!src_rate(a, p, it, a.istage, v)) {
    return;
  }
  const long so = (long)shot * a.shot_stride;
#pragma unroll
  for (int c = 0; c < kNC; c++) {
    if (v[c] == TC(0)) continue;
    const long q = so + c * cs + o;
    const TC sc = St<TS>::scaled ? TC(1) / (TC)a.isc[c] : TC(1);
    const TC is = St<TS>::scaled ? (TC)a.isc[c] : TC(1);
    // stage values take a_i dt of the source (U_{i+1} = W + a_i dt (K_i + S_i)),
    // W^{n+1} takes b3 dt of stage 3's; those of stages 0..2 reach it through
    // U1..U3 (U2's through Q, where S1Q has formed it from the sweep's K1; weight 1)
    if (a.mode == MODE_RHS) {
      St<TS>::st(a.w_out + q, ((TC)St<TS>::ld(a.w_out + q) * sc + v[c]) * is);
    } else if (a.mode == MODE_S0 || a.mode == MODE_S12 || a.mode == MODE_S1Q) {
      St<TS>::st(a.w_out + q, ((TC)St<TS>::ld(a.w_out + q) * sc + a.ca * v[c]) * is);
      if (a.mode == MODE_S1Q) St<TS>::st(a.w_end + q, ((TC)St<TS>::ld(a.w_end + q) * sc + a.ca * v[c]) * is);
    } else {
      St<TS>::st(a.w_end + q, ((TC)St<TS>::ld(a.w_end + q) * sc + a.cb * v[c]) * is);
    }
  }
}

// ---- receivers (io_recv_keep + io_recv_line_interp_pack_buff, io_funcs.cu:1624-1666, 1747-1763) ----
// Corner 5 carries both (x1,y1,z2) and (x2,y1,z2) weights and corner 4 is
// unused, as in the reference; with on-node receivers the quirk vanishes.
template <typename TS, typename TC>
__device__ __forceinline__ void record(const RecvArgs<TS, TC> &a, int t, int clock) {
  if (t >= a.nrec * kNC) return;
  const int r = t / kNC, c = t % kNC;
  const int shot = a.r_shot[r];
  if (a.shot_active && !a.shot_active[shot]) return;
  const int it = clock - a.shot_start[shot];
  if (it < 0 || it >= a.r_nt[r]) return;
  const TS *w = a.w_pre + (long)shot * a.shot_stride + c * a.cs;
  const long *ix = a.r_off + (long)r * 8;
  const TC sc = St<TS>::scaled ? (TC)a.sc[c] : TC(1);
  TC b[8];
#pragma unroll
  for (int q = 0; q < 8; q++) b[q] = (TC)St<TS>::ld(w + ix[q]) * sc;
  const TC Lx2 = a.r_frac[r * 3 + 0], Ly2 = a.r_frac[r * 3 + 1], Lz2 = a.r_frac[r * 3 + 2];
  const TC Lx1 = TC(1) - Lx2, Ly1 = TC(1) - Ly2, Lz1 = TC(1) - Lz2;
  const TC s = b[0] * Lx1 * Ly1 * Lz1 + b[1] * Lx2 * Ly1 * Lz1 + b[2] * Lx1 * Ly2 * Lz1 + b[3] * Lx2 * Ly2 * Lz1 +
               b[5] * Lx1 * Ly1 * Lz2 + b[5] * Lx2 * Ly1 * Lz2 + b[6] * Lx1 * Ly2 * Lz2 + b[7] * Lx2 * Ly2 * Lz2;
  const long pitch = a.ring > 0 ? a.ring : a.r_nt[r];
  a.seismo[a.r_out[r] + (long)c * pitch + (a.ring > 0 ? it % a.ring : it)] = s;
}

// ---- the head of a step ----
// One launch before the four stages: receivers sample W^n (blocks below
// recv_blocks), the source rates of all four stages are tabulated over each
// shot's box (the blocks after), and the step number for the next step is
// written to the other of two clocks, so no block reads a clock that another
// block of the launch writes.  The work is a few thousand threads of dependent
// loads: one launch instead of six (receivers, one source injection per stage,
// clock), each of which took 5-10 us of latency and 3-7 us between launches;
// per step on 64^3 343 -> 200 us with the small z chunks of the sweep.
template <typename TS, typename TC>
__global__ __launch_bounds__(256) void k_step_head(RecvArgs<TS, TC> r, SrcArgs<TS, TC> s, const int *clock,
                                                   int *clock_next, int recv_blocks) {
  const int now = *clock;
  if (blockIdx.x == 0 && threadIdx.x == 0) *clock_next = now + 1;
  if ((int)blockIdx.x < recv_blocks) {
    record(r, blockIdx.x * blockDim.x + threadIdx.x, now);
    return;
  }
  const int t = (blockIdx.x - recv_blocks) * blockDim.x + threadIdx.x;
  if (!s.src_v || t >= 4 * s.npt_box) return;
  const int p = t >> 2, istage = t & 3;
  const int shot = s.pt_shot[p];
  if (!s.shot_active[shot]) return;
  TC v[kNC];
  src_rate(s, p, now - s.shot_start[shot], istage, v);
  const int vol = s.sbox[shot].vol();
  TC *out = s.src_v + s.sbox[shot].off + istage * kNC * vol + s.pt_cell[p];
#pragma unroll
  for (int c = 0; c < kNC; c++) out[c * vol] = v[c];
}

template <typename T> __global__ __launch_bounds__(256) void k_fill(T *p, long n, T v) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long stride = (long)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

// ---- peak ground motion on the free surface (PG_calcu_gpu, src/forward/wav_t.cu:281-360) ----
// After each step, from W^{n+1} (w_new) and W^n (w_old) on the top plane:
// running maxima of |V|, |V_h|, |V_x|, |V_y|, |V_z|, the same for the
// acceleration |dV|/dt and for the displacement integrated with the trapezoid
// rule (accumulated in double, as the reference's 0.5 literal promotes it).
// Maps per shot: [15 maps + 3 displacements][nj][ni].
template <typename TS, typename TC>
__global__ __launch_bounds__(256) void k_peak(const TS *w_new, const TS *w_old, long shot_stride, Layout L, TC *pg,
                                              TC dt, float sx, float sy, float sz, const int *shot_active) {
  const int shot = blockIdx.y;
  if (shot_active && !shot_active[shot]) return;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = L.ni * L.nj;
  if (t >= n) return;
  const int i = t % L.ni, j = t / L.ni;
  const long o = L.off(i, j, L.nk - 1) + (long)shot * shot_stride;
  const long cs = L.cs;
  const TC vx1 = (TC)St<TS>::ld(w_new + o) * (TC)sx, vy1 = (TC)St<TS>::ld(w_new + cs + o) * (TC)sy;
  const TC vz1 = (TC)St<TS>::ld(w_new + 2 * cs + o) * (TC)sz;
  const TC vx0 = (TC)St<TS>::ld(w_old + o) * (TC)sx, vy0 = (TC)St<TS>::ld(w_old + cs + o) * (TC)sy;
  const TC vz0 = (TC)St<TS>::ld(w_old + 2 * cs + o) * (TC)sz;
  TC *m = pg + (long)shot * 18 * n + t;
  const TC Ax = fabs((vx1 - vx0) / dt), Ay = fabs((vy1 - vy0) / dt), Az = fabs((vz1 - vz0) / dt);
  TC Dx = m[15 * n], Dy = m[16 * n], Dz = m[17 * n];
  Dx = (TC)((double)Dx + 0.5 * (double)(vx1 + vx0) * (double)dt);
  Dy = (TC)((double)Dy + 0.5 * (double)(vy1 + vy0) * (double)dt);
  Dz = (TC)((double)Dz + 0.5 * (double)(vz1 + vz0) * (double)dt);
  m[15 * n] = Dx; m[16 * n] = Dy; m[17 * n] = Dz;
  const TC V = sqrt(vx1 * vx1 + vy1 * vy1 + vz1 * vz1), Vh = sqrt(vx1 * vx1 + vy1 * vy1);
  const TC A = sqrt(Ax * Ax + Ay * Ay + Az * Az), Ah = sqrt(Ax * Ax + Ay * Ay);
  const TC D = sqrt(Dx * Dx + Dy * Dy + Dz * Dz), Dh = sqrt(Dx * Dx + Dy * Dy);
  const TC val[15] = {V, Vh, fabs(vx1), fabs(vy1), fabs(vz1), A, Ah, Ax, Ay, Az, D, Dh, fabs(Dx), fabs(Dy), fabs(Dz)};
#pragma unroll
  for (int q = 0; q < 15; q++)
    if (m[q * n] < val[q]) m[q * n] = val[q];
}

// ---- strided sub-volume gather (io_snap_pack_buff, io_funcs.cu:1568-1596) ----
template <typename TS, typename TC>
__global__ __launch_bounds__(256) void k_gather(const TS *w, Layout L, int i1, int j1, int k1, int ni, int nj, int nk,
                                                int di, int dj, int dk, TC scale, TC *out) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long n = (long)ni * nj * nk;
  if (t >= n) return;
  const int i = (int)(t % ni);
  const long r = t / ni;
  const int j = (int)(r % nj), k = (int)(r / nj);
  out[t] = (TC)St<TS>::ld(w + L.off(i1 + i * di, j1 + j * dj, k1 + k * dk)) * scale;
}

// ---- launchers ------------------------------------------------------------------
template <typename TS, typename TC>
hipError_t launch_peak(const TS *w_new, const TS *w_old, long shot_stride, const Layout &L, TC *pg, TC dt,
                       const float *sc, const int *shot_active, int nshots, hipStream_t st) {
  const int n = L.ni * L.nj;
  hipLaunchKernelGGL((k_peak<TS, TC>), dim3((unsigned)((n + 255) / 256), (unsigned)nshots), dim3(256), 0, st, w_new,
                     w_old, shot_stride, L, pg, dt, sc[0], sc[1], sc[2], shot_active);
  return hipGetLastError();
}

template <typename TS, typename TC>
hipError_t launch_gather(const TS *w, const Layout &L, int i1, int j1, int k1, int ni, int nj, int nk, int di,
                         int dj, int dk, TC scale, TC *out, hipStream_t st) {
  const long n = (long)ni * nj * nk;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL((k_gather<TS, TC>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, w, L, i1, j1, k1, ni,
                     nj, nk, di, dj, dk, scale, out);
  return hipGetLastError();
}

// one RK mode's kernel for the operator directions sel = 4 dx + 2 dy + dz
#define CGFD_DIRS(sel)            \
  switch (sel) {                  \
    case 0: CGFD_L(0, 0, 0); break; \
    case 1: CGFD_L(0, 0, 1); break; \
    case 2: CGFD_L(0, 1, 0); break; \
    case 3: CGFD_L(0, 1, 1); break; \
    case 4: CGFD_L(1, 0, 0); break; \
    case 5: CGFD_L(1, 0, 1); break; \
    case 6: CGFD_L(1, 1, 0); break; \
    default: CGFD_L(1, 1, 1); break; \
  }
template <int MODE, typename TS, typename TC>
static void launch_point_m(const StageArgs<TS, TC> &a, dim3 grid, int sel, hipStream_t st) {
  const dim3 block(256);
#define CGFD_L(X, Y, Z) hipLaunchKernelGGL((k_point<X, Y, Z, MODE, TS, TC>), grid, block, 0, st, a)
  CGFD_DIRS(sel)
#undef CGFD_L
}
template <int MODE, int MET, typename TS, typename TC>
static void launch_surface_m(const StageArgs<TS, TC> &a, dim3 grid, int ntx, int nty, int sel, hipStream_t st) {
  const dim3 block(kSurfX * kSurfY);
#define CGFD_L(X, Y, Z) hipLaunchKernelGGL((k_surface<X, Y, Z, MODE, MET, TS, TC>), grid, block, 0, st, a, ntx, nty)
  CGFD_DIRS(sel)
#undef CGFD_L
}

// calls f with the RK mode as a compile-time constant (the modes this storage uses)
template <typename TS, typename F> static void with_mode(int mode, F f) {
  if constexpr (St<TS>::scaled) {
    if (mode == MODE_S3) f(std::integral_constant<int, MODE_S3>{});
  } else {
    if (mode == MODE_S1Q) f(std::integral_constant<int, MODE_S1Q>{});
    if (mode == MODE_S3Q) f(std::integral_constant<int, MODE_S3Q>{});
  }
  if (mode == MODE_S0) f(std::integral_constant<int, MODE_S0>{});
  if (mode == MODE_S12) f(std::integral_constant<int, MODE_S12>{});
  if (mode == MODE_RHS) f(std::integral_constant<int, MODE_RHS>{});
}

template <typename TS, typename TC>
hipError_t launch_point(const StageArgs<TS, TC> &a, int dx, int dy, int dz, int nshots, hipStream_t st) {
  const long n = a.nbox ? a.box_end[a.nbox - 1] : 0;
  if (n == 0) return hipSuccess;
  const dim3 grid((unsigned)((n + 255) / 256), (unsigned)nshots);
  with_mode<TS>(a.mode, [&](auto m) { launch_point_m<decltype(m)::value>(a, grid, dx * 4 + dy * 2 + dz, st); });
  return hipGetLastError();
}

template <typename TS, typename TC>
hipError_t launch_surface(const StageArgs<TS, TC> &a, int dx, int dy, int dz, int nshots, hipStream_t st) {
  if constexpr (St<TS>::scaled) return hipErrorInvalidValue;  // its surface rows go to k_point
  const int ntx = (a.L.ni + kSurfX - 1) / kSurfX, nty = (a.L.nj + kSurfY - 1) / kSurfY;
  const dim3 grid((unsigned)(8L * ((ntx * nty * 4 + 7) / 8) * nshots));
  if constexpr (!St<TS>::scaled)
    with_mode<TS>(a.mode, [&](auto m) {
      constexpr int M = decltype(m)::value;
      const int sel = dx * 4 + dy * 2 + dz;
      if (a.surf_class == MET_CONST) launch_surface_m<M, MET_CONST>(a, grid, ntx, nty, sel, st);
      else if (a.surf_class == MET_VERT) launch_surface_m<M, MET_VERT>(a, grid, ntx, nty, sel, st);
      else launch_surface_m<M, MET_ALL>(a, grid, ntx, nty, sel, st);
    });
  return hipGetLastError();
}

template <typename TS, typename TC> hipError_t launch_source(const SrcArgs<TS, TC> &a, hipStream_t st) {
  if (a.npt <= a.p0) return hipSuccess;
  hipLaunchKernelGGL((k_source<TS, TC>), dim3((a.npt - a.p0 + 255) / 256), dim3(256), 0, st, a);
  return hipGetLastError();
}

template <typename TS, typename TC>
hipError_t launch_step_head(const RecvArgs<TS, TC> &r, const SrcArgs<TS, TC> &s, const int *clock, int *clock_next,
                            hipStream_t st) {
  const int rb = (r.nrec * kNC + 255) / 256, sb = s.src_v ? (4 * s.npt_box + 255) / 256 : 0;
  hipLaunchKernelGGL((k_step_head<TS, TC>), dim3(rb + sb > 0 ? rb + sb : 1), dim3(256), 0, st, r, s, clock, clock_next,
                     rb);
  return hipGetLastError();
}

template <typename T> hipError_t launch_fill(T *p, long n, T v, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  long blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL((k_fill<T>), dim3((unsigned)blocks), dim3(256), 0, st, p, n, v);
  return hipGetLastError();
}

#define CGFD_INST(TS, TC)                                                                                   \
  template hipError_t launch_point<TS, TC>(const StageArgs<TS, TC> &, int, int, int, int, hipStream_t);    \
  template hipError_t launch_surface<TS, TC>(const StageArgs<TS, TC> &, int, int, int, int, hipStream_t);  \
  template hipError_t launch_peak<TS, TC>(const TS *, const TS *, long, const Layout &, TC *, TC, const float *, \
                                          const int *, int, hipStream_t);                                      \
  template hipError_t launch_gather<TS, TC>(const TS *, const Layout &, int, int, int, int, int, int, int, int,   \
                                            int, TC, TC *, hipStream_t);                                        \
  template hipError_t launch_source<TS, TC>(const SrcArgs<TS, TC> &, hipStream_t);                          \
  template hipError_t launch_step_head<TS, TC>(const RecvArgs<TS, TC> &, const SrcArgs<TS, TC> &, const int *, \
                                               int *, hipStream_t);
// CGFD_TYPE selects one storage type per object so the four compile in
// parallel; without it every type is instantiated here.
#if !defined(CGFD_TYPE) || CGFD_TYPE == 0
CGFD_INST(float, float)
#endif
#if !defined(CGFD_TYPE) || CGFD_TYPE == 1
CGFD_INST(double, double)
#endif
#if !defined(CGFD_TYPE) || CGFD_TYPE == 2
CGFD_INST(__half, float)
#endif
#if !defined(CGFD_TYPE) || CGFD_TYPE == 3
CGFD_INST(__hip_bfloat16, float)
#endif
#undef CGFD_INST
#if !defined(CGFD_TYPE) || CGFD_TYPE == 0
template hipError_t launch_fill<float>(float *, long, float, hipStream_t);
template hipError_t launch_fill<double>(double *, long, double, hipStream_t);
template hipError_t launch_fill<uint16_t>(uint16_t *, long, uint16_t, hipStream_t);
template hipError_t launch_fill<int>(int *, long, int, hipStream_t);
#endif

}  // namespace cgfd
