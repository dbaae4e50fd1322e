// el_iso_launch.h -- host-callable launchers of the el_iso kernels.
#pragma once
#include "el_iso_device.h"

namespace cgfd {

template <typename TS, typename TC>
hipError_t launch_point(const StageArgs<TS, TC> &a, int dx, int dy, int dz, int nshots, hipStream_t st);

// the 4 free-surface rows of the whole grid
template <typename TS, typename TC>
hipError_t launch_surface(const StageArgs<TS, TC> &a, int dx, int dy, int dz, int nshots, hipStream_t st);

template <typename TS, typename TC> hipError_t launch_source(const SrcArgs<TS, TC> &a, hipStream_t st);

// receivers, source rates of the step (s.src_v set) and *clock_next = *clock + 1
template <typename TS, typename TC>
hipError_t launch_step_head(const RecvArgs<TS, TC> &r, const SrcArgs<TS, TC> &s, const int *clock, int *clock_next,
                            hipStream_t st);

// peak ground motion maps of every shot after one step (free surface only)
template <typename TS, typename TC>
hipError_t launch_peak(const TS *w_new, const TS *w_old, long shot_stride, const Layout &L, TC *pg, TC dt,
                       const float *sc, const int *shot_active, int nshots, hipStream_t st);

// one component's points (i1 + n*di, j1 + m*dj, k1 + l*dk), physical indices,
// into out [nk][nj][ni], multiplied by scale
template <typename TS, typename TC>
hipError_t launch_gather(const TS *w, const Layout &L, int i1, int j1, int k1, int ni, int nj, int nk, int di,
                         int dj, int dk, TC scale, TC *out, hipStream_t st);

template <typename T> hipError_t launch_fill(T *p, long n, T v, hipStream_t st);

// Boxes swept by the z-marching kernel ([i0,i1]x[j0,j1]x[k0,k1], physical,
// inclusive).  Every point must lie at least 4 rows below a free surface.
// With pml set the kernel applies the CFS-PML terms to points inside a face
// box; without it no point of the set may lie in one.
struct MarchSet {
  int nbox;
  int box[6][6];
  int zchunk;  // planes per workgroup along z
  int shape;   // tile shape id, index into kTile
  int pml;     // the boxes reach into PML face boxes
  int surface; // the launch also updates the free-surface rows (see launch_interior)
};

// per-box tile counts, filled by the launcher for the chosen tile shape
struct MarchGrid {
  int ntx[6], nty[6], nzc[6];
  int wg_beg[7];
  int sntx, snty;  // tiles of a free-surface row (0: none)
};

// tile shapes the autotuner chooses from (TX x TY threads, one per column)
constexpr int kNumShapes = 4;
constexpr int kTile[kNumShapes][2] = {{64, 4}, {32, 8}, {64, 8}, {32, 16}};
// Shapes with a sweep of their own for grids of vertical lines (MET_VERT); the
// others, which no FP32 or FP64 grid has chosen, stream all nine components.
// 16-bit storage streams them on every shape: the products that drop would move
// its stored roundings.
template <typename TS> constexpr bool kVertShape(int shape) { return !St<TS>::scaled && shape < 2; }
// the shape whose PML sweep can take the free-surface rows into its launch (its
// workgroup is that of a surface tile); not with 16-bit storage
constexpr int kSurfShape = 1;

template <typename TS, typename TC, int SHAPE>
hipError_t launch_interior_shape(const StageArgs<TS, TC> &a, const MarchSet &b, int dx, int dy, int dz, int nshots,
                                 hipStream_t st);

template <typename TS, typename TC>
hipError_t launch_interior(const StageArgs<TS, TC> &a, const MarchSet &b, int dx, int dy, int dz, int nshots,
                           hipStream_t st) {
  if (b.nbox < 1) return hipSuccess;
  switch (b.shape) {
    case 0: return launch_interior_shape<TS, TC, 0>(a, b, dx, dy, dz, nshots, st);
    case 1: return launch_interior_shape<TS, TC, 1>(a, b, dx, dy, dz, nshots, st);
    case 2: return launch_interior_shape<TS, TC, 2>(a, b, dx, dy, dz, nshots, st);
    default: return launch_interior_shape<TS, TC, 3>(a, b, dx, dy, dz, nshots, st);
  }
}

}  // namespace cgfd
