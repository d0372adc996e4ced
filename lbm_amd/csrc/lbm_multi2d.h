// Several D2Q9 steps per launch on tiles held in LDS: argument block, tile
// geometry (shared by host and device) and the launcher.
#pragma once
#include <hip/hip_runtime.h>

#include "lbm_launch.h"

namespace lbm {

constexpr int MULTI2D_LDS = 80 * 1024;  // LDS of a block: two blocks share a CU's 160 KB

// population slots per direction of a block
constexpr int multi2d_cap(int esize, bool faces) { return (MULTI2D_LDS - 256) / (9 * esize + (faces ? 2 : 0)) / 16 * 16; }

// What a domain's faces ask of the kernel.
enum : int {
  MULTI2D_BOX = 0,    // periodic, no solids
  MULTI2D_WALLS = 1,  // bounce-back walls (resting or moving) and solids
  MULTI2D_OPEN = 2,   // also Zou-He, NEEM or anti-bounce-back faces across x
  MULTI2D_NONE = -1   // anything else: one step per launch
};
inline int multi2d_class(const FaceDev *face, bool solids) {
  int c = solids ? MULTI2D_WALLS : MULTI2D_BOX;
  for (int f = 0; f < 4; ++f) {
    const int k = face[f].kind;
    if (k == LBM_FACE_PERIODIC) continue;
    if (k == LBM_FACE_WALL) {
      if (c == MULTI2D_BOX) c = MULTI2D_WALLS;
    } else if (f < 2 && (k == LBM_FACE_PRESSURE_ABB || k == LBM_FACE_VELOCITY_ZH || k == LBM_FACE_PRESSURE_ZH ||
                         k == LBM_FACE_PRESSURE_NEEM || k == LBM_FACE_VELOCITY_NEEM)) {
      c = MULTI2D_OPEN;
    } else {
      return MULTI2D_NONE;
    }
  }
  return c;
}

// One tile of a batch: the cells [x0, x0 + w) x [y0, y0 + h) of domain d.
struct MultiTile {
  int d, x0, y0, w, h;
};

struct Multi2dArgs {
  const void *src;
  void *dst;
  int steps;
  int ntiles;
  // one domain (tiles null): tile t covers column t % ntx, row t / ntx of a
  // grid of tw x th cells
  long long plane;
  int nx, ny, px, per[2];
  const FaceDev *face;
  const uint32_t *links;
  double omega, F[3];
  int ntx, tw, th;
  // a batch
  const MultiTile *tiles;
  const DomainDev *doms;
  const int *active;
};

// Extent along one axis of a tile's cells [b, e] `back` steps before the
// tile's last state: a cell needs its neighbours one step earlier, and a
// cell on an open face the two cells inward (the anti-bounce-back
// extrapolation, the NEEM neighbour's upstream cells), which only adds
// something where the tile's edge lies on the face's side.
struct Extent {
  int lo, hi;
};
__host__ __device__ inline Extent multi2d_extent(int b, int e, int back, int n, bool periodic) {
  if (periodic) return Extent{b - back, e + back};
  if (back > 0) {
    b = b < n - 2 ? b : n - 2;
    e = e > 1 ? e : 1;
  }
  const int lo = b - back, hi = e + back;
  return Extent{lo > 0 ? lo : 0, hi < n - 1 ? hi : n - 1};
}

// Slots a tile of w x h cells takes at most (k_multi2d: the region with its
// halo and what the in-place shift adds).
__host__ __device__ inline int multi2d_slots(int w, int h, int steps) {
  return (w + 2 * steps) * (h + 2 * steps) + 4 * steps;
}

// Whether the kernel's row of a linear index is exact for a tile of `slots`
// slots in lines of `pitch`: i * (2^20 / w + 1) is above 2^20 i / w by at most
// i, less than the 2^20 / w to the next row.  The general plan's lines are at
// most 144 long (128 cells and 8 steps) and every tile fits multi2d_cap.
constexpr bool multi2d_exact(int slots, int pitch) { return (long long)slots * pitch < 1 << 20; }
static_assert(multi2d_exact(multi2d_cap(2, false), 144), "the widest tiles of the general plan");

// What a plan depends on: a domain of nx x ny cells, `cells` in the whole
// launch.
struct Multi2dDomain {
  int nx, ny;
  long long cells;
  int esize;
  bool faces;   // not MULTI2D_BOX
  bool pery;    // the y axis is periodic
  bool solids;
  int force;    // force_kind
};
// Steps per launch and tile.  steps 1: the single-step kernels are faster.
struct Multi2dPlan {
  int steps, tw, th;
  bool wide;
};
Multi2dPlan multi2d_plan(const Multi2dDomain &d);

template <typename ST>
struct Multi2dL {
  // cls: MULTI2D_BOX, _WALLS or _OPEN; wide: 1024 threads per block instead
  // of 512
  static void run(const Multi2dArgs &a, hipStream_t s, int cls, bool wide);
};

}  // namespace lbm
