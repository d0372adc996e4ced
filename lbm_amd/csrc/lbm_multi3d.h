// Two D3Q19 steps per pass over memory (k_multi3d): argument block, tile
// geometry and the launcher.
#pragma once
#include <hip/hip_runtime.h>

#include "lbm_launch.h"

namespace lbm {

// What a domain's faces ask of the kernel.
enum : int {
  MULTI3D_BOX = 0,    // periodic, no solids
  MULTI3D_WALLS = 1,  // bounce-back walls (resting or moving), solids; FP64 also NEEM faces across x
  MULTI3D_NONE = -1   // anything else: one step per launch
};
// Threads of a block, one per (x, y) column of its region.  Two planes of 19
// populations per column: 512 columns take 78 KB in FP32, two blocks to a CU
// (FP64: 156 KB, one).  With walls the kernel runs at three waves per SIMD,
// and three blocks of 256 columns run faster than one of 768 (256 x 128 x
// 128 cavity FP32 126 against 136 us a step).
constexpr int multi3d_threads(int esize, int cls) { return cls == MULTI3D_WALLS && esize != 8 ? 256 : 512; }

// Two steps in one pass take longer than two launches with too few columns to
// fill the chip (microseconds per step, this kernel against single steps: FP32
// box of 64^3 9.9 against 8.6; FP32 cavity of 128 x 64 x 64 20.5 against 19.6;
// FP16 box of 128^3 37 against 33; FP64 box of 40^3 6.6 against 6.7; FP64 walls of
// 128 x 32 x 32 9.7 against 8.3, of 256 x 24 x 25 with NEEM faces 1.2 times as
// long, of 128 x 38 x 36 the same; of 24 domains from 131072 to 262144 cells those
// above 196608 all gain, 1 to 37 %), in 16-bit storage with walls, where the masks
// cost more than the halved traffic (512 x 128 x 128 sphere channel 187 against
// 181), and in FP32 with NEEM faces, whose FP64 arithmetic is done for the halo
// too (the same channel 289 against 249; FP64 of 300 x 200 x 101 258 against 437).
// Beyond these bounds multi3d_ratio decides.
inline int multi3d_class(const FaceDev *face, bool solids, long long cells, int esize) {
  int c = solids ? MULTI3D_WALLS : MULTI3D_BOX;
  for (int f = 0; f < 6; ++f) {
    const int k = face[f].kind;
    if (k == LBM_FACE_PERIODIC) continue;
    if (k != LBM_FACE_WALL && !(esize == 8 && f < 2 && (k == LBM_FACE_PRESSURE_NEEM || k == LBM_FACE_VELOCITY_NEEM)))
      return MULTI3D_NONE;
    c = MULTI3D_WALLS;
  }
  const long long least = esize == 8 ? (c == MULTI3D_WALLS ? 3ll << 16 : 1ll << 17)
                          : esize == 4 ? (c == MULTI3D_WALLS ? 3ll << 18 : 1ll << 19)
                                       : (c == MULTI3D_WALLS ? 1ll << 62 : 3ll << 20);
  return cells > least ? c : MULTI3D_NONE;
}

struct Multi3dArgs {
  const void *src;
  void *dst;
  long long plane;
  int nx, ny, nz, px, per[3];
  const FaceDev *face;
  const uint32_t *links;       // null without solids
  const unsigned char *solid;  // per block: it reads link masks (multi3d_solid)
  double omega, F[3];
  // tiles of tw columns along x, nty along y and slabs along z cut evenly; a
  // block takes one tile of one slab
  int tw, ntx, nty, slabs;
};

struct Multi3dPlan {
  int tw, ntx, nty, slabs;
  double cost;  // planes that the busiest CU works through
};
Multi3dPlan multi3d_plan(int nx, int ny, int nz, int esize, int cls);

// Time of the two-step kernel over that of single steps.  lanes: threads of a
// single-step launch, force: a force_kind.
double multi3d_ratio(const Multi3dPlan &p, int nx, int ny, int nz, int esize, int cls, const FaceDev *face, bool solids,
                     int force, double lanes);

// solid[0 .. ntx * nty * slabs) of the plan in a, from a.links
void multi3d_solid(const Multi3dArgs &a, unsigned char *solid, hipStream_t s);

template <typename ST>
struct Multi3dL {
  static void run(const Multi3dArgs &a, hipStream_t s, int cls);
};

}  // namespace lbm
