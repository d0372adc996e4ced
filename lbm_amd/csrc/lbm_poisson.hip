// Poisson (screened Poisson / diffusion-reaction) lattice-Boltzmann step for
// gfx950 and the C ABI of include/lbm_poisson.h.
//
// The reference solves -D lap(phi) + kappa^2-type reaction with a scalar
// BGK scheme (src/lbm/solver.cpp:542-545, 589-611): phi = sum_{i<Q-1} fold_i /
// (1 - w_rest); feq_i = w_i phi, feq_rest = (w_rest - 1) phi; f = (1 - omega)
// fold + omega feq + source * w'_i * phi for the moving populations.  Here
// a step is in pull form on a structured window; the cells of a face with a
// boundary object are rebuilt from their extrapolation cell (non-equilibrium
// extrapolation, bnd_dirichlet.h:367-376) in the same pass, and a launch
// takes several steps (k_poisson_multi).  FP64 storage, unshifted populations
// (the reference's values, ~w phi).  The rest population is not held: nothing
// reads it, phi being a sum over the moving ones.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/lbm_hip.h"
#include "../../include/lbm_poisson.h"
#include "lbm_readback.h"

namespace lbmp {

template <int Q>
struct PLat;
template <>
struct PLat<3> {
  static constexpr int D = 1;
  static constexpr int cx[3] = {-1, 1, 0};
  static constexpr int cy[3] = {0, 0, 0};
  static constexpr double w[3] = {1.0 / 6.0, 1.0 / 6.0, 2.0 / 3.0};
  static constexpr double wp[3] = {0.5, 0.5, 0.0};
};
template <>
struct PLat<5> {
  static constexpr int D = 2;
  static constexpr int cx[5] = {-1, 1, 0, 0, 0};
  static constexpr int cy[5] = {0, 0, -1, 1, 0};
  static constexpr double w[5] = {1.0 / 6.0, 1.0 / 6.0, 1.0 / 6.0, 1.0 / 6.0, 1.0 / 3.0};
  static constexpr double wp[5] = {0.25, 0.25, 0.25, 0.25, 0.0};
};
template <>
struct PLat<9> {
  static constexpr int D = 2;
  static constexpr int cx[9] = {-1, 1, 0, 0, 1, 1, -1, -1, 0};
  static constexpr int cy[9] = {0, 0, -1, 1, 1, -1, -1, 1, 0};
  static constexpr double w[9] = {1.0 / 9.0,  1.0 / 9.0,  1.0 / 9.0,  1.0 / 9.0, 1.0 / 36.0,
                                  1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0, 4.0 / 9.0};
  static constexpr double wp[9] = {0.125, 0.125, 0.125, 0.125, 0.125, 0.125, 0.125, 0.125, 0.0};
};

struct PArgs {
  const double *src;
  double *dst;
  long long plane;  // elements between population planes
  int nx, ny, px;
  const double *phi_old;   // phi of the previous step
  const double *phi_old2;  // phi of the step before that
  double *phi_new;         // phi of this step
  double omega, source;
  int kind[4], prio[4];   // boundary object per face (0: none)
  const double *val[4];   // Dirichlet values along each face
  double *partials;       // check steps: per-block sums of the change of vars
};

// main-direction vectors of the grid (cartesian::dirVec order, 2D diagonals
// 4..7 = +x+y, +x-y, -x-y, -x+y)
__device__ __forceinline__ void dir_vec(int d, int &dx, int &dy) {
  const int tx[8] = {-1, 1, 0, 0, 1, 1, -1, -1};
  const int ty[8] = {0, 0, -1, 1, 1, -1, -1, 1};
  dx = tx[d];
  dy = ty[d];
}
// cartesian::oppositeDir<NDIM> (include/common/math/cartesian.h:22-34)
__device__ __forceinline__ int opposite_dir(int d, int dim) {
  if (d < 2 * dim) return d + 1 - 2 * (d % 2);
  return d > 5 ? d - 2 : d + 2;
}

// Whether the object on face f recomputes vars of cell (x, y) from the
// post-streaming populations while it applies: layer 1 holds its
// extrapolation cells (every object, bnd_dirichlet.h:359), layer 2 the
// second cells of a Neumann object (bnd_neumann.h:50-56); along the face both
// span the cells 1 .. n-2, the corners' extrapolation cells being diagonal.
__device__ __forceinline__ bool recomputed(const PArgs &a, int f, int layer, int x, int y, int dim) {
  const bool yin = dim == 1 || (y >= 1 && y <= a.ny - 2), xin = x >= 1 && x <= a.nx - 2;
  switch (f) {
    case 0: return x == layer && yin;
    case 1: return x == a.nx - 1 - layer && yin;
    case 2: return y == layer && xin;
    default: return y == a.ny - 1 - layer && xin;
  }
}

template <int Q>
__device__ __forceinline__ double phi_of(const double (&g)[Q - 1]) {
  double s = 0;
#pragma unroll
  for (int i = 0; i < Q - 1; ++i) s += g[i];
  return (1.0 / (1.0 - PLat<Q>::w[Q - 1])) * s;
}

// Where a cell's post-streaming populations come from: an interior cell
// gathers its own, a face cell those of its extrapolation cell (gx, gy), with
// the rule of the boundary object it belongs to.
struct PCell {
  int kind;      // 0: interior, else the kind of the object
  int face;      // the object's face
  int gx, gy;    // cell gathered at
  int g2x, g2y;  // Neumann: the second cell inward
  bool fresh;    // Neumann: vars(e) is this step's phi
};
template <int Q>
__device__ __forceinline__ PCell poisson_cell(const PArgs &a, int x, int y) {
  using L = PLat<Q>;
  PCell c = {0, 0, x, y, x, y, false};
  if (x > 0 && x < a.nx - 1 && (L::D == 1 || (y > 0 && y < a.ny - 1))) return c;
  // faces the cell lies on, in direction order -x +x -y +y
  const bool on[4] = {x == 0, x == a.nx - 1, L::D == 2 && y == 0, L::D == 2 && y == a.ny - 1};
  int prio = 0;
#pragma unroll
  for (int f = 0; f < 2 * L::D; ++f)
    if (on[f] && a.kind[f] != 0 && (c.kind == 0 || a.prio[f] > prio)) {
      c.face = f;
      c.kind = a.kind[f];
      prio = a.prio[f];
    }
  // extrapolation direction (bnd_dirichlet.h:289-312): the first missing
  // main direction; a second one makes it the corner diagonal
  int ed = -1;
#pragma unroll
  for (int d = 0; d < 2 * L::D; ++d) {
    if (!on[d]) continue;
    if (ed < 0) ed = d;
    else if (ed == 0 && d == 2) ed = 6;
    else if (ed == 0 && d == 3) ed = 7;
    else if (ed == 1 && d == 3) ed = 4;
    else if (ed == 1 && d == 2) ed = 5;
  }
  const int in = opposite_dir(ed, L::D);
  int dx, dy;
  dir_vec(in, dx, dy);
  c.gx = x + dx;
  c.gy = y + dy;
  c.g2x = c.gx + dx;
  c.g2y = c.gy + dy;
#pragma unroll
  for (int f = 0; f < 2 * L::D; ++f)
    if (a.kind[f] && a.prio[f] < prio)
      c.fresh = c.fresh || recomputed(a, f, 1, c.gx, c.gy, L::D) ||
                (a.kind[f] == LBM_POISSON_NEUMANN && recomputed(a, f, 2, c.gx, c.gy, L::D));
  return c;
}

// The rule of a face cell on its extrapolation cell's populations g (pe their
// phi): non-equilibrium extrapolation to the boundary value pb.
template <int Q>
__device__ __forceinline__ void poisson_face(double pb, double pe, double (&g)[Q - 1]) {
  using L = PLat<Q>;
#pragma unroll
  for (int i = 0; i < Q - 1; ++i) g[i] = L::w[i] * pb + g[i] - L::w[i] * pe;
}
// Neumann, zero gradient (bnd_neumann.h:50-58), from vars(e) and the
// post-streaming phi two cells in.  vars(e) is the previous step's phi unless
// an object applied earlier in the same step recomputed it from the
// post-streaming populations (PCell::fresh).
__device__ __forceinline__ double poisson_neumann(double vars_e, double phi2) { return (4.0 * vars_e - phi2 + 0.0) / 3.0; }

// collision and reaction of population i
template <int Q>
__device__ __forceinline__ double poisson_relax(const PArgs &a, int i, double g, double phi) {
  using L = PLat<Q>;
  const double f = (1.0 - a.omega) * g + a.omega * (L::w[i] * phi);
  return f + a.source * L::wp[i] * phi;
}

// One step per launch: the check steps and a call for a single step.
template <int Q, bool CHECK>
__global__ void __launch_bounds__(256) k_poisson_step(const PArgs a) {
  using L = PLat<Q>;
  const int x = blockIdx.x * 256 + threadIdx.x, y = blockIdx.y;
  double red = 0;
  if (x < a.nx) {
    const long long cell = (long long)x + (long long)a.px * y;
    auto gather = [&](int gx, int gy, double (&v)[Q - 1]) {
#pragma unroll
      for (int i = 0; i < Q - 1; ++i) {
        const long long s = (long long)(gx - L::cx[i]) + (long long)a.px * (gy - L::cy[i]);
        v[i] = __builtin_nontemporal_load(&a.src[i * a.plane + s]);  // streamed once: 2.195 -> 2.076 ms at 8192^2
      }
    };
    const PCell c = poisson_cell<Q>(a, x, y);
    double g[Q - 1];
    gather(c.gx, c.gy, g);
    if (c.kind) {
      const double pe = phi_of<Q>(g);
      double pb;
      if (c.kind == LBM_POISSON_DIRICHLET) {
        pb = a.val[c.face][c.face < 2 ? y : x];
      } else {
        double g2[Q - 1];
        gather(c.g2x, c.g2y, g2);
        pb = poisson_neumann(c.fresh ? pe : a.phi_old[(long long)c.gx + (long long)a.px * c.gy], phi_of<Q>(g2));
      }
      poisson_face<Q>(pb, pe, g);
    }
    const double phi = phi_of<Q>(g);
    if (CHECK) {
      // sumAbsDiff (solver.cpp:809-815) as the check of the next iteration
      // sees it: vars holds the previous step's phi, except where a boundary
      // object rewrote it from this step's post-streaming populations (its
      // face cells and the cells it recomputes), and varsold holds the same
      // one step earlier
      bool touched = c.kind != 0;
#pragma unroll
      for (int f = 0; f < 2 * L::D; ++f)
        if (a.kind[f])
          touched = touched || recomputed(a, f, 1, x, y, L::D) ||
                    (a.kind[f] == LBM_POISSON_NEUMANN && recomputed(a, f, 2, x, y, L::D));
      red = touched ? fabs(phi - a.phi_old[cell]) : fabs(a.phi_old[cell] - a.phi_old2[cell]);
    }
    a.phi_new[cell] = phi;
#pragma unroll
    for (int i = 0; i < Q - 1; ++i) __builtin_nontemporal_store(poisson_relax<Q>(a, i, g[i], phi), &a.dst[i * a.plane + cell]);
  }
  if (CHECK) {
    __shared__ double s[256];
    s[threadIdx.x] = red;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
      if ((int)threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
      __syncthreads();
    }
    if (threadIdx.x == 0) a.partials[blockIdx.x + (long long)gridDim.x * blockIdx.y] = s[0];
  }
}

// Several steps per launch: a block holds a tile with its halo in LDS,
// advances it there and writes the tile's cells once.  The step it replaces
// was bound by the launch on small windows and by HBM on large ones, both
// paid once per `steps` here; the arithmetic (20 FP64 operations a cell) is
// far below either.  What bounds it now: large windows, LDS (8 reads and 8
// writes of 8 bytes per cell update, 1.6 updates per cell and step with the
// halo of 16 x 24 tiles, which load 2.6 times their cells).
// LDS holds one state: a step's cells, at most two per thread, stay in
// registers until every thread has read (no order of the cells to keep,
// which the rules of a face, reaching three cells inward, would ask for).
// On small windows one wave's chain of instructions is what is left, so a
// thread keeps its cells, and all that does not change with the step is
// worked out once: where it gathers, the face's rule and value, the step from
// which the cell is no longer needed.
constexpr int MULTI_CELLS = 1024, MULTI_THREADS = 512, MULTI_RIM = 128;

struct PMulti {
  int steps, tw, th, ntx, ntiles;
  double *phi_prev;  // phi one step before the last, null where nothing will read it
  int write_phi;     // phi of the last step is wanted
};

// Extent along one axis of a tile's cells [b, e] `back` steps earlier: one
// cell more at either end, and a face cell reads up to three cells inward.
struct PExtent {
  int lo, hi;
};
__host__ __device__ inline PExtent multi_extent(int b, int e, int back, int n) {
  if (back == 0 || n == 1) return PExtent{b, e};
  const int lo = (b < n - 3 ? b : n - 3) - back, hi = (e > 2 ? e : 2) + back;
  return PExtent{lo > 0 ? lo : 0, hi < n - 1 ? hi : n - 1};
}

template <int Q>
__global__ void __launch_bounds__(MULTI_THREADS) __attribute__((amdgpu_waves_per_eu(4, 4)))
k_poisson_multi(const PArgs a, const PMulti m) {
  using L = PLat<Q>;
  constexpr int NP = Q - 1, NT = MULTI_THREADS, PER = MULTI_CELLS / NT;
  __shared__ double pop[NP * MULTI_CELLS];
  // phi of the last two steps on the first layer inside each face
  __shared__ double rim[2][4 * MULTI_RIM];
  // contiguous ranges of tiles per XCD, so that tiles sharing a halo share an L2
  const int chunk = (m.ntiles + 7) / 8, id = (int)(blockIdx.x % 8) * chunk + (int)(blockIdx.x / 8);
  if (id >= m.ntiles) return;  // uniform per block (the grid is 8 * chunk)
  const int x0 = (id % m.ntx) * m.tw, y0 = (id / m.ntx) * m.th;
  const int x1 = min(x0 + m.tw, a.nx) - 1, y1 = min(y0 + m.th, a.ny) - 1;
  const PExtent rx = multi_extent(x0, x1, m.steps, a.nx), ry = multi_extent(y0, y1, m.steps, a.ny);
  const int pitch = rx.hi - rx.lo + 1, n = pitch * (ry.hi - ry.lo + 1), tid = (int)threadIdx.x;
  // whether the tile and its halo hold face cells
  const bool faces = rx.lo == 0 || rx.hi == a.nx - 1 || (L::D == 2 && (ry.lo == 0 || ry.hi == a.ny - 1));
  // row of a linear index: exact for indices below 2^10 and widths below 2^7
  // (D1Q3 has one row)
  const unsigned recip = (unsigned)((1 << 20) / pitch + 1);
  auto slot_of = [&](int x, int y) { return (x - rx.lo) + pitch * (y - ry.lo); };
  // a first-layer cell's place in rim, -1 for the others
  auto rim_of = [&](int x, int y) {
    if (x == 1 || x == a.nx - 2) return (x == 1 ? 0 : MULTI_RIM) + y - ry.lo;
    if (L::D == 2 && (y == 1 || y == a.ny - 2)) return (y == 1 ? 2 : 3) * MULTI_RIM + x - rx.lo;
    return -1;
  };
  // steps before the last from which on a cell is needed along one axis
  auto need_of = [](int x, int b, int e, int len) {
    return x >= b && x <= e ? 0 : max(max(min(b, len - 3) - x, x - max(e, 2)), 1);
  };
  // per cell: need; at, its gather slot, with its place in rim plus one in the
  // upper half; rule, 0 or the second cell's slot, 1 Dirichlet / 2 Neumann on
  // this step's phi / 3 on the last one's, and the extrapolation cell's place
  // in rim; val, the Dirichlet value or the extrapolation cell's phi one step
  // before the first
  int need[PER], at[PER], rule[PER] = {};
  double val[PER] = {};
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = tid + k * NT;
    need[k] = m.steps;
    if (i >= n) continue;
    const int ly = L::D == 1 ? 0 : (int)(((unsigned)i * recip) >> 20), x = rx.lo + i - ly * pitch, y = ry.lo + ly;
    const long long cell = (long long)x + (long long)a.px * y;
#pragma unroll
    for (int j = 0; j < NP; ++j) pop[j * MULTI_CELLS + i] = a.src[j * a.plane + cell];
    at[k] = i;
    need[k] = max(need_of(x, x0, x1, a.nx), L::D == 1 ? 0 : need_of(y, y0, y1, a.ny));
    if (!faces) continue;  // uniform
    const PCell c = poisson_cell<Q>(a, x, y);
    if (c.kind && need[k] < m.steps) {
      at[k] = slot_of(c.gx, c.gy);
      const bool fixed = c.kind == LBM_POISSON_DIRICHLET;
      rule[k] = slot_of(c.g2x, c.g2y) | (fixed ? 1 : c.fresh ? 2 : 3) << 12 | rim_of(c.gx, c.gy) << 16;
      val[k] = fixed ? a.val[c.face][c.face < 2 ? y : x] : a.phi_old[(long long)c.gx + (long long)a.px * c.gy];
    }
    at[k] |= (rim_of(x, y) + 1) << 16;
  }
  __syncthreads();
  for (int back = m.steps - 1;; --back) {
    double f[PER][NP], phi[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      if (back < need[k]) continue;
      auto gather = [&](int slot, double (&v)[NP]) {
        // opaque: the compiler otherwise keeps every population's address over
        // the steps, 40 registers
        asm volatile("" : "+v"(slot));
        const double *row[3] = {pop + slot - pitch - 1, pop + slot - 1, pop + slot + pitch - 1};
#pragma unroll
        for (int j = 0; j < NP; ++j) v[j] = row[1 - L::cy[j]][j * MULTI_CELLS + 1 - L::cx[j]];
      };
      gather(at[k] & 0xffff, f[k]);
      phi[k] = phi_of<Q>(f[k]);
      if (rule[k]) {
        const double pe = phi[k];
        const int kind = (rule[k] >> 12) & 15;
        double pb = val[k];
        if (kind > 1) {
          double g2[NP];
          gather(rule[k] & 0xfff, g2);
          const double before = back == m.steps - 1 ? val[k] : rim[back & 1][rule[k] >> 16];
          pb = poisson_neumann(kind == 2 ? pe : before, phi_of<Q>(g2));
        }
        poisson_face<Q>(pb, pe, f[k]);
        phi[k] = phi_of<Q>(f[k]);
      }
#pragma unroll
      for (int j = 0; j < NP; ++j) f[k][j] = poisson_relax<Q>(a, j, f[k][j], phi[k]);
    }
    if (back > 0) {
      __syncthreads();  // every read of this step is done
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        if (back < need[k]) continue;
#pragma unroll
        for (int j = 0; j < NP; ++j) pop[j * MULTI_CELLS + tid + k * NT] = f[k][j];
        if (at[k] >> 16) rim[(back & 1) ^ 1][(at[k] >> 16) - 1] = phi[k];
      }
    }
    if (back == 0 || (back == 1 && m.phi_prev)) {
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        if (need[k] != 0) continue;
        const int i = tid + k * NT, ly = L::D == 1 ? 0 : (int)(((unsigned)i * recip) >> 20);
        const long long cell = (long long)(rx.lo + i - ly * pitch) + (long long)a.px * (ry.lo + ly);
        if (back == 1) {
          m.phi_prev[cell] = phi[k];
          continue;
        }
#pragma unroll
        for (int j = 0; j < NP; ++j) __builtin_nontemporal_store(f[k][j], &a.dst[j * a.plane + cell]);
        if (m.write_phi) a.phi_new[cell] = phi[k];
      }
      if (back == 0) return;
    }
    __syncthreads();
  }
}

// initialCondition: fold = feq(phi0); then phi and the collision of the
// first step.  phi0 itself (the initial vars) also goes to vars0, the slot
// the first step reads as the step before the previous one (the first
// check's varsold)
template <int Q>
__global__ void __launch_bounds__(256) k_poisson_init(const PArgs a, const double *phi0, double *vars0) {
  using L = PLat<Q>;
  const int x = blockIdx.x * 256 + threadIdx.x, y = blockIdx.y;
  if (x >= a.nx) return;
  const long long cell = (long long)x + (long long)a.px * y;
  const double p0 = phi0[x + (long long)a.nx * y];
  vars0[cell] = p0;
  double g[Q - 1];
#pragma unroll
  for (int i = 0; i < Q - 1; ++i) g[i] = L::w[i] * p0;
  const double phi = phi_of<Q>(g);
  a.phi_new[cell] = phi;
#pragma unroll
  for (int i = 0; i < Q - 1; ++i) a.dst[i * a.plane + cell] = poisson_relax<Q>(a, i, g[i], phi);
}

// fixed-order sum of the block partials
__global__ void __launch_bounds__(1024) k_poisson_sum(const double *partials, long long n, double *out) {
  __shared__ double s[1024];
  double acc = 0;
  for (long long b = threadIdx.x; b < n; b += 1024) acc += partials[b];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int k = 512; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = s[0];
}

// phi (padded layout) -> compact host order
__global__ void __launch_bounds__(256) k_poisson_compact(const double *phi, int nx, int ny, int px, double *out) {
  const int x = blockIdx.x * 256 + threadIdx.x, y = blockIdx.y;
  if (x < nx) out[x + (long long)nx * y] = phi[x + (long long)px * y];
}

}  // namespace lbmp

using namespace lbmp;

struct lbm_poisson {
  int Q = 0, nx = 0, ny = 0, px = 0;
  long long plane = 0;
  double omega = 1, source = 0;
  double *buf[2] = {nullptr, nullptr};
  double *phi[3] = {nullptr, nullptr, nullptr};
  int cur = 0;   // buffer holding the current state
  int pcur = 0;  // phi slot of the current state; pcur+2, pcur+1 (mod 3) the two before
  int kind[4] = {0, 0, 0, 0}, prio[4] = {0, 0, 0, 0};
  double *val[4] = {nullptr, nullptr, nullptr, nullptr};
  double *partials = nullptr, *sum = nullptr, *io = nullptr;
  lbm::Readback out;  // staging of the read-backs
  bool faces_set = false, ready = false;
  hipStream_t stream = nullptr;
  std::string err;
};

static thread_local std::string g_perr;

static int pfail(lbm_poisson *h, int code, const std::string &msg) {
  if (h) h->err = msg;
  g_perr = msg;
  return code;
}

#define PCHK(h, call)                                                                       \
  do {                                                                                      \
    hipError_t e_ = (call);                                                                 \
    if (e_ != hipSuccess) return pfail((h), LBM_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

static PArgs pargs(const lbm_poisson *h) {
  PArgs a;
  memset(&a, 0, sizeof(a));
  a.src = h->buf[h->cur];
  a.dst = h->buf[h->cur ^ 1];
  a.plane = h->plane;
  a.nx = h->nx;
  a.ny = h->ny;
  a.px = h->px;
  a.phi_old = h->phi[h->pcur];
  a.phi_old2 = h->phi[(h->pcur + 2) % 3];
  a.phi_new = h->phi[(h->pcur + 1) % 3];
  a.omega = h->omega;
  a.source = h->source;
  for (int f = 0; f < 4; ++f) {
    a.kind[f] = h->kind[f];
    a.prio[f] = h->prio[f];
    a.val[f] = h->val[f];
  }
  a.partials = h->partials;
  return a;
}

static dim3 pgrid(const lbm_poisson *h) { return dim3((h->nx + 255) / 256, h->ny, 1); }

template <bool CHECK>
static void launch_step(lbm_poisson *h) {
  const PArgs a = pargs(h);
  const dim3 g = pgrid(h), b(256);
  if (h->Q == 3) hipLaunchKernelGGL((k_poisson_step<3, CHECK>), g, b, 0, h->stream, a);
  else if (h->Q == 5) hipLaunchKernelGGL((k_poisson_step<5, CHECK>), g, b, 0, h->stream, a);
  else hipLaunchKernelGGL((k_poisson_step<9, CHECK>), g, b, 0, h->stream, a);
  h->cur ^= 1;
  h->pcur = (h->pcur + 1) % 3;
}

// Tiles of a power of two of cells, about one per CU (two at most of 32 x 16)
// and at least 64 cells; windows beyond that take 16 x 24 cells and 6 steps,
// the best of what 1024 cells hold with the halo.  Microseconds per step, next
// best of a sweep and one step per launch last:
//   D2Q5 128^2    8 x 8, 8 steps    1.07   16 x 4, 8    1.11     4.3
//   D2Q9 200x150  16 x 8, 8         1.65   8 x 16, 8    1.55     5.7
//   D2Q9 512^2    32 x 16, 4        3.6    16 x 32, 4   3.7      9.9
//   D2Q9 4096^2   16 x 24, 6        156    32 x 16, 4   176      489
//   D1Q3 100000   512, 48           0.64   512, 16      0.75     4.7
// A window lower than the tile takes wider ones of the same size at most, as far
// as rim holds their lines (its region has the window's rows): 1000000 x 5 D2Q5
// @P5@.
static PMulti multi_plan(const lbm_poisson *h) {
  constexpr int NCU = 256;
  const long long cells = (long long)h->nx * h->ny;
  PMulti m;
  memset(&m, 0, sizeof(m));
  int lg = 6;
  while (lg < 9 && ((long long)NCU << lg) < cells) ++lg;
  if (h->Q == 3) {
    m.tw = 1 << lg;
    m.th = 1;
    m.steps = 48;
  } else if (cells > 2ll * NCU << 9) {
    m.tw = 16;
    m.th = 24;
    m.steps = 6;
  } else {
    m.tw = 1 << (lg + 1) / 2;
    m.th = 1 << lg / 2;
    m.steps = lg < 9 ? 8 : 4;
  }
  const int size = m.tw * m.th;
  m.th = std::min(m.th, h->ny);
  while (2 * m.tw * m.th <= size && 2 * (m.tw + m.steps) <= MULTI_RIM && 2 * (m.tw + m.steps) * m.th <= MULTI_CELLS) m.tw *= 2;
  m.tw = std::min(m.tw, h->nx);
  m.ntx = (h->nx + m.tw - 1) / m.tw;
  m.ntiles = m.ntx * ((h->ny + m.th - 1) / m.th);
  return m;
}

// nsteps > 1 plain steps, split evenly over the launches.  The last two
// states of phi go to the two slots that the next step reads and the one
// after it.
static int launch_multi(lbm_poisson *h, int nsteps) {
  PMulti m = multi_plan(h);
  const int n = nsteps / m.steps + (nsteps % m.steps != 0);
  bool neumann = false;
  for (int f = 0; f < 4; ++f) neumann = neumann || h->kind[f] == LBM_POISSON_NEUMANN;
  const dim3 g((m.ntiles + 7) / 8 * 8), b(MULTI_THREADS);
  for (int i = 0; i < n; ++i) {
    const bool last = i == n - 1;
    m.steps = nsteps / n + (i < nsteps % n ? 1 : 0);
    PArgs a = pargs(h);
    a.phi_new = h->phi[(h->pcur + 2) % 3];
    m.phi_prev = last ? h->phi[(h->pcur + 1) % 3] : nullptr;
    m.write_phi = last || neumann;
    if (h->Q == 3) hipLaunchKernelGGL(k_poisson_multi<3>, g, b, 0, h->stream, a, m);
    else if (h->Q == 5) hipLaunchKernelGGL(k_poisson_multi<5>, g, b, 0, h->stream, a, m);
    else hipLaunchKernelGGL(k_poisson_multi<9>, g, b, 0, h->stream, a, m);
    PCHK(h, hipGetLastError());
    h->cur ^= 1;
    h->pcur = (h->pcur + 2) % 3;
  }
  return LBM_OK;
}

extern "C" {

int lbm_poisson_create(const lbm_poisson_params *p, lbm_poisson **out) {
  if (!p || !out) return pfail(nullptr, LBM_EINVAL, "lbm_poisson_create: null argument");
  *out = nullptr;
  if (p->lattice != 3 && p->lattice != 5 && p->lattice != 9)
    return pfail(nullptr, LBM_EINVAL, "lbm_poisson_create: lattice must be 3 (D1Q3), 5 (D2Q5) or 9 (D2Q9)");
  const int dim = p->lattice == 3 ? 1 : 2;
  if (p->nx < 5 || (dim == 1 && p->ny != 1) || (dim == 2 && p->ny < 5))
    return pfail(nullptr, LBM_EINVAL, "lbm_poisson_create: extents >= 5 (ny = 1 for D1Q3)");
  if (!(p->omega > 0 && p->omega < 2)) return pfail(nullptr, LBM_EINVAL, "lbm_poisson_create: omega must be in (0,2)");
  lbm_poisson *h = new lbm_poisson();
  h->Q = p->lattice;
  h->nx = p->nx;
  h->ny = p->ny;
  h->px = (p->nx + 63) / 64 * 64;
  h->plane = (long long)h->px * h->ny;
  h->omega = p->omega;
  h->source = p->source;
  auto bail = [&](int code, const std::string &msg) {
    pfail(nullptr, code, msg);
    lbm_poisson_destroy(h);
    return code;
  };
  if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) return bail(LBM_EHIP, "lbm_poisson_create: stream");
  const size_t pb = (size_t)h->plane * (h->Q - 1) * sizeof(double);
  for (int k = 0; k < 2; ++k) {
    if (hipMalloc(&h->buf[k], pb) != hipSuccess) return bail(LBM_ENOMEM, "lbm_poisson_create: device memory");
    if (hipMemset(h->buf[k], 0, pb) != hipSuccess) return bail(LBM_EHIP, "lbm_poisson_create: memset");
  }
  for (int k = 0; k < 3; ++k) {
    if (hipMalloc(&h->phi[k], h->plane * sizeof(double)) != hipSuccess)
      return bail(LBM_ENOMEM, "lbm_poisson_create: device memory");
    if (hipMemset(h->phi[k], 0, h->plane * sizeof(double)) != hipSuccess)
      return bail(LBM_EHIP, "lbm_poisson_create: memset");
  }
  const dim3 g = pgrid(h);
  if (hipMalloc(&h->partials, (size_t)g.x * g.y * sizeof(double)) != hipSuccess ||
      hipMalloc(&h->sum, sizeof(double)) != hipSuccess ||
      hipMalloc(&h->io, (size_t)h->nx * h->ny * sizeof(double)) != hipSuccess)
    return bail(LBM_ENOMEM, "lbm_poisson_create: device memory");
  *out = h;
  return LBM_OK;
}

int lbm_poisson_set_faces(lbm_poisson *h, const lbm_poisson_face *faces, int32_t n) {
  if (!h || !faces || n < 0) return pfail(h, LBM_EINVAL, "lbm_poisson_set_faces: bad argument");
  const int nf = h->Q == 3 ? 2 : 4;
  int kind[4] = {0, 0, 0, 0}, prio[4] = {0, 0, 0, 0};
  const double *val[4] = {nullptr, nullptr, nullptr, nullptr};
  for (int i = 0; i < n; ++i) {
    const lbm_poisson_face &f = faces[i];
    if (f.face < 0 || f.face >= nf) return pfail(h, LBM_EINVAL, "lbm_poisson_set_faces: face index out of range");
    if (kind[f.face]) return pfail(h, LBM_EINVAL, "lbm_poisson_set_faces: face described twice");
    if (f.kind != LBM_POISSON_DIRICHLET && f.kind != LBM_POISSON_NEUMANN)
      return pfail(h, LBM_EINVAL, "lbm_poisson_set_faces: kind must be LBM_POISSON_DIRICHLET or LBM_POISSON_NEUMANN");
    if (f.kind == LBM_POISSON_DIRICHLET && !f.value)
      return pfail(h, LBM_EINVAL, "lbm_poisson_set_faces: a Dirichlet face needs its values");
    kind[f.face] = f.kind;
    prio[f.face] = f.priority;
    val[f.face] = f.value;
  }
  for (int f = 0; f < nf; ++f)
    if (!kind[f]) return pfail(h, LBM_EINVAL, "lbm_poisson_set_faces: every face needs a boundary object");
  PCHK(h, hipStreamSynchronize(h->stream));
  for (int f = 0; f < nf; ++f) {
    if (h->val[f]) PCHK(h, hipFree(h->val[f]));
    h->val[f] = nullptr;
    if (kind[f] == LBM_POISSON_DIRICHLET) {
      const int len = f < 2 ? h->ny : h->nx;
      PCHK(h, hipMalloc(&h->val[f], len * sizeof(double)));
      PCHK(h, hipMemcpy(h->val[f], val[f], len * sizeof(double), hipMemcpyHostToDevice));
    }
    h->kind[f] = kind[f];
    h->prio[f] = prio[f];
  }
  h->faces_set = true;
  return LBM_OK;
}

int lbm_poisson_init(lbm_poisson *h, const double *phi0) {
  if (!h || !phi0) return pfail(h, LBM_EINVAL, "lbm_poisson_init: null argument");
  if (!h->faces_set) return pfail(h, LBM_EINVAL, "lbm_poisson_init: lbm_poisson_set_faces first");
  PCHK(h, hipMemcpyAsync(h->io, phi0, (size_t)h->nx * h->ny * sizeof(double), hipMemcpyHostToDevice, h->stream));
  h->cur = 0;
  h->pcur = 0;
  PArgs a = pargs(h);
  a.dst = h->buf[0];
  a.phi_new = h->phi[0];
  const dim3 g = pgrid(h), b(256);
  if (h->Q == 3) hipLaunchKernelGGL(k_poisson_init<3>, g, b, 0, h->stream, a, (const double *)h->io, h->phi[2]);
  else if (h->Q == 5) hipLaunchKernelGGL(k_poisson_init<5>, g, b, 0, h->stream, a, (const double *)h->io, h->phi[2]);
  else hipLaunchKernelGGL(k_poisson_init<9>, g, b, 0, h->stream, a, (const double *)h->io, h->phi[2]);
  PCHK(h, hipGetLastError());
  PCHK(h, hipStreamSynchronize(h->stream));
  h->ready = true;
  return LBM_OK;
}

int lbm_poisson_step(lbm_poisson *h, int32_t nsteps) {
  if (!h || nsteps < 0) return pfail(h, LBM_EINVAL, "lbm_poisson_step: bad argument");
  if (!h->ready) return pfail(h, LBM_EINVAL, "lbm_poisson_step: lbm_poisson_init first");
  if (nsteps > 1) return launch_multi(h, nsteps);
  if (nsteps == 1) launch_step<false>(h);
  PCHK(h, hipGetLastError());
  return LBM_OK;
}

int lbm_poisson_step_check(lbm_poisson *h, double *abs_diff) {
  if (!h || !abs_diff) return pfail(h, LBM_EINVAL, "lbm_poisson_step_check: null argument");
  if (!h->ready) return pfail(h, LBM_EINVAL, "lbm_poisson_step_check: lbm_poisson_init first");
  launch_step<true>(h);
  const dim3 g = pgrid(h);
  hipLaunchKernelGGL(k_poisson_sum, dim3(1), dim3(1024), 0, h->stream, (const double *)h->partials,
                     (long long)g.x * g.y, h->sum);
  PCHK(h, hipGetLastError());
  PCHK(h, hipMemcpyAsync(abs_diff, h->sum, sizeof(double), hipMemcpyDeviceToHost, h->stream));
  PCHK(h, hipStreamSynchronize(h->stream));
  if (!std::isfinite(*abs_diff)) return pfail(h, LBM_DIVERGED, "non-finite values (solution diverged)");
  return LBM_OK;
}

int lbm_poisson_get(lbm_poisson *h, double *phi) {
  if (!h || !phi) return pfail(h, LBM_EINVAL, "lbm_poisson_get: null argument");
  const auto staging = h->out.hold();
  hipLaunchKernelGGL(k_poisson_compact, pgrid(h), dim3(256), 0, h->stream, (const double *)h->phi[h->pcur], h->nx, h->ny,
                     h->px, h->io);
  PCHK(h, hipGetLastError());
  PCHK(h, h->out.copy(phi, h->io, (size_t)h->nx * h->ny * sizeof(double), h->stream));
  return LBM_OK;
}

int lbm_poisson_destroy(lbm_poisson *h) {
  if (!h) return LBM_OK;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  for (int k = 0; k < 2; ++k)
    if (h->buf[k]) (void)hipFree(h->buf[k]);
  for (int k = 0; k < 3; ++k)
    if (h->phi[k]) (void)hipFree(h->phi[k]);
  for (int f = 0; f < 4; ++f)
    if (h->val[f]) (void)hipFree(h->val[f]);
  if (h->partials) (void)hipFree(h->partials);
  if (h->sum) (void)hipFree(h->sum);
  if (h->io) (void)hipFree(h->io);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  return LBM_OK;
}

const char *lbm_poisson_last_error(const lbm_poisson *h) { return h ? h->err.c_str() : g_perr.c_str(); }

}  // extern "C"
