// Several D2Q9 steps per launch: every block holds a tile of the domain with
// its halo in LDS, advances it `steps` times there and writes the tile's
// cells once.
//
// What bounds the single-step kernel it replaces: on small domains the
// launch (3.5-4.5 us a step whatever the cell count), on large ones HBM (72 B
// per FP32 cell update, every step).  Here both are paid once per `steps`
// updates; what is left is the FP64 (FP32 for 16-bit storage) arithmetic of
// the updates, for the halo too: 1.2 times as many as cells in 64 x 20 tiles and
// 4 steps, 1.35 in 32 x 32 and 6, 1.8 in 32 x 16 and 8, 3.8 in 8 x 8 and 8, where
// the launch is what counts.
//
// In place: a step overwrites the tile's old state, so LDS holds it once.
// The cells of a step are taken in the order of their slots (row-major, or by
// columns at an open x face), one per thread and round; a round's new values
// are written, after a barrier, a line (pitch or rows) + 2 slots below their
// cells' old ones, two lines where a face's rules reach two lines back, which
// is below whatever a later round still reads.  As the valid region shrinks
// by a row and a column per step the shifted region stays within the slots it
// started from, except along a clipped lower edge, where `pad` slots are left
// in front.
//
// The arithmetic is that of the single-step kernels, and between steps a
// population takes its storage form, so the result equals that many single
// steps bit for bit.
#include "lbm_multi2d.h"

#include <algorithm>

namespace lbm {

// Per-cell word of a domain with faces or solids: bits 0..7, the population
// bounces back (its upstream cell is solid or across a face); WORD_RULE, the
// cell lies on a moving wall or an open face; WORD_SOLID, no update.  Walls
// and obstacles cost a select per load this way; the boundary code of the
// single-step kernels, run every step by every edge wave, took 3-4 us a step.
constexpr uint32_t WORD_RULE = 0x4000u, WORD_SOLID = 0x8000u;

__device__ __forceinline__ int wrap(int c, int n) {
  c %= n;
  return c < 0 ? c + n : c;
}

// The face rules of a cell whose populations h are gathered and bounced back:
// moving walls (Ladd), anti-bounce-back, Zou-He and NEEM across x.  src, word:
// the tile, c: the cell, on: bit f set where the cell lies on face f, kind /
// prio: the faces' in scalar registers, face: the table in LDS.
template <typename ST, int CLS, int CAP>
__device__ __forceinline__ void face_rules(const ST *src, const uint16_t *word, int sx, int sy, int c, unsigned on,
                                           const int (&kind)[4], const int (&prio)[4], const FaceDev *face,
                                           const double *F, typename Store<ST>::R (&h)[9]) {
  using L = Lat<9>;
  using C = typename Store<ST>::C;
  using R = typename Store<ST>::R;
  // population j of a cell on the faces `at` enters across face f and f owns
  // the crossing (the higher priority, ties to the x face)
  auto owned = [&](int j, int f, unsigned at) {
    const int fx = L::cx[j] > 0 ? 0 : 1, fy = L::cy[j] > 0 ? 2 : 3;
    if (!((at >> f) & 1u) || (f < 2 ? L::cx[j] == 0 || f != fx : L::cy[j] == 0 || f != fy)) return false;
    if (L::cx[j] == 0 || L::cy[j] == 0) return true;
    return f < 2 ? !(((at >> fy) & 1u) && prio[fy] > prio[fx]) : !((at >> fx) & 1u) || prio[fy] > prio[fx];
  };
  auto ladd = [&](unsigned at, R (&v)[9]) {
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      if (kind[f] != LBM_FACE_WALL) continue;  // uniform
      const C u0 = C(face[f].u[0]), u1 = C(face[f].u[1]);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (owned(j, f, at)) v[j] = R(C(v[j]) + C(6) * C(L::w[j]) * cdot<9>(j, u0, u1, C(0)));
    }
  };
  ladd(on, h);
  if (CLS != MULTI2D_OPEN) return;
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const int in = f == 0 ? 1 : -1;
    if (kind[f] == LBM_FACE_PRESSURE_ABB) {
      if (!((on >> f) & 1u)) continue;
      C u1[3], u2[3], ue[3];
      cell_velocity<9, ST>(src, CAP, c + in * sx, F[0], F[1], F[2], u1);
      cell_velocity<9, ST>(src, CAP, c + 2 * in * sx, F[0], F[1], F[2], u2);
#pragma unroll
      for (int d = 0; d < 3; ++d) ue[d] = C(1.5) * u1[d] - C(0.5) * u2[d];
      const C vsq = ue[0] * ue[0] + ue[1] * ue[1] + ue[2] * ue[2];
      const C p2 = C(2) * C(face[f].rho);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (L::cx[j] != in || !owned(j, f, on)) continue;
        const C cu = cdot<9>(j, ue[0], ue[1], ue[2]);
        h[j] = R(-C(h[j]) + C(L::w[j]) * (p2 * (C(1) + C(4.5) * cu * cu - C(1.5) * vsq) - C(2)));
      }
    } else if (kind[f] == LBM_FACE_VELOCITY_ZH || kind[f] == LBM_FACE_PRESSURE_ZH) {
      if ((on >> f) & 1u)
        zou_he<9, R>(h, 0, -in, kind[f] == LBM_FACE_VELOCITY_ZH, R(face[f].u[0]), R(face[f].u[1]), R(face[f].u[2]),
                     R(face[f].rho));
    } else if (kind[f] == LBM_FACE_PRESSURE_NEEM || kind[f] == LBM_FACE_VELOCITY_NEEM) {
      if (!((on >> f) & 1u)) continue;
      const int n1 = c + in * sx;
      const uint32_t w1 = word[n1];
      if (w1 & WORD_SOLID) continue;  // the cell keeps its bounce-back values
      // the inward neighbour's populations after streaming
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        const bool back = j < 8 && ((w1 >> j) & 1u);
        h[j] = Store<ST>::ld(src + (back ? L::opp[j] * CAP + n1 : j * CAP + n1 - sx * L::cx[j] - sy * L::cy[j]));
      }
      ladd(on & 12u, h);
      struct {
        const FaceDev *face;
        const double *F;
      } view{face, F};
      neem_correct<9, ST>(view, f, h);
    }
  }
}

// On large lattices the kernel is bound by issuing its FP64 operations, so a
// force that is not there is compiled out (FORCE): 4096 x 2048 FP32, periodic
// without a force 87 -> 67 us a step, channel with a force along x 96 -> 86.
template <typename ST, int CLS, int FORCE, int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 4))) k_multi2d(const Multi2dArgs m) {
  using L = Lat<9>;
  using C = typename Store<ST>::C;
  using R = typename Store<ST>::R;
  constexpr bool FACES = CLS != MULTI2D_BOX;
  constexpr int CAP = multi2d_cap((int)sizeof(ST), FACES);
  __shared__ __align__(16) ST pop[9 * CAP];
  __shared__ uint16_t word[FACES ? CAP : 1];
  __shared__ FaceDev face[FACES ? 4 : 1];
  // contiguous ranges of tiles per XCD, so that tiles sharing a halo share an L2
  constexpr int NXCD = 8;
  const int chunk = (m.ntiles + NXCD - 1) / NXCD;
  const int id = (int)(blockIdx.x % NXCD) * chunk + (int)(blockIdx.x / NXCD);
  if (id >= m.ntiles || (int)(blockIdx.x / NXCD) >= chunk) return;  // uniform per block
  const ST *src = static_cast<const ST *>(m.src);
  ST *dst = static_cast<ST *>(m.dst);
  const uint32_t *links = m.links;
  const FaceDev *gface = m.face;
  long long plane = m.plane;
  int nx = m.nx, ny = m.ny, px = m.px, x0, y0, x1, y1;
  bool perx = !FACES || m.per[0], pery = !FACES || m.per[1];
  double omega_ = m.omega;
  if (FACES && m.tiles) {
    const MultiTile t = m.tiles[id];
    if (!m.active[t.d]) return;
    const DomainDev &d = m.doms[t.d];
    src += d.pop_off;
    dst += d.pop_off;
    links += d.cell_off;
    plane = d.plane;
    nx = d.nx;
    ny = d.ny;
    px = d.px;
    perx = d.per[0] != 0;
    pery = d.per[1] != 0;
    gface = d.face;
    omega_ = d.omega;
    x0 = t.x0;
    y0 = t.y0;
    x1 = x0 + t.w - 1;
    y1 = y0 + t.h - 1;
  } else {
    x0 = (id % m.ntx) * m.tw;
    y0 = (id / m.ntx) * m.th;
    x1 = min(x0 + m.tw, nx) - 1;
    y1 = min(y0 + m.th, ny) - 1;
  }
  const int tid = (int)threadIdx.x;
  // face kinds and priorities in scalar registers; `rules`, faces whose cells
  // need more than bounce-back
  int kind[4] = {0, 0, 0, 0}, prio[4] = {0, 0, 0, 0};
  unsigned rules = 0;
  if (FACES) {
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      kind[f] = gface[f].kind;
      prio[f] = gface[f].prio;
      const bool rest = kind[f] == LBM_FACE_WALL && gface[f].u[0] == 0.0 && gface[f].u[1] == 0.0;
      if (kind[f] != LBM_FACE_PERIODIC && !rest) rules |= 1u << f;
    }
    if (tid < 4) face[tid] = gface[tid];
    __syncthreads();
  }
  const int T = m.steps;
  const Extent rx = multi2d_extent(x0, x1, T, nx, perx), ry = multi2d_extent(y0, y1, T, ny, pery);
  const int pitch = rx.hi - rx.lo + 1, rows = ry.hi - ry.lo + 1;
  // Tiles at an open x face go column by column, in LDS and in the order of
  // the cells: the face's rules, as long as the rest of the update, are then
  // taken by the wave that holds the column and not by every wave (NEEM
  // channel of 256 x 128 FP32 3.3 -> 2.85 us a step, of 512^2 FP64 7.7 -> 5.8,
  // of 512^2 FP32 8.1 -> 5.5 against 7.5 with one step per launch).  A cell on
  // the upper face reaches two columns back.
  const bool columns = CLS == MULTI2D_OPEN && !perx && ((rx.lo == 0 && kind[0] != LBM_FACE_WALL) || (rx.hi == nx - 1 && kind[1] != LBM_FACE_WALL));
  const int sx = columns ? rows : 1, sy = columns ? 1 : pitch;  // slots from a cell to the next
  // slots a step's state moves down by; hx: the last column it updates
  auto shift_of = [&](int hx) { return columns ? (hx == nx - 1 && kind[1] != LBM_FACE_WALL ? 2 : 1) * rows + 2 : pitch + 2; };
  int pad = 0;
  for (int s = 1, down = 0; s < T; ++s) {
    const Extent ex = multi2d_extent(x0, x1, T - s, nx, perx), ey = multi2d_extent(y0, y1, T - s, ny, pery);
    down += shift_of(ex.hi);
    pad = max(pad, down - (ey.lo - ry.lo) * sy - (ex.lo - rx.lo) * sx);
  }
  // the domain's first and last cell in the tile's coordinates (beyond reach
  // on a periodic axis)
  const int flo0 = perx ? -1 : -rx.lo, fhi0 = perx ? -1 : nx - 1 - rx.lo, flo1 = pery ? -1 : -ry.lo,
            fhi1 = pery ? -1 : ny - 1 - ry.lo;
  auto faces_of = [&](int x, int y) {
    return (x == flo0 ? 1u : 0u) | (x == fhi0 ? 2u : 0u) | (y == flo1 ? 4u : 0u) | (y == fhi1 ? 8u : 0u);
  };
  // row of a linear index: exact where index * width < 2^20 (multi2d_exact)
  auto recip = [](int w) { return (unsigned)((1 << 20) / w + 1); };
  {
    const unsigned rp = recip(pitch);
    for (int i = tid; i < rows * pitch; i += NT) {
      const int ly = (int)(((unsigned)i * rp) >> 20), lx = i - ly * pitch;
      int gx = rx.lo + lx, gy = ry.lo + ly;
      if (perx) gx = wrap(gx, nx);
      if (pery) gy = wrap(gy, ny);
      const unsigned cell = (unsigned)gx + (unsigned)px * (unsigned)gy;
#pragma unroll
      for (int j = 0; j < 9; ++j) pop[j * CAP + pad + lx * sx + ly * sy] = src[j * plane + cell];
      if (FACES) {
        uint32_t w = 0;
        if (links) {
          const uint32_t l = links[cell];
          w = (l & 0xffu) | ((l & LINK_SELF_SOLID) >> 16);
        }
        const unsigned on = faces_of(lx, ly);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (on & ((L::cx[j] > 0 ? 1u : (L::cx[j] < 0 ? 2u : 0u)) | (L::cy[j] > 0 ? 4u : (L::cy[j] < 0 ? 8u : 0u))))
            w |= 1u << j;
        if (on & rules) w |= WORD_RULE;
        word[lx * sx + ly * sy] = (uint16_t)w;
      }
    }
  }
  const C omega = scalar(C(omega_));
  const C Fx = C(m.F[0]), Fy = C(m.F[1]), Fz = C(m.F[2]);
  int at = pad;  // where the state starts
  for (int s = 1; s <= T; ++s) {
    const Extent ex = multi2d_extent(x0, x1, T - s, nx, perx), ey = multi2d_extent(y0, y1, T - s, ny, pery);
    const int w = ex.hi - ex.lo + 1, rs = ey.hi - ey.lo + 1, cells = w * rs;
    const int line = columns ? rs : w;
    const unsigned rl = recip(line);
    const bool last = s == T;
    const ST *in = pop + at;
    at -= shift_of(ex.hi);
    ST *out = pop + at;  // not used in the last step
    __syncthreads();  // the load, or the previous step's last writes
    for (int base = 0; base < cells; base += NT) {
      const int k = base + tid;
      const bool here = k < cells;
      const int q = (int)(((unsigned)k * rl) >> 20), r = k - q * line;
      const int x = (columns ? q : r) + (ex.lo - rx.lo), y = (columns ? r : q) + (ey.lo - ry.lo);
      const int c = x * sx + y * sy;
      ST f[9];
#pragma unroll
      for (int j = 0; j < 9; ++j) f[j] = ST(0.0f);  // a solid cell's populations stay zero
      const uint32_t cw = FACES && here ? word[c] : 0u;
      const bool live = here && !(cw & WORD_SOLID);
      if (live) {
        R h[9];
        if (FACES && __ballot(cw != 0)) {
#pragma unroll
          for (int j = 0; j < 9; ++j) {
            const bool back = j < 8 && ((cw >> j) & 1u);
            h[j] = Store<ST>::ld(in + (back ? L::opp[j] * CAP + c : j * CAP + c - sx * L::cx[j] - sy * L::cy[j]));
          }
          if (__ballot(cw & WORD_RULE))
            face_rules<ST, CLS, CAP>(in, word, sx, sy, c, faces_of(x, y), kind, prio, face, m.F, h);
        } else {
#pragma unroll
          for (int j = 0; j < 9; ++j) h[j] = Store<ST>::ld(in + j * CAP + c - sx * L::cx[j] - sy * L::cy[j]);
        }
        const Moments<9, C> mo = moments<9, C, FORCE>(h, Fx, Fy, Fz);
        collide<9, ST, FORCE>(h, mo, omega, Fx, Fy, Fz, true, [&](int j, C value) { Store<ST>::st(&f[j], value); });
      }
      if (!last) {
        __syncthreads();  // every read of this round is done
        if (here)
#pragma unroll
          for (int j = 0; j < 9; ++j) out[j * CAP + c] = f[j];
      } else if (live) {
        const unsigned cell = (unsigned)(x + rx.lo) + (unsigned)px * (unsigned)(y + ry.lo);
#pragma unroll
        for (int j = 0; j < 9; ++j) dst[j * plane + cell] = f[j];
      }
    }
  }
}

// Microseconds per step of a plan, and of one step per launch, fitted to 1300
// timings of domains of 3 to 40 rows (5 % in the mean for tiles of the least
// time, up to 25 % for FP64 and for tiles with idle threads).  A tile's work
// counts whole waves and a fixed part per step, more where cells have masks;
// `rounds` as in general_plan.
static double multi2d_time(const Multi2dDomain &d, const Multi2dPlan &p) {
  constexpr int NCU = 256;
  const int tw = p.tw, th = p.th, t = p.steps, whole = d.faces ? 256 : 128;
  auto at = [&](int back) { return (long long)(tw + 2 * back) * (d.pery ? th + 2 * back : std::min(th + 2 * back, d.ny)); };
  auto full = [&](long long n) { return (double)((n + whole - 1) / whole * whole); };
  double work = full(at(t));
  for (int s = 0; s < t; ++s) work += full(at(s)) + (d.faces ? 350.0 : 250.0);
  const long long columns = (d.cells + (long long)tw * d.ny - 1) / ((long long)tw * d.ny),
                  tiles = columns * ((d.ny + th - 1) / th), rest = tiles % (2 * NCU);
  const double rounds = 2.0 * (double)(tiles / (2 * NCU)) + (rest == 0 ? 0.0 : rest <= NCU ? 1.3 : 2.0);
  const double unit = (d.esize == 4 ? 1.02e-3 : d.esize == 8 ? 0.95e-3 : 0.85e-3) * (d.faces ? 1.14 : 1.0) *
                      (1.0 + d.force * (d.esize == 4 ? 0.12 : d.esize == 8 ? 0.06 : 0.1));
  const double us = unit * (rounds * work + 3000.0) / t;
  // beyond the cache: 4.8 TB/s
  const double moved = (double)d.cells * 9 * d.esize * (1.0 + (double)at(t) / (tw * th)) / t / 4.8e6;
  return 2 * 9 * d.esize * d.cells > (256ll << 20) ? std::max(us, moved) : us;
}
static double single2d_time(const Multi2dDomain &d) {
  const int bx = d.nx > 128 ? 256 : d.nx > 64 ? 128 : 64;
  // lanes, at the rate of cells without solids; 10 % of solids take 1.67 times
  const double lanes = (double)((d.nx + bx - 1) / bx * bx) * (double)(d.cells / d.nx) * (d.solids ? 1.35 : 1.0);
  if (d.esize == 2) return d.faces ? 3.9 + 8.8e-6 * lanes : 2.6 + 6.6e-6 * lanes;
  return (d.faces ? 3.5 : 2.8) + (d.esize == 4 ? 12.8e-6 : 24.5e-6) * lanes;
}

// Tiles of a power of two of cells, as square as it gets: about one per CU as
// long as that leaves at least 64 cells and at most 4 KB per direction (512,
// 1024 or 2048 cells), which with the halo is what two blocks of a CU hold.
// Small tiles take 8 steps (the launch is shared by more of them), large ones
// 6, fewer where the halo would not fit.  For a single domain the height may
// then grow to twice that where it saves a round of blocks: 512 run at once,
// the last 256 or fewer of them alone on their CU in about 0.65 of the time
// (in the formula, the cells updated per block, 1.5 per cell loaded, and 1000
// for the launch; 909 x 1366 BF16 17.8 to 13.2 us a step).
// 1024 threads where a CU has one block anyway.
// Where both buffers exceed the 256 MB of cache, rows of 256 bytes and fewer
// steps: the lines of a tile's ragged edge then come from memory.
// Best and next of a sweep over tiles of 8 x 4 to 128 x 32 cells and 2 to 12
// steps, microseconds per step, single-step launches last:
//   256 x 64 FP64     8 x 8, 8 steps   1.5     8 x 8, 6     1.6      4.1
//   256 x 128 FP32    16 x 8, 8        2.85    8 x 16, 8    2.92     5.4
//   512 x 256 FP32    32 x 16, 8       2.7     32 x 20, 6   3.0      4.7
//   1024^2 FP32       32 x 32, 6      11.0     64 x 16, 4  11.5     17.2
//   4096 x 2048 FP32  64 x 20, 4      68       32 x 32, 6   70      119
//   2048^2 FP64       32 x 16, 4      51       32 x 20, 3   58      113
//   4096 x 2048 FP16  128 x 20, 4     56       64 x 32, 6   56       81
static Multi2dPlan general_plan(const Multi2dDomain &d) {
  constexpr int NCU = 256;
  constexpr long long CACHE = 256ll << 20;
  const int nx = d.nx, ny = d.ny, esize = d.esize;
  const long long cells = d.cells;
  const bool faces = d.faces;
  const int cap = multi2d_cap(esize, faces), most = 4096 / esize;
  Multi2dPlan p;
  if (2 * 9 * esize * cells > CACHE) {
    p.tw = std::min(256 / esize, nx);
    p.th = std::min(24, ny);
    p.steps = 4;
    p.wide = false;
    while (multi2d_slots(p.tw, p.th, p.steps) > cap) p.th -= 4;
    return p;
  }
  int lg = 6;
  while ((1 << lg) < most && ((long long)NCU << lg) < cells) ++lg;
  p.tw = std::min(1 << (lg + 1) / 2, nx);
  const int low = std::min(1 << lg / 2, ny), high = cells == (long long)nx * ny ? std::min(2 * low, ny) : low;
  double least = 0.0;
  for (int th = low; th <= high; ++th) {
    int t = lg >= 10 ? 6 : 8;
    while (t > 4 && multi2d_slots(p.tw, th, t) > cap) --t;
    if (multi2d_slots(p.tw, th, t) > cap) break;
    const long long columns = (cells + (long long)p.tw * ny - 1) / ((long long)p.tw * ny);
    const long long tiles = columns * ((ny + th - 1) / th), rest = tiles % (2 * NCU);
    double work = 1.5 * (p.tw + 2 * t) * (th + 2 * t);
    for (int s = 0; s < t; ++s) work += (p.tw + 2 * s) * (th + 2 * s);
    const double rounds = 2.0 * (double)(tiles / (2 * NCU)) + (rest == 0 ? 0.0 : rest <= NCU ? 1.3 : 2.0);
    const double cost = (rounds * work + 1000.0) / t;
    if (th > low && cost >= least) continue;
    least = cost;
    p.th = th;
    p.steps = t;
    p.wide = tiles <= NCU && p.tw * th >= 256;
  }
  return p;
}

// Domains of few rows: a tile of the rule above holds too few cells for its
// threads there, and the rows of a periodic axis are updated several times
// over (3 rows and 6 steps: 3 times).  Wider or lower tiles with fewer steps, or one
// step per launch where even these take longer, by multi2d_time (below 2^15
// cells the launch is all there is to save, and the rule above holds).
// Microseconds per step, one step per launch, the rule above, this one:
//   333333 x 3 FP32 periodic   15.5   30.6   14.2 (256 x 3, 2 steps)
//   333333 x 3 FP16 periodic    8.9   18.1    8.8 (one step per launch)
//   1333333 x 3 FP16 walls     46     63     33   (256 x 3, 4 steps)
//   250000 x 4 FP32 NEEM       16.7   29.6   14.1 (128 x 4, 4 steps)
//   100000 x 10 FP32 periodic  15.5   13.8   12.0
//   20000 x 50 FP16 periodic, force along x and y   9.0   11.7   8.9
// From 64 rows on the rule above is at most 1.02 times as slow as one step per
// launch; below, of 3000 timed cases this one is in 15, by 1.03 to 1.11.
Multi2dPlan multi2d_plan(const Multi2dDomain &d) {
  constexpr int THIN = 64;
  const Multi2dPlan general = general_plan(d);
  if (d.ny >= THIN || d.cells < 1 << 15) return general;
  Multi2dPlan best = general;
  const int cap = multi2d_cap(d.esize, d.faces);
  // another tile has to be faster by more than the fit's error, which is larger
  // in FP64 (41666 x 24 periodic 12.6 us with the rule above; 14.6 with the tile
  // that the fit gives three quarters of its time)
  double time = multi2d_time(d, general), least = (d.esize == 8 ? 0.74 : 0.8) * time;
  for (int rows = 1; rows <= 3; ++rows)
    for (int width = 32; width <= 512; width *= 2)
      for (int t : {2, 3, 4, 6, 8}) {
        const Multi2dPlan p{t, std::min(width, d.nx), (d.ny + rows - 1) / rows, false};
        const int slots = multi2d_slots(p.tw, p.th, t);
        if (slots > cap || !multi2d_exact(slots, p.tw + 2 * t)) continue;
        const double us = multi2d_time(d, p);
        if (us >= least) continue;
        time = least = us;
        best = p;
      }
  return time > single2d_time(d) ? Multi2dPlan{1, 0, 0, false} : best;
}

template <typename ST, int FORCE, int NT>
static void launch_multi2d(const Multi2dArgs &a, hipStream_t s, int cls) {
  const dim3 g((unsigned)((a.ntiles + 7) / 8 * 8)), b(NT);
  if (cls == MULTI2D_BOX) hipLaunchKernelGGL((k_multi2d<ST, MULTI2D_BOX, FORCE, NT>), g, b, 0, s, a);
  else if (cls == MULTI2D_WALLS) hipLaunchKernelGGL((k_multi2d<ST, MULTI2D_WALLS, FORCE, NT>), g, b, 0, s, a);
  else hipLaunchKernelGGL((k_multi2d<ST, MULTI2D_OPEN, FORCE, NT>), g, b, 0, s, a);
}

template <typename ST>
void Multi2dL<ST>::run(const Multi2dArgs &a, hipStream_t s, int cls, bool wide) {
  const int force = force_kind(a.F);
  if (force == FORCE_NONE) wide ? launch_multi2d<ST, FORCE_NONE, 1024>(a, s, cls) : launch_multi2d<ST, FORCE_NONE, 512>(a, s, cls);
  else if (force == FORCE_X) wide ? launch_multi2d<ST, FORCE_X, 1024>(a, s, cls) : launch_multi2d<ST, FORCE_X, 512>(a, s, cls);
  else wide ? launch_multi2d<ST, FORCE_ANY, 1024>(a, s, cls) : launch_multi2d<ST, FORCE_ANY, 512>(a, s, cls);
}

template struct Multi2dL<float>;
template struct Multi2dL<double>;
template struct Multi2dL<__half>;
template struct Multi2dL<__hip_bfloat16>;

}  // namespace lbm
