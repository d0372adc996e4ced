// Two D3Q19 steps per pass over memory.
//
// The single-step kernel reads and writes every population once per step and
// runs at 74 % of the HBM peak, within 12 % of a plain copy: only fewer bytes
// per step can make it faster.  Here a block walks a column of x-y tiles along
// z.  At plane p it takes the first step (populations gathered from memory, as
// the single-step kernel does), leaves the plane in LDS, and takes the second
// step of plane p - 1 from the planes p and p - 1 it holds there; the five
// populations that plane p - 2 contributes were read from LDS one plane
// earlier and wait in registers.  Memory sees one read and one write per two
// steps, plus the one-cell halo of the tile (its first step is taken by
// several blocks).
//
// One thread owns one (x, y) column of the region, so the boundary masks of
// the x and y faces, the gather offsets and the LDS slots are fixed for the
// walk.  The next plane's loads are issued before the second step's
// arithmetic.  Values are rounded to the storage form between the two steps
// and the arithmetic is that of the single-step kernel: the result equals two
// single steps bit for bit.
#include "lbm_multi3d.h"

#include <algorithm>
#include <cmath>

namespace lbm {

constexpr uint32_t POP_BITS = (1u << 18) - 1u;
constexpr uint32_t FROM_NEIGHBOUR = 1u << 30;  // NEEM cell: gathers at its inward neighbour

// an LDS barrier that leaves global loads and stores in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Forget what the compiler knows of h: FP32 populations are then converted
// to FP64 a second time for the collision instead of being held as 38
// registers from the moments on (the kernel has 128).
template <typename R>
__device__ __forceinline__ void reconvert(R (&h)[19]) {
  if constexpr (sizeof(R) == 4) {
#pragma unroll
    for (int j = 0; j < 19; ++j) asm volatile("" : "+v"(h[j]));
  }
}

// A uniform pointer plus a 32-bit byte offset per lane, as the scalar-base
// form of the memory instructions takes them.  Both are made opaque: the
// compiler otherwise moves their loop-invariant parts, widened to 64 bits,
// out of the loop and keeps a register pair per population for them.
template <typename ST>
using Bits = typename std::conditional<sizeof(ST) == 2, uint16_t, typename std::conditional<sizeof(ST) == 4, uint32_t, uint64_t>::type>::type;
template <typename ST>
__device__ __forceinline__ auto *at_offset(const ST *base, unsigned bytes) {
  using T = __attribute__((address_space(1))) Bits<ST>;
  auto *b = (__attribute__((address_space(1))) char *)base;
  asm("" : "+s"(b));
  asm volatile("" : "+v"(bytes));
  return (T *)(b + bytes);
}

// bits of the populations that enter across face f
__host__ __device__ constexpr uint32_t entering(int f) {
  using L = Lat<19>;
  uint32_t m = 0;
  for (int j = 0; j < 18; ++j) {
    const int c = f < 2 ? L::cx[j] : (f < 4 ? L::cy[j] : L::cz[j]);
    if (c == ((f & 1) ? -1 : 1)) m |= 1u << j;
  }
  return m;
}

// The tile and slab of a block, and its region with the halo.  A NEEM cell's
// second step reads three columns, also where the tile is narrower.
struct Box3d {
  int x0, x1, y0, y1, z0, z1, rx0, rx1, ry0, ry1;
};
__device__ __forceinline__ Box3d box_of(const Multi3dArgs &m, int id, bool perx, bool pery) {
  const int tx = id % m.ntx, ty = (id / m.ntx) % m.nty, sl = id / (m.ntx * m.nty);
  Box3d b;
  b.x0 = tx * m.tw;
  b.x1 = min(b.x0 + m.tw, m.nx) - 1;
  b.y0 = (int)((long long)ty * m.ny / m.nty);
  b.y1 = (int)((long long)(ty + 1) * m.ny / m.nty) - 1;
  b.z0 = (int)((long long)sl * m.nz / m.slabs);
  b.z1 = (int)((long long)(sl + 1) * m.nz / m.slabs) - 1;
  b.rx0 = perx ? b.x0 - 1 : max(min(b.x0 - 1, m.nx - 3), 0);
  b.rx1 = perx ? b.x1 + 1 : min(max(b.x1 + 1, 2), m.nx - 1);
  b.ry0 = pery ? b.y0 - 1 : max(b.y0 - 1, 0);
  b.ry1 = pery ? b.y1 + 1 : min(b.y1 + 1, m.ny - 1);
  return b;
}
__device__ __forceinline__ int wrapped(int c, int n) { return c < 0 ? c + n : (c >= n ? c - n : c); }

// solid[id] = 1 where block id has a solid, or a link to one, among the cells
// whose masks it reads: the others then read no masks.
__global__ void __launch_bounds__(256) k_multi3d_solid(const Multi3dArgs m, unsigned char *solid) {
  __shared__ int any;
  if (threadIdx.x == 0) any = 0;
  __syncthreads();
  const Box3d b = box_of(m, blockIdx.x, m.per[0], m.per[1]);
  const int w = b.rx1 - b.rx0 + 1, h = b.ry1 - b.ry0 + 1, n = w * h * (b.z1 - b.z0 + 3);
  int found = 0;
  for (int i = threadIdx.x; i < n; i += 256) {
    const int z = b.z0 - 1 + i / (w * h), r = i % (w * h);
    if (!m.per[2] && (z < 0 || z >= m.nz)) continue;
    const int x = wrapped(b.rx0 + r % w, m.nx), y = wrapped(b.ry0 + r / w, m.ny);
    if (m.links[x + (long long)m.px * (y + (long long)m.ny * wrapped(z, m.nz))]) found = 1;
  }
  if (found) any = 1;
  __syncthreads();
  if (threadIdx.x == 0) solid[blockIdx.x] = (unsigned char)any;
}

template <typename ST, int CLS, int FORCE>
__global__ void __launch_bounds__(multi3d_threads(sizeof(ST), CLS))
__attribute__((amdgpu_waves_per_eu(sizeof(ST) == 8 ? 2 : (CLS == MULTI3D_BOX ? 4 : 3)))) k_multi3d(const Multi3dArgs m) {
  using L = Lat<19>;
  using C = typename Store<ST>::C;
  using R = typename Store<ST>::R;
  constexpr int NT = multi3d_threads(sizeof(ST), CLS);
  constexpr bool WALLS = CLS != MULTI3D_BOX;
  __shared__ ST lds[2][19][NT];
  // the masks of the two planes: a second step's column reads the one its
  // first step formed (80 KB in all, two blocks to a CU)
  __shared__ uint32_t mask[WALLS ? 2 : 1][WALLS ? NT : 1];
  // blocks of one XCD take neighbouring tiles of one slab
  const int nblk = m.ntx * m.nty * m.slabs, chunk = (nblk + 7) / 8;
  const int id = (int)(blockIdx.x % 8) * chunk + (int)(blockIdx.x / 8);
  if (id >= nblk || (int)(blockIdx.x / 8) >= chunk) return;  // uniform per block
  const bool perx = !WALLS || m.per[0], pery = !WALLS || m.per[1], perz = !WALLS || m.per[2];
  const int nx = m.nx, ny = m.ny, nz = m.nz, px = m.px;
  const Box3d b = box_of(m, id, perx, pery);
  const int z0 = b.z0, z1 = b.z1;
  const int pitch = b.rx1 - b.rx0 + 1, cols = pitch * (b.ry1 - b.ry0 + 1);
  unsigned moving = 0;  // uniform: the faces that are moving walls
  constexpr bool OPEN = WALLS && sizeof(ST) == 8;  // NEEM faces (multi3d_class)
  bool any_neem = false;
  const uint32_t *links = nullptr;
  if (WALLS) {
#pragma unroll
    for (int f = 0; f < 6; ++f)
      if (m.face[f].kind == LBM_FACE_WALL && (m.face[f].u[0] != 0.0 || m.face[f].u[1] != 0.0 || m.face[f].u[2] != 0.0)) moving |= 1u << f;
    // only the blocks at the x faces have NEEM cells
    any_neem = OPEN && !perx && ((b.rx0 == 0 && m.face[0].kind != LBM_FACE_WALL) || (b.rx1 == nx - 1 && m.face[1].kind != LBM_FACE_WALL));
    if (m.links && m.solid[id]) links = m.links;
  }
  const int zs = px * ny;  // cells per plane of z
  const ST *src = static_cast<const ST *>(m.src);
  ST *dst = static_cast<ST *>(m.dst);
  auto exists = [&](int z) { return perz || (z >= 0 && z < nz); };
  // first step: one column of the region per thread
  const int t = min((int)threadIdx.x, cols - 1);
  const bool mine = (int)threadIdx.x < cols;
  const int x = wrapped(b.rx0 + t % pitch, nx), y = wrapped(b.ry0 + t / pitch, ny);
  // The column's part of the mask: the populations that enter across the x
  // and y faces it lies on, and which faces these are (bits ON ..).  On a
  // NEEM face (bit NEEM) the cell gathers at its inward neighbour, which lies
  // on the y faces only.
  constexpr int ON = 24;  // bits 24..27: on face -x, +x, -y, +y
  constexpr uint32_t NEEM = 1u << 28;
  uint32_t faces = 0;
  if (WALLS) {
    if (!perx && x == 0) faces |= entering(0) | (1u << ON) | (m.face[0].kind != LBM_FACE_WALL ? NEEM : 0u);
    if (!perx && x == nx - 1) faces |= entering(1) | (2u << ON) | (m.face[1].kind != LBM_FACE_WALL ? NEEM : 0u);
    if (!pery && y == 0) faces |= entering(2) | (4u << ON);
    if (!pery && y == ny - 1) faces |= entering(3) | (8u << ON);
  }
  auto inward = [&](uint32_t w) { return OPEN && (w & FROM_NEIGHBOUR) ? ((w >> ON) & 1u ? 1 : -1) : 0; };
  // mask of the column's cell in plane z: populations that bounce back, the
  // bits above, LINK_SELF_SOLID, FROM_NEIGHBOUR
  auto mask_of = [&](int z) -> uint32_t {
    if (!WALLS || !exists(z)) return 0u;
    const int zz = wrapped(z, nz);
    uint32_t fz = 0;
    if (!perz && zz == 0) fz = entering(4);
    if (!perz && zz == nz - 1) fz = entering(5);
    uint32_t w = faces | fz;
    const long long cell = (long long)zz * zs + px * y + x;
    if (links) w |= links[cell];
    if (any_neem && (w & NEEM)) {
      const uint32_t l1 = links ? links[cell + ((w >> ON) & 1u ? 1 : -1)] : 0u;
      if (!(l1 & LINK_SELF_SOLID)) {
        const uint32_t fy = ((w >> ON) & 4u ? entering(2) : 0u) | ((w >> ON) & 8u ? entering(3) : 0u);
        w = (w & ~POP_BITS) | (l1 & POP_BITS) | fy | fz | FROM_NEIGHBOUR;
      }
    }
    return w;
  };
  const C omega = scalar(C(m.omega));
  const C Fx = C(m.F[0]), Fy = C(m.F[1]), Fz = C(m.F[2]);
  // the rules beyond bounce-back, on populations h of a cell with mask w in
  // plane z: the Ladd terms of moving walls and the NEEM correction
  auto rules = [&](uint32_t w, int z, R (&h)[19]) {
    // bit f: the cell (or the inward neighbour of a NEEM cell) is on face f
    const uint32_t on = ((w >> ON) & (OPEN && (w & FROM_NEIGHBOUR) ? 12u : 15u)) | (!perz && z == 0 ? 16u : 0u) |
                        (!perz && z == nz - 1 ? 32u : 0u);
    if (__ballot((on & moving) != 0)) {
#pragma unroll
      for (int f = 0; f < 6; ++f) {
        if (!((moving >> f) & 1u)) continue;  // uniform
        const C u0 = C(m.face[f].u[0]), u1 = C(m.face[f].u[1]), u2 = C(m.face[f].u[2]);
#pragma unroll
        for (int j = 0; j < 18; ++j) {
          if (!((entering(f) >> j) & 1u)) continue;
          // the other face the population crosses owns the crossing when its
          // priority is higher, or equal on a lower axis
          const int c[3] = {L::cx[j], L::cy[j], L::cz[j]};
          bool owned = (on >> f) & 1u;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            if (d == (f >> 1) || c[d] == 0) continue;
            const int g = 2 * d + (c[d] > 0 ? 0 : 1);
            const bool wins = d < (f >> 1) ? m.face[g].prio >= m.face[f].prio : m.face[g].prio > m.face[f].prio;
            owned = owned && !(((on >> g) & 1u) && wins);
          }
          if (owned) h[j] = R(C(h[j]) + C(6) * C(L::w[j]) * cdot<19>(j, u0, u1, u2));
        }
      }
    }
    if (any_neem && (w & FROM_NEIGHBOUR)) neem_correct<19, ST>(m, (w >> ON) & 1u ? 0 : 1, h);
  };

  // columns the populations are pulled from (clamped across a face)
  unsigned xs[3], ys[3];
  xs[0] = (unsigned)(x == 0 ? (perx ? nx - 1 : 0) : x - 1);
  xs[1] = (unsigned)x;
  xs[2] = (unsigned)(x == nx - 1 ? (perx ? 0 : nx - 1) : x + 1);
  ys[0] = (unsigned)px * (unsigned)(y == 0 ? (pery ? ny - 1 : 0) : y - 1);
  ys[1] = (unsigned)px * (unsigned)y;
  ys[2] = (unsigned)px * (unsigned)(y == ny - 1 ? (pery ? 0 : ny - 1) : y + 1);
  ST g[19];
  auto load = [&](int z, uint32_t w) {
    if (!exists(z)) return;
    // source planes (clamped across a face)
    const int zz = wrapped(z, nz);
    const int zsrc[3] = {exists(z - 1) ? wrapped(z - 1, nz) : zz, zz, exists(z + 1) ? wrapped(z + 1, nz) : zz};
    if (WALLS && __ballot(w != 0)) {
      // A missing population loads its bounce-back source S(x, opp j) of the
      // own plane: another uniform base, reached from the first one by a
      // 32-bit difference (the host checks the range).
      const unsigned in = any_neem ? (unsigned)inward(w) : 0u;
      unsigned x0 = xs[1] + in, xm = in ? x0 - 1u : xs[0], xp = in ? x0 + 1u : xs[2];
      // formed here each time: as loop invariants the 37 offsets would be
      // kept in registers (and spilled) by every wave
      asm volatile("" : "+v"(x0), "+v"(xm), "+v"(xp));
      const unsigned centre = x0 + ys[1];
#pragma unroll
      for (int j = 0; j < 19; ++j) {
        const int low = j < L::opp[j] ? j : L::opp[j];
        const ST *base = src + (long long)low * m.plane;  // uniform
        const unsigned xc = L::cx[j] > 0 ? xm : (L::cx[j] < 0 ? xp : x0);
        const unsigned pull = (unsigned)(j - low) * (unsigned)m.plane + (unsigned)zsrc[1 - L::cz[j]] * (unsigned)zs + (xc + ys[1 - L::cy[j]]);
        const unsigned back = (unsigned)(L::opp[j] - low) * (unsigned)m.plane + (unsigned)zz * (unsigned)zs + centre;
        const unsigned cell = j < 18 && ((w >> j) & 1u) ? back : pull;
        g[j] = __builtin_bit_cast(ST, (Bits<ST>)*at_offset(base, cell * (unsigned)sizeof(ST)));
      }
    } else {
#pragma unroll
      for (int j = 0; j < 19; ++j) {
        const ST *base = src + (long long)j * m.plane + (long long)zsrc[1 - L::cz[j]] * zs;  // uniform
        g[j] = __builtin_bit_cast(ST, (Bits<ST>)*at_offset(base, (xs[1 - L::cx[j]] + ys[1 - L::cy[j]]) * (unsigned)sizeof(ST)));
      }
    }
  };
  // second step: one column of the tile per thread, rows of the tile's width
  // so that a wave stores whole lines (with the region's threads, whose rows
  // are two columns longer, the stores alone took 2/3 of the time)
  const int ox = (int)threadIdx.x % m.tw, oy = (int)threadIdx.x / m.tw;
  const bool inner = b.x0 + ox <= b.x1 && b.y0 + oy <= b.y1;
  const int x2 = inner ? b.x0 + ox : b.x0, y2 = inner ? b.y0 + oy : b.y0;
  const unsigned own2 = (unsigned)x2 + (unsigned)px * (unsigned)y2;
  const int slot = (x2 - b.rx0) + pitch * (y2 - b.ry0);

  const int pa = exists(z0 - 1) ? z0 - 1 : z0;
  uint32_t wp = mask_of(pa), wn = mask_of(pa + 1);
  load(pa, wp);
  ST up[5];  // the populations with c_z = 1 of the next second step
#pragma unroll
  for (int k = 0; k < 5; ++k) up[k] = ST(0.0f);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): see below
  for (int p = pa; p <= z1 + 1; ++p) {
    ST(*const cur)[NT] = lds[p & 1];
    ST(*const prev)[NT] = lds[(p & 1) ^ 1];
    const bool first = exists(p);
    ST v[19];
    if (first) {
      R h[19];
#pragma unroll
      for (int j = 0; j < 19; ++j) h[j] = Store<ST>::ld(&g[j]);
      if (p <= z1) load(p + 1, wn);
      if (WALLS && __ballot(wp != 0)) rules(wp, wrapped(p, nz), h);
      const Moments<19, C> mo = moments<19, C, FORCE>(h, Fx, Fy, Fz);
      if (std::is_same<C, double>::value) reconvert(h);
      collide<19, ST, FORCE>(h, mo, omega, Fx, Fy, Fz, true, [&](int j, C value) { Store<ST>::st(&v[j], value); });
    }
    lds_barrier();  // the previous plane's reads of the slot are done
    if (first && mine) {
#pragma unroll
      for (int j = 0; j < 19; ++j) cur[j][t] = v[j];
      if (WALLS) mask[p & 1][t] = wp;
    }
    lds_barrier();
    wp = wn;
    wn = p < z1 ? mask_of(p + 2) : 0u;
    const int q = p - 1;
    if (q >= z0) {
      // second step of plane q
      R h[19];
      const uint32_t vq = WALLS ? mask[(p & 1) ^ 1][slot] : 0u;
      const bool masked = WALLS && __ballot(vq != 0);
      const int at = slot + (masked ? inward(vq) : 0);
      int k = 0;
#pragma unroll
      for (int j = 0; j < 19; ++j) {
        if (L::cz[j] == 1) {
          h[j] = Store<ST>::ld(&up[k++]);
          continue;
        }
        const ST *pull = L::cz[j] == 0 ? &prev[j][at - L::cx[j] - pitch * L::cy[j]] : &cur[j][at - L::cx[j] - pitch * L::cy[j]];
        if (masked && j < 18 && ((vq >> j) & 1u)) pull = &prev[L::opp[j]][at];
        h[j] = Store<ST>::ld(pull);
      }
      if (masked) rules(vq, wrapped(q, nz), h);
      const Moments<19, C> mo = moments<19, C, FORCE>(h, Fx, Fy, Fz);
      if (std::is_same<C, double>::value) reconvert(h);
      // The next plane's loads have to be in before the stores go out: both
      // count down one counter in order, and a wait for the loads placed
      // after the stores would wait for the stores' completion as well.
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
      if (inner && !(WALLS && (vq & LINK_SELF_SOLID))) {
        const long long zo = (long long)wrapped(q, nz) * zs;
        collide<19, ST, FORCE>(h, mo, omega, Fx, Fy, Fz, true, [&](int j, C value) {
          const ST *base = dst + (long long)j * m.plane + zo;  // uniform
          ST out;
          Store<ST>::st(&out, value);
          __builtin_nontemporal_store(__builtin_bit_cast(Bits<ST>, out), at_offset(base, own2 * (unsigned)sizeof(ST)));
        });
      }
    } else {
      __builtin_amdgcn_s_waitcnt(0x0f70);  // on every way to the next plane
    }
    // what plane p - 1 contributes to the second step of plane p
    if (p >= z0 && p <= z1) {
      const uint32_t vp = WALLS ? mask[p & 1][slot] : 0u;
      const bool masked = WALLS && __ballot(vp != 0);
      const int at = slot + (masked ? inward(vp) : 0);
      int k = 0;
#pragma unroll
      for (int j = 0; j < 19; ++j) {
        if (L::cz[j] != 1) continue;
        const ST *pull = &prev[j][at - L::cx[j] - pitch * L::cy[j]];
        if (masked && ((vp >> j) & 1u)) pull = &cur[L::opp[j]][at];
        up[k++] = *pull;
      }
    }
  }
}

// Tiles of 32 columns along x (64 for 16-bit storage, the same 128 bytes),
// as high as the block's threads reach with the halo.  Slabs along z: a CU
// works through k blocks, each for its planes and about one more (the extra
// first-step planes at both ends); below the number of blocks it can hold
// its lanes idle between barriers, which costs 1.4 times.  The least of
// k * (nz / slabs + 1) picks within 3 % of the best of 1 to 32 slabs on 22 of
// 23 swept domains (13 % off on the last), microseconds per step:
//   256^3 FP32 box             16 slabs 339   best 8: 332     single 430
//   128^3 FP32 box             12 slabs  49.4                 single  59
//   256 x 128 x 128 FP64 box    3 slabs 132                   single 218
//   300 x 200 x 101 FP64 sphere 8 slabs 260                   single 443
//   256 x 192 x 160 FP16 box    8 slabs 102                   single 116
// More than 32 planes per slab lose once a CU runs its blocks in turns (256^3
// in 3 slabs: 377), so those are left out.
// FP64 domains that fit the 256 MB of cache also try equal tiles of other
// widths: 97 columns in three tiles of 32 and one of 1 waste a quarter of the
// blocks (97 x 61 x 45 cavity 20.4 us a step, five tiles of 20 18.5; 400 x 40 x
// 24 23.4 and 19.9).  Rows that don't start on whole lines cost 15 to 20 % (200
// x 64 x 64 in 25 columns 50 against 42), more in the smaller storage forms,
// so the formula has to promise a fifth.
Multi3dPlan multi3d_plan(int nx, int ny, int nz, int esize, int cls) {
  constexpr int NCU = 256;
  constexpr long long CACHE = 256ll << 20;
  const int nt = multi3d_threads(esize, cls), line = esize == 2 ? 64 : 32;
  const int held = esize == 8 ? 1 : nt == 256 ? 3 : 2;  // blocks a CU holds
  Multi3dPlan best{};
  double least = 0.0;
  auto width = [&](int tw) {
    Multi3dPlan p;
    p.tw = std::min(tw, nx);
    p.ntx = (nx + p.tw - 1) / p.tw;
    const int rh = nt / (p.tw + 2) - 2;  // tw * rh <= nt as well
    p.nty = (ny + rh - 1) / rh;
    for (p.slabs = 1; p.slabs <= std::max(1, std::min(32 + nz / 32, nz / 2)); ++p.slabs) {
      const long long k = ((long long)p.ntx * p.nty * p.slabs + NCU - 1) / NCU;
      if (k > held && nz > 32 * p.slabs) continue;
      const double cost = (double)k * ((double)nz / p.slabs + 1.0) * (k < held ? 1.4 : 1.0);
      if (least == 0.0 || cost < (p.tw == best.tw ? 1.0 : 0.8) * least) {
        least = cost;
        best = p;
        best.cost = cost;
      }
    }
  };
  width(line);
  if (esize == 8 && 2ll * 19 * esize * nx * ny * nz <= CACHE)
    for (int n = (nx + 63) / 64; n <= (nx + 15) / 16; ++n) width((nx + n - 1) / n);
  return best;
}

// FP64 storage halves its traffic and hardly adds to its arithmetic: two steps
// win on every domain above multi3d_class's bounds but those with walls, beyond
// the cache and a few rows high (1024 x 4 x 1024 1.17 times as long, 512 x 5 x 400
// with NEEM faces 1.08).  In FP32 and 16-bit storage the second step's arithmetic,
// for the halo too, takes up much of what the traffic gives.  The logarithm of
// the ratio is fitted, closely where it is near zero, to 950 pairs of timings:
// idle lanes of the single step (its rows are rounded up to its blocks), the
// planes a CU works through here per cell, the body force (a general one costs
// a quarter: FP16 box of 256^3 232 us a step single; two steps 200, with a force
// along x 219, along y 278), solids and walls across x (single steps slow down
// more), moving walls (256 x 128 x 128 with three of them 135 single, 170; with
// none 121 single, 114).  Of the 700 pairs of at least 20 cells each way 6 are
// more than 3 % slower than single steps, the worst 9 %.  In three or four rows
// most of a block's threads idle (1024 x 3 x 1024 FP32 box 85 single, 114).
double multi3d_ratio(const Multi3dPlan &p, int nx, int ny, int nz, int esize, int cls, const FaceDev *face, bool solids,
                     int force, double lanes) {
  const double cells = (double)nx * ny * nz, idle = std::log(cells / lanes);
  if (esize == 8)
    return cls == MULTI3D_WALLS && !solids && ny < 6 && idle > -0.4 && 2 * 19 * 8 * cells > (double)(256 << 20) ? 1.1 : 0.9;
  if (ny < (solids ? 4 : 5)) return 1.1;
  // (beyond a wall there is no plane to take the first step of)
  const double beyond = p.slabs == 1 && face[4].kind != LBM_FACE_PERIODIC ? (double)nz / (nz + 1) : 1.0;
  const double planes = std::log(p.cost * beyond * 131072.0 / cells),
               mb = std::log(cells * esize * 38 / (1 << 20));
  if (esize == 2) {
    const double f[3] = {0.0, 0.104, 0.243};
    return std::exp(0.055 + 0.576 * idle + 0.27 * planes - 0.048 * mb + f[force]);
  }
  if (cls == MULTI3D_BOX) {
    const double f[3] = {0.0, 0.022, 0.083};
    return std::exp(-0.526 + 0.449 * idle + 0.148 * planes + 0.041 * mb + 0.184e6 / cells + f[force]);
  }
  int moving = 0;
  bool movx = false, movy = false;
  for (int i = 0; i < 6; ++i) {
    if (face[i].kind != LBM_FACE_WALL || (face[i].u[0] == 0.0 && face[i].u[1] == 0.0 && face[i].u[2] == 0.0)) continue;
    ++moving;
    movx = movx || i < 2;
    movy = movy || i == 2 || i == 3;
  }
  const double f[3] = {0.0, 0.051, 0.122};
  return std::exp(-0.507 + 0.476 * idle + 0.504 * planes - 0.033 * mb + f[force] - (solids ? 0.219 : 0.0) -
                  (face[0].kind != LBM_FACE_PERIODIC ? 0.346 / ((nx + 63) / 64) : 0.0) +
                  (movx ? 0.208 : movy ? 0.08 : 0.0) + 0.056 * std::max(0, moving - 1));
}

void multi3d_solid(const Multi3dArgs &a, unsigned char *solid, hipStream_t s) {
  hipLaunchKernelGGL(k_multi3d_solid, dim3((unsigned)(a.ntx * a.nty * a.slabs)), dim3(256), 0, s, a, solid);
}

template <typename ST, int CLS>
static void launch_multi3d(const Multi3dArgs &a, hipStream_t s) {
  const int n = a.ntx * a.nty * a.slabs, force = force_kind(a.F);
  const dim3 g((unsigned)((n + 7) / 8 * 8)), b(multi3d_threads(sizeof(ST), CLS));
  if (force == FORCE_NONE) hipLaunchKernelGGL((k_multi3d<ST, CLS, FORCE_NONE>), g, b, 0, s, a);
  else if (force == FORCE_X) hipLaunchKernelGGL((k_multi3d<ST, CLS, FORCE_X>), g, b, 0, s, a);
  else hipLaunchKernelGGL((k_multi3d<ST, CLS, FORCE_ANY>), g, b, 0, s, a);
}

template <typename ST>
void Multi3dL<ST>::run(const Multi3dArgs &a, hipStream_t s, int cls) {
  if (cls == MULTI3D_BOX) launch_multi3d<ST, MULTI3D_BOX>(a, s);
  else if constexpr (sizeof(ST) != 2) launch_multi3d<ST, MULTI3D_WALLS>(a, s);
}

template struct Multi3dL<float>;
template struct Multi3dL<double>;
template struct Multi3dL<__half>;
template struct Multi3dL<__hip_bfloat16>;

}  // namespace lbm
