// fluid.hip -- lattice kernels of libmfc_lbm for gfx950.
//
// Storage: populations are SoA, direction i of node (x, y, z) at
// pop[i * pitch + x + rs * (y + ny*z)]: by default the 19 directions' rows of
// one (y, z) side by side (pitch = nx or a little more, rs = 19 pitch), else
// whole planes (rs = nx, pitch = the node count plus 512 B); in FP64 or FP32
// (deviations f_i - w_i*rho0).  The resident buffer holds the post-collision (pre-streaming) field; streaming is never a separate pass:
// every consumer pulls f_i(x) = buf[i][x - c_i] (half-way bounce-back at the
// y walls when they are on).  One kernel therefore streams, takes moments,
// evaluates the forcing field and collides, reading 19 and writing 19
// populations per node: the 152 B (FP32) / 304 B (FP64) per node that bound
// the step.  Each lane owns one node; consecutive lanes are consecutive x,
// so every plane access of a wavefront is a contiguous 256 B (FP32) or
// 512 B (FP64) run.
#include <algorithm>

#include "force_table.h"
#include "field_sums.h"
#include "internal.h"
#include "lbm_access.h"
#include "lbm_collide.h"
#include "step_args.h"

namespace mfc {


// Forcing field at node x of row `row` from a per-row table
//   F_c = Re G_c0 + 2 Re(e1 G_c1) + 2 Re(e2 G_c2),  e_k = exp(i 2 pi k x / nx),
// the direct form of the reference's inverse real FFT of its few modes
// (gaussian.f90:325-369, mpifft.f90:111-158).
__device__ __forceinline__ void force_at(const double* __restrict__ G, const double* __restrict__ phx,
                                         uint32_t row, int x, int nx, double& Fx, double& Fy,
                                         double& Fz) {
  const double* t = G + 18ull * row;
  const int x2 = (2 * x >= nx) ? 2 * x - nx : 2 * x;
  const double c1 = phx[2 * x], s1 = phx[2 * x + 1];
  const double c2 = phx[2 * x2], s2 = phx[2 * x2 + 1];
  double v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double* q = t + 6 * c;
    v[c] = q[0] + 2.0 * (q[2] * c1 - q[3] * s1) + 2.0 * (q[4] * c2 - q[5] * s2);
  }
  Fx = v[0];
  Fy = v[1];
  Fz = v[2];
}

// Forcing field at node x from one row of a forcing table, in precision R.
template <typename R>
__device__ __forceinline__ void force_row(const double* __restrict__ t, R c1, R s1, R c2, R s2,
                                          R& Fx, R& Fy, R& Fz) {
  R v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double* q = t + 6 * c;
    v[c] = (R)q[0] + (R)2 * ((R)q[2] * c1 - (R)q[3] * s1) + (R)2 * ((R)q[4] * c2 - (R)q[5] * s2);
  }
  Fx = v[0];
  Fy = v[1];
  Fz = v[2];
}


// A density change as an integer whose maximum is the residual's: one above the
// bits of a non-negative double, which order as integers; 0 for a change that is
// no number, so that those count only where there is no other.
__device__ __forceinline__ uint64_t residual_bits(double change) {
  return change == change ? (uint64_t)__double_as_longlong(change) + 1 : 0;
}

// Fused stream + macro + forcing + MRT collision.
//
// One wavefront per tile of 64 consecutive x nodes of a row (kTileX):
// everything that depends on (y, z) only -- the nine neighbour-row offsets,
// the wall test and the forcing-table rows -- is wave-uniform and lives in
// scalar registers; per lane only x +- 1 wraps.
//
// ARR: conserved moments from the rho/u arrays (the reference's literal data
// flow, used while they are authoritative, e.g. the pre-relaxation);
// otherwise recomputed from the pulled populations plus half the forcing
// captured at the last macrovar, which is exactly what those arrays hold.
//
// LAY: layout of the input field.  LAY_AB reads buffer A and writes buffer B.
// The in-place (AA) layouts use one buffer: every node reads its 19 streamed
// values and writes post-collision value i where it read opp(i), so each
// node touches exactly the locations it read and nodes never race.  From
// LAY_AA_ODD that is all in the node's own slots; from LAY_AA_EVEN it is the
// neighbours' (the result is in LAY_AA_ODD, and the other way round).
// NTL, NTS: non-temporal loads of the two-buffer field, non-temporal stores
// (CollideShape says when).
// RES (with ARR): the density is taken from the populations as rhoupdat takes it
// and stored; `diff` receives the residual_bits of its change.
template <typename T, typename R, bool ARR, bool WALLS, int LAY, bool NTL, bool NTS, bool RES = false>
__device__ __forceinline__ void collide_node(const CollideArgs& a, int x, int y, int z, uint64_t* diff = nullptr) {
  const T* __restrict__ A = (const T*)a.A;
  T* __restrict__ B = (T*)a.B;
  T* F = (T*)a.B;   // the one buffer of the in-place layouts (A == B)
  const uint32_t* __restrict__ mask = a.mask;
  const Grid& g = a.g;
  const CollideConsts& k = a.k;
  const ForceArgs& fa = a.fa;
  const double* __restrict__ rho_a = a.rho;
  const double* __restrict__ ux_a = a.ux;
  const double* __restrict__ uy_a = a.uy;
  const double* __restrict__ uz_a = a.uz;
  const uint32_t nx = (uint32_t)g.nx, ny = (uint32_t)g.ny;
  const uint32_t ym = y == 0 ? ny - 1 : y - 1, yp = y == g.ny - 1 ? 0 : y + 1;
  const uint32_t zm = z == 0 ? g.nz - 1 : z - 1, zp = z == g.nz - 1 ? 0 : z + 1;
  const uint32_t row = (uint32_t)y + ny * (uint32_t)z;
  // neighbour rows, indexed [dy+1][dz+1] for the source row (y - cy, z - cz)
  const uint32_t yy[3] = {yp, (uint32_t)y, ym};   // cy = -1, 0, +1
  const uint32_t zz[3] = {zp, (uint32_t)z, zm};   // cz = -1, 0, +1
  const uint32_t xm = x == 0 ? nx - 1 : x - 1, xpp = x == g.nx - 1 ? 0 : x + 1;
  const uint32_t xs[3] = {xpp, (uint32_t)x, xm};   // cx = -1, 0, +1
  const uint32_t n = (uint32_t)x + nx * row;            // node index (mask, moment arrays)
  const uint64_t own = (uint64_t)x + g.rs * row;        // in-plane offset of the node
  const bool wall_lo = WALLS && y == 0, wall_hi = WALLS && y == g.ny - 1;
  // location of the streamed value of direction i: plane offset (pl * pitch,
  // a select between two compile-time planes on the wave-uniform wall test,
  // so it stays a scalar) and in-plane offset
  auto src_of = [&](int i, uint64_t& pbase, uint64_t& src) {
    if (LAY == LAY_AA_ODD) {
      pbase = (uint64_t)i * g.pitch;
      src = own;
      return;
    }
    const int ccx = cx(i), ccy = cy(i), ccz = cz(i);
    const bool wall = (ccy > 0 && wall_lo) || (ccy < 0 && wall_hi);
    src = wall ? own : xs[ccx + 1] + g.rs * (yy[ccy + 1] + ny * zz[ccz + 1]);
    const int p_in = LAY == LAY_AB ? i : opp(i);       // plane of an interior pull
    const int p_wall = LAY == LAY_AB ? opp(i) : i;     // plane beyond a wall
    const uint64_t b_in = (uint64_t)p_in * g.pitch, b_wall = (uint64_t)p_wall * g.pitch;
    pbase = wall ? b_wall : b_in;
  };
  R f[NPOP];
#pragma unroll
  for (int i = 0; i < NPOP; ++i) {
    uint64_t pb;
    uint64_t src;
    src_of(i, pb, src);
    f[i] = LAY == LAY_AB ? (NTL ? (R)__builtin_nontemporal_load(&A[pb + src]) : (R)A[pb + src])
                         : (R)F[pb + src];
  }
  const bool solid = mask != nullptr && ((mask[n >> 5] >> (n & 31u)) & 1u);
  if (!solid) {
    const int x2 = (2 * x >= g.nx) ? 2 * x - g.nx : 2 * x;
    const R c1 = (R)fa.phx[2 * x], s1 = (R)fa.phx[2 * x + 1];
    const R c2 = (R)fa.phx[2 * x2], s2 = (R)fa.phx[2 * x2 + 1];
    R rho, ux, uy, uz;
    R mx = (R)fa.bfx, my = (R)fa.bfy, mz = (R)fa.bfz;   // force of the macrovar moments
    if (ARR) {
      if (RES) {
        double r = (double)f[0];
#pragma unroll
        for (int i = 1; i < NPOP; ++i) r = r + (double)f[i];
        const double old = a.rho[n];
        *diff = residual_bits(fabs(r - old));
        a.rho[n] = r;
        rho = (R)r;
      } else {
        rho = (R)rho_a[n];
      }
      ux = (R)ux_a[n];
      uy = (R)uy_a[n];
      uz = (R)uz_a[n];
    } else {
      R jx, jy, jz;
      density_momentum<R>(f, rho, jx, jy, jz);
      if (fa.gmac) {
        R gx, gy, gz;
        force_row<R>(fa.gmac + 18ull * row, c1, s1, c2, s2, gx, gy, gz);
        mx += gx;
        my += gy;
        mz += gz;
      }
      ux = jx + (R)0.5 * mx;
      uy = jy + (R)0.5 * my;
      uz = jz + (R)0.5 * mz;
    }
    R Fx = (R)fa.bfx, Fy = (R)fa.bfy, Fz = (R)fa.bfz;
    if (fa.gcur) {
      R gx, gy, gz;
      force_row<R>(fa.gcur + 18ull * row, c1, s1, c2, s2, gx, gy, gz);
      Fx += gx;
      Fy += gy;
      Fz += gz;
    }
    // FP32 arithmetic takes the conserved corrections in closed form; FP64
    // keeps the reference's own arithmetic
    if (!ARR && sizeof(R) == 4)
      mrt_collide<R, true>(f, rho, ux, uy, uz, Fx, Fy, Fz, k, mx, my, mz);
    else
      mrt_collide<R, false>(f, rho, ux, uy, uz, Fx, Fy, Fz, k);
  }
  if (LAY == LAY_AB) {
    // one running pointer over the planes: no per-plane 64-bit base to keep
    T* q = B + own;
#pragma unroll
    for (int i = 0; i < NPOP; ++i) {
      if (NTS)
        __builtin_nontemporal_store((T)f[i], q);
      else
        *q = (T)f[i];
      q += g.pitch;
    }
  } else {
#pragma unroll
    for (int i = 0; i < NPOP; ++i) {
      uint64_t pb;
      uint64_t dst;
      src_of(opp(i), pb, dst);
      __builtin_nontemporal_store((T)f[i], &F[pb + dst]);
    }
  }
}

// Workgroups are dealt to the 8 XCDs round-robin in launch order, and each XCD
// has its own L2.  With per = grid / 8 each XCD takes a contiguous range of
// workgroups instead (per = 0: launch order).
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t per) {
  return b < per * kXcds ? (b % kXcds) * per + b / kXcds : b;
}

// The tiles of a lattice, `waves` per workgroup, numbered x fastest.
struct TileGrid {
  FastDiv tpr;        // tiles per row
  uint32_t ntiles, per, waves;
};

// FP32 storage with FP64 arithmetic, two buffers: 4 waves per SIMD (128
// VGPRs, 20-28 B/lane of spills) instead of 3 (132 VGPRs) measured 6 % faster
// at 256^3; the same bound on the FP64 kernel made it 3 % slower there and at
// 512^3 (897 against 872 us, 7.16 against 6.93 ms).
template <typename T, typename R, bool ARR, bool WALLS, int LAY, bool NTL, bool NTS>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 && sizeof(R) == 8 && LAY == LAY_AB ? 4 : 1)))
    k_collide(CollideArgs a, TileGrid g) {
  const uint32_t b = xcd_block(blockIdx.x, g.per);
  // the wavefront's index is uniform: keep it (and the tile, row, y, z) scalar
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t t = b * g.waves + w;
  if (t >= g.ntiles) return;
  const uint32_t row = div_by(t, g.tpr);
  const int x = (int)((t - row * g.tpr.d) * (uint32_t)kTileX + (threadIdx.x & 63u));
  if (x >= a.g.nx) return;
  const uint32_t z = div_by(row, a.g.dy);
  collide_node<T, R, ARR, WALLS, LAY, NTL, NTS>(a, x, (int)(row - z * a.g.dy.d), (int)z);
}

// Pre-relaxation at frozen velocity: the rhoupdat that ends one iteration and
// the collide that begins the next in one pass over the populations.  Each
// wavefront leaves its largest density change in one of kRelaxSlots words
// (as in rhoupdat), zero before.  The collide is wasted once, when
// the change has become small enough.  Bound: the populations read and written,
// rho and u read, rho written.  An iteration of two grids took 843 us at 256^3
// FP32, 1536 in FP64, 150 at 128 x 120 x 110 FP64 and 17.9 at 32^3 FP32; now
// 573, 1013, 106 and 14.0 (6.3 TB/s at 128 x 120 x 110).
constexpr uint32_t kRelaxSlots = 1024;
template <typename T, typename R, bool WALLS, bool NTL, bool NTS>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 && sizeof(R) == 8 ? 4 : 1)))
    k_collide_relax(CollideArgs a, TileGrid g, unsigned long long* __restrict__ slots) {
  const uint32_t b = xcd_block(blockIdx.x, g.per);
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t t = b * g.waves + w;
  if (t >= g.ntiles) return;
  const uint32_t row = div_by(t, g.tpr);
  const int x = (int)((t - row * g.tpr.d) * (uint32_t)kTileX + (threadIdx.x & 63u));
  const uint32_t z = div_by(row, a.g.dy);
  uint64_t d = 0;
  if (x < a.g.nx) collide_node<T, R, true, WALLS, LAY_AB, NTL, NTS, true>(a, x, (int)(row - z * a.g.dy.d), (int)z, &d);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) d = max(d, (uint64_t)__shfl_down((unsigned long long)d, o, 64));
  if ((threadIdx.x & 63u) == 0) atomicMax(&slots[t % kRelaxSlots], (unsigned long long)d);
}

// The collide of the tiles of a list (overlapped step): one tile per
// wavefront, four per workgroup, the grid sized to the list, each XCD a
// contiguous range of it: neighbouring rows then meet in one L2.
// Occupancy as the plain collide reaches it: FP32 storage with FP64
// arithmetic held to 4 waves per SIMD with two buffers; FP64 arithmetic in
// place held to 3 (the in-place layouts with walls otherwise take 178 VGPRs,
// 2 waves).
template <typename T, typename R>
constexpr int tile_waves(int lay) {
  return sizeof(R) == 8 ? (lay == LAY_AB ? (sizeof(T) == 4 ? 4 : 1) : 3) : 1;
}

template <typename T, typename R, bool WALLS, int LAY>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(tile_waves<T, R>(LAY))))
    k_collide_tiles(CollideArgs a, const uint32_t* __restrict__ list, uint32_t n, uint32_t tpr) {
  const uint32_t b = xcd_block(blockIdx.x, gridDim.x / kXcds);
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t L = b * 4u + w;
  if (L >= n) return;
  const uint32_t t = list[L];
  const uint32_t row = t / tpr;
  const int x = (int)((t - row * tpr) * (uint32_t)kTileX + (threadIdx.x & 63u));
  if (x >= a.g.nx) return;
  collide_node<T, R, false, WALLS, LAY, true, true>(a, x, (int)(row % (uint32_t)a.g.ny), (int)(row / (uint32_t)a.g.ny));
}

// Several boxes in one grid (ensemble engine): block b belongs to box c with
// off[c] <= b < off[c+1]; the box's nodes are numbered x fastest and taken
// BS per block, so consecutive lanes still read consecutive x (and rows
// continue into the next row without a gap).
__device__ __forceinline__ int case_of_block(const int* __restrict__ off, int nc, int b) {
  int lo = 0, hi = nc;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= b) lo = mid; else hi = mid;
  }
  return lo;
}

// ARR_ANY: some member takes its moments from the rho/u arrays (a.arr, its
// first step after joining); without it only the recomputing path is built.
// remap = 1 deals the grid to the 8 XCDs in contiguous ranges: consecutive
// node ranges, whose neighbour rows overlap, then share one L2.  The
// block-to-nodes map is a bijection either way, so results do not depend on it.
// NTL: non-temporal loads, where most nodes lie in rows of whole 64-B half lines (32
// boxes of 32 to 128 nodes an edge FP64 1697 us a step against 1748 plain, FP32 928
// against 935).  In other rows neighbouring blocks need the same lines: plain
// loads (100 x 90 x 96 FP32 44 to 35 us, 262 x 257 x 227 774 to 683, FP64 1066 to
// 1026; 130 x 118 x 126 FP32 99 to 72).  One grid, one kind: with both in one
// kernel it needs 99 instead of 71 VGPRs (FP64 176 instead of 132) and loses.
template <typename T, typename R, bool WALLS, int BS, bool ARR_ANY, bool NTL>
__global__ void __launch_bounds__(BS)
    kb_collide(const CollideArgs* __restrict__ t, const int* __restrict__ off, int nc, int remap) {
  const uint32_t b = xcd_block(blockIdx.x, remap ? gridDim.x / kXcds : 0);
  const int c = case_of_block(off, nc, (int)b);
  const CollideArgs a = t[c];
  const uint64_t n = (uint64_t)((int)b - off[c]) * BS + threadIdx.x;
  if (n >= a.g.ncell) return;
  int x, y, z;
  uint32_t row;
  node_coords((uint32_t)n, a.g, x, y, z, row);
  if (ARR_ANY && a.arr)
    collide_node<T, R, true, WALLS, LAY_AB, NTL, true>(a, x, y, z);
  else
    collide_node<T, R, false, WALLS, LAY_AB, NTL, true>(a, x, y, z);
}

// Forcing table of one step (force_table.h): one thread per (row, component).
__global__ void __launch_bounds__(256)
    k_force_table(ModeSet M, const double* __restrict__ phy, const double* __restrict__ phz, int ny,
                  int nz, double* __restrict__ G) {
  force_table_block(M, phy, phz, ny, nz, G, blockIdx.x);
}

// macrovar (collision.f90:232-332): rho = sum f, u = sum c f + F/2, then the
// rigid-body velocity and rho = rhopart at solid nodes.
struct MacroArgs {
  const void* A;
  Grid g;
  ForceArgs fa;
  const uint32_t* mask;
  const int32_t* isn;
  const double *ypglb, *wp, *omgp;
  double rhopart;
  double *rho, *ux, *uy, *uz;
};
template <typename T, bool PULLED, bool WALLS>
__device__ __forceinline__ void macro_node(const MacroArgs& a, uint32_t n, double& r, double& u, double& v, double& w) {
  const T* __restrict__ A = (const T*)a.A;
  const Grid& g = a.g;
  const ForceArgs& fa = a.fa;
  int x, y, z;
  uint32_t row;
  node_coords(n, g, x, y, z, row);
  double f[NPOP];
  if (PULLED)
    load_pulled<T, double, WALLS>(A, g, x, y, z, n, f);
  else
    load_direct<T, double, WALLS>(A, g, x, y, z, n, f);
  double jx, jy, jz;
  density_momentum<double>(f, r, jx, jy, jz);
  double Fx = fa.bfx, Fy = fa.bfy, Fz = fa.bfz;
  if (fa.gmac) {
    double gx, gy, gz;
    force_at(fa.gmac, fa.phx, row, x, g.nx, gx, gy, gz);
    Fx += gx;
    Fy += gy;
    Fz += gz;
  }
  u = jx + Fx / 2.0;
  v = jy + Fy / 2.0;
  w = jz + Fz / 2.0;
  if (a.mask != nullptr && ((a.mask[n >> 5] >> (n & 31u)) & 1u)) {
    const double *ypglb = a.ypglb, *wp = a.wp, *omgp = a.omgp;
    const int id = a.isn[n] - 1;
    const double xp = (double)(x + 1) - 0.5, yp = (double)(y + 1) - 0.5, zp = (double)(z + 1) - 0.5;
    const double xc = near_image(ypglb[3 * id], xp, g.nx);
    const double yc = WALLS ? ypglb[3 * id + 1] : near_image(ypglb[3 * id + 1], yp, g.ny);
    const double zc = near_image(ypglb[3 * id + 2], zp, g.nz);
    const double xx = xp - xc, yy = yp - yc, zz = zp - zc;
    const double* W = wp + 3 * id;
    const double* O = omgp + 3 * id;
    u = W[0] + (O[1] * zz - O[2] * yy);
    v = W[1] + (O[2] * xx - O[0] * zz);
    w = W[2] + (O[0] * yy - O[1] * xx);
    r = a.rhopart;
  }
  a.rho[n] = r;
  a.ux[n] = u;
  a.uy[n] = v;
  a.uz[n] = w;
}
template <typename T, bool PULLED, bool WALLS>
__global__ void __launch_bounds__(256) k_macro(MacroArgs a) {
  const uint32_t n = blockIdx.x * 256u + threadIdx.x;
  double r, u, v, w;
  if (n < a.g.ncell) macro_node<T, PULLED, WALLS>(a, n, r, u, v, w);
}

// The same with the first level of the field sums, taken from the registers: a
// thread's nodes and their order are those of the sums' own kernel.  The driver asks for the sums before the
// spectrum, so its statistics read the arrays once less: 354 us at 256^3 FP32
// (populations read, arrays written; 5.1 TB/s) against 312 and 108 us, 3.13 ms
// at 512^3 against 2.79 and 0.73, 14 us at 64^3 FP64 against 11 and 7.
template <typename T, bool PULLED, bool WALLS>
__global__ void __launch_bounds__(kSumThreads) k_macro_sums(MacroArgs a, double* __restrict__ part) {
  FieldSums f;
  for (uint64_t n = (uint64_t)blockIdx.x * kSumThreads + threadIdx.x; n < a.g.ncell;
       n += (uint64_t)gridDim.x * kSumThreads) {
    double r, u, v, w;
    macro_node<T, PULLED, WALLS>(a, (uint32_t)n, r, u, v, w);
    f.add(r, u, v, w);
  }
  f.store(part);
}

// rhoupdat (collision.f90:213-229) plus the pre-relaxation residual
// max|rho_new - rho_old| (main.f90:91-96): each workgroup walks its share of
// the nodes and leaves one maximum in part.  A node whose change is no number
// is passed over, as maxval passes it over.  Bound: 19 populations and rho
// read, rho written.  One atomic per 256 nodes on a single word, behind a
// barrier tree in LDS, set the time before: 796 us at 256^3 FP32 and 88 us at
// 128 x 120 x 110 FP64, now 338 and 48 us (4.6 and 5.9 TB/s).  16384
// workgroups: with 4096 it took 351 and 50 us, with one per 256 nodes 325 us at
// 256^3, but then 20 us more for the final maximum.
__device__ __forceinline__ uint64_t block_max(uint64_t d) {   // 256 threads; valid in thread 0
  __shared__ uint64_t red[4];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) d = max(d, (uint64_t)__shfl_down((unsigned long long)d, o, 64));
  if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = d;
  __syncthreads();
  return max(max(red[0], red[1]), max(red[2], red[3]));
}

template <typename T, bool PULLED, bool WALLS>
__global__ void __launch_bounds__(256)
    k_rhoupdat(const T* __restrict__ A, Grid g, double* __restrict__ rho, uint64_t* __restrict__ part) {
  uint64_t d = 0;
  for (uint32_t n = blockIdx.x * 256u + threadIdx.x; n < g.ncell; n += gridDim.x * 256u) {
    int x, y, z;
    uint32_t row;
    node_coords(n, g, x, y, z, row);
    const double old = rho[n];
    double f[NPOP];
    if (PULLED)
      load_pulled<T, double, WALLS>(A, g, x, y, z, n, f);
    else
      load_direct<T, double, WALLS>(A, g, x, y, z, n, f);
    double r = f[0];
#pragma unroll
    for (int i = 1; i < NPOP; ++i) r = r + f[i];
    d = max(d, residual_bits(fabs(r - old)));
    rho[n] = r;
  }
  d = block_max(d);
  if (threadIdx.x == 0) part[blockIdx.x] = d;
}

// The maximum of the workgroups' maxima, stored where the host reads it, and
// then seq in the word the host polls (pinned memory: no copy, no stream
// synchronisation follows).  CLEAR: the maxima are set to zero for the next use.
template <bool CLEAR>
__global__ void __launch_bounds__(256)
    k_rho_residual(uint64_t* __restrict__ part, int n, uint64_t* __restrict__ out, uint32_t seq) {
  uint64_t d = 0;
#pragma unroll 8
  for (int i = threadIdx.x; i < n; i += 256) {
    d = max(d, part[i]);
    if (CLEAR) part[i] = 0;
  }
  d = block_max(d);
  if (threadIdx.x == 0) {
    *out = d ? d - 1 : 0x7ff8000000000000ull;   // no number anywhere: NaN
    __hip_atomic_store((uint32_t*)(out + 1), seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// initpop (initial.f90:3-28): deviation equilibrium with rho = 0.
template <typename T, bool WALLS>
__global__ void __launch_bounds__(256)
    k_initpop(T* __restrict__ A, Grid g, CollideConsts k, bool pulled, double* __restrict__ rho,
              const double* __restrict__ ux, const double* __restrict__ uy,
              const double* __restrict__ uz) {
  const uint32_t n = blockIdx.x * 256u + threadIdx.x;
  if (n >= g.ncell) return;
  int x, y, z;
  uint32_t row;
  node_coords(n, g, x, y, z, row);
  rho[n] = 0.0;
  const double u = ux[n], v = uy[n], w = uz[n];
  const double usqr = 1.5 * (u * u + v * v + w * w);
#pragma unroll
  for (int i = 0; i < NPOP; ++i) {
    const double G = (double)cx(i) * u + (double)cy(i) * v + (double)cz(i) * w;
    const double wt = i == 0 ? k.ww0 : (i <= 6 ? k.ww1 : k.ww2);
    const double fe = i == 0 ? wt * (0.0 - usqr) : wt * (0.0 + 3.0 * G + 4.5 * G * G - usqr);
    store_phase<T, WALLS>(A, g, i, x, y, z, n, pulled, fe);
  }
}

// SoA (resident, current phase) -> AoS double f(0:18, ...) for z in [z0, z0+nzs)
template <typename T, bool WALLS>
__global__ void __launch_bounds__(256)
    k_pop_to_aos(const T* __restrict__ A, Grid g, double* __restrict__ dst, int z0, uint32_t count,
                 bool pulled) {
  const uint32_t q = blockIdx.x * 256u + threadIdx.x;
  if (q >= count) return;
  const uint32_t n = q + (uint32_t)z0 * (uint32_t)g.nx * (uint32_t)g.ny;
  int x, y, z;
  uint32_t row;
  node_coords(n, g, x, y, z, row);
  double f[NPOP];
  if (pulled)
    load_pulled<T, double, WALLS>(A, g, x, y, z, n, f);
  else
    load_direct<T, double, WALLS>(A, g, x, y, z, n, f);
#pragma unroll
  for (int i = 0; i < NPOP; ++i) dst[19ull * q + i] = f[i];
}

template <typename T, bool WALLS>
__global__ void __launch_bounds__(256)
    k_aos_to_pop(T* __restrict__ A, Grid g, const double* __restrict__ src, int z0, uint32_t count,
                 bool pulled) {
  const uint32_t q = blockIdx.x * 256u + threadIdx.x;
  if (q >= count) return;
  const uint32_t n = q + (uint32_t)z0 * (uint32_t)g.nx * (uint32_t)g.ny;
  int x, y, z;
  uint32_t row;
  node_coords(n, g, x, y, z, row);
#pragma unroll
  for (int i = 0; i < NPOP; ++i) store_phase<T, WALLS>(A, g, i, x, y, z, n, pulled, src[19ull * q + i]);
}

__global__ void __launch_bounds__(256)
    k_force_field(Grid g, ForceArgs fa, double* __restrict__ fx, double* __restrict__ fy,
                  double* __restrict__ fz) {
  const uint32_t n = blockIdx.x * 256u + threadIdx.x;
  if (n >= g.ncell) return;
  int x, y, z;
  uint32_t row;
  node_coords(n, g, x, y, z, row);
  double Fx = fa.bfx, Fy = fa.bfy, Fz = fa.bfz;
  if (fa.gcur) {
    double gx, gy, gz;
    force_at(fa.gcur, fa.phx, row, x, g.nx, gx, gy, gz);
    Fx += gx;
    Fy += gy;
    Fz += gz;
  }
  fx[n] = Fx;
  fy[n] = Fy;
  fz[n] = Fz;
}

// ---------------------------------------------------------------------------
static inline unsigned nblocks(uint64_t n) { return (unsigned)((n + 255) / 256); }

static ForceArgs force_args(const Ctx& c) {
  ForceArgs fa;
  fa.gcur = c.ft.live[c.ft.cur] ? c.ft.g[c.ft.cur] : nullptr;
  fa.gmac = c.ft.live[c.ft.mac] ? c.ft.g[c.ft.mac] : nullptr;
  fa.phx = c.ft.phx;
  fa.bfx = c.p.body_force[0];
  fa.bfy = c.p.body_force[1];
  fa.bfz = c.p.body_force[2];
  return fa;
}

hipError_t launch_force_table(Ctx& c, int slot, const ModeSet& m) {
  const uint32_t rows = (uint32_t)c.g.ny * (uint32_t)c.g.nz;
  hipLaunchKernelGGL(k_force_table, dim3((3 * rows + 255) / 256), dim3(256), 0, c.stream, m,
                     c.ft.phy, c.ft.phz, c.g.ny, c.g.nz, c.ft.g[slot]);
  return hipGetLastError();
}

// Arguments of one box's collide launch (also used by the ensemble engine).
CollideArgs collide_args(Ctx& c) {
  CollideArgs a;
  a.A = c.pop[c.cur];
  a.B = c.g.lay == LAY_AB ? c.pop[c.cur ^ 1] : c.pop[c.cur];
  a.mask = (c.pt.np > 0 && c.pt.map_np[c.pt.map_cur] > 0) ? c.pt.mask[c.pt.map_cur] : nullptr;
  a.g = c.g;
  a.k = c.cc;
  a.fa = force_args(c);
  a.rho = c.rho; a.ux = c.ux; a.uy = c.uy; a.uz = c.uz;
  a.arr = 0;
  return a;
}

// How the collide of a box is launched.  Measured on one MI355X, us per
// collide, in fluid-only steps (f) and in steps with spheres (s), whose other
// kernels run between two collides:
//  waves   4 wavefronts per workgroup, 3 where rows are a multiple of three
//          tiles, so that workgroups hold whole rows (192 x 176 x 208 FP32 step
//          with spheres 282 against 284); 1 where the lattice has at most
//          16 tiles per CU (48^3 FP64 f 8.7 against 9.1), and in FP64 rows of
//          up to three quarters of a tile, whose idle lanes leave the wavefront
//          slots as the bound (24 million nodes: nx = 5 f 5.62 against 6.79 ms,
//          17 1.87 against 2.20, 48 1.15 against 1.21; nx = 50 1.32 against
//          1.24; FP32 nx = 17 0.96 and 0.99).  In place with FP64 arithmetic one
//          or two tiles of a row, with ranges: FP32 storage (24 x 256 x 3906 f
//          1207 against 1297 us, 64 x 256 x 1464 676 against 703, 128 x 256 x 732
//          681 against 719, 128 x 160 x 400 s 316 against 323), FP64 from a GiB a
//          tile (64 x 256 x 600 s 590 against 669, 128 x 256 x 732 f 1346 against
//          1358; 100 x 256 x 500, 1.8 GiB, 749 against 717).
//  cached  plain stores where both buffers stay in the 256 MiB last-level
//          cache between steps: from 48 MiB (64^3 FP32, 38 MiB, s 13.1 against
//          11.6 non-temporal; 64^3 FP64, 76 MiB, s 18.6 against 20.2, f 14.0
//          against 17.3) to 260 MiB (96^3 FP64, 257 MiB, f 43 against 47, s 49
//          against 53; 130 x 118 x 126 FP32, 280 MiB, f 64 against 60).
//  ntl     non-temporal loads.  Small lattices (up to 48 MiB: 48^3 FP32 f 5.6
//          against 6.3).  FP64 with spheres (256^3 s 860 against 897, 448 x
//          256 x 256 s 1536 against 1570; without them f 877 against 875, 262
//          x 257 x 227 f 841 against 811; in ragged rows with spheres it is
//          nearly even: 262 x 257 x 227 s 937 against 929, 200 x 190 x 210 s 518
//          against 530, 150 x 141 x 162 s 241 against 243), and large FP64
//          lattices without spheres in rows of whole 64-B half lines (64 x 160
//          x 1000 f 494 against 518, 192 x 256 x 488 1174 against 1187; 75 x 256 x
//          1250 1346-1480 and 1412-1515).  FP32 storage with FP64 arithmetic
//          with spheres (256^3 s 454 against 474, 262 x 257 x 227 s 486
//          against 491) and in rows of whole workgroups (256^3 f 442 against
//          451, but 262 x 257 x 227 f 468 against 450).  FP32 with spheres
//          where a workgroup holds whole rows (256^3 s 430 against 443; 290 x
//          280 x 270 s 722 against 663, where workgroups end inside rows and
//          the next one needs the same cache lines; 256^3 f 451 against 438).
//  per     contiguous workgroups per XCD instead of launch order.  Two
//          buffers: when the 19 populations of a plane reach 18 MiB (512^3
//          FP32 f 3.36 against 3.45-3.61 ms, 1024^3 26.6 against 29.1 ms; 320
//          x 288 x 304 FP32 f 759 against 719), and in lattices up to 128 MiB,
//          whose nodes then meet the same L2 in the next step (40^3 FP32 f 5.0
//          against 6.2).  FP64 without spheres from 2.5 GiB (64 x 256 x 1464 f
//          1173 against 1280 us, 100 x 256 x 937 1306 against 1453, 256^3 822
//          against 867; 200^3, 2.3 GiB, 426 against 413), in rows of more than four
//          tiles from 6 GiB (384 x 256 x 256 1261 against 1315; 262 x 200 x 200
//          575 against 545), in rows of 32 nodes or more (20 x 256 x 2000 771
//          against 721).  In place: always (1024^3 FP64 f 52.5 against 64 ms,
//          130 x 118 x 126 FP32 47 against 58), but rows of up to four tiles
//          that outgrow the last-level cache (200 x 190 x 210 FP64 f 461
//          against 441) up to 2 GiB of FP64 (256 x 256 x 320 f 1052 against 1173).
// One workgroup per row or 256-node chunk of a row, the shape before, left
// half of its lanes idle where a row ends in a short chunk: 320 x 288 x 304
// FP32 f 912 us (now 715) and FP64 in place 1790 (now 1575), 262 x 257 x 227
// FP32 f 773 (now 436), s 785 (now 444) and FP64 f 1226 (now 800), s 1224 (now
// 825); other rows gain from the plain loads and the padding: 150 x 141 x 162
// FP32 f 136 (98), s 134 (97) and FP64 s 232 (195), 96^3 FP64 s 55 (49).
struct CollideShape {
  TileGrid t;
  unsigned grid, block;
  bool cached, ntl;
};
template <typename T, typename R>
static CollideShape collide_shape(const Ctx& c, bool spheres) {
  CollideShape s;
  const uint32_t tpr = (uint32_t)((c.g.nx + kTileX - 1) / kTileX);
  s.t.tpr = fast_div(tpr);
  s.t.ntiles = tpr * (uint32_t)c.g.ny * (uint32_t)c.g.nz;
  const bool ab = c.g.lay == LAY_AB, all64 = sizeof(T) == 8;
  const uint64_t mib = (uint64_t)1 << 20;
  const uint64_t buf = (uint64_t)NPOP * sizeof(T) * c.g.ncell;
  // in place with FP64 arithmetic: a workgroup per row
  const bool row_groups = !ab && sizeof(R) == 8 && tpr <= 2 && (!all64 || c.g.nx <= 48 || buf >= tpr * 1024 * mib);
  s.t.waves = s.t.ntiles <= 4096 || (all64 && c.g.nx <= 48) ? 1 : (tpr % 4 != 0 && tpr % 3 == 0 ? 3 : 4);
  if (row_groups && s.t.ntiles > 4096) s.t.waves = tpr;
  s.block = (unsigned)kTileX * s.t.waves;
  s.grid = (s.t.ntiles + s.t.waves - 1) / s.t.waves;
  const uint64_t plane = (uint64_t)NPOP * sizeof(T) * (uint64_t)c.g.nx * (uint64_t)c.g.ny;
  const bool small = 2 * buf <= 48 * mib;
  s.cached = ab && !small && 2 * buf <= 260 * mib;
  const bool streams64 = ab && all64 && !spheres && c.g.nx >= 32 && 2 * buf >= (tpr <= 4 ? 2560 : 6144) * mib;
  if (sizeof(T) != sizeof(R))
    s.ntl = small || spheres || c.g.nx % 256 == 0;
  else
    s.ntl = small || (streams64 && c.g.nx % 8 == 0) ||
            (spheres && (all64 || (c.g.nx % kTileX == 0 && s.t.waves % tpr == 0)));
  bool ranges;
  if (c.xcd_remap >= 0)
    ranges = c.xcd_remap != 0;
  else if (ab)
    ranges = plane >= 18 * mib || 2 * buf <= 128 * mib || streams64;
  else
    ranges = row_groups || !(tpr <= 4 && buf > 256 * mib) || (all64 && buf >= 2048 * mib);
  s.t.per = ranges ? s.grid / kXcds : 0;
  return s;
}

template <typename T, typename R, int LAY, bool NTL, bool NTS>
static void collide_launch(Ctx& c, bool arrays, const CollideArgs& a, const CollideShape& s) {
  const dim3 grid(s.grid), blk(s.block);
#define MFC_COLLIDE(ARR, W) \
  hipLaunchKernelGGL((k_collide<T, R, ARR, W, LAY, NTL, NTS>), grid, blk, 0, c.stream, a, s.t)
  if (arrays) {
    if (c.g.walls_y) MFC_COLLIDE(true, true); else MFC_COLLIDE(true, false);
  } else {
    if (c.g.walls_y) MFC_COLLIDE(false, true); else MFC_COLLIDE(false, false);
  }
#undef MFC_COLLIDE
}

template <typename T, typename R, int LAY>
static void collide_dispatch_lay(Ctx& c, bool arrays, const CollideArgs& a) {
  const CollideShape s = collide_shape<T, R>(c, a.mask != nullptr);
  if constexpr (LAY == LAY_AB) {
    if (s.cached) {
      collide_launch<T, R, LAY, false, false>(c, arrays, a, s);
      return;
    }
    if (s.ntl) {
      collide_launch<T, R, LAY, true, true>(c, arrays, a, s);
      return;
    }
  }
  collide_launch<T, R, LAY, false, true>(c, arrays, a, s);
}

template <typename T, typename R>
static void collide_dispatch(Ctx& c, bool arrays, const CollideArgs& a) {
  if (c.g.lay == LAY_AA_ODD)
    collide_dispatch_lay<T, R, LAY_AA_ODD>(c, arrays, a);
  else if (c.g.lay == LAY_AA_EVEN)
    collide_dispatch_lay<T, R, LAY_AA_EVEN>(c, arrays, a);
  else
    collide_dispatch_lay<T, R, LAY_AB>(c, arrays, a);
}

template <typename T, typename R, int LAY>
static void collide_tiles_lay(Ctx& c, const CollideArgs& a, const uint32_t* list, uint32_t n) {
  const uint32_t tpr = (uint32_t)((c.g.nx + kTileX - 1) / kTileX);
  const dim3 grid((n + 3) / 4);
  if (c.g.walls_y)
    hipLaunchKernelGGL((k_collide_tiles<T, R, true, LAY>), grid, dim3(256), 0, c.stream, a, list, n, tpr);
  else
    hipLaunchKernelGGL((k_collide_tiles<T, R, false, LAY>), grid, dim3(256), 0, c.stream, a, list, n, tpr);
}

template <typename T, typename R>
static void collide_tiles_dispatch(Ctx& c, const CollideArgs& a, const uint32_t* list, uint32_t n) {
  if (c.g.lay == LAY_AA_ODD)
    collide_tiles_lay<T, R, LAY_AA_ODD>(c, a, list, n);
  else if (c.g.lay == LAY_AA_EVEN)
    collide_tiles_lay<T, R, LAY_AA_EVEN>(c, a, list, n);
  else
    collide_tiles_lay<T, R, LAY_AB>(c, a, list, n);
}

hipError_t launch_collide_tiles(Ctx& c, const uint32_t* list, uint32_t n, bool far) {
  if (n == 0) return hipSuccess;
  CollideArgs a = collide_args(c);
  if (far) a.mask = nullptr;   // no node of a far tile is solid in any map of the step
  if (c.prec == MFC_PREC_FP64)
    collide_tiles_dispatch<double, double>(c, a, list, n);
  else if (c.prec == MFC_PREC_FP32_F64MATH)
    collide_tiles_dispatch<float, double>(c, a, list, n);
  else
    collide_tiles_dispatch<float, float>(c, a, list, n);
  return hipGetLastError();
}

hipError_t launch_collide(Ctx& c, bool arrays) {
  const CollideArgs a = collide_args(c);
  if (c.prec == MFC_PREC_FP64)
    collide_dispatch<double, double>(c, arrays, a);
  else if (c.prec == MFC_PREC_FP32_F64MATH)
    collide_dispatch<float, double>(c, arrays, a);
  else
    collide_dispatch<float, float>(c, arrays, a);
  return hipGetLastError();
}

template <typename T>
static void macro_dispatch(Ctx& c, bool pulled, double* part) {
  const bool parts = c.pt.np > 0 && c.pt.map_np[c.pt.map_cur] > 0;
  const MacroArgs a = {c.pop[c.cur], c.g, force_args(c),
                       parts ? c.pt.mask[c.pt.map_cur] : nullptr, parts ? c.pt.isn[c.pt.map_cur] : nullptr,
                       c.pt.ypglb, c.pt.wp, c.pt.omgp, c.p.rhopart, c.rho, c.ux, c.uy, c.uz};
  const dim3 grid(nblocks(c.g.ncell)), blk(256);
#define MFC_MACRO(P, W)                                                                                        \
  do {                                                                                                         \
    if (part)                                                                                                  \
      hipLaunchKernelGGL((k_macro_sums<T, P, W>), dim3(sum_blocks(c.g.ncell)), dim3(kSumThreads), 0, c.stream, a, part);  \
    else                                                                                                       \
      hipLaunchKernelGGL((k_macro<T, P, W>), grid, blk, 0, c.stream, a);                                       \
  } while (0)
  if (pulled) {
    if (c.g.walls_y) MFC_MACRO(true, true); else MFC_MACRO(true, false);
  } else {
    if (c.g.walls_y) MFC_MACRO(false, true); else MFC_MACRO(false, false);
  }
#undef MFC_MACRO
}

hipError_t launch_macro(Ctx& c, bool pulled) { return launch_macro_sums(c, pulled, nullptr); }

hipError_t launch_macro_sums(Ctx& c, bool pulled, double* part) {
  if (c.prec == MFC_PREC_FP64)
    macro_dispatch<double>(c, pulled, part);
  else
    macro_dispatch<float>(c, pulled, part);
  return hipGetLastError();
}

template <typename T>
static void rhoupdat_dispatch(Ctx& c, bool pulled, dim3 grid, double* part) {
  const T* A = (const T*)c.pop[c.cur];
  const dim3 blk(256);
  if (pulled) {
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_rhoupdat<T, true, true>), grid, blk, 0, c.stream, A, c.g, c.rho, (uint64_t*)part);
    else
      hipLaunchKernelGGL((k_rhoupdat<T, true, false>), grid, blk, 0, c.stream, A, c.g, c.rho, (uint64_t*)part);
  } else {
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_rhoupdat<T, false, true>), grid, blk, 0, c.stream, A, c.g, c.rho, (uint64_t*)part);
    else
      hipLaunchKernelGGL((k_rhoupdat<T, false, false>), grid, blk, 0, c.stream, A, c.g, c.rho, (uint64_t*)part);
  }
}

int rhoupdat_blocks(const Ctx& c) { return (int)std::min(nblocks(c.g.ncell), 16384u); }

hipError_t launch_rhoupdat(Ctx& c, bool pulled, double* part, double* out, uint32_t seq) {
  const unsigned nb = (unsigned)rhoupdat_blocks(c);
  if (c.prec == MFC_PREC_FP64)
    rhoupdat_dispatch<double>(c, pulled, dim3(nb), part);
  else
    rhoupdat_dispatch<float>(c, pulled, dim3(nb), part);
  if (out) hipLaunchKernelGGL(k_rho_residual<false>, dim3(1), dim3(256), 0, c.stream, (uint64_t*)part, (int)nb,
                              (uint64_t*)out, seq);
  return hipGetLastError();
}

template <typename T, typename R>
static void relax_dispatch(Ctx& c, const CollideArgs& a, unsigned long long* slots) {
  const CollideShape s = collide_shape<T, R>(c, false);
  const dim3 grid(s.grid), blk(s.block);
#define MFC_RELAX(NTL, NTS)                                                                                     \
  do {                                                                                                          \
    if (c.g.walls_y)                                                                                            \
      hipLaunchKernelGGL((k_collide_relax<T, R, true, NTL, NTS>), grid, blk, 0, c.stream, a, s.t, slots);       \
    else                                                                                                        \
      hipLaunchKernelGGL((k_collide_relax<T, R, false, NTL, NTS>), grid, blk, 0, c.stream, a, s.t, slots);      \
  } while (0)
  if (s.cached)
    MFC_RELAX(false, false);
  else if (s.ntl)
    MFC_RELAX(true, true);
  else
    MFC_RELAX(false, true);
#undef MFC_RELAX
}

int relax_slots() { return (int)kRelaxSlots; }

hipError_t launch_collide_relax(Ctx& c, double* slots, double* out, uint32_t seq) {
  const CollideArgs a = collide_args(c);
  unsigned long long* sl = (unsigned long long*)slots;
  if (c.prec == MFC_PREC_FP64)
    relax_dispatch<double, double>(c, a, sl);
  else if (c.prec == MFC_PREC_FP32_F64MATH)
    relax_dispatch<float, double>(c, a, sl);
  else
    relax_dispatch<float, float>(c, a, sl);
  hipLaunchKernelGGL(k_rho_residual<true>, dim3(1), dim3(256), 0, c.stream, (uint64_t*)slots, (int)kRelaxSlots,
                     (uint64_t*)out, seq);
  return hipGetLastError();
}

hipError_t launch_initpop(Ctx& c) {
  const dim3 grid(nblocks(c.g.ncell)), blk(256);
  const bool pulled = c.phase == PHASE_POST_STREAM;
  if (c.prec == MFC_PREC_FP64) {
    double* A = (double*)c.pop[c.cur];
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_initpop<double, true>), grid, blk, 0, c.stream, A, c.g, c.cc, pulled, c.rho, c.ux, c.uy, c.uz);
    else
      hipLaunchKernelGGL((k_initpop<double, false>), grid, blk, 0, c.stream, A, c.g, c.cc, pulled, c.rho, c.ux, c.uy, c.uz);
  } else {
    float* A = (float*)c.pop[c.cur];
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_initpop<float, true>), grid, blk, 0, c.stream, A, c.g, c.cc, pulled, c.rho, c.ux, c.uy, c.uz);
    else
      hipLaunchKernelGGL((k_initpop<float, false>), grid, blk, 0, c.stream, A, c.g, c.cc, pulled, c.rho, c.ux, c.uy, c.uz);
  }
  return hipGetLastError();
}

hipError_t launch_pop_to_aos(Ctx& c, double* dst, int z0, int nzs, bool pulled) {
  const uint32_t count = (uint32_t)c.g.nx * (uint32_t)c.g.ny * (uint32_t)nzs;
  const dim3 grid(nblocks(count)), blk(256);
  if (c.prec == MFC_PREC_FP64) {
    const double* A = (const double*)c.pop[c.cur];
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_pop_to_aos<double, true>), grid, blk, 0, c.stream, A, c.g, dst, z0, count, pulled);
    else
      hipLaunchKernelGGL((k_pop_to_aos<double, false>), grid, blk, 0, c.stream, A, c.g, dst, z0, count, pulled);
  } else {
    const float* A = (const float*)c.pop[c.cur];
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_pop_to_aos<float, true>), grid, blk, 0, c.stream, A, c.g, dst, z0, count, pulled);
    else
      hipLaunchKernelGGL((k_pop_to_aos<float, false>), grid, blk, 0, c.stream, A, c.g, dst, z0, count, pulled);
  }
  return hipGetLastError();
}

hipError_t launch_aos_to_pop(Ctx& c, const double* src, int z0, int nzs, bool pulled) {
  const uint32_t count = (uint32_t)c.g.nx * (uint32_t)c.g.ny * (uint32_t)nzs;
  const dim3 grid(nblocks(count)), blk(256);
  if (c.prec == MFC_PREC_FP64) {
    double* A = (double*)c.pop[c.cur];
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_aos_to_pop<double, true>), grid, blk, 0, c.stream, A, c.g, src, z0, count, pulled);
    else
      hipLaunchKernelGGL((k_aos_to_pop<double, false>), grid, blk, 0, c.stream, A, c.g, src, z0, count, pulled);
  } else {
    float* A = (float*)c.pop[c.cur];
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_aos_to_pop<float, true>), grid, blk, 0, c.stream, A, c.g, src, z0, count, pulled);
    else
      hipLaunchKernelGGL((k_aos_to_pop<float, false>), grid, blk, 0, c.stream, A, c.g, src, z0, count, pulled);
  }
  return hipGetLastError();
}

hipError_t launch_force_field(Ctx& c, int slot, double* fx, double* fy, double* fz) {
  ForceArgs fa = force_args(c);
  fa.gcur = c.ft.live[slot] ? c.ft.g[slot] : nullptr;
  hipLaunchKernelGGL(k_force_field, dim3(nblocks(c.g.ncell)), dim3(256), 0, c.stream, c.g, fa, fx, fy, fz);
  return hipGetLastError();
}

}  // namespace mfc

namespace mfc {

template <typename T, typename R, int BS, bool ARR_ANY>
static void batched_collide_k(int walls, const CollideArgs* t, const int* off, int nc, int blocks, int remap,
                              bool ntl, hipStream_t s) {
#define MFC_BATCHED(W, N) \
  hipLaunchKernelGGL((kb_collide<T, R, W, BS, ARR_ANY, N>), dim3(blocks), dim3(BS), 0, s, t, off, nc, remap)
  // a first step after joining (ARR_ANY) is rare: non-temporal only
  if (ARR_ANY || ntl) {
    if (walls) MFC_BATCHED(true, true); else MFC_BATCHED(false, true);
  } else {
    if (walls) MFC_BATCHED(true, ARR_ANY); else MFC_BATCHED(false, ARR_ANY);
  }
#undef MFC_BATCHED
}

template <int BS, bool ARR_ANY>
static void batched_collide_bs(int prec, int walls, const void* t, const int* off, int nc, int blocks,
                               int remap, bool ntl, hipStream_t s) {
  const CollideArgs* tab = (const CollideArgs*)t;
  if (prec == MFC_PREC_FP64)
    batched_collide_k<double, double, BS, ARR_ANY>(walls, tab, off, nc, blocks, remap, ntl, s);
  else if (prec == MFC_PREC_FP32_F64MATH)
    batched_collide_k<float, double, BS, ARR_ANY>(walls, tab, off, nc, blocks, remap, ntl, s);
  else
    batched_collide_k<float, float, BS, ARR_ANY>(walls, tab, off, nc, blocks, remap, ntl, s);
}

hipError_t launch_batched_collide(int prec, int walls, int bs, int remap, const void* t, const int* off,
                                  int nc, int blocks, bool arr_any, bool ntl, hipStream_t s) {
  if (nc <= 0 || blocks <= 0) return hipSuccess;
  switch (bs) {
    case 64:
      arr_any ? batched_collide_bs<64, true>(prec, walls, t, off, nc, blocks, remap, ntl, s)
              : batched_collide_bs<64, false>(prec, walls, t, off, nc, blocks, remap, ntl, s);
      break;
    case 128:
      arr_any ? batched_collide_bs<128, true>(prec, walls, t, off, nc, blocks, remap, ntl, s)
              : batched_collide_bs<128, false>(prec, walls, t, off, nc, blocks, remap, ntl, s);
      break;
    case 256:
      arr_any ? batched_collide_bs<256, true>(prec, walls, t, off, nc, blocks, remap, ntl, s)
              : batched_collide_bs<256, false>(prec, walls, t, off, nc, blocks, remap, ntl, s);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace mfc
