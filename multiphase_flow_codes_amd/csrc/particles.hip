// particles.hip -- finite-size moving spheres: node maps, boundary links,
// interpolated bounce-back with momentum exchange, lubrication, Newton-Euler
// motion and refilling of uncovered nodes (BOX/partlib.f90).
//
// Data layout.  Node maps are double-buffered (current / previous step):
// an int32 id map (particle id, 1-based, or 0) and a 1-bit solid mask read by
// the collide kernel.  Boundary links (node index, direction, wall fraction)
// are listed per segment of a particle's bounding box, each segment in a slot
// of its own (Particles::lk_seg links), in a deterministic order by the workgroup
// that scans the segment; no dense 18-per-node link arrays exist.  Maps are maintained incrementally: a build
// first clears the nodes its buffer marked two steps earlier, so no pass
// ever touches the whole lattice.  All particle state is FP64.
//
// Compiled with -ffp-contract=off: the geometry is evaluated exactly as the
// reference writes it, so maps and wall fractions match the FP64 oracle bit
// for bit.
#include <algorithm>

#include <math.h>

#include "force_table.h"
#include "internal.h"
#include "lbm_access.h"
#include "lbm_particle_math.h"
#include "step_args.h"

namespace mfc {

constexpr int PB = 256;  // threads per particle workgroup
// A segment is one z-slab (G.slab planes: 1, 2, 4 or 8) of one particle's bounding
// box: the unit of work of every box-scan kernel, so a sphere spreads over
// several workgroups.  Segment s of particle p is block p * nseg + s.


struct AxisRange {
  int lo, cnt;
};

__device__ __forceinline__ int wrap_any(int a, int n) {
  int r = a % n;
  return r < 0 ? r + n : r;
}

__device__ __forceinline__ bool sane_coord(double c, int n) { return isfinite(c) && c >= 0.0 && c < (double)n; }

// Candidate node indices (unwrapped, 0-based) whose centre i+0.5 can lie
// within radp2 of c: a superset of the reference's test |pnt - c_img| <= radp2.
__device__ __forceinline__ AxisRange axis_range(double c, double radp2) {
  AxisRange r;
  r.lo = (int)floor(c - radp2 - 0.5) - 1;
  const int hi = (int)ceil(c + radp2 - 0.5) + 1;
  r.cnt = hi - r.lo + 1;
  return r;
}

// Per-particle constants of a box scan, computed by thread 0.
struct BoxInfo {
  int ok;
  double x0, y0, z0, xr, yr;   // original centre and sweep-rest bases
  int kfirst, jfirst;          // first k (index order) in the box, first j of that row
  AxisRange ax, ay, az;
};

__device__ double y_image(double ybase, double ypnt, const PGeom& G) {
  return G.walls_y ? ybase : near_image(ybase, ypnt, G.ny);
}

// one-period wrap (the box candidate ranges never span more than a period)
__device__ __forceinline__ int wrap1(int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); }

__device__ __forceinline__ bool bit_at(const uint32_t* __restrict__ mask, uint32_t n) {
  return (mask[n >> 5] >> (n & 31u)) & 1u;
}

// ---- pair-search cells ------------------------------------------------------
// Cell of coordinate v in [0, n) on an axis of nc cells (each at least as
// wide as the longest pair range, so partners sit in adjacent cells).
__device__ __forceinline__ int cell_of(double v, int n, int nc) {
  int c = (int)(v * (double)nc / (double)n);
  return c < 0 ? 0 : (c >= nc ? nc - 1 : c);
}

__device__ __forceinline__ void cell_coords(const double* __restrict__ ypglb, int p, const PGeom& G,
                                            const CellArgs& C, int& cx_, int& cy_, int& cz_) {
  cx_ = cell_of(ypglb[3 * p], G.nx, C.ncx);
  cy_ = cell_of(ypglb[3 * p + 1], G.ny, C.ncy);
  cz_ = cell_of(ypglb[3 * p + 2], G.nz, C.ncz);
}

// Index of neighbour cell k (0..26) of (cx_, cy_, cz_), or -1 beyond a wall.
__device__ __forceinline__ int cell_neighbour(const CellArgs& C, const PGeom& G, int cx_, int cy_,
                                              int cz_, int k) {
  const int dx = k % 3 - 1, dy = (k / 3) % 3 - 1, dz = k / 9 - 1;
  int y = cy_ + dy;
  if (G.walls_y) {
    if (y < 0 || y >= C.ncy) return -1;
  } else {
    y = wrap1(y, C.ncy);
  }
  const int x = wrap1(cx_ + dx, C.ncx), z = wrap1(cz_ + dz, C.ncz);
  return x + C.ncx * (y + C.ncy * z);
}

__global__ void k_cell_zero(int32_t* __restrict__ cnt, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) cnt[i] = 0;
}

// Enters particle p, centre (x, y, z), in its cell.
__device__ __forceinline__ void cell_insert(int p, double x, double y, double z, const PGeom& G,
                                            const CellArgs& C, int32_t* __restrict__ status) {
  if (!(sane_coord(x, G.nx) && sane_coord(y, G.ny) && sane_coord(z, G.nz)))
    return;   // reported by the move / links kernels
  const int cell = cell_of(x, G.nx, C.ncx) + C.ncx * (cell_of(y, G.ny, C.ncy) + C.ncy * cell_of(z, G.nz, C.ncz));
  const int slot = atomicAdd(&C.cnt[cell], 1);
  if (slot < kCellCap)
    C.list[cell * kCellCap + slot] = p;
  else
    atomicAdd(&status[ST_CELL_OVERFLOW], 1);
}

__global__ void __launch_bounds__(256)
    k_cell_build(const double* __restrict__ ypglb, int np, PGeom G, CellArgs C,
                 int32_t* __restrict__ status) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < np) cell_insert(p, ypglb[3 * p], ypglb[3 * p + 1], ypglb[3 * p + 2], G, C, status);
}

// Overlap test of ovlpchk (partlib.f90:118-171) for the pair (p, q), q > p.
__device__ __forceinline__ bool pair_overlaps(const double* __restrict__ ypglb, int p, int q,
                                              const PGeom& G) {
  const double xc = ypglb[3 * p], yc = ypglb[3 * p + 1], zc = ypglb[3 * p + 2];
  const double xb = near_image(ypglb[3 * q], xc, G.nx);
  const double yb = G.walls_y ? ypglb[3 * q + 1] : near_image(ypglb[3 * q + 1], yc, G.ny);
  const double zb = near_image(ypglb[3 * q + 2], zc, G.nz);
  const double dist = sqrt((xc - xb) * (xc - xb) + (yc - yb) * (yc - yb) + (zc - zb) * (zc - zb));
  return dist - 2.0 * G.rad < 0.0;
}

// Does particle p overlap a later one?  Evaluated by the calling block: all
// later particles (no cells) or one neighbour cell per thread.
__device__ bool block_overlap(const double* __restrict__ ypglb, int p, int np, const PGeom& G,
                              const CellArgs& C) {
  __shared__ int hit;
  if (threadIdx.x == 0) hit = 0;
  __syncthreads();
  if (C.cnt) {
    if (threadIdx.x < 27) {
      int a, b, c;
      cell_coords(ypglb, p, G, C, a, b, c);
      const int cell = cell_neighbour(C, G, a, b, c, (int)threadIdx.x);
      if (cell >= 0) {
        const int n = min(C.cnt[cell], kCellCap);
        for (int k = 0; k < n; ++k) {
          const int q = C.list[cell * kCellCap + k];
          if (q > p && pair_overlaps(ypglb, p, q, G)) hit = 1;
        }
      }
    }
  } else {
    for (int q = p + 1 + threadIdx.x; q < np; q += PB)
      if (pair_overlaps(ypglb, p, q, G)) hit = 1;
  }
  __syncthreads();
  return hit != 0;
}

// Per-particle constants of a box scan (shared memory), computed by the whole
// block: thread 0 sets the centre and candidate ranges, then every thread
// tests one z or y candidate and the first passing index wins by atomicMin.
__device__ void box_info(const double* __restrict__ pos, int p, const PGeom& G, BoxInfo& B) {
  if (threadIdx.x == 0) {
    B.x0 = pos[3 * p];
    B.y0 = pos[3 * p + 1];
    B.z0 = pos[3 * p + 2];
    B.ok = sane_coord(B.x0, G.nx) && sane_coord(B.y0, G.ny) && sane_coord(B.z0, G.nz);
    if (B.ok) {
      B.xr = sweep_rest_base(B.x0, G.nx);
      B.yr = G.walls_y ? B.y0 : sweep_rest_base(B.y0, G.ny);
      B.ax = axis_range(B.x0, G.radp2);
      B.ay = axis_range(B.y0, G.radp2);
      B.az = axis_range(B.z0, G.radp2);
      if (B.ax.cnt > G.nx || B.ay.cnt > G.ny || B.az.cnt > G.nz) B.ok = 0;
    }
    B.kfirst = 1 << 30;
    B.jfirst = 1 << 30;
  }
  __syncthreads();
  if (B.ok) {
    for (int t = threadIdx.x; t < B.az.cnt; t += blockDim.x) {
      const int kw = wrap1(B.az.lo + t, G.nz);
      const double zp = (double)(kw + 1) - 0.5;
      const double zz0 = zp - near_image(B.z0, zp, G.nz);
      if (fabs(zz0) <= G.radp2) atomicMin(&B.kfirst, kw);
    }
    for (int t = threadIdx.x; t < B.ay.cnt; t += blockDim.x) {
      const int jw = G.walls_y ? B.ay.lo + t : wrap1(B.ay.lo + t, G.ny);
      if (jw < 0 || jw >= G.ny) continue;
      const double yp = (double)(jw + 1) - 0.5;
      const double yy0 = yp - y_image(B.y0, yp, G);
      if (fabs(yy0) <= G.radp2) atomicMin(&B.jfirst, jw);
    }
  }
  __syncthreads();
}

__device__ __forceinline__ int block_exclusive_scan(int v, int* sh, int& total);

// Rows (y, z) of one segment's walk: the x run of each row that can hold
// nodes within r + 1.5 of the centre (a superset: the node test decides).  A
// segment has at most PB rows (one thread per row): slab planes of at most
// PB / slab candidate rows each, which the choice of slab guarantees
// (segment_planes).
struct SegRow {
  uint32_t n0;         // node index of the row's x = 0
  int xs;              // flattened index t of the row is at x = xs + t (unwrapped)
  int jw, kw;
  double yimg, zimg;   // imaged centre used for the row's nodes
};

// Geometry of the node at unwrapped x `ux` of row w (iw: its wrapped x).
// Returns false if the node is outside the reference's bounding box
// (partlib.f90:965-985); rows outside it or beyond a wall have no run.
__device__ __forceinline__ bool node_geom(const BoxInfo& B, const PGeom& G, const SegRow& w, int ux, int& iw, LinkGeom& L) {
  iw = wrap1(ux, G.nx);
  const double zp = (double)(w.kw + 1) - 0.5;
  L.zimg = w.zimg;
  L.zz0 = zp - L.zimg;
  const double yp = (double)(w.jw + 1) - 0.5;
  L.yimg = w.yimg;
  L.yy0 = yp - L.yimg;
  const double xp = (double)(iw + 1) - 0.5;
  L.ximg = near_image((w.kw == B.kfirst && w.jw == B.jfirst) ? B.x0 : B.xr, xp, G.nx);
  L.xx0 = xp - L.ximg;
  L.rr0 = L.xx0 * L.xx0 + L.yy0 * L.yy0 + L.zz0 * L.zz0;
  return fabs(L.xx0) <= G.radp2;
}

// Walk of one segment (z-slab s) of the box in passes of PB candidate nodes,
// the slab's row runs flattened x-fastest so every lane of a pass has a node.
// Every thread runs the same number of passes (barriers are allowed in fn);
// fn(active, row, ux) is called once per pass, in row-major, x-ascending
// node order.  rowof: LDS bytes, one per node of the walk, for its row's
// number (written by the row's thread; a search of the rows' starts by every
// node is a chain of six dependent LDS reads).
template <typename F>
__device__ __forceinline__ void walk_segment(const BoxInfo& B, const PGeom& G, int s, SegRow* rows,
                                             uint8_t* rowof, int* sh, F&& fn) {
  const int z0 = s * G.slab;
  const int nzs = max(0, min(G.slab, B.az.cnt - z0));
  const int nrows = nzs * B.ay.cnt;   // <= PB
  // x run of each row (a row at most PB nodes)
  int run = 0;
  SegRow w;
  const int r = (int)threadIdx.x;
  if (r < nrows) {
    const int tz = r / B.ay.cnt, ty = r - tz * B.ay.cnt;
    const int kw = wrap1(B.az.lo + z0 + tz, G.nz);
    const int jw = G.walls_y ? B.ay.lo + ty : wrap1(B.ay.lo + ty, G.ny);
    if (jw >= 0 && jw < G.ny) {
      const double zp = (double)(kw + 1) - 0.5;
      w.zimg = near_image(B.z0, zp, G.nz);
      const double zz0 = zp - w.zimg;
      const double yp = (double)(jw + 1) - 0.5;
      w.yimg = y_image(kw == B.kfirst ? B.y0 : B.yr, yp, G);
      const double yy0 = yp - w.yimg;
      const double rem = G.rlink2 - yy0 * yy0 - zz0 * zz0;
      if (fabs(zz0) <= G.radp2 && fabs(yy0) <= G.radp2 && rem >= 0.0) {
        // node i (unwrapped) sits at i + 0.5; keep |i + 0.5 - x0| <= sqrt(rem) + 1
        const double dx = sqrt(rem) + 1.0;
        const int ilo = max((int)ceil(B.x0 - dx - 0.5), B.ax.lo);
        const int ihi = min((int)floor(B.x0 + dx - 0.5), B.ax.lo + B.ax.cnt - 1);
        if (ihi >= ilo) {
          run = ihi - ilo + 1;
          w.xs = ilo;
          w.jw = jw;
          w.kw = kw;
          w.n0 = (uint32_t)G.nx * ((uint32_t)jw + (uint32_t)G.ny * (uint32_t)kw);
        }
      }
    }
  }
  int total;
  const int st = block_exclusive_scan(run, sh, total);
  if (run > 0) {
    w.xs -= st;
    rows[r] = w;
    for (int i = 0; i < run; ++i) rowof[st + i] = (uint8_t)r;
  }
  __syncthreads();
  for (int t0 = 0; t0 < total; t0 += PB) {
    const int t = t0 + (int)threadIdx.x;
    const bool act = t < total;
    const int row = act ? (int)rowof[t] : 0;
    fn(act, row, act ? rows[row].xs + t : 0);
  }
}

// Directions q (bit q) along which the neighbour of a node is inside the
// sphere (rr1 - r2 <= 0, the squares of the three possible offsets per axis
// taken once; the sums are those of link_end).
__device__ __forceinline__ uint32_t link_hits(const LinkGeom& L, int iw, int jw, int kw, double r2) {
  double X[3], Y[3], Z[3];
#pragma unroll
  for (int o = 0; o < 3; ++o) {
    const double x = (double)(iw + o) - 0.5 - L.ximg;
    const double y = (double)(jw + o) - 0.5 - L.yimg;
    const double z = (double)(kw + o) - 0.5 - L.zimg;
    X[o] = x * x;
    Y[o] = y * y;
    Z[o] = z * z;
  }
  uint32_t hits = 0;
#pragma unroll
  for (int q = 1; q < NPOP; ++q)
    if (X[cx(q) + 1] + Y[cy(q) + 1] + Z[cz(q) + 1] - r2 <= 0.0) hits |= 1u << q;
  return hits;
}

// The neighbour of node (iw, jw, kw) along q: its offsets from the centre.
__device__ __forceinline__ void link_end(const LinkGeom& L, int iw, int jw, int kw, int q, double& xx1,
                                         double& yy1, double& zz1, double& rr1) {
  xx1 = (double)(iw + 1 + cx(q)) - 0.5 - L.ximg;
  yy1 = (double)(jw + 1 + cy(q)) - 0.5 - L.yimg + 0.0;
  zz1 = (double)(kw + 1 + cz(q)) - 0.5 - L.zimg + 0.0;
  rr1 = xx1 * xx1 + yy1 * yy1 + zz1 * zz1;
}

// Wavefront-wide inclusive scans through DPP lane moves (no LDS round trip):
// within each row of 16 lanes by shifts of 1, 2, 4 and 8 (lanes shifted in
// from outside the row contribute 0), then lane 15 of each row into the next
// row and lane 31 into the upper half.  Every lane of the wavefront must be
// active.  DPP controls: row_shr:n = 0x110 + n, row_bcast:15 = 0x142,
// row_bcast:31 = 0x143; rows left out by the row mask keep the old value 0.
__device__ __forceinline__ int wave_inclusive_add(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return x;
}

// Bitwise OR of x over the wavefront (every lane active), in every lane.
__device__ __forceinline__ uint32_t wave_or(uint32_t x) {
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);
  x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);
  return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

// Exclusive prefix sum over the PB threads of a block: a DPP scan inside
// each 64-lane wavefront, then the wavefront totals through LDS.
__device__ __forceinline__ int block_exclusive_scan(int v, int* sh, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int x = wave_inclusive_add(v);
  if (lane == 63) sh[w] = x;
  __syncthreads();
  int before = 0, tot = 0;
#pragma unroll
  for (int q = 0; q < PB / 64; ++q) {
    const int t = sh[q];
    before += (q < w) ? t : 0;
    tot += t;
  }
  __syncthreads();
  total = tot;
  return before + x - v;
}


// Set (or clear) the solid bit of node n for every lane with `on`, issuing
// one atomic per distinct mask word per wavefront: lanes walking a box row
// share one or two words, and same-address atomics from one instruction
// would otherwise serialise.  Must be called by every lane of the wavefront.
__device__ __forceinline__ void mask_update(uint32_t* __restrict__ mask, bool on, uint32_t n, bool set) {
  uint64_t pending = __ballot(on);
  const uint32_t wd = n >> 5;
  const uint32_t bit = on ? (1u << (n & 31u)) : 0u;
  const int lane = threadIdx.x & 63;
  while (pending) {
    const int leader = __ffsll((unsigned long long)pending) - 1;
    const uint32_t wl = (uint32_t)__builtin_amdgcn_readlane((int)wd, leader);
    const bool mem = on && wd == wl;
    const uint32_t v = wave_or(mem ? bit : 0u);
    if (lane == leader) {
      if (set)
        atomicOr(&mask[wl], v);
      else
        atomicAnd(&mask[wl], ~v);
    }
    pending &= ~__ballot(mem);
  }
}

// Position of each flagged lane in a deterministic block-wide order (pass
// order, then thread order) for two flags at once, with one barrier per call:
// wave totals go through LDS slots that alternate between calls.  base_* hold
// the running totals of earlier calls and are advanced by this one.
__device__ __forceinline__ void block_place2(bool fa, bool fb, int (*wt)[PB / 64][2], int& parity,
                                             int& base_a, int& base_b, int& at_a, int& at_b) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t ba = __ballot(fa), bb = __ballot(fb);
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  if (lane == 0) {
    wt[parity][w][0] = __popcll(ba);
    wt[parity][w][1] = __popcll(bb);
  }
  __syncthreads();
  int pa = 0, pb = 0, ta = 0, tb = 0;
#pragma unroll
  for (int q = 0; q < PB / 64; ++q) {
    const int ca = wt[parity][q][0], cb = wt[parity][q][1];
    pa += (q < w) ? ca : 0;
    pb += (q < w) ? cb : 0;
    ta += ca;
    tb += cb;
  }
  at_a = base_a + pa + __popcll(ba & below);
  at_b = base_b + pb + __popcll(bb & below);
  base_a += ta;
  base_b += tb;
  parity ^= 1;
}

// beads_links, first half of the map rebuild (partlib.f90:945-949): reset the
// nodes the same map buffer marked two steps earlier, from that build's solid
// lists.  Every marked node of the buffer is to be reset before any new mark
// (the marks come in a later grid), so each listed node's id and its whole
// 32-node mask word are stored as zero: no read, no atomic; a word or a node
// listed by several spheres receives the same zero from each.
__device__ void clear_segment(int b, int seg_cap, const uint32_t* __restrict__ sol_list,
                              const int32_t* __restrict__ sol_cnt, int32_t* __restrict__ isn,
                              uint32_t* __restrict__ mask) {
  const int cnt = sol_cnt[b];
  const uint32_t* lst = sol_list + (size_t)b * seg_cap;
  for (int e = (int)threadIdx.x; e < cnt; e += PB) {
    const uint32_t n = lst[e];
    isn[n] = 0;
    mask[n >> 5] = 0u;
  }
}

__global__ void __launch_bounds__(PB)
    k_map_clear(int seg_cap, const uint32_t* __restrict__ sol_list,
                const int32_t* __restrict__ sol_cnt, int32_t* __restrict__ isn,
                uint32_t* __restrict__ mask) {
  clear_segment(blockIdx.x, seg_cap, sol_list, sol_cnt, isn, mask);
}

// beads_links (partlib.f90:934-1043) for one segment of a particle's box:
// classify every box node (solid: mark the id map and mask, list it; fluid
// within r + 1.5: keep it in LDS), then test the 18 directions of the kept
// nodes, one node per lane, list their links (node, direction) in LDS and
// write them with their wall fractions (partlib.f90:1013-1024), one link per
// lane, into the segment's slot, in (node, direction) order.  With `ovl` set the
// first segment of each particle also performs the overlap check of
// beads_redistribute (partlib.f90:2631-2646) on the freshly wrapped positions.
// Dynamic LDS: shell_bytes for the kept nodes, packed_bytes for a pass's links
// (during the walk: its rows' numbers), then the segment's rows.
// Bound: instructions (FP64 geometry of the candidates, then of the kept nodes
// and the links); more waves per SIMD change nothing.  Slots of fixed size
// need no offsets: with links placed by a prefix sum over all segments (shell
// lists in memory, a grid for the sum, a grid to write the links and find the
// nodes to refill) the rebuild and the refill took 88 us at 256^3 with 300
// spheres of radius 8, 82 us with 900 of radius 4, 284 us with 2500 of radius
// 6 and 33 us at 64^3 in FP64 with 8 of radius 4; with slots 68, 58, 248 and 21
// us, and 62 to 70, 49, 189 and 17 with the segment sizes chosen since and no list
// of contact links.  Of the slots' times the scan was 66, 52, 220 and 13.5 us while each node searched the
// rows' starts for its row and took the image of the centre by itself and each
// direction squared its own offsets: 44, 34, 144 and 11.3 us with the rows'
// numbers and geometry in LDS and the squares shared.
constexpr int kPassLinks = 9 * PB;   // a node outside a sphere has at most 9 links
__host__ __device__ constexpr int shell_bytes(int seg_cap) { return (2 * seg_cap + 7) & ~7; }
__host__ __device__ constexpr int packed_bytes(int seg_cap) {
  return seg_cap > 4 * kPassLinks ? (seg_cap + 7) & ~7 : 4 * kPassLinks;
}
__device__ __forceinline__ void links_scan_body(int b_, const double* __restrict__ ypglb, int np, int nseg, int seg_cap, PGeom G,
                 int32_t* __restrict__ isn, uint32_t* __restrict__ mask,
                 uint32_t* __restrict__ sol_list, int32_t* __restrict__ sol_cnt,
                 const LinkSlots& lk, int32_t* __restrict__ ct_count, int ovl, int istep,
                 int32_t* __restrict__ status, CellArgs cells) {
  extern __shared__ uint64_t scan_mem[];
  uint16_t* shell = (uint16_t*)scan_mem;                                  // row << 8 | x in the box
  uint32_t* packed = (uint32_t*)((char*)scan_mem + shell_bytes(seg_cap));   // shell index | direction << 24
  uint8_t* rowof = (uint8_t*)packed;                                      // before the links
  SegRow* rows = (SegRow*)((char*)packed + packed_bytes(seg_cap));
  __shared__ BoxInfo B;
  __shared__ int wt[2][PB / 64][2];
  __shared__ int sh[PB / 64];
  const int b = b_;
  const int p = (int)div_by((uint32_t)b, G.dseg), s = b - p * nseg;
  if (p >= np) return;
  if (b == 0 && threadIdx.x == 0) *ct_count = 0;   // listed again once the map is complete
  if (ovl && s == 0) {
    // ovlpchk: flag p if any later particle is closer than 2r
    const bool hit = block_overlap(ypglb, p, np, G, cells);
    if (threadIdx.x == 0 && hit) {
      atomicAdd(&status[ST_OVERLAP], 1);
      atomicCAS(&status[ST_OVERLAP_STEP], 0, istep);
    }
  }
  box_info(ypglb, p, G, B);
  if (!B.ok) {
    if (threadIdx.x == 0) {
      lk.cnt[b] = 0;
      sol_cnt[b] = 0;
      if (s == 0) atomicAdd(&status[ST_BOX_FAULT], 1);
    }
    return;
  }
  uint32_t* sol = sol_list + (size_t)b * seg_cap;
  int parity = 0, nsol = 0, nshell = 0;
  walk_segment(B, G, s, rows, rowof, sh, [&](bool act, int row, int ux) {
    LinkGeom L;
    int iw = 0;
    const bool in = act && node_geom(B, G, rows[row], ux, iw, L) && L.rr0 <= G.rlink2;
    const bool solid = in && (L.rr0 - G.r2 <= 0.0);
    const bool near = in && !solid;
    const uint32_t n = act ? rows[row].n0 + (uint32_t)iw : 0u;
    if (solid) atomicMax(&isn[n], p + 1);   // the highest id containing the node wins
    mask_update(mask, solid, n, true);
    int at_s, at_n;
    block_place2(solid, near, wt, parity, nsol, nshell, at_s, at_n);
    if (solid && at_s < seg_cap) sol[at_s] = n;
    if (near && at_n < seg_cap) shell[at_n] = (uint16_t)(row << 8 | (ux - B.ax.lo));
  });
  __syncthreads();
  const int nsh = min(nshell, seg_cap);
  const int64_t slot = (int64_t)b * lk.cap;
  int nl = 0, alpha_bad = 0;
  for (int e0 = 0; e0 < nsh; e0 += PB) {
    const int e = e0 + (int)threadIdx.x;
    uint32_t hits = 0;
    if (e < nsh) {
      const uint32_t at = shell[e];
      const SegRow w = rows[at >> 8];
      LinkGeom L;
      int iw;
      node_geom(B, G, w, B.ax.lo + (int)(at & 255u), iw, L);
      hits = link_hits(L, iw, w.jw, w.kw, G.r2);
    }
    int tot;
    int at = block_exclusive_scan(__popc(hits), sh, tot);
    while (hits) {
      const int q = __ffs(hits) - 1;
      hits &= hits - 1;
      if (at < kPassLinks) packed[at] = (uint32_t)e | ((uint32_t)q << 24);
      ++at;
    }
    __syncthreads();
    tot = min(tot, kPassLinks);
    for (int l = (int)threadIdx.x; l < tot; l += PB) {
      const uint32_t pk = packed[l];
      const uint32_t from = shell[pk & 0xffffffu];
      const int q = (int)(pk >> 24);
      const SegRow w = rows[from >> 8];
      LinkGeom L;
      int iw;
      node_geom(B, G, w, B.ax.lo + (int)(from & 255u), iw, L);
      double xx1, yy1, zz1, rr1;
      link_end(L, iw, w.jw, w.kw, q, xx1, yy1, zz1, rr1);
      const double alpha = link_alpha(L, xx1, yy1, zz1, rr1, G.r2);
      if (alpha < 0.0 || alpha > 1.0) ++alpha_bad;
      if (nl + l < lk.cap) {
        lk.node[slot + nl + l] = w.n0 + (uint32_t)iw;
        lk.dir[slot + nl + l] = (uint8_t)q;
        lk.alpha[slot + nl + l] = alpha;
      }
    }
    nl += tot;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    lk.cnt[b] = min(nl, lk.cap);
    sol_cnt[b] = min(nsol, seg_cap);
    if (nl > lk.cap) atomicAdd(&status[ST_LINK_OVERFLOW], 1);
  }
  if (alpha_bad) atomicAdd(&status[ST_ALPHA_FAULT], alpha_bad);
}

// Links and solid nodes of the current build (status words read on demand).
__global__ void __launch_bounds__(1024)
    k_link_totals(const int32_t* __restrict__ cnt, const int32_t* __restrict__ scnt, int nsegs,
                  int32_t* __restrict__ status) {
  __shared__ unsigned long long sum[2];
  if (threadIdx.x < 2) sum[threadIdx.x] = 0;
  __syncthreads();
  unsigned long long a = 0, b = 0;
  for (int i = threadIdx.x; i < nsegs; i += 1024) {
    a += (unsigned long long)cnt[i];
    b += (unsigned long long)scnt[i];
  }
  atomicAdd(&sum[0], a);
  atomicAdd(&sum[1], b);
  __syncthreads();
  if (threadIdx.x == 0) {
    status[ST_NLINKS] = (int32_t)min(sum[0], 0x7fffffffull);
    status[ST_NSOLID] = (int32_t)min(sum[1], 0x7fffffffull);
  }
}

// Lists the contact links of one segment: links whose node is solid for
// another sphere in the (now complete) map.
__device__ __forceinline__ void list_contacts(int b, const ContactArgs& a) {
  const int cnt = a.lk.cnt[b];
  const int64_t slot = (int64_t)b * a.lk.cap;
  for (int l = (int)threadIdx.x; l < cnt; l += PB) {
    if (!bit_at(a.mask, a.lk.node[slot + l])) continue;
    const int at = atomicAdd(a.ct_count, 1);
    if (at < a.ct_cap) a.ct_list[at] = ((uint64_t)(uint32_t)div_by((uint32_t)b, a.dseg) << 40) | (uint64_t)(slot + l);
  }
}
__global__ void __launch_bounds__(PB) k_contacts(ContactArgs a) { list_contacts((int)blockIdx.x, a); }

// beads_lubforce (partlib.f90:2211-2292): one workgroup sums the pair forces
// of particle a; each pair is evaluated as the reference does, from the lower
// id's side (so both partners see bitwise opposite pair forces).
// Sphere-wall lubrication (channel beads_lubforce, CHAN/partlib.f90:2316-2355,
// with its wall axis moved to y): the wall at y = 0 pushes up, the wall at
// y = ny down.  Added to the y pair sum.
__device__ __forceinline__ double wall_lub(double yd, const PGeom& G, const LubArgs& L) {
  const double dist0 = L.mingap_w + G.rad;
  double s = 0.0;
  double dist = yd, hgap = dist - G.rad;
  if (dist < dist0) {
    const double d1 = hgap < 0.0 ? -hgap : 0.0, t = (dist0 - dist) / L.mingap_w;
    s += (t * t / L.stf0_w + d1 / L.mingap_w / L.stf1_w) * L.fpc;
  }
  dist = (double)G.ny - yd;
  hgap = dist - G.rad;
  if (dist < dist0) {
    const double d1 = hgap < 0.0 ? -hgap : 0.0, t = (dist0 - dist) / L.mingap_w;
    s -= (t * t / L.stf0_w + d1 / L.mingap_w / L.stf1_w) * L.fpc;
  }
  return s;
}

__device__ void lub_block(int a, const double* __restrict__ ypglb, int np, const PGeom& G,
                          const LubArgs& L) {
  __shared__ double red[3][PB / 64];
  const double dist0 = 2.0 * G.rad + L.mingap;
  const double pre = (dist0 + 1e-6) * (dist0 + 1e-6);
  double fx = 0.0, fy = 0.0, fz = 0.0;
  for (int b = threadIdx.x; b < np; b += PB) {
    if (b == a) continue;
    const int lo = a < b ? a : b, hi = a < b ? b : a;
    const double xc = ypglb[3 * lo], yc = ypglb[3 * lo + 1], zc = ypglb[3 * lo + 2];
    const double xb = near_image(ypglb[3 * hi], xc, G.nx);
    const double yb = G.walls_y ? ypglb[3 * hi + 1] : near_image(ypglb[3 * hi + 1], yc, G.ny);
    const double zb = near_image(ypglb[3 * hi + 2], zc, G.nz);
    const double dx = xc - xb, dy = yc - yb, dz = zc - zb;
    const double d2 = dx * dx + dy * dy + dz * dz;
    if (!(d2 < pre)) continue;
    const double dist = sqrt(d2);
    const double fpd = lub_fpd(dist, G.rad, L.mingap, L.fpc, L.stf0, L.stf1);
    const double sgn = (a == lo) ? 1.0 : -1.0;
    fx += sgn * (fpd * dx);
    fy += sgn * (fpd * dy);
    fz += sgn * (fpd * dz);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double v[3] = {fx, fy, fz};
#pragma unroll
  for (int c = 0; c < 3; ++c) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v[c] += __shfl_down(v[c], o, 64);
    if (lane == 0) red[c][w] = v[c];
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < PB / 64; ++q) s += red[threadIdx.x][q];
    if (G.walls_y && threadIdx.x == 1) s += wall_lub(ypglb[3 * a + 1], G, L);
    L.flubp[3 * a + threadIdx.x] = s;
  }
}

// Pair force of the pair (a, b) on a (the reference evaluates each pair from
// the lower id's side, so both partners get bitwise opposite forces); false
// if the pair is out of range.
__device__ __forceinline__ bool lub_pair(const double* __restrict__ ypglb, int a, int b,
                                         const PGeom& G, const LubArgs& L, double pre, double& fx,
                                         double& fy, double& fz) {
  const int lo = a < b ? a : b, hi = a < b ? b : a;
  const double xc = ypglb[3 * lo], yc = ypglb[3 * lo + 1], zc = ypglb[3 * lo + 2];
  const double xb = near_image(ypglb[3 * hi], xc, G.nx);
  const double yb = G.walls_y ? ypglb[3 * hi + 1] : near_image(ypglb[3 * hi + 1], yc, G.ny);
  const double zb = near_image(ypglb[3 * hi + 2], zc, G.nz);
  const double dx = xc - xb, dy = yc - yb, dz = zc - zb;
  const double d2 = dx * dx + dy * dy + dz * dz;
  if (!(d2 < pre)) return false;
  const double fpd = lub_fpd(sqrt(d2), G.rad, L.mingap, L.fpc, L.stf0, L.stf1);
  const double sgn = (a == lo) ? 1.0 : -1.0;
  fx = sgn * (fpd * dx);
  fy = sgn * (fpd * dy);
  fz = sgn * (fpd * dz);
  return true;
}

// beads_lubforce of particle a from the cells, by one wavefront: every lane
// tests one (cell, slot) of the 27 cells around a at a time (at least three
// cells on every axis: no partner is met twice), the partners in range are
// listed in LDS with their pair forces, ranked by id and summed in increasing
// id (a fixed order); then the walls.  Bound: three dependent loads (cell
// count, slot, position).  One thread per particle, walking its cells serially,
// took 39 us of a step with 900 spheres, this takes 9 us.  A sphere with more
// than kLubList partners falls back to lane 0 finding each next id by a
// further pass over the cells.  Called by every wavefront of a workgroup, with
// lub_lds bytes of dynamic LDS (static LDS would cost the workgroups of boxes
// without cells 2 us).
constexpr int kLubList = 128;
struct LubList {
  int32_t id[kLubList];
  double f[kLubList][3];
  double sorted[kLubList][3];
};
__device__ void lub_cells(int a, const double* __restrict__ ypglb, int np, const PGeom& G,
                          const LubArgs& L, LubList& W) {
  const CellArgs& C = L.cells;
  const double dist0 = 2.0 * G.rad + L.mingap;
  const double pre = (dist0 + 1e-6) * (dist0 + 1e-6);
  const int lane = threadIdx.x & 63;
  int ca = 0, cb = 0, cc = 0;
  const bool on = a < np;
  if (on) cell_coords(ypglb, a, G, C, ca, cb, cc);
  int m = 0;   // partners so far (the same in every lane)
  for (int k0 = 0; k0 < 27 * kCellCap && on; k0 += 64) {
    const int k = (k0 + lane) / kCellCap, e = (k0 + lane) % kCellCap;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    int b = -1;
    bool in = false;
    if (k < 27) {
      const int cell = cell_neighbour(C, G, ca, cb, cc, k);
      if (cell >= 0 && e < min(C.cnt[cell], kCellCap)) {
        b = C.list[cell * kCellCap + e];
        in = b != a && lub_pair(ypglb, a, b, G, L, pre, fx, fy, fz);
      }
    }
    const uint64_t bal = __ballot(in);
    const int at = m + __popcll(bal & ((1ull << lane) - 1ull));
    if (in && at < kLubList) {
      W.id[at] = b;
      W.f[at][0] = fx;
      W.f[at][1] = fy;
      W.f[at][2] = fz;
    }
    m += __popcll(bal);
  }
  const bool full = m > kLubList;
  __syncthreads();
  if (on && !full) {
    for (int i = lane; i < m; i += 64) {
      const int b = W.id[i];
      int rank = 0;
      for (int j = 0; j < m; ++j) rank += W.id[j] < b;
#pragma unroll
      for (int c = 0; c < 3; ++c) W.sorted[rank][c] = W.f[i][c];
    }
  }
  __syncthreads();
  if (!on) return;
  if (!full) {
    if (lane < 3) {
      double s = 0.0;
      for (int i = 0; i < m; ++i) s += W.sorted[i][lane];
      if (lane == 1 && G.walls_y) s += wall_lub(ypglb[3 * a + 1], G, L);
      L.flubp[3 * a + lane] = s;
    }
    return;
  }
  if (lane != 0) return;
  double sx = 0.0, sy = 0.0, sz = 0.0;
  int last = -1;
  for (int guard = 0; guard < 27 * kCellCap; ++guard) {
    int next = 0x7fffffff;
    for (int k = 0; k < 27; ++k) {
      const int cell = cell_neighbour(C, G, ca, cb, cc, k);
      if (cell < 0) continue;
      const int n = min(C.cnt[cell], kCellCap);
      for (int e = 0; e < n; ++e) {
        const int b = C.list[cell * kCellCap + e];
        if (b <= last || b >= next || b == a) continue;
        double fx, fy, fz;
        if (lub_pair(ypglb, a, b, G, L, pre, fx, fy, fz)) next = b;
      }
    }
    if (next == 0x7fffffff) break;
    double fx, fy, fz;
    lub_pair(ypglb, a, next, G, L, pre, fx, fy, fz);
    sx += fx;
    sy += fy;
    sz += fz;
    last = next;
  }
  if (G.walls_y) sy += wall_lub(ypglb[3 * a + 1], G, L);
  L.flubp[3 * a] = sx;
  L.flubp[3 * a + 1] = sy;
  L.flubp[3 * a + 2] = sz;
}

__global__ void __launch_bounds__(PB)
    k_lubforce(const double* __restrict__ ypglb, int np, PGeom G, LubArgs L, int32_t* __restrict__ status) {
  if (L.cells.cnt) {
    extern __shared__ double lds_f64[];
    lub_cells((int)(blockIdx.x * (PB / 64) + (threadIdx.x >> 6)), ypglb, np, G, L,
              ((LubList*)lds_f64)[threadIdx.x >> 6]);
  } else if ((int)blockIdx.x < np)
    lub_block(blockIdx.x, ypglb, np, G, L);
}


// Bounce-back of one link (partlib.f90:1363-1703): the wall point and its
// rigid-body velocity, then the interpolated value f9 sent back into the
// fluid and ff1 = f_q(x) post-collision; ff1 + f9 is the link's momentum
// exchange.  (xx0, yy0, zz0) is the wall point relative to the centre.
// With `gather` false only the geometry is evaluated.  With kSub the values
// read at x itself can be replaced: f_q(x) by sub_q (has_q) and, for
// alpha > 1/2, f_qbar(x) by sub_qbar (has_qbar).
template <typename T, bool kSub = false>
__device__ __forceinline__ void link_bounce(const T* A, const Grid& g, const PGeom& G,
                                            const uint32_t* __restrict__ mask, uint32_t n, int q,
                                            double alpha, double xcp, double ycp, double zcp,
                                            double w1, double w2, double w3, double o1, double o2,
                                            double o3, double ww1, double ww2, bool gather,
                                            double& ff1, double& f9, double& xx0, double& yy0,
                                            double& zz0, bool has_q = false, double sub_q = 0.0,
                                            bool has_qbar = false, double sub_qbar = 0.0) {
  int x, y, z;
  uint32_t row;
  node_coords(n, g, x, y, z, row);
  const int ix = cx(q), iy = cy(q), iz = cz(q);
  const double xp = (double)(x + 1) - 0.5, yp = (double)(y + 1) - 0.5, zp = (double)(z + 1) - 0.5;
  const double xc = near_image(xcp, xp, g.nx);
  const double yc = G.walls_y ? ycp : near_image(ycp, yp, g.ny);
  const double zc = near_image(zcp, zp, g.nz);
  xx0 = xp + (double)ix * alpha - xc;
  yy0 = yp + (double)iy * alpha - yc;
  zz0 = zp + (double)iz * alpha - zc;
  if (!gather) return;
  const double uwx = w1 + o2 * zz0 - o3 * yy0;
  const double uwy = w2 + o3 * xx0 - o1 * zz0;
  const double uwz = w3 + o1 * yy0 - o2 * xx0;
  const double uwpro = uwx * (double)ix + uwy * (double)iy + uwz * (double)iz;
  // x - c and x - 2c (periodic; beyond a wall counts as solid)
  const int y1 = y - iy, y2 = y - 2 * iy;
  const bool out1 = g.walls_y && (y1 < 0 || y1 >= g.ny);
  const bool out2 = g.walls_y && (y2 < 0 || y2 >= g.ny);
  const uint32_t m1 = out1 ? n : (uint32_t)wrap1(x - ix, g.nx) + (uint32_t)g.nx * ((uint32_t)wrap1(y1, g.ny) + (uint32_t)g.ny * (uint32_t)wrap1(z - iz, g.nz));
  const uint32_t m2 = out2 ? n : (uint32_t)wrap1(x - 2 * ix, g.nx) + (uint32_t)g.nx * ((uint32_t)wrap1(y2, g.ny) + (uint32_t)g.ny * (uint32_t)wrap1(z - 2 * iz, g.nz));
  // the values the interpolation may use are gathered together with the
  // solidity tests of x - c and x - 2c (one dependent load stage less; a
  // value at a solid node is read but not used): the alpha <= 1/2 branch
  // takes f_q at x, x - c and x - 2c, the alpha > 1/2 branch f_q at x and
  // f_qbar at x and x - c
  const int qo = opp(q);
  const double wt = q <= 6 ? ww1 : ww2;
  const bool lo = alpha <= 0.5;
  ff1 = post_value(A, g, q, n);
  double v1 = post_value(A, g, lo ? q : qo, lo ? m1 : n);
  const double v2 = post_value(A, g, lo ? q : qo, lo ? m2 : m1);
  if (kSub) {
    if (has_q) ff1 = sub_q;
    if (has_qbar && !lo) v1 = sub_qbar;
  }
  const bool sol1 = out1 || bit_at(mask, m1);
  const bool sol2 = out2 || bit_at(mask, m2);
  if (lo)
    f9 = bounce_back_value(alpha, ff1, sol1 ? 0.0 : v1, (sol1 || sol2) ? 0.0 : v2, sol1, sol1 || sol2,
                           0.0, 0.0, wt, uwpro);
  else
    f9 = bounce_back_value(alpha, ff1, 0.0, 0.0, sol1, true, v1, sol1 ? 0.0 : v2, wt, uwpro);
}

// Contact links in the reference's order (one workgroup).  The reference
// runs its links in (k, j, i, q) loop order and stores each value at once into
// the solid node x + c (partlib.f90:1363-1621).  A link reads f_q and, for
// alpha > 1/2, f_qbar at its own node x; every other value it uses is at a
// fluid node, which no link writes.  So only a contact link (x solid for
// another sphere) can read a stored value: the one its writer stored at x if
// the loop ran that writer earlier and the store reached x in place, not
// through the halo copy of a periodic y or z face, which the reference
// applies after the loop (partlib.f90:1605-1621, 2101-2171).  Non-contact
// links keep their snapshot values; the contact links' values are the fixed
// point of f9(C) = F(the values of C's earlier writers), found by Jacobi
// passes over the contact list until no value changes (writers run earlier,
// so the dependencies are acyclic and pass m settles chains of length m).
// The writer of f_q(x) is the link of x's owner at x + c_q along -c_q, the
// writer of f_qbar(x) its link at x - c_q along c_q.
constexpr int kOrderBatch = 16;
template <typename T>
__device__ void bb_contact_ordered(const BounceArgs& a) {
  __shared__ int changed;
  const T* A = (const T*)a.A;
  const Grid& g = a.g;
  const int64_t total = min((int64_t)*a.ct_count, a.ct_cap);
  if (total > a.ord_cap) {
    if (threadIdx.x == 0) atomicAdd(&a.status[ST_ORDER_CAP], 1);
    return;
  }
  for (int64_t e = threadIdx.x; e < total; e += PB) {
    const uint64_t ent = a.ct_list[e];
    const int p = (int)(ent >> 40);
    const int64_t l = (int64_t)(ent & ((1ull << 40) - 1));
    OrderEntry o;
    o.dep[0] = o.dep[1] = -1;
    o.val[0] = o.val[1] = o.f9 = o.ff1 = 0.0;
    const bool in = p < a.np && l < (int64_t)a.nsegs * a.lk.cap;
    const uint32_t n = in ? a.lk.node[l] : 0u;
    const int q = in ? a.lk.dir[l] : 0;
    if (in && n < g.ncell && q >= 1 && q < NPOP) {
      const double alpha = a.lk.alpha[l];
      double ff1, f9, xx0, yy0, zz0;
      link_bounce<T>(A, g, a.G, a.mask, n, q, alpha, a.ypglb[3 * p], a.ypglb[3 * p + 1],
                     a.ypglb[3 * p + 2], a.wp[3 * p], a.wp[3 * p + 1], a.wp[3 * p + 2], a.omgp[3 * p],
                     a.omgp[3 * p + 1], a.omgp[3 * p + 2], a.ww1, a.ww2, true, ff1, f9, xx0, yy0, zz0);
      a.lk_out[l] = make_double2(f9, ff1);
      int x, y, z;
      uint32_t row;
      node_coords(n, g, x, y, z, row);
      const int own = a.isn[n] - 1;
      for (int s = 0; s < 2 && own >= 0 && own < a.np; ++s) {
        if (s == 1 && !(alpha > 0.5)) break;
        const int sg = s == 0 ? 1 : -1;
        const int xw = x + sg * cx(q), yw = y + sg * cy(q), zw = z + sg * cz(q);
        if (yw < 0 || yw >= g.ny || zw < 0 || zw >= g.nz) continue;   // stored through a halo
        const uint32_t nw = (uint32_t)wrap1(xw, g.nx) + (uint32_t)g.nx * ((uint32_t)yw + (uint32_t)g.ny * (uint32_t)zw);
        if (nw > n) continue;   // the loop runs the writer later
        const int qw = s == 0 ? opp(q) : q;
        // the owner's link (a writer is listed once), kOrderBatch independent
        // loads per round trip
        int64_t lw = -1;
        for (int sg2 = own * a.nseg; sg2 < (own + 1) * a.nseg && lw < 0; ++sg2) {
          const int64_t lo = (int64_t)sg2 * a.lk.cap, hi = lo + a.lk.cnt[sg2];
          for (int64_t k0 = lo; k0 < hi && lw < 0; k0 += kOrderBatch) {
            uint32_t nn[kOrderBatch];
            int dd[kOrderBatch];
#pragma unroll
            for (int j = 0; j < kOrderBatch; ++j) {
              const bool here = k0 + j < hi;
              nn[j] = here ? a.lk.node[k0 + j] : ~0u;
              dd[j] = here ? (int)a.lk.dir[k0 + j] : -1;
            }
#pragma unroll
            for (int j = 0; j < kOrderBatch; ++j)
              if (lw < 0 && nn[j] == nw && dd[j] == qw) lw = k0 + j;
          }
        }
        if (lw < 0) continue;
        if (bit_at(a.mask, nw)) {
          o.dep[s] = lw | kOrderContact;
        } else {
          double wf1, wf9, wx, wy, wz;
          link_bounce<T>(A, g, a.G, a.mask, nw, qw, a.lk.alpha[lw], a.ypglb[3 * own],
                         a.ypglb[3 * own + 1], a.ypglb[3 * own + 2], a.wp[3 * own], a.wp[3 * own + 1],
                         a.wp[3 * own + 2], a.omgp[3 * own], a.omgp[3 * own + 1], a.omgp[3 * own + 2],
                         a.ww1, a.ww2, true, wf1, wf9, wx, wy, wz);
          o.dep[s] = lw;
          o.val[s] = (double)(T)wf9;   // what the writer stores
        }
      }
    }
    a.ord[e] = o;
  }
  for (int64_t pass = 0; pass <= total + 1; ++pass) {
    if (threadIdx.x == 0) changed = 0;
    __syncthreads();   // phase-1 entries and the previous pass's values are visible
    for (int64_t e = threadIdx.x; e < total; e += PB) {
      OrderEntry& o = a.ord[e];
      if (o.dep[0] < 0 && o.dep[1] < 0) continue;
      const uint64_t ent = a.ct_list[e];
      const int p = (int)(ent >> 40);
      const int64_t l = (int64_t)(ent & ((1ull << 40) - 1));
      double v[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int64_t d = o.dep[s];
        v[s] = d < 0 ? 0.0 : ((d & kOrderContact) ? (double)(T)a.lk_out[d & ~kOrderContact].x : o.val[s]);
      }
      double ff1, f9, xx0, yy0, zz0;
      link_bounce<T, true>(A, g, a.G, a.mask, a.lk.node[l], a.lk.dir[l], a.lk.alpha[l], a.ypglb[3 * p],
                           a.ypglb[3 * p + 1], a.ypglb[3 * p + 2], a.wp[3 * p], a.wp[3 * p + 1],
                           a.wp[3 * p + 2], a.omgp[3 * p], a.omgp[3 * p + 1], a.omgp[3 * p + 2],
                           a.ww1, a.ww2, true, ff1, f9, xx0, yy0, zz0, o.dep[0] >= 0, v[0],
                           o.dep[1] >= 0, v[1]);
      o.f9 = f9;
      o.ff1 = ff1;
    }
    __syncthreads();   // every next value is computed before any is stored
    for (int64_t e = threadIdx.x; e < total; e += PB) {
      const OrderEntry& o = a.ord[e];
      if (o.dep[0] < 0 && o.dep[1] < 0) continue;
      const int64_t l = (int64_t)(a.ct_list[e] & ((1ull << 40) - 1));
      const double2 cur = a.lk_out[l];
      if (__double_as_longlong(cur.x) != __double_as_longlong(o.f9) ||
          __double_as_longlong(cur.y) != __double_as_longlong(o.ff1)) {
        a.lk_out[l] = make_double2(o.f9, o.ff1);
        changed = 1;
      }
    }
    __syncthreads();
    const int more = changed;
    __syncthreads();   // every thread has read the flag before it is reset
    if (!more) break;
  }
}

// Streamed value of direction i at node n of a two-buffer field.
template <typename T>
__device__ __forceinline__ double pulled_value(const T* A, const Grid& g, int i, uint32_t n) {
  int x, y, z, pl;
  uint32_t row;
  uint64_t s;
  node_coords(n, g, x, y, z, row);
  if (g.walls_y)
    pull_src_lay<true>(LAY_AB, i, x, y, z, g, pl, s);
  else
    pull_src_lay<false>(LAY_AB, i, x, y, z, g, pl, s);
  return (double)A[(uint64_t)pl * g.pitch + s];
}

// Pre-pass of the bounce-back.  Contact links (node x solid for another
// sphere, spheres almost touching) read post-collision values at a solid
// node, which the bounce-back grid overwrites: their values are taken first,
// from the untouched field, into lk_out (f9, ff1).  Every other link reads
// fluid nodes only and writes only solid ones, so the bounce-back grid can
// scatter as it goes; all links see the one post-collision snapshot.  nct
// blocks stride over the contact list.  With two buffers neither is needed: a
// solid node's post-collision values are the streamed ones the collide copied,
// which the other buffer still holds, and a contact link reads them there
// (one launch less, and the refill grid lists no contact links: 192 x 176 x 208
// FP32 with 900 spheres 293 to 290 us a step, 64^3 FP64 with 8 48.2 to 46.3, 512^3
// with 2500 4154 to 4137, 32 boxes in one grid 938 to 932).
template <typename T>
__device__ __forceinline__ void bb_contact_body(int b_, const BounceArgs& a) {
  if (a.ref_order) {
    if (b_ == 0) bb_contact_ordered<T>(a);
    return;
  }
  const int nblk = a.nct;
  const T* A = (const T*)a.A;
  const int64_t total = min((int64_t)*a.ct_count, a.ct_cap);
  for (int64_t e = (int64_t)b_ * PB + threadIdx.x; e < total; e += (int64_t)nblk * PB) {
    const uint64_t ent = a.ct_list[e];
    const int p = (int)(ent >> 40);
    const int64_t l = (int64_t)(ent & ((1ull << 40) - 1));
    if (p >= a.np || l >= (int64_t)a.nsegs * a.lk.cap) continue;   // never true for a consistent list
    const uint32_t n = a.lk.node[l];
    const int q = a.lk.dir[l];
    if (n >= a.g.ncell || q < 1 || q >= NPOP) continue;
    double ff1 = 0.0, f9 = 0.0, xx0, yy0, zz0;
    link_bounce<T>(A, a.g, a.G, a.mask, n, q, a.lk.alpha[l], a.ypglb[3 * p], a.ypglb[3 * p + 1],
                   a.ypglb[3 * p + 2], a.wp[3 * p], a.wp[3 * p + 1], a.wp[3 * p + 2], a.omgp[3 * p],
                   a.omgp[3 * p + 1], a.omgp[3 * p + 2], a.ww1, a.ww2, true, ff1, f9, xx0, yy0, zz0);
    a.lk_out[l] = make_double2(f9, ff1);
  }
}

// Workgroups are dealt to the 8 XCDs round-robin in launch order.  Launch
// index L of the first nsegs blocks is mapped so that all segments of a
// particle run on one XCD (particle p on XCD p % 8): neighbouring segments
// read overlapping stencils and that XCD's L2 then holds them once.
__device__ __forceinline__ int xcd_segment(int L, int nsegs, int nseg) {
  const int group = 8 * nseg;
  const int full = (nsegs / group) * group;
  if (L >= full) return L;
  const int q = L / group, r = L - q * group;
  return (q * 8 + r % 8) * nseg + r / 8;
}

// beads_collision (partlib.f90:1363-1703), one unit (1/split of a segment's
// links) per block: the bounce-back value of every link, written at once into
// the opposite population of the solid neighbour x + c (partlib.f90:1605-1621),
// and the unit's momentum-exchange force and torque (FP64, fixed reduction
// order) into seg_ft.  In the fused step nlub blocks before the units compute
// beads_lubforce: beside the links they cost nothing, in the pre-pass 5 us (900
// spheres at 192 x 176 x 208: pre-pass 9.2 to 4.6 us, this grid 62 to 63 us, a step
// 299 to 293 us; 64^3 FP64 with 8 49 to 48 us).  Blocks past the units reset one segment
// of the map buffer the coming beads_links rebuilds (built two steps ago), and
// blocks past those the counts of the pair-search cells.
template <typename T>
__device__ __forceinline__ void bounce_back_body(int b_, const BounceArgs& a) {
  __shared__ double red[6][PB / 64];
  T* A = (T*)a.A;
  const Grid& g = a.g;
  if (b_ < a.nlub) {   // beads_lubforce, which no link reads
    if (a.lub.cells.cnt) {
      extern __shared__ double lds_f64[];
      lub_cells(b_ * (PB / 64) + (int)(threadIdx.x >> 6), a.ypglb, a.np, a.G, a.lub,
                ((LubList*)lds_f64)[threadIdx.x >> 6]);
    } else {
      lub_block(b_, a.ypglb, a.np, a.G, a.lub);
    }
    return;
  }
  const int nunits = a.nsegs * a.split;
  const int u = b_ - a.nlub;
  if (u >= nunits) {
    if (u - nunits < a.nclr) {
      clear_segment(u - nunits, a.seg_cap, a.clr_list, a.clr_cnt, a.clr_isn, a.clr_mask);
    } else {   // the counts of the pair-search cells the coming move fills
      const int i = (u - nunits - a.nclr) * PB + (int)threadIdx.x;
      if (i < a.ncell) a.clr_cells[i] = 0;
    }
    return;
  }
  const int b = a.split == 1 ? u : u / a.split, h = u - b * a.split;
  const int p = (int)div_by((uint32_t)b, a.G.dseg);
  const int64_t s0 = (int64_t)b * a.lk.cap, s1 = s0 + a.lk.cnt[b];
  const int64_t per = (max(s1 - s0, (int64_t)0) + a.split - 1) / a.split;
  const int64_t l0 = s0 + h * per;
  const int64_t e = min(s1, l0 + per);
  const double xcp = a.ypglb[3 * p], ycp = a.ypglb[3 * p + 1], zcp = a.ypglb[3 * p + 2];
  const double w1 = a.wp[3 * p], w2 = a.wp[3 * p + 1], w3 = a.wp[3 * p + 2];
  const double o1 = a.omgp[3 * p], o2 = a.omgp[3 * p + 1], o3 = a.omgp[3 * p + 2];
  double acc[6] = {0, 0, 0, 0, 0, 0};
  int contact = 0;
  for (int64_t l = l0 + threadIdx.x; l < e; l += PB) {
    const uint32_t n = a.lk.node[l];
    const int q = a.lk.dir[l];
    const double alpha = a.lk.alpha[l];
    if (n >= g.ncell || q < 1 || q >= NPOP) continue;  // never true for a consistent list
    const bool cont = bit_at(a.mask, n);
    const bool own = cont && a.old;
    double ff1 = 0.0, f9 = 0.0, xx0, yy0, zz0, was_q = 0.0, was_qbar = 0.0;
    if (own) {
      was_q = pulled_value((const T*)a.old, g, q, n);
      was_qbar = pulled_value((const T*)a.old, g, opp(q), n);
    }
    link_bounce<T, true>(A, g, a.G, a.mask, n, q, alpha, xcp, ycp, zcp, w1, w2, w3, o1, o2, o3, a.ww1,
                         a.ww2, own || !cont, ff1, f9, xx0, yy0, zz0, own, was_q, own, was_qbar);
    if (cont) {
      if (!own) {
        const double2 v = a.lk_out[l];
        f9 = v.x;
        ff1 = v.y;
      }
      ++contact;
    }
    // scatter: the post-collision value of opp(q) at the solid node x + c
    int x, y, z;
    uint32_t row;
    node_coords(n, g, x, y, z, row);
    const int yt = y + cy(q);
    if (!(g.walls_y && (yt < 0 || yt >= g.ny))) {
      const int xt = wrap1(x + cx(q), g.nx), zt = wrap1(z + cz(q), g.nz), ytw = wrap1(yt, g.ny);
      int pl;
      uint64_t s;
      if (g.walls_y)
        post_src<true>(g.lay, opp(q), xt, ytw, zt, g, pl, s);
      else
        post_src<false>(g.lay, opp(q), xt, ytw, zt, g, pl, s);
      A[(uint64_t)pl * g.pitch + s] = (T)f9;
    }
    const double dff = ff1 + f9;
    const double dxm = dff * (double)cx(q), dym = dff * (double)cy(q), dzm = dff * (double)cz(q);
    acc[0] += dxm;
    acc[1] += dym;
    acc[2] += dzm;
    acc[3] += dzm * yy0 - dym * zz0;
    acc[4] += dxm * zz0 - dzm * xx0;
    acc[5] += dym * xx0 - dxm * yy0;
  }
  // wavefront tree reduction (fixed order), then the four wave partials
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    double v = acc[c];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if (lane == 0) red[c][w] = v;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < PB / 64; ++q) v += red[threadIdx.x][q];
    a.seg_ft[6ll * u + threadIdx.x] = v;
  }
  if (contact) atomicAdd(&a.status[ST_CONTACT_LINKS], contact);
}

// fHIp / torqp of each particle: its units' sums (nunit per particle), in
// unit order.
__device__ __forceinline__ void seg_sum(const double* __restrict__ seg_ft, int nunit, int p,
                                        double (&f)[3], double (&t)[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double v = 0.0, u = 0.0;
    for (int s = 0; s < nunit; ++s) {
      v += seg_ft[6ll * ((int64_t)p * nunit + s) + c];
      u += seg_ft[6ll * ((int64_t)p * nunit + s) + 3 + c];
    }
    f[c] = v;
    t[c] = u;
  }
}

__global__ void __launch_bounds__(256)
    k_seg_reduce(const double* __restrict__ seg_ft, int nseg, int np, double* __restrict__ fHIp,
                 double* __restrict__ torqp) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  double f[3], t[3];
  seg_sum(seg_ft, nseg, p, f, t);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    fHIp[3 * p + c] = f[c];
    torqp[3 * p + c] = t[c];
  }
}


__device__ __forceinline__ bool wrap_particle(double* yp, double* ypglb, double* ypglbp, int p,
                                              const PGeom& G) {
  const int ns[3] = {G.nx, G.ny, G.nz};
  bool bad = false;
  for (int c = 0; c < 3; ++c) {
    const int q = 3 * p + c;
    const double v = yp[q], N = (double)ns[c];
    if (!(G.walls_y && c == 1)) {
      if (v >= N) yp[q] = yp[q] - N;
      if (v < 0.0) yp[q] = yp[q] + N;
    }
    if (!sane_coord(yp[q], ns[c])) bad = true;
    ypglbp[q] = ypglb[q];
    ypglb[q] = yp[q];
  }
  return bad;
}

// beads_move (partlib.f90:2295-2394): second-order Newton-Euler update, one
// component per lane, the lanes of a particle in a quad (the fourth idles).
// With `wrap` set the periodic wrap of beads_redistribute
// (partlib.f90:2600-2626) follows in the same lane; with seg_ft set the
// hydrodynamic force and torque are first summed from the bounce-back segments
// (and stored), in unit order; with cells.cnt set the particle enters its
// pair-search cell.  Every input is loaded before the first store (the
// argument arrays are distinct, but the compiler cannot know it).  Bound: the
// latency of one round of loads and stores over few lanes; one thread per
// particle with all components took 8.7-10.8 us
// (300 to 900 spheres), this takes 5.0.
constexpr int kMoveBlock = 64;
__device__ __forceinline__ void move_body(int b_, MoveArgs m, int np, int first, int wrap, PGeom G,
                                          int32_t* __restrict__ status,
                                          const double* __restrict__ seg_ft, int nseg, CellArgs cells) {
  const int t = b_ * kMoveBlock + (int)threadIdx.x;
  const int p = t >> 2, c = t & 3;
  const bool on = p < np && c < 3;
  const double dt = 1.0;
  const int q = on ? 3 * p + c : 0;
  bool fast = false, bad = false;
  double yg = 0.0;
  if (on) {
    const double bf = c == 0 ? m.bfx : (c == 1 ? m.bfy : m.bfz);
    const double pf = c == 0 ? m.pfx : (c == 1 ? m.pfy : m.pfz);
    double yp = m.yp[q], wp = m.wp[q], omgp = m.omgp[q], fpp = m.forcepp[q], tpp = m.torqpp[q];
    double dwdt = m.dwdt[q], domgdt = m.domgdt[q];
    const double flub = m.flubp[q];
    double th = first ? 0.0 : m.thetap[q];
    yg = m.ypglb[q];
    double fhi, torq;
    if (seg_ft) {
      fhi = torq = 0.0;
#pragma unroll 8
      for (int s = 0; s < nseg; ++s) {
        fhi += seg_ft[6ll * ((int64_t)p * nseg + s) + c];
        torq += seg_ft[6ll * ((int64_t)p * nseg + s) + 3 + c];
      }
    } else {
      fhi = m.fHIp[q];
      torq = m.torqp[q];
    }
    const double wpp = wp, omgpp = omgp;
    double F = fhi + flub;
    if (c == 1) F = F - m.volp * m.rhog;
    if (bf != 0.0) F = F + m.volp * bf;
    if (pf != 0.0) F = F + m.volp * pf;
    if (first) fpp = F;
    const double dwn = 0.5 * (F + fpp) / m.amp;
    if (first) dwdt = dwn;
    wp = wpp + 0.5 * dt * (dwdt + dwn);
    const double d = 0.5 * dt * (wp + wpp);
    yp = yp + d;
    // the overlapped step assumes a centre moves less than one node per step
    fast = !(fabs(d) < 1.0);
    if (first) tpp = torq;
    const double don = 0.5 * (torq + tpp) / m.aip;
    if (first) domgdt = don;
    omgp = omgpp + 0.5 * dt * (domgdt + don);
    th = th + 0.5 * dt * (omgp + omgpp);
    const double ygp = yg;
    if (wrap) {
      // beads_redistribute: wrap into the periodic box (not across a wall),
      // ypglbp <- ypglb, ypglb <- yp
      const int n = c == 0 ? G.nx : (c == 1 ? G.ny : G.nz);
      const double v = yp, N = (double)n;
      if (!(G.walls_y && c == 1)) {
        if (v >= N) yp = yp - N;
        if (v < 0.0) yp = yp + N;
      }
      bad = !sane_coord(yp, n);
      yg = yp;
    }
    m.wpp[q] = wpp;
    m.omgpp[q] = omgpp;
    m.forcep[q] = F;
    m.wp[q] = wp;
    m.yp[q] = yp;
    m.omgp[q] = omgp;
    m.thetap[q] = th;
    m.dwdt[q] = dwn;
    m.domgdt[q] = don;
    m.forcepp[q] = F;
    m.torqpp[q] = torq;
    if (seg_ft) {
      m.fHIp[q] = fhi;
      m.torqp[q] = torq;
    }
    if (wrap) {
      m.ypglbp[q] = ygp;
      m.ypglb[q] = yg;
    }
  }
  // once per particle: the quad's first lane speaks for it
  const int lane = (int)threadIdx.x & 63;
  const uint64_t quad = 7ull << (lane & ~3);
  const uint64_t fastm = __ballot(fast), badm = __ballot(bad);
  const double y1 = __shfl(yg, lane | 1, 64), y2 = __shfl(yg, lane | 2, 64);
  if (!on || c != 0) return;
  if (fastm & quad) atomicAdd(&status[ST_FAST], 1);
  if (badm & quad) atomicAdd(&status[ST_NONFINITE], 1);
  if (cells.cnt) cell_insert(p, yg, y1, y2, G, cells, status);
}

// beads_redistribute, one-rank content (partlib.f90:2600-2626): periodic wrap,
// ypglbp <- ypglb, ypglb <- yp.
__global__ void __launch_bounds__(256)
    k_wrap(double* __restrict__ yp, double* __restrict__ ypglb, double* __restrict__ ypglbp, int np,
           PGeom G, int32_t* __restrict__ status) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  if (wrap_particle(yp, ypglb, ypglbp, p, G)) atomicAdd(&status[ST_NONFINITE], 1);
}

// ovlpchk (partlib.f90:118-171): one workgroup per particle flags it if any
// later particle is closer than 2r.
__global__ void __launch_bounds__(PB)
    k_overlap(const double* __restrict__ ypglb, int np, PGeom G, int istep, CellArgs cells,
              int32_t* __restrict__ status) {
  const int a = blockIdx.x;
  if (a >= np) return;
  const bool hit = block_overlap(ypglb, a, np, G, cells);
  if (threadIdx.x == 0 && hit) {
    atomicAdd(&status[ST_OVERLAP], 1);
    atomicCAS(&status[ST_OVERLAP_STEP], 0, istep);
  }
}


// beads_filling for one segment of the previous build (partlib.f90:2846-3089).
// First the nodes that were solid for particle p in the previous map (p owns
// them there) and are fluid in the new one, from the previous build's solid
// list, kFillPass listed entries at a time; then one wavefront per such node: lane
// l examines neighbour l+1 (fluid in both maps?  its density; the
// non-equilibrium part if it lies along the back-traced normal), and lane i
// writes population i of the node: equilibrium at the rigid-body velocity
// (new w, omega; old centre) and the neighbours' mean density, plus the
// non-equilibrium part.  Written into the pull sources of the node.  The
// neighbours read are fluid in both maps, so no refilled node is read and the
// order of the refills does not matter.  Bound: two rounds of dependent loads
// (list, new map), then two more for the few nodes uncovered.
constexpr int kFillPass = 4 * PB;
template <typename T, bool WALLS>
__device__ __forceinline__ void refill_nodes(const uint32_t* todo, int total, int id, T* __restrict__ A,
                                             const Grid& g, const FillArgs& fa) {
  __shared__ double fneq[4][NPOP];
  __shared__ double srho[4][NPOP];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // the trip count is the same for every wavefront of the block (barriers inside)
  for (int base = 0; base < total; base += 4) {
    const int e = base + w;
    const bool active = e < total;
    const uint32_t n = active ? todo[e] : 0u;
    int i, j, k;
    uint32_t row;
    node_coords(n, g, i, j, k, row);
    const double xp = (double)(i + 1) - 0.5, yp = (double)(j + 1) - 0.5, zp = (double)(k + 1) - 0.5;
    const double xc = near_image(fa.ypglbp[3 * id] * 1.0, xp, g.nx);
    const double yc = WALLS ? fa.ypglbp[3 * id + 1] : near_image(fa.ypglbp[3 * id + 1] * 1.0, yp, g.ny);
    const double zc = near_image(fa.ypglbp[3 * id + 2] * 1.0, zp, g.nz);
    const double w1 = -0.5 * (fa.wp[3 * id] * 1.0 + fa.wpp[3 * id] * 1.0);
    const double w2 = -0.5 * (fa.wp[3 * id + 1] * 1.0 + fa.wpp[3 * id + 1] * 1.0);
    const double w3 = -0.5 * (fa.wp[3 * id + 2] * 1.0 + fa.wpp[3 * id + 2] * 1.0);
    const double o1 = -0.5 * (fa.omgp[3 * id] * 1.0 + fa.omgpp[3 * id] * 1.0);
    const double o2 = -0.5 * (fa.omgp[3 * id + 1] * 1.0 + fa.omgpp[3 * id + 1] * 1.0);
    const double o3 = -0.5 * (fa.omgp[3 * id + 2] * 1.0 + fa.omgpp[3 * id + 2] * 1.0);
    const int ipmx = refill_direction(xp, yp, zp, xc, yc, zc, w1, w2, w3, o1, o2, o3, fa.rad);
    // lane l < 18: neighbour d = l + 1
    bool fluid = false;
    if (active && lane < NPOP - 1) {
      const int d = lane + 1;
      const int a = i + cx(d), bb = j + cy(d), c = k + cz(d);
      const bool out = WALLS && (bb < 0 || bb >= g.ny);
      if (!out) {
        const uint32_t q = (uint32_t)wrap1(a, g.nx) + (uint32_t)g.nx * ((uint32_t)wrap1(bb, g.ny) + (uint32_t)g.ny * (uint32_t)wrap1(c, g.nz));
        fluid = !bit_at(fa.mask_new, q) && !bit_at(fa.mask_old, q);
        double s = 0.0;
        if (fluid) {
          int qx, qy, qz;
          uint32_t r2;
          node_coords(q, g, qx, qy, qz, r2);
          double f9[NPOP];
          load_pulled<T, double, WALLS>(A, g, qx, qy, qz, q, f9);
          for (int ii = 0; ii < NPOP; ++ii) s = s + f9[ii];
          if (d == ipmx) {
            double rho9 = 0.0, u9 = 0.0, v9 = 0.0, w9 = 0.0;
            for (int ip = 0; ip < NPOP; ++ip) {
              rho9 = rho9 + f9[ip];
              u9 = u9 + (double)cx(ip) * f9[ip];
              v9 = v9 + (double)cy(ip) * f9[ip];
              w9 = w9 + (double)cz(ip) * f9[ip];
            }
            // feq_point's expressions one direction at a time (no array of 19)
            const double usqr = 1.5 * (u9 * u9 + v9 * v9 + w9 * w9);
            fneq[w][0] = f9[0] - fa.ww0 * (rho9 - usqr);
            for (int ip = 1; ip < NPOP; ++ip) {
              const double G = (double)cx(ip) * u9 + (double)cy(ip) * v9 + (double)cz(ip) * w9;
              fneq[w][ip] = f9[ip] - (ip <= 6 ? fa.ww1 : fa.ww2) * (rho9 + 3.0 * G + 4.5 * G * G - usqr);
            }
          }
        }
        srho[w][lane] = s;
      } else {
        srho[w][lane] = 0.0;
      }
    }
    const uint64_t fl = __ballot(fluid);
    const bool have_neq = (fl >> (ipmx - 1)) & 1ull;
    __syncthreads();
    if (active && lane < NPOP) {
      const int nghb = __popcll(fl);
      double rho9 = 0.0;
      for (int l = 0; l < NPOP - 1; ++l)
        if ((fl >> l) & 1ull) rho9 = rho9 + srho[w][l];
      rho9 = (nghb > 0) ? rho9 / (double)nghb : fa.rho0;
      const double xx0 = xp - xc, yy0 = yp - yc, zz0 = zp - zc;
      const double W1 = fa.wp[3 * id], W2 = fa.wp[3 * id + 1], W3 = fa.wp[3 * id + 2];
      const double O1 = fa.omgp[3 * id], O2 = fa.omgp[3 * id + 1], O3 = fa.omgp[3 * id + 2];
      const double u9 = W1 + O2 * zz0 - O3 * yy0;
      const double v9 = W2 + O3 * xx0 - O1 * zz0;
      const double w9 = W3 + O1 * yy0 - O2 * xx0;
      const double usqr = 1.5 * (u9 * u9 + v9 * v9 + w9 * w9);
      const int ip = lane;
      const double G = (double)cx(ip) * u9 + (double)cy(ip) * v9 + (double)cz(ip) * w9;
      const double feq = ip == 0 ? fa.ww0 * (rho9 - usqr)
                                 : (ip <= 6 ? fa.ww1 : fa.ww2) * (rho9 + 3.0 * G + 4.5 * G * G - usqr);
      const double fn = have_neq ? fneq[w][ip] : 0.0;
      store_phase<T, WALLS>(A, g, ip, i, j, k, n, true, fn + feq);
    }
    __syncthreads();
  }
}

template <typename T, bool WALLS>
__device__ __forceinline__ void fill_segment(int b, T* __restrict__ A, const Grid& g, const FillArgs& fa, FastDiv dseg) {
  __shared__ uint32_t todo[kFillPass];
  __shared__ int ntodo;
  const int id = (int)div_by((uint32_t)b, dseg);
  const int cnt = fa.sol_cnt_old[b];
  const uint32_t* lst = fa.sol_old + (size_t)b * fa.seg_cap;
  for (int e0 = 0; e0 < cnt; e0 += kFillPass) {
    __syncthreads();   // the previous pass's list has been refilled
    if (threadIdx.x == 0) ntodo = 0;
    __syncthreads();
    constexpr int kEach = kFillPass / PB;
    uint32_t cand[kEach];
    bool open[kEach];
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
      const int e = e0 + k * PB + (int)threadIdx.x;
      cand[k] = e < cnt ? lst[e] : ~0u;
    }
    // the new map's bit first: nearly every node stays solid
#pragma unroll
    for (int k = 0; k < kEach; ++k) open[k] = cand[k] != ~0u && !bit_at(fa.mask_new, cand[k]);
    // (a node of several spheres is refilled by its owner)
#pragma unroll
    for (int k = 0; k < kEach; ++k)
      if (open[k] && fa.isn_old[cand[k]] == id + 1) todo[atomicAdd(&ntodo, 1)] = cand[k];
    __syncthreads();
    const int total = ntodo;
    if (threadIdx.x == 0 && total) atomicAdd(&fa.status[ST_REFILL], total);
    refill_nodes<T, WALLS>(todo, total, id, A, g, fa);
  }
}

// ---------------------------------------------------------------------------
// Launch forms of the step kernels.  Each kernel body takes its block index;
// k_* launches one box (arguments by value), kb_* one grid over several boxes
// at once: block b belongs to box c with off[c] <= b < off[c+1] and reads that
// box's arguments from the table t (the ensemble engine's per-case tables).
__device__ __forceinline__ int case_of(const int* __restrict__ off, int nc, int b) {
  int lo = 0, hi = nc;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= b) lo = mid; else hi = mid;
  }
  return lo;
}

__global__ void __launch_bounds__(PB) k_links_scan(ScanArgs a) {
  links_scan_body((int)blockIdx.x, a.ypglb, a.np, a.nseg, a.seg_cap, a.G, a.isn, a.mask, a.sol_list, a.sol_cnt, a.lk, a.ct_count, a.ovl, a.istep, a.status, a.cells);
}
__global__ void __launch_bounds__(PB)
    kb_links_scan(const ScanArgs* __restrict__ t, const int* __restrict__ off, int nc) {
  const int c = case_of(off, nc, (int)blockIdx.x);
  const ScanArgs a = t[c];
  links_scan_body((int)blockIdx.x - off[c], a.ypglb, a.np, a.nseg, a.seg_cap, a.G, a.isn, a.mask, a.sol_list, a.sol_cnt, a.lk, a.ct_count, a.ovl, a.istep, a.status, a.cells);
}

template <typename T>
__global__ void __launch_bounds__(PB) k_bb_contact(BounceArgs a) {
  bb_contact_body<T>((int)blockIdx.x, a);
}
template <typename T>
__global__ void __launch_bounds__(PB)
    kb_bb_contact(const BounceArgs* __restrict__ t, const int* __restrict__ off, int nc) {
  const int c = case_of(off, nc, (int)blockIdx.x);
  const BounceArgs a = t[c];
  bb_contact_body<T>((int)blockIdx.x - off[c], a);
}

template <typename T>
__global__ void __launch_bounds__(PB) k_bounce_back(BounceArgs a) {
  const int b = (int)blockIdx.x;
  bounce_back_body<T>(b < a.nlub ? b : a.nlub + xcd_segment(b - a.nlub, a.nsegs * a.split, a.nseg * a.split), a);
}
template <typename T>
__global__ void __launch_bounds__(PB)
    kb_bounce_back(const BounceArgs* __restrict__ t, const int* __restrict__ off, int nc) {
  const int c = case_of(off, nc, (int)blockIdx.x);
  const BounceArgs a = t[c];
  bounce_back_body<T>((int)blockIdx.x - off[c], a);
}

__global__ void __launch_bounds__(kMoveBlock) k_move(MoveKArgs a) {
  move_body((int)blockIdx.x, a.m, a.np, a.first, a.wrap, a.G, a.status, a.seg_ft, a.nseg, a.cells);
}
__global__ void __launch_bounds__(kMoveBlock)
    kb_move(const MoveKArgs* __restrict__ t, const int* __restrict__ off, int nc) {
  const int c = case_of(off, nc, (int)blockIdx.x);
  const MoveKArgs a = t[c];
  move_body((int)blockIdx.x - off[c], a.m, a.np, a.first, a.wrap, a.G, a.status, a.seg_ft, a.nseg, a.cells);
}

// The refill of the previous build's segments, the contact links of the new
// build's (where the bounce-back wants their list) and, in blocks past those, the next step's forcing table.  4 waves
// per SIMD (at most 128 VGPRs; 5 or more spill: 24 to 31 us with 900 spheres of
// radius 4).  The search in a grid of its own that lists the nodes for a refill
// grid was no faster but with 15,000 segments (12 + 12 us against 24 with 900
// spheres, 3.6 + 9.2 against 9.8 with 8, 58 + 26 against 105 with 2500).
template <typename T, bool WALLS>
__device__ __forceinline__ bool fill_block(int b, const FillKArgs& a) {
  if (b < a.nfill) {
    fill_segment<T, WALLS>(b, (T*)a.A, a.g, a.fa, a.ct.dseg);
  } else if (b < a.nfill + a.nct) {
    list_contacts(b - a.nfill, a.ct);
  } else {
    return false;
  }
  return true;
}
template <typename T, bool WALLS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
    k_fill(FillKArgs a, TableJob tj) {
  if (!fill_block<T, WALLS>((int)blockIdx.x, a))
    force_table_block(tj.M, tj.phy, tj.phz, tj.ny, tj.nz, tj.G, blockIdx.x - (uint32_t)(a.nfill + a.nct));
}
static_assert(sizeof(FillKArgs) + sizeof(TableJob) <= 4096, "refill kernel arguments over 4 KB");
template <typename T, bool WALLS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
    kb_fill(const FillKArgs* __restrict__ t, const int* __restrict__ off, int nc) {
  const int c = case_of(off, nc, (int)blockIdx.x);
  const FillKArgs a = t[c];
  fill_block<T, WALLS>((int)blockIdx.x - off[c], a);
}

// trilinear velocity at the particle centres (initpartvel,
// partlib.f90:177-263 with trilinear :320-831); node (i) sits at i - 0.5.
__global__ void k_initpartvel(const double* __restrict__ ypglb, int np, Grid g,
                              const double* __restrict__ ux, const double* __restrict__ uy,
                              const double* __restrict__ uz, double* __restrict__ wp) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const double xc = ypglb[3 * p], yc = ypglb[3 * p + 1], zc = ypglb[3 * p + 2];
  if (!(sane_coord(xc, g.nx) && sane_coord(yc, g.ny) && sane_coord(zc, g.nz))) return;
  const int i = (int)(xc + 0.5), j = (int)(yc + 0.5), k = (int)(zc + 0.5);
  const double tx = xc + 0.5 - (double)i, ty = yc + 0.5 - (double)j, tz = zc + 0.5 - (double)k;
  const double tx0 = 1.0 - tx, ty0 = 1.0 - ty, tz0 = 1.0 - tz;
  const int i0 = wrap_any(i - 1, g.nx), i1 = wrap_any(i, g.nx);
  const int j0 = wrap_any(j - 1, g.ny), j1 = wrap_any(j, g.ny);
  const int k0 = wrap_any(k - 1, g.nz), k1 = wrap_any(k, g.nz);
  const double* us[3] = {ux, uy, uz};
  for (int c = 0; c < 3; ++c) {
    const double* u = us[c];
    auto at = [&](int a, int b, int d) {
      return u[(uint64_t)a + (uint64_t)g.nx * ((uint64_t)b + (uint64_t)g.ny * (uint64_t)d)];
    };
    wp[3 * p + c] = tx0 * ty0 * tz0 * at(i0, j0, k0) + tx * ty0 * tz0 * at(i1, j0, k0) +
                    tx * ty * tz0 * at(i1, j1, k0) + tx0 * ty * tz0 * at(i0, j1, k0) +
                    tx0 * ty0 * tz * at(i0, j0, k1) + tx * ty0 * tz * at(i1, j0, k1) +
                    tx * ty * tz * at(i1, j1, k1) + tx0 * ty * tz * at(i0, j1, k1);
  }
}

__global__ void k_maps_dense(Grid g, const int32_t* __restrict__ isn, const uint32_t* __restrict__ mask,
                             int32_t* __restrict__ ib, int32_t* __restrict__ is) {
  const uint32_t n = blockIdx.x * 256u + threadIdx.x;
  if (n >= g.ncell) return;
  const bool solid = mask != nullptr && bit_at(mask, n);
  ib[n] = solid ? 1 : -1;
  is[n] = (isn != nullptr && isn[n] > 0) ? isn[n] : -1;
}

__global__ void k_links_dense(Grid g, FastDiv dseg, LinkSlots lk, int32_t* __restrict__ ilink,
                              int32_t* __restrict__ mlink, double* __restrict__ alink) {
  const int b = blockIdx.x;
  const int p = (int)div_by((uint32_t)b, dseg);
  const int64_t a = (int64_t)b * lk.cap, e = a + lk.cnt[b];
  for (int64_t l = a + threadIdx.x; l < e; l += blockDim.x) {
    if (lk.node[l] >= g.ncell || lk.dir[l] < 1 || lk.dir[l] >= NPOP) continue;
    const uint64_t d = (uint64_t)(lk.dir[l] - 1) + 18ull * lk.node[l];
    ilink[d] = 1;
    mlink[d] = p + 1;
    alink[d] = lk.alpha[l];
  }
}

// ---------------------------------------------------------------------------
static PGeom pgeom(const Ctx& c) {
  PGeom G;
  G.nx = c.g.nx;
  G.ny = c.g.ny;
  G.nz = c.g.nz;
  G.walls_y = c.g.walls_y;
  G.rad = c.p.rad;
  G.radp2 = c.p.rad * 1.0 + 2.0;
  G.r2 = (c.p.rad * 1.0) * (c.p.rad * 1.0);
  G.rlink2 = (c.p.rad + 1.5) * (c.p.rad + 1.5);
  G.slab = c.pt.slab;
  G.dseg = fast_div((uint32_t)c.pt.nseg);
  return G;
}

// the widest candidate range axis_range() can return, in nodes
static int box_candidates(double rad) {
  const double radp2 = rad + 2.0;
  return (int)ceil(2.0 * radp2 + 1.0) + 4;
}

int segments_per_particle(double rad, int slab) {
  return (box_candidates(rad) + slab - 1) / slab;
}

int segment_capacity(double rad, int slab) {
  const int maxcnt = box_candidates(rad);
  return slab * maxcnt * maxcnt;
}

// Links a segment can hold: a lattice line along a direction enters a sphere
// once, so a direction within the planes has at most as many links as lines
// meet the disc of each plane (2r + 1 along an axis, 2 sqrt(2) r + 1 along a
// diagonal), and a direction across the planes as many as lines meet the sphere
// or the part of its surface in the segment, whichever is fewer (a band of
// height h has the projected area pi r h, a cap 2 pi r h; sqrt(2) lines per unit
// area along a diagonal), each with a margin of a node.  Over radii from 2 to 27
// and random centres it is 1.7 (8 planes) to 5.7 times (1 plane, radius 2) the
// largest count met.
int segment_links(double rad, int slab) {
  const double r = rad + 1.0, disc = M_PI * r * r, h = slab + 1.0;
  const double in_plane = slab * (4.0 * (2.0 * r) + 4.0 * (2.0 * sqrt(2.0) * rad + 2.0));
  const double across = 2.0 * std::min(disc, 2.0 * M_PI * r * h) + 8.0 * sqrt(2.0) * std::min(disc, M_PI * r * h);
  return (int)ceil(in_plane + across) + 64;
}

// Planes per segment.  The fewer planes, the shorter a workgroup's chain of
// passes; the more, the fewer workgroups.  1 or 2 where the spheres are few:
// their workgroups fit the 256 CUs at once, five or six each (step at 64^3 FP32
// with 8 spheres of radius 4: 46.0 us with 1, 47.7 with 2, 54.1 with 4; 96^3 with
// 20 of radius 6 69.6, 72.0, 82.9; 100^3 with 4 of radius 13 81, 91, 118; 128^3
// with 60 of radius 6 (1260 segments of 1 plane) 107.3, 109.7, 117.7; with 100
// of radius 4 (1700) 106.6, 105.0, 107.0; 150 x 141 x 162 with 140 of radius 6
// (1540 of 2 planes) 178.9, 171.8, 177.4; 160^3 with 250 of radius 4 (2250)
// 189.1, 180.2, 175.1).  Many small boxes in one grid fill the GPU anyhow (32
// boxes 1003 us a step with 1, 953 with 2, 939 with 4): their contexts ask for
// 4.  8 where the spheres are many and small, whose segments of 4 leave most of
// a pass idle: radius up to 4 from 500 segments of 8 (160^3 with 400 of radius 3
// 175 us against 193 with 4; 192^3 with 400 of radius 4 259 against 264; 128^3
// with 150 of radius 3, 300 segments, 105 against 109), up to 6 from 2048 (352^3
// with 1500 of radius 6 1667 against 1684, 256^3 with 700 637 against 640; 224^3
// with 350, 1050 segments, 435 against 437 with 4 but 428 with 2).  Larger
// spheres have enough in 4 (radius 7 at 400^3 2420 and 2418; radius 8 at 288^3
// 899 against 1002, at 448^3 with 8400 segments of 8 3298 against 3683).  8 also
// needs at most PB / 8 candidate rows per plane and keeps the scan's shell list
// within 10 KB of LDS, so only for box_candidates <= 25 (rad <= 8).  `want` (a
// context's own choice) and MFC_SEG_PLANES = 1, 2, 4 or 8 force one (8 only
// where it fits).
constexpr int64_t kSlab1MaxSegments = 1280, kSlab2MaxSegments = 1600;
int segment_planes(double rad, int npart, int want) {
  const int rows = box_candidates(rad);
  const char* e = getenv("MFC_SEG_PLANES");
  if (e && (e[0] == '1' || e[0] == '2' || e[0] == '4' || e[0] == '8')) want = e[0] - '0';
  if (want == 8 && rows > 25) want = 4;
  if (want) return want;
  auto segs = [&](int planes) { return (int64_t)npart * segments_per_particle(rad, planes); };
  if (segs(8) >= (rows <= 17 ? 500 : 2048) && rows <= 21) return 8;   // radius up to 4, 6
  if (segs(1) <= kSlab1MaxSegments) return 1;
  return segs(2) <= kSlab2MaxSegments ? 2 : 4;
}

// Reset map buffer `buf` to empty (no-op if it is empty already).
hipError_t launch_map_clear(Ctx& c, int buf) {
  Particles& P = c.pt;
  if (P.map_np[buf] > 0)
    hipLaunchKernelGGL(k_map_clear, dim3(P.map_np[buf] * P.nseg), dim3(PB), 0, c.stream, P.seg_cap,
                       P.sol_list[buf], P.sol_cnt[buf], P.isn[buf], P.mask[buf]);
  P.map_np[buf] = 0;
  return hipGetLastError();
}

// Arguments of beads_filling for the maps `old` (previous) and `neu` (new);
// false if there is nothing to refill.
static bool make_fill_args(Ctx& c, int old, int neu, FillArgs& fa) {
  Particles& P = c.pt;
  if (P.map_np[old] == 0 || old == neu) return false;
  fa.ypglbp = P.ypglbp; fa.wp = P.wp; fa.wpp = P.wpp; fa.omgp = P.omgp; fa.omgpp = P.omgpp;
  fa.sol_old = P.sol_list[old];
  fa.sol_cnt_old = P.sol_cnt[old];
  fa.seg_cap = P.seg_cap;
  fa.isn_old = P.isn[old];
  fa.mask_new = P.mask[neu];
  fa.mask_old = P.mask[old];
  fa.rad = c.p.rad; fa.rho0 = c.p.rho0; fa.ww0 = c.p.ww0; fa.ww1 = c.p.ww1; fa.ww2 = c.p.ww2;
  fa.status = c.d_status;
  return true;
}

static int cell_count(const Particles& P) { return P.cell_n[0] * P.cell_n[1] * P.cell_n[2]; }

// The cell grid if it is on (else cnt = nullptr: all pairs).  The lists must
// be current (ensure_cells) before a kernel reads them.
static CellArgs cell_args(const Ctx& c) {
  const Particles& P = c.pt;
  CellArgs C;
  C.cnt = c.ens || !P.cell_cnt ? nullptr : P.cell_cnt + P.cell_half * cell_count(P);   // ensemble members search all pairs
  C.list = P.cell_list;
  C.ncx = P.cell_n[0];
  C.ncy = P.cell_n[1];
  C.ncz = P.cell_n[2];
  return C;
}

static size_t lub_lds(const Ctx& c) { return cell_args(c).cnt ? sizeof(LubList) * (PB / 64) : 0; }

// Blocks of the lubrication part of a grid: one per particle (all pairs) or
// one wavefront per particle (cells).
static int lub_blocks(const Ctx& c) {
  return cell_args(c).cnt ? (c.pt.np + PB / 64 - 1) / (PB / 64) : c.pt.np;
}

hipError_t ensure_cells(Ctx& c) {
  Particles& P = c.pt;
  if (!cell_args(c).cnt || P.cells_ok) return hipSuccess;
  const int ncell = cell_count(P);
  hipLaunchKernelGGL(k_cell_zero, dim3((ncell + 255) / 256), dim3(256), 0, c.stream, cell_args(c).cnt, ncell);
  hipLaunchKernelGGL(k_cell_build, dim3((P.np + 255) / 256), dim3(256), 0, c.stream, P.ypglb, P.np,
                     pgeom(c), cell_args(c), c.d_status);
  P.cells_ok = true;
  return hipGetLastError();
}

static LubArgs lub_args(Ctx& c) {
  LubArgs L;
  L.mingap = c.p.mingap;
  L.fpc = c.p.volp * c.p.rho0 * 9.8 / c.p.gscale;
  L.stf0 = c.p.stf0;
  L.stf1 = c.p.stf1;
  L.mingap_w = c.p.mingap_w;
  L.stf0_w = c.p.stf0_w;
  L.stf1_w = c.p.stf1_w;
  L.flubp = c.pt.flubp;
  L.cells = cell_args(c);
  return L;
}

static LinkSlots link_slots(const Particles& P) {
  return LinkSlots{P.lk_node, P.lk_dir, P.lk_alpha, P.lk_cnt, P.lk_seg};
}

static ContactArgs contact_args(const Particles& P) {
  ContactArgs a;
  a.lk = link_slots(P);
  a.mask = P.mask[P.map_cur];
  a.ct_list = P.ct_list;
  a.ct_count = P.ct_count;
  a.ct_cap = P.lk_cap;
  a.dseg = fast_div((uint32_t)P.nseg);
  return a;
}

// ---- argument builders: one box's arguments of each step kernel ------------
// (used by the single-box launchers below and by the ensemble engine)

ScanArgs scan_args(Ctx& c, int target, int ovl, int istep) {
  c.pt.ct_ok = false;   // the scan empties the contact list
  Particles& P = c.pt;
  ScanArgs a;
  a.ypglb = P.ypglb; a.np = P.np; a.nseg = P.nseg; a.seg_cap = P.seg_cap; a.G = pgeom(c);
  a.isn = P.isn[target]; a.mask = P.mask[target]; a.sol_list = P.sol_list[target];
  a.sol_cnt = P.sol_cnt[target]; a.lk = link_slots(P); a.ct_count = P.ct_count; a.ovl = ovl; a.istep = istep; a.status = c.d_status;
  a.cells = cell_args(c);
  return a;
}

size_t scan_lds(const Ctx& c) {
  return (size_t)shell_bytes(c.pt.seg_cap) + packed_bytes(c.pt.seg_cap) +
         sizeof(SegRow) * (size_t)(c.pt.slab * box_candidates(c.p.rad));
}

// fused (mfc_step): lubrication blocks, and the map buffer the coming links
// rebuild (map_cur ^ 1, built two steps ago) cleared in the same grid and
// marked empty
BounceArgs bounce_args(Ctx& c, bool fused, int nct, int* bb_blocks, int* pre_blocks) {
  Particles& P = c.pt;
  BounceArgs a;
  a.A = c.pop[c.cur]; a.g = c.g; a.G = pgeom(c); a.mask = P.mask[P.map_cur]; a.nseg = P.nseg;
  a.lk = link_slots(P); a.lk_out = P.lk_out;
  a.ct_list = P.ct_list; a.ct_count = P.ct_count; a.ct_cap = P.lk_cap;
  a.ypglb = P.ypglb; a.wp = P.wp; a.omgp = P.omgp;
  a.ww1 = c.p.ww1; a.ww2 = c.p.ww2; a.seg_ft = P.seg_ft; a.status = c.d_status;
  a.nsegs = P.np * P.nseg; a.np = P.np; a.lub = lub_args(c);
  a.split = P.bb_split;
  a.ref_order = P.bb_order == MFC_BB_REFERENCE;
  a.old = !a.ref_order && c.g.lay == LAY_AB && c.old_version == c.f_version ? c.pop[c.cur ^ 1] : nullptr;
  a.nct = a.old ? 0 : (a.ref_order ? 1 : nct);
  a.ord = P.ord; a.ord_cap = P.ord_cap; a.isn = P.isn[P.map_cur];
  a.nlub = fused ? lub_blocks(c) : 0;
  const int t = P.map_cur ^ 1;
  const int nclr = (fused && P.map_np[t] > 0) ? P.map_np[t] * P.nseg : 0;
  a.seg_cap = P.seg_cap;
  a.clr_list = P.sol_list[t]; a.clr_cnt = P.sol_cnt[t]; a.clr_isn = P.isn[t]; a.clr_mask = P.mask[t];
  if (nclr) P.map_np[t] = 0;
  a.nclr = nclr;
  a.ncell = fused && a.lub.cells.cnt ? cell_count(P) : 0;
  a.clr_cells = a.ncell ? P.cell_cnt + (P.cell_half ^ 1) * a.ncell : nullptr;
  P.cells_zeroed = a.ncell > 0;
  *bb_blocks = a.nlub + a.nsegs * a.split + nclr + (a.ncell + PB - 1) / PB;
  *pre_blocks = a.nct;
  return a;
}

MoveKArgs move_args(Ctx& c, int first, int wrap, bool from_seg, int* blocks) {
  Particles& P = c.pt;
  MoveKArgs a;
  MoveArgs& m = a.m;
  m.yp = P.yp; m.ypglb = P.ypglb; m.ypglbp = P.ypglbp;
  m.wp = P.wp; m.wpp = P.wpp; m.omgp = P.omgp; m.omgpp = P.omgpp;
  m.fHIp = P.fHIp; m.flubp = P.flubp; m.torqp = P.torqp; m.forcep = P.forcep;
  m.forcepp = P.forcepp; m.torqpp = P.torqpp; m.dwdt = P.dwdt; m.domgdt = P.domgdt;
  m.thetap = P.thetap;
  m.volp = c.p.volp; m.rhog = c.p.rhog; m.amp = c.p.amp; m.aip = c.p.aip;
  m.bfx = c.p.body_force[0]; m.bfy = c.p.body_force[1]; m.bfz = c.p.body_force[2];
  m.pfx = c.p.particle_force[0]; m.pfy = c.p.particle_force[1]; m.pfz = c.p.particle_force[2];
  a.np = P.np; a.first = first; a.wrap = wrap; a.G = pgeom(c); a.status = c.d_status;
  a.seg_ft = from_seg ? P.seg_ft : nullptr; a.nseg = P.nseg * P.bb_split;
  // the cells the fused bounce-back grid has cleared: filled at the new centres
  const bool fill = wrap && from_seg && P.cells_zeroed;
  if (fill) P.cell_half ^= 1;
  a.cells = fill ? cell_args(c) : CellArgs{};
  P.cells_zeroed = false;
  if (wrap) P.cells_ok = fill;   // the wrapped positions are the new ypglb
  *blocks = (4 * P.np + kMoveBlock - 1) / kMoveBlock;
  return a;
}

// refill: beads_filling between the maps map_old and map_cur (no blocks if there
// is nothing to refill); contacts: list the contact links of the current build
FillKArgs fill_args(Ctx& c, bool refill, bool contacts, int* blocks) {
  Particles& P = c.pt;
  FillKArgs a;
  a.fa = FillArgs{};
  a.nfill = refill && make_fill_args(c, P.map_old, P.map_cur, a.fa) ? P.map_np[P.map_old] * P.nseg : 0;
  a.nct = contacts ? P.np * P.nseg : 0;
  if (a.nct) P.ct_ok = true;
  a.ct = contact_args(P);
  a.A = c.pop[c.cur];
  a.g = c.g;
  *blocks = a.nfill + a.nct;
  return a;
}

// ---- far and near tiles of the overlapped step ----------------------------------
// A tile is kTileX consecutive x nodes of one row (tile t = tx + tpr * row).
// The particle phase of step n (bounce-back, lubrication, move, links,
// refill, with the clearing of the map built two steps back) reads and
// writes no node farther than r + 3 sqrt 2 + 2 from the centres it starts
// from, as long as no sphere moves a node or more in one step (k_move counts
// such steps); the next collide touches only nodes within sqrt 2 of its
// own.  Tiles with no node within reach = r + 3 sqrt 2 + 2 + sqrt 2 of a
// centre (periodic images; none across the y walls) are "far": their collide
// for step n + 1 can run while the particle phase of step n does.

// One workgroup per sphere marks the tiles of every row whose node centres
// come within `reach` of the centre.
__global__ void __launch_bounds__(PB)
    k_tile_mark(const double* __restrict__ ypglb, int np, PGeom G, double reach, int tpr,
                uint8_t* __restrict__ mark) {
  const int p = blockIdx.x;
  if (p >= np) return;
  const double cx = ypglb[3 * p], cy = ypglb[3 * p + 1], cz = ypglb[3 * p + 2];
  const int j0 = (int)floor(cy - reach - 0.5), j1 = (int)ceil(cy + reach - 0.5);
  const int k0 = (int)floor(cz - reach - 0.5), k1 = (int)ceil(cz + reach - 0.5);
  const int nj = j1 - j0 + 1, nk = k1 - k0 + 1;
  const double r2 = reach * reach;
  for (int t = threadIdx.x; t < nj * nk; t += PB) {
    const int jj = j0 + t % nj, kk = k0 + t / nj;
    const double dy = (double)jj + 0.5 - cy, dz = (double)kk + 0.5 - cz;
    const double d2 = dy * dy + dz * dz;
    if (d2 > r2) continue;
    if (G.walls_y && (jj < 0 || jj >= G.ny)) continue;
    const int j = ((jj % G.ny) + G.ny) % G.ny, k = ((kk % G.nz) + G.nz) % G.nz;
    uint8_t* row = mark + (size_t)tpr * ((size_t)j + (size_t)G.ny * k);
    const double e = sqrt(r2 - d2);
    const int i0 = (int)ceil(cx - e - 0.5), i1 = (int)floor(cx + e - 0.5);
    if (i1 - i0 + 1 >= G.nx) {
      for (int b = 0; b < tpr; ++b) row[b] = 1;
      continue;
    }
    for (int i = i0; i <= i1;) {
      const int iw = ((i % G.nx) + G.nx) % G.nx;
      const int b = iw / kTileX;
      row[b] = 1;
      // first node past this tile (the last tile of a row may be short)
      const int end = kTileX * (b + 1) < G.nx ? kTileX * (b + 1) : G.nx;
      i += end - iw;
    }
  }
}

// Near tiles per chunk of kTileChunk tiles.
__global__ void __launch_bounds__(PB)
    k_tile_count(const uint8_t* __restrict__ mark, uint64_t ntiles, int32_t* __restrict__ cnt) {
  __shared__ int red[PB / 64];
  const uint64_t base = (uint64_t)blockIdx.x * kTileChunk;
  int c = 0;
  for (int i = threadIdx.x; i < kTileChunk; i += PB) {
    const uint64_t t = base + (uint64_t)i;
    if (t < ntiles && mark[t]) ++c;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    int s = 0;
    for (int w = 0; w < PB / 64; ++w) s += red[w];
    cnt[blockIdx.x] = s;
  }
}

// Exclusive offsets of the near and far tiles of each chunk; totals in
// tot[0] (near) and tot[1] (far).  One workgroup.
__global__ void __launch_bounds__(1024)
    k_tile_offsets(const int32_t* __restrict__ cnt, int nchunk, uint64_t ntiles,
                   uint32_t* __restrict__ off_near, uint32_t* __restrict__ off_far,
                   uint32_t* __restrict__ tot) {
  __shared__ uint32_t part[1024];
  const int per = (nchunk + 1023) / 1024;
  const int c0 = threadIdx.x * per, c1 = min(nchunk, c0 + per);
  uint32_t s = 0;
  for (int c = c0; c < c1; ++c) s += (uint32_t)cnt[c];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const uint32_t v = threadIdx.x >= (unsigned)o ? part[threadIdx.x - o] : 0u;
    __syncthreads();
    part[threadIdx.x] += v;
    __syncthreads();
  }
  uint32_t near = threadIdx.x ? part[threadIdx.x - 1] : 0u;
  for (int c = c0; c < c1; ++c) {
    const uint64_t first = (uint64_t)c * kTileChunk;
    off_near[c] = near;
    off_far[c] = (uint32_t)(first - near);
    near += (uint32_t)cnt[c];
  }
  if (threadIdx.x == 1023) {
    tot[0] = part[1023];
    tot[1] = (uint32_t)(ntiles - part[1023]);
  }
}

// Each chunk writes its tiles, in order, into the near and far lists, and
// clears its marks for the next step.
__global__ void __launch_bounds__(PB)
    k_tile_emit(uint8_t* __restrict__ mark, uint64_t ntiles, const uint32_t* __restrict__ off_near,
                const uint32_t* __restrict__ off_far, uint32_t* __restrict__ near_list,
                uint32_t* __restrict__ far_list) {
  __shared__ uint32_t wsum[PB / 64];
  const uint64_t base = (uint64_t)blockIdx.x * kTileChunk;
  uint32_t near = off_near[blockIdx.x], far = off_far[blockIdx.x];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int i0 = 0; i0 < kTileChunk; i0 += PB) {
    const uint64_t t = base + (uint64_t)(i0 + threadIdx.x);
    const bool in = t < ntiles;
    const bool nr = in && mark[t] != 0;
    const uint64_t bal = __ballot(nr);
    const uint64_t bin = __ballot(in);
    const uint32_t below = (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
    const uint32_t below_in = (uint32_t)__popcll(bin & ((1ull << lane) - 1ull));
    if (lane == 0) wsum[w] = (uint32_t)__popcll(bal);
    __syncthreads();
    uint32_t pre = 0, tot = 0;
    for (int q = 0; q < PB / 64; ++q) {
      if (q < w) pre += wsum[q];
      tot += wsum[q];
    }
    // tiles of earlier waves in this pass: 64 each (all in range until the end)
    const uint32_t pre_in = (uint32_t)(64 * w);
    if (in) {
      if (nr) {
        near_list[near + pre + below] = (uint32_t)t;
        mark[t] = 0;
      } else {
        far_list[far + (pre_in - pre) + (below_in - below)] = (uint32_t)t;
      }
    }
    near += tot;
    far += (uint32_t)PB - tot;
    __syncthreads();
  }
}

hipError_t launch_tiles(Ctx& c, TileLists& T) {
  Particles& P = c.pt;
  const PGeom G = pgeom(c);
  hipLaunchKernelGGL(k_tile_mark, dim3(P.np), dim3(PB), 0, c.stream, P.ypglb, P.np, G, T.reach, T.tpr,
                     T.mark);
  const int nchunk = (int)((T.ntiles + kTileChunk - 1) / kTileChunk);
  hipLaunchKernelGGL(k_tile_count, dim3(nchunk), dim3(PB), 0, c.stream, T.mark, T.ntiles, T.cnt);
  hipLaunchKernelGGL(k_tile_offsets, dim3(1), dim3(1024), 0, c.stream, T.cnt, nchunk, T.ntiles, T.off_near,
                     T.off_far, T.tot);
  hipLaunchKernelGGL(k_tile_emit, dim3(nchunk), dim3(PB), 0, c.stream, T.mark, T.ntiles, T.off_near,
                     T.off_far, T.near_list, T.far_list);
  return hipGetLastError();
}

// ---- single-box launchers -------------------------------------------------------
hipError_t launch_links(Ctx& c, int target, int overlap_check, int istep) {
  Particles& P = c.pt;
  const int nsegs = P.np * P.nseg;
  hipError_t e = launch_map_clear(c, target);
  if (e != hipSuccess) return e;
  if (P.np <= 0) return hipGetLastError();
  if (overlap_check) {
    e = ensure_cells(c);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_links_scan, dim3(nsegs), dim3(PB), scan_lds(c), c.stream,
                     scan_args(c, target, overlap_check, istep));
  P.map_np[target] = P.np;
  return hipGetLastError();
}

bool wants_contacts(const Ctx& c) { return c.g.lay != LAY_AB || c.pt.bb_order == MFC_BB_REFERENCE; }

hipError_t ensure_contacts(Ctx& c) {
  Particles& P = c.pt;
  if (P.ct_ok || P.np <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_contacts, dim3(P.np * P.nseg), dim3(PB), 0, c.stream, contact_args(P));
  P.ct_ok = true;
  return hipGetLastError();
}

hipError_t launch_link_totals(Ctx& c) {
  Particles& P = c.pt;
  if (P.np <= 0 || P.map_np[P.map_cur] == 0) return hipSuccess;
  hipLaunchKernelGGL(k_link_totals, dim3(1), dim3(1024), 0, c.stream, P.lk_cnt, P.sol_cnt[P.map_cur],
                     P.np * P.nseg, c.d_status);
  return hipGetLastError();
}

constexpr int kContactBlocks = 16;   // grid of the contact pre-pass (contacts are rare)

hipError_t launch_bounce_back(Ctx& c, bool fused) {
  Particles& P = c.pt;
  if (fused) {
    const hipError_t e = ensure_cells(c);
    if (e != hipSuccess) return e;
  }
  int nb = 0, npre = 0;
  const BounceArgs ba = bounce_args(c, fused, kContactBlocks, &nb, &npre);
  const size_t lds = fused ? lub_lds(c) : 0;
  if (npre) {
    const hipError_t e = ensure_contacts(c);
    if (e != hipSuccess) return e;
  }
  if (c.prec == MFC_PREC_FP64) {
    if (npre) hipLaunchKernelGGL(k_bb_contact<double>, dim3(npre), dim3(PB), 0, c.stream, ba);
    hipLaunchKernelGGL(k_bounce_back<double>, dim3(nb), dim3(PB), lds, c.stream, ba);
  } else {
    if (npre) hipLaunchKernelGGL(k_bb_contact<float>, dim3(npre), dim3(PB), 0, c.stream, ba);
    hipLaunchKernelGGL(k_bounce_back<float>, dim3(nb), dim3(PB), lds, c.stream, ba);
  }
  if (!fused)
    hipLaunchKernelGGL(k_seg_reduce, dim3((P.np + 255) / 256), dim3(256), 0, c.stream, P.seg_ft,
                       P.nseg * P.bb_split, P.np, P.fHIp, P.torqp);
  return hipGetLastError();
}

hipError_t launch_lubforce(Ctx& c) {
  Particles& P = c.pt;
  const hipError_t e = ensure_cells(c);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_lubforce, dim3(lub_blocks(c)), dim3(PB), lub_lds(c), c.stream, P.ypglb, P.np, pgeom(c),
                     lub_args(c), c.d_status);
  return hipGetLastError();
}

hipError_t launch_move(Ctx& c, int first, int wrap, bool from_seg) {
  int nb = 0;
  const MoveKArgs a = move_args(c, first, wrap, from_seg, &nb);
  hipLaunchKernelGGL(k_move, dim3(nb), dim3(kMoveBlock), 0, c.stream, a);
  return hipGetLastError();
}

hipError_t launch_redistribute(Ctx& c, int istep) {
  Particles& P = c.pt;
  hipLaunchKernelGGL(k_wrap, dim3((P.np + 255) / 256), dim3(256), 0, c.stream, P.yp, P.ypglb,
                     P.ypglbp, P.np, pgeom(c), c.d_status);
  P.cells_ok = false;
  const hipError_t e = ensure_cells(c);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_overlap, dim3(P.np), dim3(PB), 0, c.stream, P.ypglb, P.np, pgeom(c), istep,
                     cell_args(c), c.d_status);
  return hipGetLastError();
}

hipError_t launch_filling(Ctx& c, bool contacts, const TableJob* job) {
  int nb = 0;
  const FillKArgs a = fill_args(c, true, contacts, &nb);
  TableJob tj;
  if (job)
    tj = *job;
  else
    tj.nblk = 0;
  const dim3 grid(nb + tj.nblk), blk(256);
  if (grid.x == 0) return hipSuccess;
  if (c.prec == MFC_PREC_FP64) {
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_fill<double, true>), grid, blk, 0, c.stream, a, tj);
    else
      hipLaunchKernelGGL((k_fill<double, false>), grid, blk, 0, c.stream, a, tj);
  } else {
    if (c.g.walls_y)
      hipLaunchKernelGGL((k_fill<float, true>), grid, blk, 0, c.stream, a, tj);
    else
      hipLaunchKernelGGL((k_fill<float, false>), grid, blk, 0, c.stream, a, tj);
  }
  return hipGetLastError();
}

hipError_t launch_initpartvel(Ctx& c) {
  Particles& P = c.pt;
  hipLaunchKernelGGL(k_initpartvel, dim3((P.np + 255) / 256), dim3(256), 0, c.stream, P.ypglb, P.np,
                     c.g, c.ux, c.uy, c.uz, P.wp);
  return hipGetLastError();
}

hipError_t launch_maps_to_host_layout(Ctx& c, int which, int32_t* ib, int32_t* is) {
  Particles& P = c.pt;
  const int b = which == 0 ? P.map_cur : P.map_old;
  const bool have = P.isn[b] != nullptr && P.map_np[b] > 0;
  hipLaunchKernelGGL(k_maps_dense, dim3((unsigned)((c.g.ncell + 255) / 256)), dim3(256), 0, c.stream,
                     c.g, have ? P.isn[b] : nullptr, have ? P.mask[b] : nullptr, ib, is);
  return hipGetLastError();
}

hipError_t launch_links_dense(Ctx& c, int32_t* ilink, int32_t* mlink, double* alink) {
  Particles& P = c.pt;
  hipLaunchKernelGGL(k_links_dense, dim3(P.np * P.nseg), dim3(256), 0, c.stream, c.g,
                     fast_div((uint32_t)P.nseg), link_slots(P), ilink, mlink, alink);
  return hipGetLastError();
}

}  // namespace mfc

namespace mfc {

size_t stage_arg_bytes(Stage st) {
  switch (st) {
    case SG_BOUNCE: return sizeof(BounceArgs);
    case SG_CONTACT: return sizeof(BounceArgs);
    case SG_MOVE: return sizeof(MoveKArgs);
    case SG_SCAN: return sizeof(ScanArgs);
    case SG_FILL: return sizeof(FillKArgs);
  }
  return 0;
}

hipError_t launch_batched(Stage st, int prec, int walls, const void* t, const int* off, int nc,
                          int blocks, size_t lds, hipStream_t s) {
  if (nc <= 0 || blocks <= 0) return hipSuccess;
  const bool f64 = prec == MFC_PREC_FP64;
  switch (st) {
    case SG_BOUNCE:
      if (f64)
        hipLaunchKernelGGL(kb_bounce_back<double>, dim3(blocks), dim3(PB), 0, s, (const BounceArgs*)t, off, nc);
      else
        hipLaunchKernelGGL(kb_bounce_back<float>, dim3(blocks), dim3(PB), 0, s, (const BounceArgs*)t, off, nc);
      break;
    case SG_CONTACT:
      if (f64)
        hipLaunchKernelGGL(kb_bb_contact<double>, dim3(blocks), dim3(PB), 0, s, (const BounceArgs*)t, off, nc);
      else
        hipLaunchKernelGGL(kb_bb_contact<float>, dim3(blocks), dim3(PB), 0, s, (const BounceArgs*)t, off, nc);
      break;
    case SG_MOVE:
      hipLaunchKernelGGL(kb_move, dim3(blocks), dim3(kMoveBlock), 0, s, (const MoveKArgs*)t, off, nc);
      break;
    case SG_SCAN:
      hipLaunchKernelGGL(kb_links_scan, dim3(blocks), dim3(PB), lds, s, (const ScanArgs*)t, off, nc);
      break;
    case SG_FILL:
      if (f64) {
        if (walls)
          hipLaunchKernelGGL((kb_fill<double, true>), dim3(blocks), dim3(256), 0, s, (const FillKArgs*)t, off, nc);
        else
          hipLaunchKernelGGL((kb_fill<double, false>), dim3(blocks), dim3(256), 0, s, (const FillKArgs*)t, off, nc);
      } else {
        if (walls)
          hipLaunchKernelGGL((kb_fill<float, true>), dim3(blocks), dim3(256), 0, s, (const FillKArgs*)t, off, nc);
        else
          hipLaunchKernelGGL((kb_fill<float, false>), dim3(blocks), dim3(256), 0, s, (const FillKArgs*)t, off, nc);
      }
      break;
  }
  return hipGetLastError();
}

}  // namespace mfc
