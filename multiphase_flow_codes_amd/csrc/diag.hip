// diag.hip -- FP64 diagnostics on the device: global sums of the macroscopic
// fields and the kinetic-energy spectrum of the reference's statistc
// (BOX/saveload.f90:1111-1300), with its own FFT.
//
// Sums use a fixed two-level tree (per-block partials, then one block), so
// they are bitwise repeatable.  The spectrum transforms the velocity
// components through half spectra in an FP64 scratch field, lines in
// registers and LDS (radix 8 for power-of-two lengths, the factors of n
// otherwise); each axis is normalised by 1/n as mpifft3DRC does
// (BOX/mpifft.f90:52-108), forward sign e^{-i}.
#include <algorithm>
#include <mutex>

#include "field_sums.h"
#include "internal.h"

namespace mfc {

// Scratch of the allocation-free field sums (mfc_diag_sums_noalloc): the
// kSumBlocksMax x 6 first-level partials, then the 6 results it leaves before
// they are copied out.  Every GPU the library runs on holds its own copy
// until the process ends.  The host resolves its address once per device
// (sums_scratch) and passes that pointer to the kernels; the array's name in
// host code is only a stand-in.  Each call overwrites every word it reads,
// so nothing is cleared between calls; calls that overlap on one GPU share
// the array and race.
constexpr size_t kSumsScratchDoubles = 6 * (size_t)kSumBlocksMax + 8;
static __device__ __align__(256) double scratch[kSumsScratchDoubles];

// Per-block partial sums of rho, ux, uy, uz and u.u, and the block's max |u|^2.
__global__ void __launch_bounds__(kSumThreads)
    k_field_sums(const double* __restrict__ rho, const double* __restrict__ ux,
                 const double* __restrict__ uy, const double* __restrict__ uz, uint64_t n,
                 double* __restrict__ part) {
  FieldSums f;
  for (uint64_t i = (uint64_t)blockIdx.x * kSumThreads + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kSumThreads)
    f.add(rho[i], ux[i], uy[i], uz[i]);
  f.store(part);
}

// The final sums: wavefront k adds component k's partials, each lane every
// 64th of them, then across the lanes (a fixed order).  One thread walking
// its 1024 partials, one load after another, took 245 us of each call; this
// takes 5 us.
__global__ void __launch_bounds__(6 * 64)
    k_sums_final(const double* __restrict__ part, int nblk, double* __restrict__ out) {
  const int k = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double v = 0.0;   // the max is over squares
#pragma unroll 8
  for (int b = lane; b < nblk; b += 64) {
    const double t = part[6 * b + k];
    v = (k == 5) ? fmax(v, t) : v + t;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double t = __shfl_down(v, o, 64);
    v = (k == 5) ? fmax(v, t) : v + t;
  }
  if (lane == 0) out[k] = v;
}

// ---- energy spectrum ---------------------------------------------------------
// The transform of a real component needs only the modes 0 <= kx < hx = nx/2
// that statistc counts, so the scratch field is half spectra: Z[(kx + hx * (y
// + ny * z)) + comp * hx * ny * nz].  Three passes per component:
//   AXIS_X  real rows, two packed into one complex line (row 2p + i row 2p+1,
//           separated by the symmetry of real transforms), half spectra out;
//   AXIS_Y  in place along y;
//   AXIS_Z  along z, the shells summed from the registers that hold the
//           result: the transformed field is never written.
// A workgroup takes a tile of `tx` lines: along y and z they are neighbours in
// kx, so each of the tile's rows is one contiguous run of tx complex numbers.
// Bound: memory traffic, 8 B read + 8 B written (x), 8 + 8 (y) and 8 (z) per
// node and component.  At 256^3 a component's passes take 56, 45 and 46 us
// (4.8, 6.0 and 2.9 TB/s; the last is bound by its shell sums) and the three
// components 0.47 ms; with one line per workgroup (16-B accesses a plane
// apart), full complex passes of radix 2 and a binning pass that re-read the
// field they took 4.3 ms.
enum FftAxis { AXIS_X, AXIS_Y, AXIS_Z };

struct FftArgs {
  const double* re[3];   // AXIS_X: the components' real fields
  double2* Z;            // half spectra of the launch's components
  const double2* tw;     // exp(-2 pi i j / n)
  int nx, ny, nz, hx;
  int n;                 // length of the transformed axis
  int tx, ltx;           // lines per tile, and log2
  int tiles;             // tiles of all components of the launch
  int per;               // tiles per component
  int across;            // AXIS_Y, AXIS_Z: tiles along kx
  int nek;               // AXIS_Z: shells, and their partial sums per workgroup
  double* part;
  int nf;                // general lengths: factors of n
  int f[12];
};

__device__ __forceinline__ double2 operator+(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 operator-(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 mul_mi(double2 a) { return make_double2(a.y, -a.x); }   // a * (-i)

__device__ __forceinline__ void dft2(double2& a, double2& b) {
  const double2 t = a - b;
  a = a + b;
  b = t;
}
__device__ __forceinline__ void dft4(double2& a, double2& b, double2& c, double2& d) {
  dft2(a, c);
  dft2(b, d);
  d = mul_mi(d);
  dft2(a, b);
  dft2(c, d);
  const double2 t = b;   // natural order: 0 a, 1 c, 2 b, 3 d
  b = c;
  c = t;
}
__device__ __forceinline__ void dft8(double2 (&v)[8]) {
  const double h = 0.70710678118654752440;
  dft4(v[0], v[2], v[4], v[6]);
  dft4(v[1], v[3], v[5], v[7]);
  const double2 w1 = make_double2(h * (v[3].x + v[3].y), h * (v[3].y - v[3].x));
  const double2 w2 = mul_mi(v[5]);
  const double2 w3 = make_double2(h * (v[7].y - v[7].x), -h * (v[7].x + v[7].y));
  const double2 a0 = v[0], a1 = v[2], a2 = v[4], a3 = v[6], b0 = v[1];
  v[0] = a0 + b0;
  v[4] = a0 - b0;
  v[1] = a1 + w1;
  v[5] = a1 - w1;
  v[2] = a2 + w2;
  v[6] = a2 - w2;
  v[3] = a3 + w3;
  v[7] = a3 - w3;
}

__device__ __forceinline__ int signed_k(int i, int n) { return i < n / 2 + 1 ? i : i - n; }

// Shell of a mode, int(|k| + 0.5), by integer comparison: ik holds the modes
// with ik^2 - ik < k2 <= ik^2 + ik.
__device__ __forceinline__ int shell_of(int k2) {
  int ik = (int)(sqrtf((float)k2) + 0.5f);
  if (k2 <= ik * ik - ik) --ik;
  else if (k2 > ik * ik + ik) ++ik;
  return ik;
}

// Adds |v|^2 of mode (kx, ky, kz) to its shell (statistc,
// BOX/saveload.f90:1273-1300): weight 1/2 on the kx = 0 plane, k = 0 left out.
__device__ __forceinline__ void add_mode(double* bins, int nek, int kx, int kyz2, int kz, double2 v, double sc2) {
  const int ik = shell_of(kyz2 + kz * kz);
  if (ik < 1 || ik > nek) return;
  double e = (v.x * v.x + v.y * v.y) * sc2;
  if (kx == 0) e *= 0.5;
  atomicAdd(&bins[ik - 1], e);
}

// Where a tile's lines lie.
struct Tile {
  uint64_t base;    // first element of line 0 (AXIS_X: row of line 0)
  uint64_t es;      // elements from one entry of a line to the next
  int lines;        // lines of this tile (the last one may be short)
  int comp, kx, y;
};
template <int AXIS>
__device__ __forceinline__ Tile tile_of(const FftArgs& a, int t) {
  Tile r;
  r.comp = t / a.per;
  const int q = t - r.comp * a.per;
  r.kx = r.y = 0;
  const uint64_t field = (uint64_t)r.comp * (uint64_t)a.hx * (uint64_t)a.ny * (uint64_t)a.nz;
  if (AXIS == AXIS_X) {
    const int64_t rows = (int64_t)a.ny * a.nz;
    r.base = 2ull * (uint64_t)q * (uint64_t)a.tx;   // rows
    const int64_t left = (rows - (int64_t)r.base + 1) / 2;
    r.lines = (int)(left < a.tx ? left : a.tx);
    r.es = 1;
  } else {
    const int o = q / a.across;   // z plane (AXIS_Y) or y row (AXIS_Z)
    r.kx = (q - o * a.across) * a.tx;
    r.lines = min(a.tx, a.hx - r.kx);
    r.y = o;
    if (AXIS == AXIS_Y) {
      r.base = field + (uint64_t)r.kx + (uint64_t)a.hx * (uint64_t)a.ny * (uint64_t)o;
      r.es = (uint64_t)a.hx;
    } else {
      r.base = field + (uint64_t)r.kx + (uint64_t)a.hx * (uint64_t)o;
      r.es = (uint64_t)a.hx * (uint64_t)a.ny;
    }
  }
  return r;
}

// Entry j of packed line t (AXIS_X): the rows 2t and 2t + 1 of the tile.
__device__ __forceinline__ double2 packed_row(const FftArgs& a, const Tile& T, int t, int j) {
  const double* re = a.re[T.comp];
  const uint64_t row = T.base + 2ull * (uint64_t)t;
  const uint64_t at = row * (uint64_t)a.nx + (uint64_t)j;
  return make_double2(re[at], row + 1 < (uint64_t)a.ny * (uint64_t)a.nz ? re[at + (uint64_t)a.nx] : 0.0);
}

// Half spectra of the two rows packed in line t, mode k, from V(k) and V(n-k).
__device__ __forceinline__ void unpack_rows(const FftArgs& a, const Tile& T, int t, int k, double2 p, double2 m,
                                            double sc) {
  const uint64_t row = T.base + 2ull * (uint64_t)t;
  double2* z = a.Z + (uint64_t)T.comp * (uint64_t)a.hx * (uint64_t)a.ny * (uint64_t)a.nz + row * (uint64_t)a.hx + (uint64_t)k;
  const double h = 0.5 * sc;
  z[0] = make_double2(h * (p.x + m.x), h * (p.y - m.y));
  if (row + 1 < (uint64_t)a.ny * (uint64_t)a.nz) z[a.hx] = make_double2(h * (p.y + m.y), h * (m.x - p.x));
}

// Power-of-two lengths (8..2048): every thread holds eight entries of one
// line, j = b + k n/8, in registers; passes of radix 8 (the last one 4 or 2
// where log2 n leaves a remainder) exchange them through LDS.  The first pass
// loads from memory and the last one stores to memory, so a 256-point line
// goes through LDS twice.  Entry j sits at LDS slot j + j/8, so that neither
// the strided stores of a pass nor its unit-stride loads meet in one bank.
template <int AXIS>
__global__ void __launch_bounds__(512)
    k_fft_pow2(FftArgs a) {
  extern __shared__ double2 lbuf[];
  const int n = a.n, n8 = n >> 3;
  // x lines are contiguous along j, the others across the lines
  const int t = AXIS == AXIS_X ? (int)threadIdx.x / n8 : (int)threadIdx.x & (a.tx - 1);
  const int b = AXIS == AXIS_X ? (int)threadIdx.x - t * n8 : (int)threadIdx.x >> a.ltx;
  const int span = n + n8;
  auto slot = [&](int j) {
    const int p = j + (j >> 3);
    return AXIS == AXIS_X ? t * span + p : (p << a.ltx) + t;
  };
  double* bins = (double*)(lbuf + (size_t)span * a.tx);
  if (AXIS == AXIS_Z) {
    for (int i = threadIdx.x; i < a.nek; i += blockDim.x) bins[i] = 0.0;
    __syncthreads();
  }
  const double sc = 1.0 / (double)n;
  for (int tile = blockIdx.x; tile < a.tiles; tile += gridDim.x) {
    const Tile T = tile_of<AXIS>(a, tile);
    const bool on = t < T.lines;
    double2 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      v[k] = make_double2(0.0, 0.0);
      if (on) v[k] = AXIS == AXIS_X ? packed_row(a, T, t, b + k * n8) : a.Z[T.base + (uint64_t)t + (uint64_t)(b + k * n8) * T.es];
    }
    int pos[8];
    for (int ns = 1; ns < n;) {
      if (ns > 1) {
#pragma unroll
        for (int k = 0; k < 8; ++k) lbuf[slot(pos[k])] = v[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = lbuf[slot(b + k * n8)];
        __syncthreads();
      }
      const int left = n / ns;   // uniform: one radix for every thread
      if (left >= 8) {
        const int k0 = b & (ns - 1), st = n8 / ns;
        if (ns > 1) {
#pragma unroll
          for (int m = 1; m < 8; ++m) v[m] = cmul(v[m], a.tw[k0 * m * st]);
        }
        dft8(v);
#pragma unroll
        for (int m = 0; m < 8; ++m) pos[m] = (b - k0) * 8 + k0 + m * ns;
        ns *= 8;
      } else if (left == 4) {
        // butterflies b (even entries) and b + n/8 (odd entries); ns = n/4
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k0 = b + h * n8;
#pragma unroll
          for (int m = 1; m < 4; ++m) v[2 * m + h] = cmul(v[2 * m + h], a.tw[k0 * m]);
        }
        dft4(v[0], v[2], v[4], v[6]);
        dft4(v[1], v[3], v[5], v[7]);
#pragma unroll
        for (int k = 0; k < 8; ++k) pos[k] = b + (k & 1) * n8 + (k >> 1) * ns;
        ns *= 4;
      } else {
        // four butterflies b + h n/8, each of entries h and h + 4; ns = n/2
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          v[h + 4] = cmul(v[h + 4], a.tw[b + h * n8]);
          dft2(v[h], v[h + 4]);
          pos[h] = b + h * n8;
          pos[h + 4] = b + h * n8 + ns;
        }
        ns *= 2;
      }
    }
    if (AXIS == AXIS_X) {
      // mode k needs V(k) and V(n - k): once more through LDS
#pragma unroll
      for (int k = 0; k < 8; ++k) lbuf[slot(pos[k])] = v[k];
      __syncthreads();
      for (int k = b; k < a.hx && on; k += n8)
        unpack_rows(a, T, t, k, lbuf[slot(k)], lbuf[slot(k ? n - k : 0)], sc);
      __syncthreads();
    } else if (AXIS == AXIS_Y) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (on) a.Z[T.base + (uint64_t)t + (uint64_t)pos[k] * T.es] = make_double2(v[k].x * sc, v[k].y * sc);
    } else {
      const int kx = T.kx + t, ky = signed_k(T.y, a.ny);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (on) add_mode(bins, a.nek, kx, kx * kx + ky * ky, signed_k(pos[k], n), v[k], sc * sc);
    }
  }
  if (AXIS == AXIS_Z) {
    __syncthreads();
    for (int i = threadIdx.x; i < a.nek; i += blockDim.x) a.part[(size_t)blockIdx.x * a.nek + i] = bins[i];
  }
}

// One radix-R pass over the tile's lines, src to dst (both LDS).
template <int R, typename Slot>
__device__ __forceinline__ void small_pass(const FftArgs& a, const double2* src, double2* dst, int ns, Slot&& slot) {
  const int n = a.n, nr = n / R, st = nr / ns;
  for (int w = threadIdx.x; w < nr * a.tx; w += blockDim.x) {
    const int t = w & (a.tx - 1), i = w >> a.ltx;
    const int k0 = i % ns;
    double2 v[R];
#pragma unroll
    for (int m = 0; m < R; ++m) {
      v[m] = src[slot(i + m * nr, t)];
      if (m) v[m] = cmul(v[m], a.tw[k0 * m * st]);
    }
    if (R == 2) {
      dft2(v[0], v[1]);
    } else if (R == 4) {
      dft4(v[0], v[1 % R], v[2 % R], v[3 % R]);
    } else if (R == 3) {
      const double s3 = 0.86602540378443864676;
      const double2 s = v[1] + v[2 % R], d = v[1] - v[2 % R];
      const double2 c = make_double2(v[0].x - 0.5 * s.x, v[0].y - 0.5 * s.y);
      v[0] = v[0] + s;
      v[1] = make_double2(c.x + s3 * d.y, c.y - s3 * d.x);
      v[2 % R] = make_double2(c.x - s3 * d.y, c.y + s3 * d.x);
    } else {
      const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
      const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
      const double2 p1 = v[1] + v[4 % R], d1 = v[1] - v[4 % R], p2 = v[2 % R] + v[3 % R], d2 = v[2 % R] - v[3 % R];
      const double2 e1 = make_double2(v[0].x + c1 * p1.x + c2 * p2.x, v[0].y + c1 * p1.y + c2 * p2.y);
      const double2 e2 = make_double2(v[0].x + c2 * p1.x + c1 * p2.x, v[0].y + c2 * p1.y + c1 * p2.y);
      const double2 o1 = make_double2(s1 * d1.x + s2 * d2.x, s1 * d1.y + s2 * d2.y);
      const double2 o2 = make_double2(s2 * d1.x - s1 * d2.x, s2 * d1.y - s1 * d2.y);
      v[0] = v[0] + p1 + p2;
      v[1] = make_double2(e1.x + o1.y, e1.y - o1.x);
      v[4 % R] = make_double2(e1.x - o1.y, e1.y + o1.x);
      v[2 % R] = make_double2(e2.x + o2.y, e2.y - o2.x);
      v[3 % R] = make_double2(e2.x - o2.y, e2.y + o2.x);
    }
#pragma unroll
    for (int m = 0; m < R; ++m) dst[slot((i - k0) * R + k0 + m * ns, t)] = v[m];
  }
}

// LDS entries from one index of k_fft_any's lines to the next: x lines are
// loaded along j, so the rows of several are padded.
template <int AXIS>
__host__ __device__ constexpr int any_row(int tx) { return AXIS == AXIS_X && tx > 1 ? tx + 1 : tx; }

// Any length: passes over the factors of n (4, 2, 3, 5, then the remaining
// primes by their sums, outputs m and r - m together) between two LDS buffers.
// Bound: those sums.  A spectrum of 150 x 141 x 162 nodes (141 = 3 x 47) takes
// 0.25 ms, 0.35 with every output summed by itself, 4.6 with direct sums over
// whole lines; 139 x 151 x 149 0.50 ms (1.33), 98 x 121 x 169 0.18 (0.26).
template <int AXIS>
__global__ void __launch_bounds__(256)
    k_fft_any(FftArgs a) {
  extern __shared__ double2 lbuf[];
  const int n = a.n;
  const int row = any_row<AXIS>(a.tx);
  auto slot = [&](int j, int t) { return j * row + t; };
  double* bins = (double*)(lbuf + 2 * (size_t)n * row);
  if (AXIS == AXIS_Z) {
    for (int i = threadIdx.x; i < a.nek; i += blockDim.x) bins[i] = 0.0;
  }
  const double sc = 1.0 / (double)n;
  for (int tile = blockIdx.x; tile < a.tiles; tile += gridDim.x) {
    const Tile T = tile_of<AXIS>(a, tile);
    double2 *src = lbuf, *dst = lbuf + (size_t)n * row;
    for (int w = threadIdx.x; w < n * a.tx; w += blockDim.x) {
      const int t = AXIS == AXIS_X ? w / n : w & (a.tx - 1), j = AXIS == AXIS_X ? w - t * n : w >> a.ltx;
      double2 v = make_double2(0.0, 0.0);
      if (t < T.lines) v = AXIS == AXIS_X ? packed_row(a, T, t, j) : a.Z[T.base + (uint64_t)t + (uint64_t)j * T.es];
      src[slot(j, t)] = v;
    }
    __syncthreads();
    for (int p = 0, ns = 1; p < a.nf; ++p) {
      const int r = a.f[p];
      if (r == 4) {
        small_pass<4>(a, src, dst, ns, slot);
      } else if (r == 2) {
        small_pass<2>(a, src, dst, ns, slot);
      } else if (r == 3) {
        small_pass<3>(a, src, dst, ns, slot);
      } else if (r == 5) {
        small_pass<5>(a, src, dst, ns, slot);
      } else {
        // x_q: entry i + q n/r of butterfly i, turned by exp(-2 pi i q k0 / (ns r)).
        // Outputs m and r - m share the sums over q <= (r - 1) / 2 of cos(2 pi q m / r)
        // (x_q + x_{r-q}) and sin(2 pi q m / r) (x_q - x_{r-q}): first those sums and
        // differences in place, then a pair of outputs per thread.
        const int nr = n / r, st = nr / ns, h = r / 2;
        for (int w = threadIdx.x; w < nr * h * a.tx; w += blockDim.x) {
          const int t = w & (a.tx - 1), iq = w >> a.ltx;
          const int q = iq / nr, i = iq - q * nr, k0 = i % ns;
          double2 &lo = src[slot(i + (q + 1) * nr, t)], &hi = src[slot(i + (r - 1 - q) * nr, t)];
          const double2 u = cmul(lo, a.tw[(q + 1) * k0 * st]), v = cmul(hi, a.tw[(r - 1 - q) * k0 * st]);
          lo = u + v;
          hi = u - v;
        }
        __syncthreads();
        for (int w = threadIdx.x; w < nr * (h + 1) * a.tx; w += blockDim.x) {
          const int t = w & (a.tx - 1), im = w >> a.ltx;
          const int m = im / nr, i = im - m * nr, k0 = i % ns, step = m * nr;
          double2 c = src[slot(i, t)], d = make_double2(0.0, 0.0);
          int e = 0;
          for (int q = 1; q <= h; ++q) {
            e += step;
            if (e >= n) e -= n;
            const double2 s = src[slot(i + q * nr, t)], f = src[slot(i + (r - q) * nr, t)], cs = a.tw[e];
            c.x += cs.x * s.x;
            c.y += cs.x * s.y;
            d.x -= cs.y * f.y;   // cs.y = -sin
            d.y += cs.y * f.x;
          }
          const int o = (i - k0) * r + k0;
          dst[slot(o + m * ns, t)] = c + d;
          if (m) dst[slot(o + (r - m) * ns, t)] = c - d;
        }
      }
      __syncthreads();
      double2* x = src;
      src = dst;
      dst = x;
      ns *= r;
    }
    if (AXIS == AXIS_X) {
      for (int w = threadIdx.x; w < a.hx * a.tx; w += blockDim.x) {
        const int t = w / a.hx, k = w - t * a.hx;
        if (t < T.lines) unpack_rows(a, T, t, k, src[slot(k, t)], src[slot(k ? n - k : 0, t)], sc);
      }
    } else {
      for (int w = threadIdx.x; w < n * a.tx; w += blockDim.x) {
        const int t = w & (a.tx - 1), j = w >> a.ltx;
        if (t >= T.lines) continue;
        const double2 v = src[slot(j, t)];
        if (AXIS == AXIS_Y) {
          a.Z[T.base + (uint64_t)t + (uint64_t)j * T.es] = make_double2(v.x * sc, v.y * sc);
        } else {
          const int kx = T.kx + t, ky = signed_k(T.y, a.ny);
          add_mode(bins, a.nek, kx, kx * kx + ky * ky, signed_k(j, n), v, sc * sc);
        }
      }
    }
    __syncthreads();
  }
  if (AXIS == AXIS_Z)
    for (int i = threadIdx.x; i < a.nek; i += blockDim.x) a.part[(size_t)blockIdx.x * a.nek + i] = bins[i];
}

// Shells from the workgroups' partial sums, 64 shells per workgroup: wavefront
// w adds every 16th workgroup's, then the wavefronts are added in order.  `add`:
// to what acc holds (a later component).  One thread per shell walking all
// partials took 235 us a component; this takes 7-11 us.
__global__ void __launch_bounds__(1024)
    k_spectrum_final(const double* __restrict__ part, int nblk, int nek, double* __restrict__ acc, int add) {
  __shared__ double red[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + lane;
  double v = 0.0;
  if (i < nek) {
#pragma unroll 8
    for (int b = w; b < nblk; b += 16) v += part[(size_t)b * nek + i];
  }
  red[w][lane] = v;
  __syncthreads();
  if (w == 0 && i < nek) {
    double s = add ? acc[i] : 0.0;
#pragma unroll
    for (int q = 0; q < 16; ++q) s += red[q][lane];
    acc[i] = s;
  }
}

// ---------------------------------------------------------------------------
hipError_t launch_field_sums(Ctx& c, bool fill, double* part, double* out) {
  const int nb = sum_blocks(c.g.ncell);
  if (fill) {
    const hipError_t e = launch_macro_sums(c, c.phase == PHASE_POST_STREAM, part);
    if (e != hipSuccess) return e;
  } else {
    hipLaunchKernelGGL(k_field_sums, dim3(nb), dim3(kSumThreads), 0, c.stream, c.rho, c.ux, c.uy, c.uz,
                       (uint64_t)c.g.ncell, part);
  }
  hipLaunchKernelGGL(k_sums_final, dim3(1), dim3(6 * 64), 0, c.stream, part, nb, out);
  return hipGetLastError();
}

static int ilog2_exact(int n) {
  int l = 0;
  while ((1 << l) < n) ++l;
  return (1 << l) == n ? l : -1;
}

int diag_blocks() { return kSumBlocks; }

size_t sums_scratch_doubles() { return kSumsScratchDoubles; }

// Device address of `scratch` on the current device, resolved with
// hipGetSymbolAddress the first time a context is created on that device
// and kept per device ordinal.
hipError_t sums_scratch(double** out) {
  static std::mutex mu;
  static double* ptr[kMaxDevices] = {};
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    ptr[dev] = (double*)p;
  }
  *out = ptr[dev];
  return hipSuccess;
}

// Components whose half spectra are transformed in one launch: all three while
// they fit the 256 MB last-level cache together with room to spare (small boxes
// are bound by the number of launches), else one at a time, each then read
// back from that cache up to 256^3 (half a spectrum is 8 B per node).
int spectrum_batch(const Grid& g) {
  const uint64_t half = sizeof(double2) * (uint64_t)(g.nx / 2) * (uint64_t)g.ny * (uint64_t)g.nz;
  return 3 * half <= ((uint64_t)128 << 20) ? 3 : 1;
}

size_t spectrum_scratch_bytes(const Grid& g) {
  return sizeof(double2) * (size_t)(g.nx / 2) * (size_t)g.ny * (size_t)g.nz * (size_t)spectrum_batch(g);
}

template <int AXIS>
static hipError_t launch_fft(const Grid& g, FftArgs a, int comps, hipStream_t s, int* blocks = nullptr) {
  a.n = AXIS == AXIS_X ? g.nx : (AXIS == AXIS_Y ? g.ny : g.nz);
  const bool pow2 = ilog2_exact(a.n) >= 3;
  // lines per tile: eight (runs of 128 B), more where eight are too few to
  // fill a wavefront, fewer where they would be more than 4096 (two buffers:
  // 2048) entries: at most 72 KB of LDS and the shells of the z pass, along x
  // 96 KB (two padded lines of 1023 entries)
  const int most = pow2 ? 4096 : 2048;
  a.ltx = 3;
  while ((a.n << a.ltx) < 512) ++a.ltx;
  while (a.ltx > 0 && (a.n << a.ltx) > most) --a.ltx;
  a.tx = 1 << a.ltx;
  if (AXIS == AXIS_X) {
    const int64_t pairs = ((int64_t)g.ny * g.nz + 1) / 2;
    a.per = (int)((pairs + a.tx - 1) / a.tx);
  } else {
    a.across = (a.hx + a.tx - 1) / a.tx;
    a.per = a.across * (AXIS == AXIS_Y ? g.nz : g.ny);
  }
  a.tiles = a.per * comps;
  a.nf = 0;
  for (int r = 4, m = a.n; m > 1; r = r == 4 ? 2 : (r == 2 ? 3 : r + 2))
    for (; m % r == 0; m /= r) a.f[a.nf++] = r;
  size_t lds = sizeof(double2) * (pow2 ? (size_t)(a.n + a.n / 8) * a.tx
                                       : 2 * (size_t)a.n * any_row<AXIS>(a.tx));
  int nb = a.tiles;
  if (AXIS == AXIS_Z) {
    lds += sizeof(double) * a.nek;
    nb = std::min(nb, kSumBlocks);   // each keeps its own shells over its tiles
    *blocks = nb;
  }
  if (pow2)
    hipLaunchKernelGGL((k_fft_pow2<AXIS>), dim3(nb), dim3(a.tx * a.n / 8), lds, s, a);
  else
    hipLaunchKernelGGL((k_fft_any<AXIS>), dim3(nb), dim3(256), lds, s, a);
  return hipGetLastError();
}

hipError_t launch_spectrum(Ctx& c, int nek, double2* Z, const double2* const tw[3], double* part,
                           double* acc) {
  const double* u[3] = {c.ux, c.uy, c.uz};
  FftArgs a{};
  a.Z = Z;
  a.nx = c.g.nx;
  a.ny = c.g.ny;
  a.nz = c.g.nz;
  a.hx = c.g.nx / 2;
  a.nek = nek;
  a.part = part;
  const int batch = spectrum_batch(c.g);
  for (int c0 = 0; c0 < 3; c0 += batch) {
    for (int k = 0; k < batch; ++k) a.re[k] = u[c0 + k];
    int nb = 0;
    hipError_t e;
    a.tw = tw[0];
    if ((e = launch_fft<AXIS_X>(c.g, a, batch, c.stream)) != hipSuccess) return e;
    a.tw = tw[1];
    if ((e = launch_fft<AXIS_Y>(c.g, a, batch, c.stream)) != hipSuccess) return e;
    a.tw = tw[2];
    if ((e = launch_fft<AXIS_Z>(c.g, a, batch, c.stream, &nb)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_spectrum_final, dim3((nek + 63) / 64), dim3(1024), 0, c.stream, part, nb, nek, acc,
                       c0 > 0 ? 1 : 0);
  }
  return hipGetLastError();
}

}  // namespace mfc
