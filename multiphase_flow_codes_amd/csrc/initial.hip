// initial.hip -- synthetic initial velocity fields on the device.
//
// A band-limited field u_c(x) = scale * sum_k 2 Re(a_c(k) e^{2 pi i k.x/n})
// over 0 <= kx <= 16, |ky|, |kz| <= 16 (x at the node indices), evaluated
// separably:
//   B1(kz, ky, x) = sum_kx a(kx, ky, kz) e^{2 pi i kx x/nx}   (33 x 33 x nx)
//   B2(kz, y, x)  = sum_ky B1(kz, ky, x) e^{2 pi i ky y/ny}    (33 x ny x nx)
//   u(x, y, z)    = 2 scale Re sum_kz B2(kz, y, x) e^{2 pi i kz z/nz}
// The y and z sums pair k with -k: B(k) e^{i t} + B(-k) e^{-i t} is
// (B(k) + B(-k)) cos t + i (B(k) - B(-k)) sin t, so a thread keeps the sums and
// differences of its column in registers and walks along the axis with one or
// two multiply-adds per cosine and sine.  Those are the same for every lane: a
// table of cos and sin of 2 pi k j / n for k = 1..16, one 256-B row per j, is
// read with scalar loads, in the z pass one row for two columns (one column
// each took 1.6 times as long at 256^3).  Bound: the stores of u (8 B per node,
// and of rho once) and the latency of those scalar loads.  At 256^3 a
// component's z pass takes 57 us and its y pass 25 us; one thread per whole
// column (256 workgroups), each finding its 33 phases per node by 64-bit
// remainders, took 531 us, and the y pass 124 us.
#include <algorithm>

#include "internal.h"

namespace mfc {

constexpr int KM = 16;            // largest |k| component
constexpr int NK = 2 * KM + 1;    // ky, kz values
constexpr int NKX = KM + 1;       // kx values

// (cos, sin)(2 pi k j / n) at [j * KM + k - 1], k = 1..KM, for the y axis and
// behind it the z axis, from the context's (cos, sin)(2 pi m / n) tables.
__global__ void __launch_bounds__(256)
    k_mode_phases(const double* __restrict__ phy, const double* __restrict__ phz, int ny, int nz,
                  double2* __restrict__ E) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= (uint32_t)(ny + nz) * KM) return;
  const uint32_t r = t / KM, k = t % KM + 1;
  const bool y = r < (uint32_t)ny;
  const uint32_t j = y ? r : r - (uint32_t)ny, n = (uint32_t)(y ? ny : nz);
  const double* ph = y ? phy : phz;
  const uint32_t m = (k * j) % n;
  E[t] = make_double2(ph[2 * m], ph[2 * m + 1]);
}

// B1[(iz * NK + iy) * nx + x]
__global__ void __launch_bounds__(256)
    k_modes_x(const double2* __restrict__ a, const double* __restrict__ phx, int nx,
              double2* __restrict__ B1) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  const uint32_t n1 = (uint32_t)(NK * NK) * (uint32_t)nx;
  if (t >= n1) return;
  const uint32_t x = t % (uint32_t)nx;
  const uint32_t row = t / (uint32_t)nx;   // iz * NK + iy
  double sr = 0.0, si = 0.0;
  uint32_t m = 0;   // kx * x mod nx
  for (int kx = 0; kx < NKX; ++kx) {
    const double2 v = a[row * NKX + kx];
    const double c = phx[2 * m], s = phx[2 * m + 1];
    sr += v.x * c - v.y * s;
    si += v.x * s + v.y * c;
    m += x;
    if (m >= (uint32_t)nx) m -= (uint32_t)nx;
  }
  B1[t] = make_double2(sr, si);
}

// B2[(iz * ny + y) * nx + x], y in chunk blockIdx.y of `chunk` rows
__global__ void __launch_bounds__(256)
    k_modes_y(const double2* __restrict__ B1, const double2* __restrict__ Ey, int nx, int ny, int chunk,
              double2* __restrict__ B2) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;   // iz * nx + x
  if (t >= (uint32_t)NK * (uint32_t)nx) return;
  const uint32_t iz = t / (uint32_t)nx, x = t - iz * (uint32_t)nx;
  const double2* b = B1 + (size_t)iz * NK * nx + x;
  double2 S[KM], D[KM];
  const double2 b0 = b[(size_t)KM * nx];
#pragma unroll
  for (int k = 1; k <= KM; ++k) {
    const double2 p = b[(size_t)(KM + k) * nx], m = b[(size_t)(KM - k) * nx];
    S[k - 1] = make_double2(p.x + m.x, p.y + m.y);
    D[k - 1] = make_double2(m.y - p.y, p.x - m.x);   // i (p - m)
  }
  const int y0 = (int)blockIdx.y * chunk, y1 = min(ny, y0 + chunk);
  double2* out = B2 + (size_t)iz * ny * nx + x;
  for (int y = y0; y < y1; ++y) {
    const double2* e = Ey + (size_t)y * KM;
    double sr = b0.x, si = b0.y;
#pragma unroll
    for (int k = 0; k < KM; ++k) {
      const double2 w = e[k];
      sr += S[k].x * w.x;
      sr += D[k].x * w.y;
      si += S[k].y * w.x;
      si += D[k].y * w.y;
    }
    out[(size_t)y * nx] = make_double2(sr, si);
  }
}

// One component, z in chunk blockIdx.y; with `rho` the density is cleared too.
__global__ void __launch_bounds__(256)
    k_modes_z(const double2* __restrict__ B2, const double2* __restrict__ Ez, uint32_t plane, int nz, int chunk,
              double scale, double* __restrict__ u, double* __restrict__ rho) {
  // two columns per thread share each phase row
  const uint32_t t0 = blockIdx.x * 512u + threadIdx.x;
  const double s2 = 2.0 * scale;
  double S[2][KM], D[2][KM], b0[2];
  bool on[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    on[h] = t0 + 256u * h < plane;
    const double2* b = B2 + (on[h] ? t0 + 256u * h : 0u);
    b0[h] = s2 * b[(size_t)KM * plane].x;
#pragma unroll
    for (int k = 1; k <= KM; ++k) {
      const double2 p = b[(size_t)(KM + k) * plane], m = b[(size_t)(KM - k) * plane];
      S[h][k - 1] = s2 * (p.x + m.x);
      D[h][k - 1] = s2 * (m.y - p.y);
    }
  }
  const int z0 = (int)blockIdx.y * chunk, z1 = min(nz, z0 + chunk);
  for (int z = z0; z < z1; ++z) {
    const double2* e = Ez + (size_t)z * KM;
    double acc[2] = {b0[0], b0[1]}, odd[2] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < KM; ++k) {
      const double2 w = e[k];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        acc[h] += S[h][k] * w.x;
        odd[h] += D[h][k] * w.y;
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!on[h]) continue;
      const uint64_t at = (uint64_t)z * plane + t0 + 256u * h;
      u[at] = acc[h] + odd[h];
      if (rho) rho[at] = 0.0;
    }
  }
}

int init_mode_kx() { return NKX; }
int init_mode_k() { return NK; }

// Scratch of launch_init_velocity behind the mode table, in double2 (one
// component's: allocating three would cost a small box more than the launches
// it saves).
size_t init_scratch(const Grid& g) {
  return (size_t)(g.ny + g.nz) * KM + (size_t)NK * NK * (size_t)g.nx + (size_t)NK * (size_t)g.nx * (size_t)g.ny;
}

// amp: (re, im) of a_c(kx, ky, kz) at flat index kx + NKX * ((ky + KM) + NK * ((kz + KM) + NK * c)),
// already on the device; work: init_scratch elements.
hipError_t launch_init_velocity(Ctx& c, const double2* amp, double scale, double2* work) {
  const Grid& g = c.g;
  const uint32_t plane = (uint32_t)g.nx * (uint32_t)g.ny;
  const uint32_t n1 = (uint32_t)(NK * NK) * (uint32_t)g.nx, ny1 = (uint32_t)NK * (uint32_t)g.nx;
  double2* E = work;
  double2* B1 = E + (size_t)(g.ny + g.nz) * KM;
  double2* B2 = B1 + n1;
  auto blocks = [](uint64_t n) { return (unsigned)((n + 255) / 256); };
  // chunks along the walked axis: `want` workgroups in all (2048 of the y and
  // 1024 of the z pass fill the GPU; more would only reload the columns: z at
  // 512^3 with 512, 1024, 4096 and 8192 took 465, 489, 578 and 647 us, at 256^3
  // 196, 181, 197 and 218), but walks of 16 or more
  auto chunk_of = [](unsigned across, int n, unsigned want) {
    const int per = (int)((want + across - 1) / across);
    return std::max(16, (n + per - 1) / per);
  };
  hipLaunchKernelGGL(k_mode_phases, dim3(blocks((uint64_t)(g.ny + g.nz) * KM)), dim3(256), 0, c.stream, c.ft.phy,
                     c.ft.phz, g.ny, g.nz, E);
  const int cy = chunk_of(blocks(ny1), g.ny, 2048), cz = chunk_of((plane + 511) / 512, g.nz, 1024);
  double* u[3] = {c.ux, c.uy, c.uz};
  for (int k = 0; k < 3; ++k) {
    hipLaunchKernelGGL(k_modes_x, dim3(blocks(n1)), dim3(256), 0, c.stream, amp + (size_t)k * NKX * NK * NK,
                       c.ft.phx, g.nx, B1);
    hipLaunchKernelGGL(k_modes_y, dim3(blocks(ny1), (g.ny + cy - 1) / cy), dim3(256), 0, c.stream, B1, E, g.nx,
                       g.ny, cy, B2);
    hipLaunchKernelGGL(k_modes_z, dim3((plane + 511) / 512, (g.nz + cz - 1) / cz), dim3(256), 0, c.stream, B2,
                       E + (size_t)g.ny * KM, plane, g.nz, cz, scale, u[k], k == 0 ? c.rho : nullptr);
  }
  return hipGetLastError();
}

}  // namespace mfc
