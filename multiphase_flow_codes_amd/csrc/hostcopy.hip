// hostcopy.hip -- copies from device memory to the caller's pageable host
// arrays (fields, populations, maps, particle arrays, results).
//
// A plain copy to pageable memory goes through the runtime's own staging, one
// piece and one wait after the other.  Here one kernel per window writes the
// data into pinned memory and raises a flag for every piece of 256 KB; the
// calling thread polls the flags and copies each piece on to the caller's
// arrays while the next ones cross the bus (57 GB/s), with two windows in turn.
// A small array is one workgroup and one flag: no copy command, no stream
// synchronisation.  Measured against hipMemcpyAsync and hipStreamSynchronize:
// 7 KB 11.5 against 25 us, 1.2 MB 68 against 88, 8.4 MB 330 against 477, 54 MB
// 1.75 against 2.99 ms (into fresh arrays, whose pages fault on the one
// thread, 4.4 against 6.4 ms).  Bound from 1 MB on by the calling thread's
// copy, 25-31 GB/s.  Copying with further threads was faster alone (54 MB fresh
// 2.5 ms) but starved beside a program's own thread pool (17.7 MB 0.6 to 5 ms).
//
// The windows belong to a device and are shared by its contexts: allocated at
// the first copy, freed with the last context.  The calling thread's current
// device may be another one (a thread starts on device 0): it is the context's
// while a copy allocates and launches.  A copy that finds them in use by
// another host thread takes the runtime's path.
#include <mutex>
#include <thread>

#include <string.h>

#include "internal.h"

namespace mfc {

namespace {

constexpr uint32_t kUnit = 16384;                  // bytes per workgroup
constexpr uint32_t kPieceUnits = 16;               // workgroups per flag
constexpr uint32_t kWindowUnits = 256;             // workgroups per launch
constexpr uint32_t kWindowPieces = kWindowUnits / kPieceUnits;

// The parts, each starting at a unit of the window sequence.
struct CopyJob {
  const char* dev[kMaxParts];
  uint64_t bytes[kMaxParts];
  uint32_t unit0[kMaxParts + 1];   // first unit of each part, then their number
  int nparts;
};

struct Pipe {
  std::mutex use;        // held by the copy that owns the windows
  std::mutex mu;         // guards refs and the allocation
  int refs = 0;
  char* win[2] = {};     // pinned
  uint32_t* flag = nullptr;      // pinned: [2][kWindowPieces]
  uint32_t* count = nullptr;     // device: finished workgroups per piece, back at 0 after each launch
  uint32_t seq = 0;              // value the flags of the last launch take
};

Pipe g_pipe[kMaxDevices];

__device__ __forceinline__ int part_of_unit(const CopyJob& j, uint32_t u) {
  int k = 0;
  while (k + 1 < j.nparts && u >= j.unit0[k + 1]) ++k;
  return k;
}

__global__ void __launch_bounds__(256)
    k_copy_out(CopyJob j, uint32_t first, uint32_t nunits, char* __restrict__ win, uint32_t* __restrict__ count,
               uint32_t* __restrict__ flag, uint32_t seq) {
  const uint32_t b = blockIdx.x, u = first + b;
  const int k = part_of_unit(j, u);
  const uint64_t off = (uint64_t)(u - j.unit0[k]) * kUnit;
  const uint64_t left = j.bytes[k] - off;
  const uint32_t n = left < kUnit ? (uint32_t)left : kUnit;
  const char* src = j.dev[k] + off;
  char* dst = win + (uint64_t)b * kUnit;
  if (((uintptr_t)src & 15u) == 0) {
    const uint32_t nv = n / 16;
    for (uint32_t i = threadIdx.x; i < nv; i += 256) ((uint4*)dst)[i] = ((const uint4*)src)[i];
    for (uint32_t i = nv * 16 + threadIdx.x; i < n; i += 256) dst[i] = src[i];
  } else {   // 4-byte elements
    for (uint32_t i = threadIdx.x; i < n / 4; i += 256) ((uint32_t*)dst)[i] = ((const uint32_t*)src)[i];
  }
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x != 0) return;
  const uint32_t p = b / kPieceUnits;
  const uint32_t units = min(kPieceUnits, nunits - p * kPieceUnits);
  if (__hip_atomic_fetch_add(&count[p], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) != units - 1) return;
  __hip_atomic_store(&count[p], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&flag[p], seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void k_zero_u32(uint32_t* a, uint32_t n) {
  if (threadIdx.x < n) a[threadIdx.x] = 0u;
}

void release(Pipe& P) {
  for (char*& w : P.win) {
    if (w) (void)hipHostFree(w);
    w = nullptr;
  }
  if (P.flag) (void)hipHostFree(P.flag);
  if (P.count) (void)hipFree(P.count);
  P.flag = nullptr;
  P.count = nullptr;
}

// The windows the copy needs, allocated (false: take the runtime's path).
bool prepare(Pipe& P, int windows, hipStream_t s) {
  std::lock_guard<std::mutex> lk(P.mu);
  const unsigned fl = hipHostMallocPortable | hipHostMallocCoherent;
  if (!P.flag) {
    if (hipHostMalloc((void**)&P.flag, sizeof(uint32_t) * 2 * kWindowPieces, fl) != hipSuccess ||
        hipMalloc((void**)&P.count, sizeof(uint32_t) * 2 * kWindowPieces) != hipSuccess) {
      (void)hipGetLastError();
      release(P);
      return false;
    }
    memset(P.flag, 0, sizeof(uint32_t) * 2 * kWindowPieces);
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, P.count, 2 * kWindowPieces);
    if (hipStreamSynchronize(s) != hipSuccess) return false;
    P.seq = 0;
  }
  for (int w = 0; w < windows; ++w)
    if (!P.win[w] && hipHostMalloc((void**)&P.win[w], (size_t)kUnit * kWindowUnits, fl) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
  return true;
}

}  // namespace

OnDevice::OnDevice(int dev) {
  int now = -1;
  ok = dev >= 0 && hipGetDevice(&now) == hipSuccess;
  if (!ok || now == dev) return;
  ok = hipSetDevice(dev) == hipSuccess;
  if (ok) was = now;
}
OnDevice::~OnDevice() {
  if (was >= 0) (void)hipSetDevice(was);
}

void host_pipe_ref(int dev) {
  std::lock_guard<std::mutex> lk(g_pipe[dev].mu);
  ++g_pipe[dev].refs;
}

void host_pipe_unref(int dev) {
  Pipe& P = g_pipe[dev];
  std::lock_guard<std::mutex> lk(P.mu);
  if (--P.refs == 0) release(P);
}

// Waits until a kernel queued on the stream has stored `value` in the pinned
// word; the stream's state is asked now and then, so that a failure of the
// queued work ends the wait.
hipError_t wait_flag(const uint32_t* flag, uint32_t value, hipStream_t s) {
  for (uint32_t spin = 1;; ++spin) {
    if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == value) return hipSuccess;
    if ((spin & 0xffffu) == 0) {
      const hipError_t e = hipStreamQuery(s);
      if (e == hipErrorNotReady) {
        (void)hipGetLastError();
        std::this_thread::yield();
        continue;
      }
      if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == value) return hipSuccess;
      return e != hipSuccess ? e : hipErrorUnknown;
    }
    __builtin_ia32_pause();
  }
}

// Is the target left to the runtime's own copy?  Memory the thread cannot be
// relied on to write (a device's, managed) always, pinned memory where the bus
// alone is the faster: four arrays of 2.1 MB 185 us against 308 through the
// windows, of 885 KB 102 against 165, of 262 KB 55 against 53, of 85 KB 42 against 24.
static bool runtime_target(const HostPart& part) {
  constexpr size_t kPinnedFrom = (size_t)1 << 19;
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, part.host) != hipSuccess) {
    (void)hipGetLastError();   // ordinary memory
    return false;
  }
  if (a.type == hipMemoryTypeHost) return part.bytes >= kPinnedFrom;
  return a.type != hipMemoryTypeUnregistered;
}

// Copies the parts to the host after the work queued on the context's stream
// and waits for them (no parts: for that work).
hipError_t copy_to_host(Ctx& c, const HostPart* all, int nall) {
  CopyJob j{};
  HostPart part[kMaxParts];
  int nparts = 0;
  uint32_t units = 0;
  bool plain = c.pipe_dev < 0;
  for (int k = 0; k < nall; ++k) {
    if (runtime_target(all[k])) {
      const hipError_t e = hipMemcpyAsync(all[k].host, all[k].dev, all[k].bytes, hipMemcpyDeviceToHost, c.stream);
      if (e != hipSuccess) return e;
      continue;
    }
    part[nparts] = all[k];
    j.dev[nparts] = (const char*)all[k].dev;
    j.bytes[nparts] = all[k].bytes;
    j.unit0[nparts] = units;
    const uint64_t n = (all[k].bytes + kUnit - 1) / kUnit;
    if (n == 0 || n > (1u << 24) || all[k].bytes % 4 != 0) plain = true;
    units += (uint32_t)n;
    ++nparts;
  }
  if (nparts == 0) return hipStreamSynchronize(c.stream);
  j.unit0[nparts] = units;
  j.nparts = nparts;
  const OnDevice here(plain ? -1 : c.pipe_dev);
  plain = plain || !here.ok;
  std::unique_lock<std::mutex> own;
  if (!plain) {
    own = std::unique_lock<std::mutex>(g_pipe[c.pipe_dev].use, std::try_to_lock);
    if (own.owns_lock() && !prepare(g_pipe[c.pipe_dev], units > kWindowUnits ? 2 : 1, c.stream)) own.unlock();
  }
  if (!own.owns_lock()) {
    for (int k = 0; k < nparts; ++k) {
      const hipError_t e = hipMemcpyAsync(part[k].host, part[k].dev, part[k].bytes, hipMemcpyDeviceToHost, c.stream);
      if (e != hipSuccess) return e;
    }
    return hipStreamSynchronize(c.stream);
  }
  Pipe& P = g_pipe[c.pipe_dev];
  const uint32_t nwin = (units + kWindowUnits - 1) / kWindowUnits;
  uint32_t seq[2] = {0, 0};
  auto issue = [&](uint32_t w) {
    const uint32_t h = w & 1u, first = w * kWindowUnits;
    const uint32_t n = units - first < kWindowUnits ? units - first : kWindowUnits;
    if (++P.seq == 0) ++P.seq;
    seq[h] = P.seq;
    hipLaunchKernelGGL(k_copy_out, dim3(n), dim3(256), 0, c.stream, j, first, n, P.win[h],
                       P.count + h * kWindowPieces, P.flag + h * kWindowPieces, seq[h]);
    return hipGetLastError();
  };
  hipError_t err = issue(0);
  if (err == hipSuccess && nwin > 1) err = issue(1);
  int k = 0;   // part of the current unit
  for (uint32_t w = 0; w < nwin && err == hipSuccess; ++w) {
    const uint32_t h = w & 1u, first = w * kWindowUnits;
    const uint32_t n = units - first < kWindowUnits ? units - first : kWindowUnits;
    for (uint32_t p = 0; p * kPieceUnits < n; ++p) {
      if ((err = wait_flag(P.flag + h * kWindowPieces + p, seq[h], c.stream)) != hipSuccess) break;
      const uint32_t end = first + (n < (p + 1) * kPieceUnits ? n : (p + 1) * kPieceUnits);
      for (uint32_t u = first + p * kPieceUnits; u < end;) {
        while (u >= j.unit0[k + 1]) ++k;
        const uint32_t stop = end < j.unit0[k + 1] ? end : j.unit0[k + 1];
        const uint64_t off = (uint64_t)(u - j.unit0[k]) * kUnit;
        const uint64_t run = (uint64_t)(stop - u) * kUnit;
        memcpy((char*)part[k].host + off, P.win[h] + (uint64_t)(u - first) * kUnit,
               run < j.bytes[k] - off ? run : j.bytes[k] - off);
        u = stop;
      }
    }
    if (err == hipSuccess && w + 2 < nwin) err = issue(w + 2);
  }
  if (err != hipSuccess) {
    // nothing of this copy may still write the windows when another takes them
    const hipError_t e = hipStreamSynchronize(c.stream);
    if (e != hipSuccess) err = e;
  }
  return err;
}

}  // namespace mfc
