// A HIP runtime that runs on the CPU and computes nothing: memory is host
// memory, copies happen at once, a kernel launch is only noted (name, grid,
// dynamic LDS, device, stream) -- except the kernels whose result the calling
// thread waits for, which are carried out here.  Loaded with RTLD_GLOBAL before
// libmfc_lbm.so, whose calls then come here, it shows what the host side
// allocates, copies and launches.  Two devices; the current one is per thread.
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <vector>

typedef int hipError_t;
struct dim3 {
  uint32_t x, y, z;
};

namespace {

enum Kind { DEVICE, PINNED };
struct Block {
  size_t bytes;
  int device;
  Kind kind;
};
struct Launch {
  std::string name;
  uint64_t blocks;
  size_t lds;
  int device;
};
struct Stream {
  int device;
};

std::mutex mu;
std::map<const char*, Block> blocks;
std::map<const void*, std::string> kernels;
std::vector<Launch> launches;
size_t allocated = 0, free_bytes = (size_t)288 << 30;
int copies = 0, syncs = 0, foreign = 0;
thread_local int current = 0;
thread_local hipError_t last = 0;
thread_local dim3 cfg_grid, cfg_block;
thread_local size_t cfg_lds;
thread_local void* cfg_stream;

// a launch or allocation a real second device would not see
void note_device(void* stream) {
  if (stream && ((Stream*)stream)->device != current) ++foreign;
}

const std::pair<const char* const, Block>* block_of(const void* p) {
  auto it = blocks.upper_bound((const char*)p);
  if (it == blocks.begin()) return nullptr;
  --it;
  return (const char*)p < it->first + it->second.bytes ? &*it : nullptr;
}

// hostcopy.hip's job: parts in units of 16384 bytes
struct CopyJob {
  const char* dev[4];
  uint64_t bytes[4];
  uint32_t unit0[5];
  int nparts;
};
void copy_out(void** a) {
  const CopyJob& j = *(const CopyJob*)a[0];
  const uint32_t first = *(uint32_t*)a[1], n = *(uint32_t*)a[2], seq = *(uint32_t*)a[6];
  char* win = *(char**)a[3];
  uint32_t* count = *(uint32_t**)a[4];
  uint32_t* flag = *(uint32_t**)a[5];
  // the kernel's atomics need the counters on its own device
  const auto* b = block_of(count);
  if (!b || b->second.device != current) ++foreign;
  for (uint32_t u = first; u < first + n; ++u) {
    int k = 0;
    while (k + 1 < j.nparts && u >= j.unit0[k + 1]) ++k;
    const uint64_t off = (uint64_t)(u - j.unit0[k]) * 16384;
    memcpy(win + (uint64_t)(u - first) * 16384, j.dev[k] + off, std::min<uint64_t>(16384, j.bytes[k] - off));
  }
  for (uint32_t p = 0; p * 16 < n; ++p) flag[p] = seq;
}

hipError_t allocate(void** p, size_t n, Kind kind) {
  std::lock_guard<std::mutex> lk(mu);
  if (kind == DEVICE && n > free_bytes) return 2;
  // zero pages on demand: untouched memory costs nothing
  *p = calloc(1, n ? n : 1);
  if (!*p) return 2;
  blocks[(char*)*p] = {n ? n : 1, current, kind};
  if (kind == DEVICE) {
    allocated += n;
    free_bytes -= n;
  }
  return 0;
}
hipError_t release(void* p) {
  std::lock_guard<std::mutex> lk(mu);
  auto it = blocks.find((char*)p);
  if (it == blocks.end()) return p ? 1 : 0;
  if (it->second.kind == DEVICE) free_bytes += it->second.bytes;
  blocks.erase(it);
  free(p);
  return 0;
}

}  // namespace

extern "C" {

// ---- what the tests read ----
int fake_launches(const char* part) {
  int n = 0;
  for (const Launch& l : launches) n += l.name.find(part) != std::string::npos;
  return n;
}
size_t fake_max_lds(const char* part) {
  size_t m = 0;
  for (const Launch& l : launches)
    if (l.name.find(part) != std::string::npos) m = std::max(m, l.lds);
  return m;
}
// the i-th launch since the last reset ("" past the end)
const char* fake_launch(int i) { return (size_t)i < launches.size() ? launches[i].name.c_str() : ""; }
void fake_reset() {
  launches.clear();
  copies = syncs = foreign = 0;
}
int fake_copies() { return copies; }
int fake_syncs() { return syncs; }
int fake_foreign() { return foreign; }
size_t fake_allocated() { return allocated; }
void fake_set_free(size_t n) { free_bytes = n; }

// ---- the runtime ----
hipError_t hipGetDeviceCount(int* n) { return *n = 2, 0; }
hipError_t hipGetDevice(int* d) { return *d = current, 0; }
hipError_t hipSetDevice(int d) { return d < 0 || d > 1 ? 101 : (current = d, 0); }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = 0;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e ? "error" : "no error"; }
hipError_t hipMalloc(void** p, size_t n) { return allocate(p, n, DEVICE); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return allocate(p, n, PINNED); }
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipHostFree(void* p) { return release(p); }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { return *f = free_bytes, *t = (size_t)288 << 30, 0; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, int) { return memcpy(d, s, n), ++copies, 0; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { return memcpy(d, s, n), ++copies, 0; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, void*) {
  if (v || n < ((size_t)1 << 24)) memset(d, v, n);   // large blocks are zero from the start
  return 0;
}
struct Attributes {   // hipPointerAttribute_t
  int type, device;
  void *devicePointer, *hostPointer;
  int isManaged;
  unsigned allocationFlags;
};
hipError_t hipPointerGetAttributes(Attributes* a, const void* p) {
  std::lock_guard<std::mutex> lk(mu);
  *a = Attributes{};
  const auto* b = block_of(p);
  if (!b) return 1;
  a->type = b->second.kind == PINNED ? 1 : 2;   // hipMemoryTypeHost, hipMemoryTypeDevice
  a->device = b->second.device;
  return 0;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char symbol[1 << 20];
  return *p = symbol, 0;
}
hipError_t hipStreamCreateWithFlags(void** s, unsigned) { return *s = new Stream{current}, 0; }
hipError_t hipStreamDestroy(void* s) { return delete (Stream*)s, 0; }
hipError_t hipStreamSynchronize(void*) { return ++syncs, 0; }
hipError_t hipStreamQuery(void*) { return 0; }
hipError_t hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
hipError_t hipEventCreate(void** e) { return *e = malloc(1), 0; }
hipError_t hipEventCreateWithFlags(void** e, unsigned) { return *e = malloc(1), 0; }
hipError_t hipEventDestroy(void* e) { return free(e), 0; }
hipError_t hipEventRecord(void*, void*) { return 0; }
hipError_t hipEventSynchronize(void*) { return 0; }
hipError_t hipEventElapsedTime(float* t, void*, void*) { return *t = 0.f, 0; }
hipError_t hipStreamBeginCapture(void*, int) { return 801; }
hipError_t hipStreamEndCapture(void*, void**) { return 801; }
hipError_t hipGraphInstantiate(void**, void*, void**, char*, size_t) { return 801; }
hipError_t hipGraphLaunch(void*, void*) { return 801; }
hipError_t hipGraphDestroy(void*) { return 0; }
hipError_t hipGraphExecDestroy(void*) { return 0; }

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void* stream) {
  cfg_grid = grid;
  cfg_block = block;
  cfg_lds = lds;
  cfg_stream = stream;
  return 0;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, void** stream) {
  *grid = cfg_grid;
  *block = cfg_block;
  *lds = cfg_lds;
  *stream = cfg_stream;
  return 0;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t lds, void* stream) {
  std::lock_guard<std::mutex> lk(mu);
  const uint64_t n = (uint64_t)g.x * g.y * g.z;
  const std::string& name = kernels[f];
  if (n == 0 || b.x * b.y * b.z == 0 || lds > 160 * 1024) {
    launches.push_back({"invalid " + name, n, lds, current});
    return last = 9;   // hipErrorInvalidConfiguration
  }
  note_device(stream);
  launches.push_back({name, n, lds, current});
  if (name.find("k_copy_out") != std::string::npos) copy_out(args);
  if (name.find("k_rho_residual") != std::string::npos) {
    uint64_t* out = *(uint64_t**)args[2];
    *out = 0;
    *(uint32_t*)(out + 1) = *(uint32_t*)args[3];
  }
  return 0;
}

}  // extern "C"
