// A HIP runtime for tests of the library's host code without a GPU: device
// memory is host memory (reserved, zero until written), kernels are recorded and
// not run, copies are made at once, and an allocation limit can be set.  Loaded
// with RTLD_GLOBAL before the library, whose HIP calls then end here.
#include <sys/mman.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

typedef int hipError_t;
struct dim3 {
  uint32_t x, y, z;
};
enum { kSuccess = 0, kInvalid = 1, kOutOfMemory = 2 };

namespace {
struct Launch {
  std::string name;
  dim3 grid;
  void* stream;
};
std::map<char*, size_t>& live() { static std::map<char*, size_t> m; return m; }
std::map<const void*, std::string>& names() { static std::map<const void*, std::string> m; return m; }
std::map<void*, long>& queued() { static std::map<void*, long> m; return m; }  // work put on a stream and not waited for
std::vector<Launch> launches;
struct { dim3 grid, block; size_t lds; void* stream; } config;
size_t used = 0, most = (size_t)1 << 60;
int last_error = kSuccess;
int64_t found[3];
bool have_found = false;
std::string text;

hipError_t fail(hipError_t e) {
  last_error = e;
  return e;
}
}  // namespace

extern "C" {
// ---- controls -----------------------------------------------------------------
size_t rt_used() { return used; }
void rt_set_limit(size_t bytes) { most = bytes; }
long rt_queued(void* stream) { return queued()[stream]; }
void rt_forget() { launches.clear(); }
// kernels launched since rt_forget: "name gx gy gz" a line
const char* rt_launches() {
  text.clear();
  for (const Launch& l : launches)
    text += l.name + " " + std::to_string(l.grid.x) + " " + std::to_string(l.grid.y) + " " + std::to_string(l.grid.z) + "\n";
  return text.c_str();
}
// what the inspection of a CSR window reports from now on
void rt_inspection(int64_t first, int64_t last, int64_t flags) {
  found[0] = first;
  found[1] = last;
  found[2] = flags;
  have_found = true;
}

// ---- memory -------------------------------------------------------------------
hipError_t hipMalloc(void** p, size_t bytes) {
  if (used + bytes > most) return fail(kOutOfMemory);
  void* m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (m == MAP_FAILED) return fail(kOutOfMemory);
  live()[static_cast<char*>(m)] = bytes;
  used += bytes;
  *p = m;
  return kSuccess;
}
hipError_t hipFree(void* p) {
  auto it = live().find(static_cast<char*>(p));
  if (it == live().end()) return p ? fail(kInvalid) : kSuccess;
  munmap(p, it->second);
  used -= it->second;
  live().erase(it);
  return kSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = calloc(1, bytes);
  return kSuccess;
}
hipError_t hipHostFree(void* p) {
  free(p);
  return kSuccess;
}
hipError_t hipMemGetAddressRange(void** base, size_t* bytes, void* p) {
  auto it = live().upper_bound(static_cast<char*>(p));
  if (it == live().begin()) return fail(kInvalid);
  --it;
  if (static_cast<char*>(p) >= it->first + it->second) return fail(kInvalid);
  *base = it->first;
  *bytes = it->second;
  return kSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char symbol[64];  // its contents are the kernels' business
  *p = symbol;
  return kSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, void* stream) {
  memcpy(d, s, n);
  ++queued()[stream];
  return kSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int, void* stream) {
  for (size_t i = 0; i < h; ++i) memcpy(static_cast<char*>(d) + i * dp, static_cast<const char*>(s) + i * sp, w);
  ++queued()[stream];
  return kSuccess;
}

// ---- streams, events, device ----------------------------------------------------
hipError_t hipStreamSynchronize(void* stream) {
  queued()[stream] = 0;
  return kSuccess;
}
hipError_t hipSetDevice(int) { return kSuccess; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return kSuccess;
}
hipError_t hipGetLastError() {
  const int e = last_error;
  last_error = kSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == kOutOfMemory ? "out of memory" : "error"; }
hipError_t hipEventCreate(void** e) {
  *e = &last_error;
  return kSuccess;
}
hipError_t hipEventDestroy(void*) { return kSuccess; }
hipError_t hipEventRecord(void*, void*) { return kSuccess; }
hipError_t hipEventSynchronize(void*) { return kSuccess; }
hipError_t hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0.f;
  return kSuccess;
}

// ---- kernels ------------------------------------------------------------------
void** __hipRegisterFatBinary(const void*) {
  static void* handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
  names()[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void* stream) {
  config = {grid, block, lds, stream};
  return kSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, void** stream) {
  *grid = config.grid;
  *block = config.block;
  *lds = config.lds;
  *stream = config.stream;
  return kSuccess;
}
hipError_t hipLaunchKernel(const void* host, dim3 grid, dim3, void** args, size_t, void* stream) {
  const std::string& name = names()[host];
  launches.push_back({name, grid, stream});
  ++queued()[stream];
  if (have_found && name.find("k_inspect_csr") != std::string::npos)
    memcpy(*static_cast<int64_t**>(args[5]), found, sizeof(found));  // (rowptr, rows, col, cols, room, out)
  return kSuccess;
}
}
