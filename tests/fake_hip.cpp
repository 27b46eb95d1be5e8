// A HIP runtime without a device, for tests of the library's host side: memory
// is mapped but not filled, kernels do nothing, and every call is logged.
// Loaded with RTLD_GLOBAL before libedhmc.so, whose calls it then takes.
#include <stdint.h>
#include <string.h>
#include <sys/mman.h>

#include <map>
#include <set>
#include <string>

namespace {

struct dim3_t { uint32_t x, y, z; };
struct Config { dim3_t grid, block; size_t shm; void* stream; };

std::map<void*, size_t> mem;
std::map<const void*, std::string>& names() {   // used while libraries load
  static std::map<const void*, std::string> m;
  return m;
}
std::set<void*> capturing;
std::string lines, fail_kernel;
size_t limit = SIZE_MAX, in_use = 0;
int fail_malloc = 0;
int error = 0;
Config config;
constexpr size_t kCopy = 1 << 20;   // larger memory is neither filled nor copied

void log(const std::string& s) { lines += s + "\n"; }
std::string str(const void* p) { return std::to_string((uintptr_t)p); }

}  // namespace

extern "C" {

// -- the test's side ----------------------------------------------------------
const char* fake_log() { return lines.c_str(); }
void fake_clear() { lines.clear(); }
void fake_limit(size_t bytes) { limit = bytes; }
size_t fake_in_use() { return in_use; }
void fake_fail_malloc(int nth) { fail_malloc = nth; }   // 1: the next one; 0: none
int fake_to_fail() { return fail_malloc; }
void fake_capture(void* stream, int on) {
  if (on) capturing.insert(stream);
  else capturing.erase(stream);
}
void fake_fail_kernel(const char* part_of_name) { fail_kernel = part_of_name; }

// -- the runtime's ------------------------------------------------------------
int hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if (n > limit - in_use || in_use > limit || (fail_malloc > 0 && --fail_malloc == 0)) {
    log("malloc_failed " + std::to_string(n));
    return error = 2;
  }
  void* q = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (q == MAP_FAILED) return error = 2;
  mem[q] = n;
  in_use += n;
  log("malloc " + std::to_string(n));
  *p = q;
  return 0;
}
int hipFree(void* p) {
  auto it = mem.find(p);
  if (it == mem.end()) return p ? error = 1 : 0;
  log("free " + std::to_string(it->second));
  in_use -= it->second;
  munmap(p, it->second);
  mem.erase(it);
  return 0;
}
int hipMemset(void* p, int v, size_t n) {
  if (n <= kCopy) memset(p, v, n);
  return 0;
}
int hipMemsetAsync(void* p, int v, size_t n, void* st) {
  log("memset " + str(st));
  return hipMemset(p, v, n);
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) {
  log("memcpy " + str(st));
  if (kind != 3 && n <= kCopy) memcpy(d, s, n);   // not from device to device
  return 0;
}
int hipStreamSynchronize(void* st) {
  log("sync " + str(st));
  return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int) { return 0; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipGetLastError() {
  const int e = error;
  error = 0;
  return e;
}
const char* hipGetErrorString(int) { return "fake error"; }
int hipGetSymbolAddress(void** p, const void*) { return hipMalloc(p, 64 << 20); }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 3;
  return 0;
}

int hipLaunchKernel(const void* f, dim3_t grid, dim3_t, void**, size_t, void* st) {
  const std::string& name = names()[f];
  log("launch " + str(st) + " " + std::to_string(grid.x) + "," + std::to_string(grid.y) + "," +
      std::to_string(grid.z) + " " + name);
  if (!fail_kernel.empty() && name.find(fail_kernel) != std::string::npos) return error = 98;
  return 0;
}
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t shm, void* st) {
  config = {grid, block, shm, st};
  return 0;
}
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* shm, void** st) {
  *grid = config.grid;
  *block = config.block;
  *shm = config.shm;
  *st = config.stream;
  return 0;
}
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
  names()[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

int hipEventCreateWithFlags(void** e, unsigned) {
  *e = new char;
  return 0;
}
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e) {
  delete (char*)e;
  return 0;
}
int hipEventRecord(void* e, void* st) {
  log("record " + str(st) + " " + str(e));
  return 0;
}
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0.0f;
  return 0;
}
int hipStreamWaitEvent(void* st, void* e, unsigned) {
  log("wait " + str(st) + " " + str(e));
  return 0;
}
int hipStreamIsCapturing(void* st, int* status) {
  *status = capturing.count(st) ? 1 : 0;
  return 0;
}

}  // extern "C"
