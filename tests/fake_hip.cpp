// A stand-in for the HIP runtime, for host-side tests of what the library does when a
// call of it fails: device memory is zeroed host memory, copies are memcpy, kernels are not run (but one).  Linked into a
// copy of libdgv_amd.so (tests/fake_device.py).  fake_fail_kernel / fake_fail_malloc choose
// the call that fails; the launches so far, and the widest, can be read back.
#include <sys/mman.h>

#include <cstdint>
#include <cstring>
#include <map>
#include <string>

typedef int hipError_t;   // hipSuccess 0, hipErrorOutOfMemory 2, hipErrorInvalidConfiguration 9
struct dim3_t { uint32_t x, y, z; };

static std::map<const void*, std::string> names;
static std::map<void*, size_t> sizes;
static std::string fail_kernel, launched;
static int64_t fail_malloc_above = INT64_MAX, largest = 0;
static uint64_t widest = 0;
static int capturing = 0, fastest = -1, timed = 0;
static hipError_t last = 0;
static struct { dim3_t g, b; size_t shm; void* st; } conf;

extern "C" {
void fake_fail_kernel(const char* part) { fail_kernel = part; }
void fake_fail_malloc_above(int64_t bytes) { fail_malloc_above = bytes; }
void fake_fastest(int k) { fastest = k; timed = 0; }   // the k-th time read from now on is the shortest
void fake_capturing(int on) { capturing = on; }
void fake_reset() { launched.clear(); widest = 0; largest = 0; }
const char* fake_launched() { return launched.c_str(); }
uint64_t fake_widest_launch() { return widest; }
int64_t fake_largest_malloc() { return largest; }
int64_t fake_live_bytes() {
  int64_t n = 0;
  for (const auto& s : sizes) n += (int64_t)s.second;
  return n;
}

void** __hipRegisterFatBinary(const void*) { static void* h = nullptr; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, dim3_t*, dim3_t*, int*) {
  names[host] = device;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t shm, void* st) { conf = {g, b, shm, st}; return 0; }
hipError_t __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* shm, void** st) {
  *g = conf.g; *b = conf.b; *shm = conf.shm; *st = conf.st;
  return 0;
}
// The one kernel whose result sizes what is built: quads per block, a third of its pairs
struct alignas(16) QuadBlk { int64_t sbeg; int32_t nst; int8_t a[3], b[3]; uint8_t same, pad; int32_t npairs; };
static void assign(void** arg) {
  const int64_t nq = *(const int64_t*)arg[1];
  const QuadBlk* qb = *(const QuadBlk* const*)arg[2];
  int32_t* count = *(int32_t* const*)arg[9];
  for (int64_t k = 0; k < nq; ++k) count[k] = qb[k].npairs / 3;
}
hipError_t hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** arg, size_t, void*) {
  const std::string& n = names[f];
  launched += n + "\n";
  const uint64_t items = (uint64_t)g.x * b.x;
  if (items > widest) widest = items;
  if (items >> 32) return last = 9;   // a grid dimension holds fewer than 2^32 work-items
  if (!fail_kernel.empty() && n.find(fail_kernel) != std::string::npos) return last = 9;
  if (n.find("k_quad_assign") != std::string::npos) assign(arg);
  return 0;
}
hipError_t hipGetLastError() { const hipError_t e = last; last = 0; return e; }
const char* hipGetErrorString(hipError_t e) { return e ? "fake error" : "no error"; }
// zeroed pages that take memory only where they are written: a device's memory is larger than the host's
hipError_t hipMalloc(void** p, size_t n) {
  if ((int64_t)n > fail_malloc_above) return 2;   // reported here alone
  *p = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (*p == MAP_FAILED) return 2;
  sizes[*p] = n ? n : 1;
  if ((int64_t)n > largest) largest = n;
  return 0;
}
hipError_t hipFree(void* p) {
  const auto it = sizes.find(p);
  if (it == sizes.end()) return p ? 1 : 0;
  munmap(p, it->second);
  sizes.erase(it);
  return 0;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return 0; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { memcpy(d, s, n); return 0; }
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int, void*) {
  for (size_t i = 0; i < h; ++i) memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
  return 0;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, void*) { memset(d, v, n); return 0; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { *p = const_cast<void*>(s); return 0; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return 0; }
hipError_t hipGetDevicePropertiesR0600(void*, int) { return 0; }
hipError_t hipSetDevice(int) { return 0; }
hipError_t hipDeviceSynchronize() { return 0; }
hipError_t hipStreamCreateWithFlags(void** s, unsigned) { *s = nullptr; return 0; }
hipError_t hipStreamDestroy(void*) { return 0; }
hipError_t hipStreamSynchronize(void*) { return 0; }
hipError_t hipStreamIsCapturing(void*, int* s) { *s = capturing; return 0; }
hipError_t hipStreamBeginCapture(void*, int) { return 0; }
hipError_t hipStreamEndCapture(void*, void** g) { *g = nullptr; return 0; }
hipError_t hipEventCreate(void** e) { *e = nullptr; return 0; }
hipError_t hipEventDestroy(void*) { return 0; }
hipError_t hipEventRecord(void*, void*) { return 0; }
hipError_t hipEventSynchronize(void*) { return 0; }
hipError_t hipEventElapsedTime(float* ms, void*, void*) { *ms = timed++ == fastest ? 1.f : 2.f; return 0; }
hipError_t hipGraphInstantiate(void** x, void*, void*, char*, size_t) { *x = nullptr; return 0; }
hipError_t hipGraphLaunch(void*, void*) { return 0; }
hipError_t hipGraphDestroy(void*) { return 0; }
hipError_t hipGraphExecDestroy(void*) { return 0; }
}
