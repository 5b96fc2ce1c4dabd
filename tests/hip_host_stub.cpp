// A HIP runtime for tests of the library's host code where no GPU is: device
// and pinned memory are host memory, streams are idle, and kernels are not run.
// It is loaded before libfargo_hip.so with its symbols global, so the library's
// calls end here.  Two devices.  The stub_* functions let a test make a call
// fail and look at what the library asked for.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <string>

struct dim {
  uint32_t x, y, z;
};
enum { OK = 0, INVALID = 1, OUT_OF_MEMORY = 2, LAUNCH_FAILURE = 719 };

// (created on first use: the library registers its kernels while it is loaded)
struct stub_state {
  int device = 0, last = OK;
  int fail_pinned = 0, fail_launches = 0;
  std::string fail_kernel;
  std::map<const void *, std::string> kernels;
  std::map<const void *, size_t> device_memory;
  struct pinned {
    size_t bytes;
    int device;
  };
  std::map<char *, pinned> pinned_memory;
  std::map<const void *, size_t> lds_granted, lds_asked;
  // the bytes of argument `index` of the last launch of the watched kernel
  std::string watch_kernel;
  int watch_index = -1, watch_bytes = 0;
  char watched[64];
  dim grid, block;
  size_t shm = 0;
  void *stream = nullptr;
};
static stub_state &S() {
  static stub_state *s = new stub_state;
  return *s;
}
static int fails(int e) { return S().last = e; }
static bool fail_new;

void *operator new(size_t n) {
  void *p = fail_new ? nullptr : malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

extern "C" {
int hipGetDeviceCount(int *n) { return *n = 2, OK; }
int hipSetDevice(int d) { return d < 0 || d > 1 ? fails(INVALID) : (S().device = d, OK); }
int hipGetLastError() {
  const int e = S().last;
  S().last = OK;
  return e;
}
const char *hipGetErrorString(int e) { return e == OK ? "no error" : "stub error"; }
int hipMalloc(void **p, size_t n) {
  *p = calloc(n ? n : 1, 1);
  S().device_memory[*p] = n;
  return OK;
}
int hipFree(void *p) {
  S().device_memory.erase(p);
  free(p);
  return OK;
}
int hipHostMalloc(void **p, size_t n, unsigned) {
  if (S().fail_pinned) return fails(OUT_OF_MEMORY);
  *p = calloc(n ? n : 1, 1);
  S().pinned_memory[(char *)*p] = {n, S().device};
  return OK;
}
int hipHostFree(void *p) {
  S().pinned_memory.erase((char *)p);
  free(p);
  return OK;
}
int hipHostGetDevicePointer(void **d, void *h, unsigned) { return *d = h, OK; }
int hipMemcpy(void *d, const void *s, size_t n, int) {
  if (!d || !s) return fails(INVALID);
  memcpy(d, s, n);
  return OK;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *) { return hipMemcpy(d, s, n, kind); }
int hipMemset(void *d, int v, size_t n) { return memset(d, v, n), OK; }
int hipStreamCreate(void **s) {
  int *device = (int *)malloc(sizeof(int));
  *device = S().device;
  return *s = device, OK;
}
int hipStreamDestroy(void *s) { return free(s), OK; }
int hipStreamSynchronize(void *) { return OK; }
int hipStreamQuery(void *) { return OK; }
int hipFuncSetAttribute(const void *f, int, int value) { return S().lds_granted[f] = value, OK; }
int hipGetSymbolAddress(void **p, const void *) {
  static char device_variable[4 << 20];
  return *p = device_variable, OK;
}
void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  S().kernels[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim grid, dim block, size_t shm, void *stream) {
  stub_state &s = S();
  s.grid = grid, s.block = block, s.shm = shm, s.stream = stream;
  return OK;
}
int __hipPopCallConfiguration(dim *grid, dim *block, size_t *shm, void **stream) {
  stub_state &s = S();
  *grid = s.grid, *block = s.block, *shm = s.shm, *stream = s.stream;
  return OK;
}
int hipLaunchKernel(const void *f, dim, dim, void **args, size_t shm, void *) {
  stub_state &s = S();
  const std::string &name = s.kernels[f];
  if (s.fail_launches > 0 && name.find(s.fail_kernel) != std::string::npos) {
    s.fail_launches--;
    return fails(LAUNCH_FAILURE);
  }
  if (s.lds_asked[f] < shm) s.lds_asked[f] = shm;
  if (s.watch_index >= 0 && name.find(s.watch_kernel) != std::string::npos)
    memcpy(s.watched, args[s.watch_index], s.watch_bytes);
  return OK;
}

// ---- for the tests ----
void stub_fail_pinned(int on) { S().fail_pinned = on; }
void stub_fail_new(int on) { fail_new = on; }
// the next n launches of kernels whose name contains `kernel` fail
void stub_fail_launches(const char *kernel, int n) {
  S().fail_kernel = kernel;
  S().fail_launches = n;
}
void stub_watch(const char *kernel, int index, int bytes) {
  S().watch_kernel = kernel;
  S().watch_index = index;
  S().watch_bytes = bytes;
}
void stub_watched(void *out) { memcpy(out, S().watched, S().watch_bytes); }
size_t stub_device_bytes() {
  size_t n = 0;
  for (const auto &m : S().device_memory) n += m.second;
  return n;
}
// the device a pointer into pinned memory is mapped for, -1 for other memory
int stub_pinned_device(uint64_t at) {
  for (const auto &m : S().pinned_memory)
    if ((char *)at >= m.first && (char *)at < m.first + m.second.bytes) return m.second.device;
  return -1;
}
// dynamic LDS of a kernel: the most that was asked for in a launch, and what
// hipFuncSetAttribute granted
void stub_lds(const char *kernel, size_t *asked, size_t *granted) {
  *asked = *granted = 0;
  for (const auto &k : S().kernels)
    if (k.second.find(kernel) != std::string::npos) {
      if (S().lds_asked[k.first] > *asked) *asked = S().lds_asked[k.first];
      if (S().lds_granted[k.first] > *granted) *granted = S().lds_granted[k.first];
    }
}
}
