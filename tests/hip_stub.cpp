// hip_stub.cpp -- a host stand-in for the HIP runtime, rocBLAS and rocSOLVER, preloaded by test_host_runtime.py so that
// the library's host side (set-up threads, error handling, workspaces) runs without a GPU: device memory is host
// memory filled with 1.0, copies are memcpy, kernels do nothing.  A call can be made to fail, and what the library
// asks of the runtime is counted.  As in HIP, a failed call's error stays until hipGetLastError takes it.
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>

namespace {

std::mutex mu;
std::map<char*, size_t> live;                     // allocations
std::map<const void*, std::string> names;         // kernels by host function
std::map<const void*, size_t> lds_limit;          // hipFuncSetAttribute
std::string fail_kernel, watch_kernel;
int watch_arg = 0;
long fail_malloc = 0;                             // the k-th next hipMalloc fails (0: none)
long counts[9];                                   // see stub_count
std::set<void*> watched_streams;
bool recording = false;                           // an odd number of events recorded: BETWEEN counts allocations
thread_local int last = 0;

int failed(int code) { return last = code; }
bool in_live(char* p) {
  auto it = live.upper_bound(p);
  if (it == live.begin()) return false;
  --it;
  return p < it->first + it->second;
}

struct Dim3 {
  unsigned x, y, z;
};
thread_local struct {
  Dim3 grid, block;
  size_t lds;
  void* stream;
} config;

}  // namespace

extern "C" {

enum { MALLOCS, STREAMS, WATCHED, WATCHED_OUTSIDE, LDS_BEYOND, FAILED, WATCHED_STREAMS, BETWEEN };
long stub_count(int what) {
  std::lock_guard<std::mutex> lk(mu);
  return what == WATCHED_STREAMS ? (long)watched_streams.size() : counts[what];
}
// The k-th next hipMalloc fails (0: none).
void stub_fail_malloc(long k) {
  std::lock_guard<std::mutex> lk(mu);
  fail_malloc = k;
}
// Launches of the kernels whose name contains name fail ("": none).
void stub_fail_kernel(const char* name) {
  std::lock_guard<std::mutex> lk(mu);
  fail_kernel = name;
}
// Counts launches of the kernels whose name contains name, those of them whose pointer argument arg lies in no
// allocation, and their streams.
void stub_watch(const char* name, int arg) {
  std::lock_guard<std::mutex> lk(mu);
  watch_kernel = name;
  watch_arg = arg;
  counts[WATCHED] = counts[WATCHED_OUTSIDE] = 0;
  watched_streams.clear();
}

int hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lk(mu);
  ++counts[MALLOCS];
  if (recording) ++counts[BETWEEN];
  if (fail_malloc > 0 && --fail_malloc == 0) {
    ++counts[FAILED];
    *p = nullptr;
    return failed(2);
  }
  char* q = (char*)malloc(bytes + 64);
  const double one = 1.0;
  for (size_t i = 0; i + 8 <= bytes + 64; i += 8) memcpy(q + i, &one, 8);
  live[q] = bytes;
  *p = q;
  return 0;
}
int hipFree(void* p) {
  std::lock_guard<std::mutex> lk(mu);
  live.erase((char*)p);
  free(p);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t bytes, int, void*) {
  memmove(d, s, bytes);
  return 0;
}
int hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int, void*) {
  for (size_t r = 0; r < h; ++r) memmove((char*)d + r * dp, (const char*)s + r * sp, w);
  return 0;
}
int hipStreamCreate(void** s) {
  std::lock_guard<std::mutex> lk(mu);
  ++counts[STREAMS];
  *s = malloc(8);
  return 0;
}
int hipStreamDestroy(void* s) {
  std::lock_guard<std::mutex> lk(mu);
  --counts[STREAMS];
  free(s);
  return 0;
}
int hipStreamSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) {
  *g = malloc(8);
  return 0;
}
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) {
  *x = malloc(8);
  return 0;
}
int hipGraphLaunch(void*, void*) { return 0; }
int hipGraphDestroy(void* g) {
  free(g);
  return 0;
}
int hipGraphExecDestroy(void* g) {
  free(g);
  return 0;
}
int hipEventCreate(void** e) {
  *e = malloc(8);
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) {
  free(e);
  return 0;
}
int hipEventRecord(void*, void*) {
  std::lock_guard<std::mutex> lk(mu);
  recording = !recording;
  return 0;
}
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 1.f;
  return 0;
}
int hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
int hipSetDevice(int) { return 0; }
int hipGetDeviceCount(int* d) {
  *d = 1;
  return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 163840;  // serves as the LDS bytes of a workgroup; as a CU count it only makes the grids larger
  return 0;
}
int hipFuncSetAttribute(const void* f, int, int v) {
  std::lock_guard<std::mutex> lk(mu);
  lds_limit[f] = (size_t)v;
  return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 2;
  return 0;
}
int hipGetLastError() {
  const int e = last;
  last = 0;
  return e;
}
const char* hipGetErrorString(int) { return "stub failure"; }
int hipGetSymbolAddress(void** p, const void*) {
  static void* m = mmap(nullptr, (size_t)1 << 26, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  *p = m;
  return 0;
}
int hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = (size_t)256 << 30;
  return 0;
}

int hipLaunchKernel(const void* f, Dim3, Dim3, void** args, size_t lds, void* stream) {
  std::lock_guard<std::mutex> lk(mu);
  const std::string& name = names[f];
  auto it = lds_limit.find(f);
  if (it != lds_limit.end() && lds > it->second) ++counts[LDS_BEYOND];
  if (!watch_kernel.empty() && name.find(watch_kernel) != std::string::npos) {
    ++counts[WATCHED];
    if (!in_live(*(char**)args[watch_arg])) ++counts[WATCHED_OUTSIDE];
    watched_streams.insert(stream);
  }
  if (!fail_kernel.empty() && name.find(fail_kernel) != std::string::npos) {
    ++counts[FAILED];
    return failed(1);
  }
  return 0;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, void* s) {
  config = {g, b, lds, s};
  return 0;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* lds, void** s) {
  *g = config.grid;
  *b = config.block;
  *lds = config.lds;
  *s = config.stream;
  return 0;
}
void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  std::lock_guard<std::mutex> lk(mu);
  names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}

int rocblas_create_handle(void** h) {
  *h = malloc(8);
  return 0;
}
int rocblas_destroy_handle(void* h) {
  free(h);
  return 0;
}
int rocblas_set_stream(void*, void*) { return 0; }
int rocblas_set_pointer_mode(void*, int) { return 0; }
const char* rocblas_status_to_string(int) { return "stub"; }
int rocblas_dgemm(void*, ...) { return 0; }
int rocblas_dgemv(void*, ...) { return 0; }
int rocblas_dgemm_strided_batched(void*, ...) { return 0; }
int rocblas_ddot(void*, int, const double*, int, const double*, int, double* r) {
  *r = 1.0;
  return 0;
}
int rocblas_dnrm2(void*, int, const double*, int, double* r) {
  *r = 1.0;
  return 0;
}
int rocblas_idamax(void*, int, const double*, int, int* r) {
  *r = 1;
  return 0;
}
int rocsolver_dsyevd(void*, int, int, int n, double* a, int lda, double* w, double*, int* info) {
  for (int i = 0; i < n; ++i) {
    w[i] = 1.0 + i;
    for (int j = 0; j < n; ++j) a[(size_t)i * lda + j] = i == j;
  }
  *info = 0;
  return 0;
}

}  // extern "C"
