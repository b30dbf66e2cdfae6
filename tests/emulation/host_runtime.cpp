// host_runtime.cpp -- the HIP runtime calls that librbgpu.so makes, on host
// memory, for tests of its host code without a GPU. Copies are queued and run
// when the stream or an event after them is waited for; kernels do nothing.
// fake_fail makes one wait fail (its copies stay queued); fake_pending counts
// the copies still queued, fake_stream_waits the waits for the stream,
// fake_mallocs the allocations of device memory.
#include <cstdlib>
#include <cstring>
#include <deque>

namespace {
struct Copy {
  void* dst;
  const void* src;
  size_t bytes;
};
std::deque<Copy> queue;
long done = 0;  // copies run so far
int fail_stream = 0, fail_event = 0, stream_waits = 0, mallocs = 0;
struct Event {
  long after;
};
void run_to(long upto) {
  while (done < upto && !queue.empty()) {
    std::memcpy(queue.front().dst, queue.front().src, queue.front().bytes);
    queue.pop_front();
    done++;
  }
}
long all() { return done + long(queue.size()); }
constexpr int kError = 999;
}  // namespace

extern "C" {
void fake_fail(int event, int stream) {
  fail_event = event;
  fail_stream = stream;
  stream_waits = mallocs = 0;
}
long fake_pending() { return long(queue.size()); }
int fake_stream_waits() { return stream_waits; }
int fake_mallocs() { return mallocs; }

void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
struct Dim3 {
  unsigned x, y, z;
};
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void*) { return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* m, void** s) {
  *g = *b = {1, 1, 1};
  *m = 0;
  *s = nullptr;
  return 0;
}
int hipLaunchKernel(const void*, Dim3, Dim3, void**, size_t, void*) { return 0; }

int hipGetDeviceCount(int* n) { return *n = 1, 0; }
int hipGetDevice(int* d) { return *d = 0, 0; }
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int* v, int, int) { return *v = 256, 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int e) { return e ? "injected failure" : "no error"; }
int hipGetSymbolAddress(void** p, const void*) {
  static char symbol;
  return *p = &symbol, 0;
}
int hipMalloc(void** p, size_t n) { return mallocs++, *p = std::calloc(n, 1), 0; }
int hipFree(void* p) { return run_to(all()), std::free(p), 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::calloc(n, 1), 0; }
int hipHostFree(void* p) { return hipFree(p); }
int hipStreamCreate(void** s) { return *s = nullptr, 0; }
int hipStreamDestroy(void*) { return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { return run_to(all()), std::memcpy(d, s, n), 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { return queue.push_back({d, s, n}), 0; }
int hipStreamSynchronize(void*) {
  stream_waits++;
  if (fail_stream && --fail_stream == 0) return kError;
  return run_to(all()), 0;
}
int hipEventCreate(void** e) { return *e = new Event{0}, 0; }
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) { return delete static_cast<Event*>(e), 0; }
int hipEventRecord(void* e, void*) { return static_cast<Event*>(e)->after = all(), 0; }
int hipEventSynchronize(void* e) {
  if (fail_event && --fail_event == 0) return kError;
  return run_to(static_cast<Event*>(e)->after), 0;
}
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 0.f, 0; }
}
