// The few runtime calls host_mem.h makes, on host memory, for a CPU test.  What
// a stream is given runs as late as it may: when the host waits for it (or for
// an event recorded after it) or frees memory.  A missing wait, a staging
// buffer reused too early or an array written after its call has returned
// therefore shows every time.
#pragma once
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>

typedef int hipError_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2, hipMemcpyDeviceToDevice = 3 };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };

namespace fake {
struct Stream {
  std::deque<std::function<void()>> ops;
  long long issued = 0, done = 0;
  void run(long long upto) {
    while (done < upto && !ops.empty()) {
      ops.front()();
      ops.pop_front();
      ++done;
    }
  }
};
struct Event {
  Stream *s = nullptr;
  long long at = 0;
};
struct State {
  std::recursive_mutex mu;
  std::map<void *, size_t> mem;
  std::vector<Stream *> streams;
  size_t live = 0, limit = (size_t)-1;
  int mallocs = 0, frees = 0, fail_copies = 0;  // fail_copies: the next n copies fail
};
inline State &st() {
  static State s;
  return s;
}
using Lock = std::lock_guard<std::recursive_mutex>;
}  // namespace fake
typedef fake::Stream *hipStream_t;
typedef fake::Event *hipEvent_t;

inline const char *hipGetErrorString(hipError_t) { return "fake error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipStreamCreate(hipStream_t *s) {
  fake::Lock l(fake::st().mu);
  *s = new fake::Stream;
  fake::st().streams.push_back(*s);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  fake::Lock l(fake::st().mu);
  if (s) s->run(s->issued);
  return hipSuccess;
}
inline hipError_t hipDeviceSynchronize() {
  fake::Lock l(fake::st().mu);
  for (hipStream_t s : fake::st().streams) s->run(s->issued);
  return hipSuccess;
}
inline hipError_t enqueue(hipStream_t s, std::function<void()> f) {
  fake::Lock l(fake::st().mu);
  if (!s) f();
  else s->ops.push_back(f), ++s->issued;
  return hipSuccess;
}
inline hipError_t hipMalloc(void **p, size_t n) {
  fake::Lock l(fake::st().mu);
  fake::State &t = fake::st();
  if (t.live + n > t.limit) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  std::memset(*p, 0xa5, n);  // never zero by itself
  t.mem[*p] = n;
  t.live += n;
  ++t.mallocs;
  return hipSuccess;
}
inline hipError_t hipFree(void *p) {
  fake::Lock l(fake::st().mu);
  hipDeviceSynchronize();
  fake::State &t = fake::st();
  if (!t.mem.count(p)) std::abort();
  t.live -= t.mem[p];
  t.mem.erase(p);
  ++t.frees;
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = new fake::Event;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  fake::Lock l(fake::st().mu);
  e->s = s;
  e->at = s->issued;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  fake::Lock l(fake::st().mu);
  if (e->s) e->s->run(e->at);
  return hipSuccess;
}
inline hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t s) {
  return enqueue(s, [=] { std::memset(p, v, n); });
}
inline hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *a, size_t ap, size_t w, size_t h, hipMemcpyKind,
                                   hipStream_t s) {
  {
    fake::Lock l(fake::st().mu);
    if (fake::st().fail_copies > 0) {
      --fake::st().fail_copies;
      return hipErrorUnknown;
    }
  }
  return enqueue(s, [=] {
    for (size_t r = 0; r < h; ++r) std::memcpy((char *)d + r * dp, (const char *)a + r * ap, w);
  });
}
inline hipError_t hipMemcpyAsync(void *d, const void *a, size_t n, hipMemcpyKind k, hipStream_t s) {
  return hipMemcpy2DAsync(d, n, a, n, n, 1, k, s);
}
