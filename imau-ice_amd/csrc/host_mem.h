// host_mem.h -- device memory and host copies of a context: the pool its
// buffers come from (DevPool, DBuf) and the pinned ring through which the
// caller's arrays travel (Stager).  Host code only.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/imau_vel.h"

namespace {

struct Err {
  int code;
  std::string msg;
};

#define HIPCHK(x)                                                                          \
  do {                                                                                     \
    hipError_t e_ = (x);                                                                   \
    if (e_ != hipSuccess) throw Err{IMAU_ERR_DEVICE, std::string(#x ": ") + hipGetErrorString(e_)}; \
  } while (0)

[[noreturn]] void fail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  throw Err{code, buf};
}

// Device memory of one context.  A call on host arrays needs some sixty
// buffers; asking the driver for each (hipMalloc, a synchronising clear,
// hipFree) cost more than the call's kernels: an explicit thickness update of
// 281 x 281 cells, 50 us of kernels, took 5.2 ms, now 0.48 ms.  So the blocks of
// such calls are kept and handed out again, at most limit() bytes of them (by
// default kKeep, the buffers of a DIVA problem of about 1000 x 1000 cells; the
// oldest go back to the driver first).  When the driver has no more, every
// context of the process gives back what it keeps before that is an error.
// Problems and plans that the caller owns come from the driver and go back to it
// when they are destroyed (Pool::keep false): a 726 x 426 problem holds 1.1 GB;
// it is created and destroyed in 11.0 + 2.4 ms, with kept blocks in 10.7 (twelve
// of 305 x 305, 3.9 GB: 92 + 3.3 against 37.5 ms).
// Contents are cleared on the context's stream, which also orders a block's new
// use after its last one; an owner whose buffers other streams may read
// synchronises the device before it lets them go (problem and plan destruction).
// Buffers may outlive the context: they hold the pool, and once it is closed
// their blocks go straight back to the driver.
class DevPool {
 public:
  static constexpr size_t kKeep = (size_t)4 << 30;
  explicit DevPool(hipStream_t s) : s_(s) {
    std::lock_guard<std::mutex> lock(open_pools().mu);
    open_pools().all.push_back(this);
  }
  ~DevPool() { close(); }
  // cap: the size of the block, to be handed back to put(); keep: from the kept
  // blocks if one fits
  void *get(size_t bytes, size_t &cap, bool keep) {
    cap = (bytes + kGrain - 1) / kGrain * kGrain;
    void *p = nullptr;
    if (keep) {
      std::lock_guard<std::mutex> lock(mu_);
      // the smallest kept block that holds it without wasting over a quarter
      size_t best = kept_.size();
      for (size_t q = 0; q < kept_.size(); ++q)
        if (kept_[q].cap >= cap && kept_[q].cap <= cap + cap / 4 &&
            (best == kept_.size() || kept_[q].cap < kept_[best].cap))
          best = q;
      if (best < kept_.size()) {
        p = kept_[best].p;
        cap = kept_[best].cap;
        total_ -= cap;
        kept_.erase(kept_.begin() + best);
      }
    }
    if (!p && hipMalloc(&p, cap) != hipSuccess) {
      (void)hipGetLastError();
      Scarce scarce;  // no thread keeps a block until the second try is over
      trim_all();
      HIPCHK(hipMalloc(&p, cap));
    }
    hipError_t e = hipMemsetAsync(p, 0, bytes, stream());
    if (e == hipSuccess && !stream()) e = hipDeviceSynchronize();  // closed: no stream orders what follows
    if (e != hipSuccess) put(p, cap, keep);
    HIPCHK(e);
    return p;
  }
  // the context's stream; null (the null stream) once the pool is closed
  hipStream_t stream() const { return s_.load(); }
  void put(void *p, size_t cap, bool keep) noexcept {
    if (keep) {
      std::lock_guard<std::mutex> lock(mu_);
      if (open_ && cap <= limit_ && open_pools().scarce == 0) try {
        kept_.push_back(Block{p, cap});
        total_ += cap;
        p = nullptr;
      } catch (const std::bad_alloc &) {
      }
    }
    if (p) (void)hipFree(p);
    trim(limit());
  }
  size_t limit() {
    std::lock_guard<std::mutex> lock(mu_);
    return limit_;
  }
  void set_limit(size_t most) {
    {
      std::lock_guard<std::mutex> lock(mu_);
      limit_ = most;
    }
    trim(most);
  }
  size_t kept() {
    std::lock_guard<std::mutex> lock(mu_);
    return total_;
  }
  void close() {
    {
      std::lock_guard<std::mutex> lock(open_pools().mu);
      std::vector<DevPool *> &all = open_pools().all;
      all.erase(std::remove(all.begin(), all.end(), this), all.end());
    }
    {
      std::lock_guard<std::mutex> lock(mu_);
      open_ = false;
      s_ = nullptr;
    }
    trim(0);
  }

 private:
  struct Block {
    void *p;
    size_t cap;
  };
  static constexpr size_t kGrain = 4096;
  struct OpenPools {
    std::mutex mu;  // taken before a pool's own
    std::vector<DevPool *> all;
    std::atomic<int> scarce{0};
  };
  static OpenPools &open_pools() {
    static OpenPools *p = new OpenPools;  // outlives every static object that may still hold a pool
    return *p;
  }
  struct Scarce {
    Scarce() { ++open_pools().scarce; }
    ~Scarce() { --open_pools().scarce; }
  };
  static void trim_all() {
    std::lock_guard<std::mutex> lock(open_pools().mu);
    for (DevPool *p : open_pools().all) p->trim(0);
  }
  void trim(size_t most) noexcept {
    for (;;) {
      void *p;
      {
        std::lock_guard<std::mutex> lock(mu_);
        if (total_ <= most) return;
        p = kept_.front().p;
        total_ -= kept_.front().cap;
        kept_.erase(kept_.begin());
      }
      (void)hipFree(p);
    }
  }
  std::atomic<hipStream_t> s_;
  std::mutex mu_;
  std::vector<Block> kept_;  // oldest first
  size_t total_ = 0, limit_ = kKeep;
  bool open_ = true;
};

// a context's pool, and whether what is allocated through this handle is kept
// in it afterwards
struct Pool {
  std::shared_ptr<DevPool> pool;
  bool keep = true;
  DevPool *operator->() const { return pool.get(); }
  explicit operator bool() const { return (bool)pool; }
  Pool given_back() const { return Pool{pool, false}; }
};

// a zeroed device array; the zeroing is ordered on the context's stream, as is
// everything that fills or reads it
template <class T>
struct DBuf {
  T *p = nullptr;
  size_t n = 0;
  void alloc(const Pool &pool, size_t count) {
    release();
    n = count;
    if (count) {
      p = static_cast<T *>(pool->get(count * sizeof(T), cap_, pool.keep));
      pool_ = pool;
    }
  }
  void release() {
    if (p) pool_->put(p, cap_, pool_.keep);
    p = nullptr;
    n = 0;
    pool_ = Pool{};
  }
  DBuf() = default;
  DBuf(const DBuf &) = delete;
  DBuf &operator=(const DBuf &) = delete;
  ~DBuf() { release(); }

 private:
  Pool pool_;
  size_t cap_ = 0;
};

// a copy from pageable host memory on the stream, complete on return
void h2d(hipStream_t s, void *dst, const void *src, size_t bytes) {
  HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
  HIPCHK(hipStreamSynchronize(s));
}

// Copies between the caller's (pageable) arrays and the device, through a ring
// of kSlots pinned buffers of kStage bytes: the host fills or empties one while
// others are in flight.  The runtime's own pageable path pins every array for
// its copy: the 66 MB of the producers at 281 x 281 x 15 cells took 85 ms, now
// 4 ms.  h2d() has read its source when it returns; what d2h() asks for is in
// the caller's arrays after flush().
// Several threads may be inside calls on one context: the ring is locked for one
// piece at a time, a flush completes the downloads of all of them (none has
// returned, so their arrays are there), and an error drops its own thread's only.
class Stager {
 public:
  static constexpr size_t kStage = (size_t)2 << 20;
  static constexpr int kSlots = 8;
  ~Stager() {
    for (Slot &h : slot_) {
      if (h.ev) (void)hipEventDestroy(h.ev);
      if (h.p) (void)hipHostFree(h.p);
    }
  }
  // `rows` rows of `row` bytes, contiguous on the host, `pitch` apart on the device
  void h2d(hipStream_t s, void *dst, size_t pitch, const void *src, size_t row, size_t rows) {
    pieces(s, (char *)dst, pitch, (char *)const_cast<void *>(src), row, rows, true);
  }
  void d2h(hipStream_t s, void *dst, const void *src, size_t pitch, size_t row, size_t rows) {
    pieces(s, (char *)const_cast<void *>(src), pitch, (char *)dst, row, rows, false);
  }
  // small device array into dst, complete on return
  void fetch(hipStream_t s, void *dst, const void *src, size_t bytes) {
    d2h(s, dst, src, bytes, bytes, 1);
    flush(s);
  }
  void flush(hipStream_t s) {
    std::lock_guard<std::mutex> lock(mu_);
    if (!slot_[0].p) return;
    rotate(s);
    for (int k = 0; k < kSlots; ++k) reclaim((cur_ + k) % kSlots);  // oldest first
  }
  // forget this thread's downloads that an error left unfinished: their arrays
  // may be gone.  What is in flight to the ring's own buffers may go on.
  void drop() {
    std::lock_guard<std::mutex> lock(mu_);
    const std::thread::id me = std::this_thread::get_id();
    for (Slot &h : slot_)
      h.out.erase(std::remove_if(h.out.begin(), h.out.end(), [&](const Out &o) { return o.by == me; }), h.out.end());
  }

 private:
  struct Out {
    size_t at, bytes;
    char *dst;
    std::thread::id by;
  };
  struct Slot {
    char *p = nullptr;
    hipEvent_t ev = nullptr;
    size_t used = 0;
    bool busy = false;      // ev marks the end of copies from or into it
    std::vector<Out> out;   // downloads in it
  };
  Slot slot_[kSlots];
  int cur_ = 0;
  std::mutex mu_;

  // with the lock held: create, reclaim, rotate, take
  void create() {
    if (slot_[kSlots - 1].ev) return;
    for (Slot &h : slot_) {
      if (!h.p) HIPCHK(hipHostMalloc((void **)&h.p, kStage, hipHostMallocDefault));
      if (!h.ev) HIPCHK(hipEventCreateWithFlags(&h.ev, hipEventDisableTiming));
    }
  }
  void reclaim(int b) {
    Slot &h = slot_[b];
    if (h.busy) HIPCHK(hipEventSynchronize(h.ev));
    h.busy = false;
    for (const Out &o : h.out) std::memcpy(o.dst, h.p + o.at, o.bytes);
    h.out.clear();
    h.used = 0;
  }
  // the slot in use is complete: go on with the next one
  void rotate(hipStream_t s) {
    Slot &h = slot_[cur_];
    if (h.used) {
      HIPCHK(hipEventRecord(h.ev, s));
      h.busy = true;
    }
    cur_ = (cur_ + 1) % kSlots;
    reclaim(cur_);
  }
  char *take(hipStream_t s, size_t bytes) {
    if (slot_[cur_].used + bytes > kStage) rotate(s);
    Slot &h = slot_[cur_];
    char *p = h.p + h.used;
    h.used += (bytes + 255) / 256 * 256;
    return p;
  }
  void pieces(hipStream_t s, char *dev, size_t pitch, char *host, size_t row, size_t rows, bool up) {
    if (!row || !rows) return;
    if (pitch == row) {  // one long row
      row *= rows;
      pitch = row;
      rows = 1;
    }
    // whole rows at a time, or parts of a row longer than half a slot
    constexpr size_t kPiece = kStage / 2;
    if (row > kPiece) {
      for (size_t r = 0; r < rows; ++r)
        for (size_t a = 0; a < row; a += kPiece)
          piece(s, dev + r * pitch + a, pitch, host + r * row + a, std::min(kPiece, row - a), 1, up);
      return;
    }
    const size_t most = kPiece / row;
    for (size_t r = 0; r < rows; r += most)
      piece(s, dev + r * pitch, pitch, host + r * row, row, std::min(most, rows - r), up);
  }
  void piece(hipStream_t s, char *dev, size_t pitch, char *host, size_t row, size_t rows, bool up) {
    const size_t bytes = row * rows;
    std::lock_guard<std::mutex> lock(mu_);
    create();
    char *p = take(s, bytes);
    if (up) std::memcpy(p, host, bytes);
    if (rows == 1)
      HIPCHK(hipMemcpyAsync(up ? dev : p, up ? p : dev, bytes, up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, s));
    else if (up)
      HIPCHK(hipMemcpy2DAsync(dev, pitch, p, row, row, rows, hipMemcpyHostToDevice, s));
    else
      HIPCHK(hipMemcpy2DAsync(p, row, dev, pitch, row, rows, hipMemcpyDeviceToHost, s));
    if (!up) {
      Slot &h = slot_[cur_];
      h.out.push_back(Out{(size_t)(p - h.p), bytes, host, std::this_thread::get_id()});
    }
  }
};

}  // namespace
