// Checks of csrc/host_mem.h on the CPU (hip/hip_runtime.h beside this file
// stands in for the runtime).  argv[1] names the check; 0 on success.
#include <cstdio>
#include <random>
#include <thread>

#include "host_mem.h"

#define CHECK(x)                                                        \
  do {                                                                  \
    if (!(x)) {                                                         \
      std::printf("line %d: %s\n", __LINE__, #x);                       \
      return 1;                                                         \
    }                                                                   \
  } while (0)

namespace {

using Bytes = std::vector<unsigned char>;
Bytes noise(size_t n, unsigned seed) {
  std::mt19937 g(seed);
  Bytes b(n);
  for (auto &x : b) x = (unsigned char)g();
  return b;
}

// rows of `row` bytes up to a device array of that pitch and down again
bool round_trip(Stager &st, hipStream_t s, size_t row, size_t rows, size_t pitch, unsigned seed) {
  const Bytes a = noise(row * rows, seed);
  Bytes b(row * rows, 1), src = a;
  Bytes dev(pitch * rows);
  st.h2d(s, dev.data(), pitch, src.data(), row, rows);
  std::fill(src.begin(), src.end(), 0);  // read when h2d returns
  st.d2h(s, b.data(), dev.data(), pitch, row, rows);
  st.flush(s);
  return a == b;
}

int ring() {
  hipStream_t s;
  hipStreamCreate(&s);
  Stager st;
  st.flush(s);  // nothing yet
  constexpr size_t S = Stager::kStage;
  unsigned seed = 1;
  for (size_t n : {(size_t)1, (size_t)255, (size_t)256, (size_t)257, S / 2 - 1, S / 2, S / 2 + 1, S, S + 8,
                   S * Stager::kSlots, S * Stager::kSlots + 3, 3 * S * Stager::kSlots + 11})
    CHECK(round_trip(st, s, n, 1, n, seed++));
  // pitched: rows of a piece, rows longer than half a buffer
  for (size_t row : {(size_t)8, (size_t)1000, S / 3, S / 2, S / 2 + 1, S + 40})
    for (size_t rows : {(size_t)1, (size_t)2, (size_t)7}) CHECK(round_trip(st, s, row, rows, row + 24, seed++));
  CHECK(round_trip(st, s, 24, 200000, 32, seed++));
  CHECK(round_trip(st, s, 0, 5, 8, seed++));
  // a later download of the same array wins
  Bytes d1 = noise(5000, 90), d2 = noise(5000, 91), out(5000);
  st.d2h(s, out.data(), d1.data(), 5000, 5000, 1);
  st.d2h(s, out.data(), d2.data(), 5000, 5000, 1);
  st.flush(s);
  CHECK(out == d2);
  return 0;
}

// after an error nothing more is written to the arrays of the call, and the
// ring goes on
int drop() {
  hipStream_t s;
  hipStreamCreate(&s);
  Stager st;
  const Bytes dev = noise(3 * Stager::kStage, 5);
  Bytes out(dev.size(), 7);
  st.d2h(s, out.data(), dev.data(), dev.size(), dev.size(), 1);
  const Bytes seen = out;
  bool threw = false;
  try {
    fake::st().fail_copies = 1;
    st.d2h(s, out.data(), dev.data(), 100, 100, 1);
  } catch (const Err &) {
    threw = true;
  }
  CHECK(threw);
  st.drop();
  for (unsigned k = 0; k < 20; ++k) CHECK(round_trip(st, s, Stager::kStage, 1, Stager::kStage, k));
  CHECK(out == seen);
  return 0;
}

// a call of another thread on the same context that ends on an error does not
// take this one's pending downloads with it
int drop_of_another_thread() {
  hipStream_t s;
  hipStreamCreate(&s);
  Stager st;
  const Bytes dev = noise(100000, 5), dev2 = noise(70000, 6);
  Bytes out(dev.size()), out2(dev2.size(), 7);
  st.d2h(s, out.data(), dev.data(), dev.size(), dev.size(), 1);
  std::thread([&] {
    st.d2h(s, out2.data(), dev2.data(), dev2.size(), dev2.size(), 1);
    st.drop();
  }).join();
  st.flush(s);
  CHECK(out == dev);
  CHECK(out2 == Bytes(dev2.size(), 7));
  return 0;
}

// calls of several threads on one context
int threads() {
  hipStream_t s;
  hipStreamCreate(&s);
  Stager st;
  std::atomic<int> bad{0};
  std::vector<std::thread> ts;
  for (unsigned q = 0; q < 4; ++q)
    ts.emplace_back([&, q] {
      std::mt19937 g(q);
      for (unsigned k = 0; k < 60; ++k) {
        const size_t row = 1 + g() % 50000, rows = 1 + g() % 20;
        if (!round_trip(st, s, row, rows, row + g() % 2 * 8, 100 * q + k)) ++bad;
      }
    });
  for (auto &t : ts) t.join();
  CHECK(bad == 0);
  return 0;
}

Pool new_pool() {
  hipStream_t s;
  hipStreamCreate(&s);
  return Pool{std::make_shared<DevPool>(s)};
}
bool zero(const DBuf<char> &b) {
  return std::all_of(b.p, b.p + b.n, [](char c) { return c == 0; });
}

// kept blocks are handed out again, zeroed, in the order of the stream
int reuse() {
  const Pool pool = new_pool();
  DBuf<char> a, b;
  a.alloc(pool, 10000);
  hipStreamSynchronize(pool->stream());
  CHECK(zero(a));
  hipMemsetAsync(a.p, 1, a.n, pool->stream());
  const char *was = a.p;
  a.release();
  CHECK(pool->kept() == 12288 && fake::st().live == 12288);
  b.alloc(pool, 13000);  // does not fit
  CHECK(b.p != was);
  a.alloc(pool, 9000);   // within a quarter
  CHECK(a.p == was && pool->kept() == 0);
  hipStreamSynchronize(pool->stream());
  CHECK(zero(a) && zero(b));
  return 0;
}

// at most limit() bytes are kept, the oldest go first, a limit of 0 gives all back
int limit() {
  const Pool pool = new_pool();
  pool->set_limit(5 << 20);
  DBuf<char> b[4];
  const char *last = nullptr;
  for (int k = 0; k < 4; ++k) b[k].alloc(pool, (size_t)(k + 1) << 20);
  for (auto &x : b) last = x.p, x.release();  // 1 + 2 MiB, then 3, then 4: the older ones go
  CHECK(pool->kept() == (4 << 20) && fake::st().live == (4 << 20));
  b[0].alloc(pool, 4 << 20);
  CHECK(b[0].p == last);
  b[1].alloc(pool, 6 << 20);  // more than the limit: straight back
  b[1].release();
  CHECK(pool->kept() == 0 && fake::st().live == (4 << 20));
  b[0].release();
  pool->set_limit(0);
  CHECK(pool->kept() == 0 && fake::st().live == 0);
  b[0].alloc(pool, 100);
  b[0].release();
  CHECK(fake::st().live == 0);
  return 0;
}

// what the caller owns goes back to the driver
int given_back() {
  const Pool pool = new_pool();
  DBuf<char> kept, own;
  kept.alloc(pool, 1 << 20);
  kept.release();
  own.alloc(pool.given_back(), 1 << 20);
  CHECK(pool->kept() == (1 << 20) && fake::st().live == (2 << 20));
  hipStreamSynchronize(pool->stream());
  CHECK(zero(own));
  own.release();
  CHECK(pool->kept() == (1 << 20) && fake::st().live == (1 << 20));
  return 0;
}

// when the driver has no more, every context gives back what it keeps
int out_of_memory() {
  const Pool mine = new_pool(), other = new_pool();
  DBuf<char> a, b;
  for (const Pool &p : {mine, other}) {
    a.alloc(p, 3 << 20);
    a.release();
  }
  fake::st().limit = 7 << 20;
  b.alloc(mine, 5 << 20);
  CHECK(mine->kept() == 0 && other->kept() == 0 && fake::st().live == (5 << 20));
  b.release();
  bool threw = false;
  try {
    a.alloc(other.given_back(), 8 << 20);
  } catch (const Err &) {
    threw = true;
  }
  CHECK(threw && fake::st().live == 0);
  return 0;
}

// buffers that outlive the context
int closed() {
  Pool pool = new_pool();
  DBuf<char> a, b;
  a.alloc(pool, 5000);
  b.alloc(pool, 5000);
  a.release();
  pool->close();
  CHECK(pool->kept() == 0 && fake::st().live == 8192);
  a.alloc(pool, 3000);
  CHECK(zero(a));  // nothing to wait for
  pool = Pool{};
  a.release();
  b.release();
  CHECK(fake::st().live == 0);
  return 0;
}

// allocations of several threads and contexts, with less memory than they want to keep
int pool_threads() {
  const Pool pools[2] = {new_pool(), new_pool()};
  fake::st().limit = 15 << 20;  // 4 x (1.25 x 2 + 1) MiB in use at most
  std::atomic<int> bad{0};
  std::vector<std::thread> ts;
  for (unsigned q = 0; q < 4; ++q)
    ts.emplace_back([&, q] {
      std::mt19937 g(q);
      const Pool &pool = pools[q & 1];
      for (int k = 0; k < 200; ++k) {
        DBuf<char> a, b;
        a.alloc(pool, 1 + g() % (2 << 20));
        b.alloc(pool.given_back(), 1 + g() % (1 << 20));
        hipStreamSynchronize(pool->stream());
        if (!zero(a) || !zero(b)) ++bad;
        std::fill(a.p, a.p + a.n, (char)1);
      }
    });
  for (auto &t : ts) t.join();
  CHECK(bad == 0);
  return 0;
}

}  // namespace

int main(int, char **argv) {
  const std::string w = argv[1];
  if (w == "ring") return ring();
  if (w == "drop") return drop();
  if (w == "drop_of_another_thread") return drop_of_another_thread();
  if (w == "threads") return threads();
  if (w == "reuse") return reuse();
  if (w == "limit") return limit();
  if (w == "given_back") return given_back();
  if (w == "out_of_memory") return out_of_memory();
  if (w == "closed") return closed();
  if (w == "pool_threads") return pool_threads();
  return 2;
}
