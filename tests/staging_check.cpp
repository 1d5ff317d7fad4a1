// Host-only check of csrc/vb_staging.cpp: the HIP calls it makes are stood in for
// here by a stream that is a thread, so the chunks, the workers and the pool of
// blocks run without a GPU (and under the thread sanitizer).
#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <stdexcept>
#include <thread>
#include <vector>

#include "vb_staging.hpp"

// ---- the stand-ins -----------------------------------------------------------
struct Stream {
  std::mutex mu;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  long long pushed = 0, ran = 0;
  bool stop = false;
  std::thread th{[this] {
    for (;;) {
      std::function<void()> f;
      {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return stop || !q.empty(); });
        if (q.empty()) return;
        f = std::move(q.front());
        q.pop_front();
      }
      f();
      {
        std::lock_guard<std::mutex> l(mu);
        ++ran;
      }
      cv.notify_all();
    }
  }};
  void push(std::function<void()> f) {
    {
      std::lock_guard<std::mutex> l(mu);
      q.push_back(std::move(f));
      ++pushed;
    }
    cv.notify_all();
  }
  void wait(long long n) {
    std::unique_lock<std::mutex> l(mu);
    cv.wait(l, [&] { return ran >= n; });
  }
  ~Stream() {
    {
      std::lock_guard<std::mutex> l(mu);
      stop = true;
    }
    cv.notify_all();
    th.join();
  }
};
struct Event {
  Stream* s = nullptr;
  long long at = 0;
};
static std::atomic<int> g_blocks{0}, g_events{0}, g_mallocs{0};
static std::atomic<bool> g_no_pinned{false};

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ++g_mallocs;
  if (g_no_pinned) { *p = nullptr; return hipErrorOutOfMemory; }
  *p = std::malloc(n);
  ++g_blocks;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { std::free(p); --g_blocks; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new Event);
  ++g_events;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event*>(e); --g_events; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  Event* v = reinterpret_cast<Event*>(e);
  v->s = reinterpret_cast<Stream*>(st);
  std::lock_guard<std::mutex> l(v->s->mu);
  v->at = v->s->pushed;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  Event* v = reinterpret_cast<Event*>(e);
  v->s->wait(v->at);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
  Stream* s = reinterpret_cast<Stream*>(st);
  long long n;
  {
    std::lock_guard<std::mutex> l(s->mu);
    n = s->pushed;
  }
  s->wait(n);
  return hipSuccess;
}
}

// ---- the checks ----------------------------------------------------------------
#define CHECK(c)                                                       \
  do {                                                                 \
    if (!(c)) {                                                        \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);              \
      std::exit(1);                                                    \
    }                                                                  \
  } while (0)

static unsigned pattern(long long item, size_t i, unsigned seed) {
  return unsigned(item) * 2654435761u ^ unsigned(i) * 40503u ^ seed;
}

struct Fill final : vb::StagingJob {
  Stream& s;
  size_t item;
  unsigned seed;
  long long throw_at = -1;
  std::atomic<long long> calls{0};
  Fill(Stream& q, size_t b, unsigned k) : s(q), item(b), seed(k) {}
  void produce(long long first, long long count, void* p) override {
    if (throw_at >= 0 && calls == throw_at) throw std::runtime_error("launch");
    ++calls;
    const size_t b = item;
    const unsigned k = seed;
    s.push([=] {
      unsigned* o = static_cast<unsigned*>(p);
      for (long long i = 0; i < count; ++i)
        for (size_t j = 0; j < b / 4; ++j) o[(size_t)i * (b / 4) + j] = pattern(first + i, j, k);
    });
  }
};

// false: there was no block, and nothing was launched
static bool one(long long items, size_t item, unsigned seed) {
  Stream s;
  Fill f(s, item, seed);
  std::vector<unsigned> out((size_t)items * item / 4 + 1, 0xdeadbeefu);
  if (!vb::staging_copy_out(f, items, item, out.data(), reinterpret_cast<hipStream_t>(&s))) {
    CHECK(f.calls == 0 && out[0] == 0xdeadbeefu);
    return false;
  }
  for (long long i = 0; i < items; ++i)
    for (size_t j = 0; j < item / 4; ++j) CHECK(out[(size_t)i * (item / 4) + j] == pattern(i, j, seed));
  CHECK(out.back() == 0xdeadbeefu);
  return true;
}

// a first read large enough for blocks to pay from here on
static void warm() { CHECK(one(32, (size_t)1 << 20, 77)); }

// sizes: one slot, exactly one, just past it, ragged last chunks, more chunks
// than slots, one item per slot
static void sizes() {
  vb::staging_user(1);
  warm();
  const size_t M = (size_t)1 << 20;
  CHECK(one(1, 4096, 1));
  CHECK(one(16, 16 * 16 * 8, 2));
  CHECK(one(2, M, 3));
  CHECK(one(3, M, 4));
  CHECK(one(17, M, 5));
  CHECK(one(67, M / 2, 6));
  CHECK(one(41, 4 * M, 7));
  CHECK(one(13, 3 * M, 8));
  vb::staging_user(-1);
  CHECK(g_blocks == 0 && g_events == 0);
}

// readers in several threads, solvers coming and going meanwhile
static void threads() {
  std::vector<std::thread> th;
  for (int t = 0; t < 6; ++t)
    th.emplace_back([t] {
      for (int r = 0; r < 4; ++r) {
        vb::staging_user(1);
        (void)one(t % 2 ? 9 : 37, t % 2 ? 65536 : 262144, unsigned(16 * t + r));
        vb::staging_user(-1);
      }
    });
  for (auto& t : th) t.join();
  CHECK(g_blocks == 0 && g_events == 0);
}

// blocks are kept while a solver lives, at most two of a kind, then freed
static void pool() {
  vb::staging_user(1);
  warm();
  std::vector<std::thread> th;
  for (int t = 0; t < 5; ++t) th.emplace_back([t] { CHECK(one(37, 262144, unsigned(t))); });
  for (auto& t : th) t.join();
  CHECK(g_blocks <= 2);
  const int n = g_mallocs;
  CHECK(one(37, 262144, 9));
  CHECK(g_mallocs == n);
  vb::staging_user(-1);
  CHECK(g_blocks == 0);
}

static void launch_failure() {
  vb::staging_user(1);
  warm();
  for (long long at : {0, 1, 9}) {
    Stream s;
    Fill f(s, 262144, 3);
    f.throw_at = at;
    std::vector<unsigned> out((size_t)200 * 65536);
    bool threw = false;
    try {
      (void)vb::staging_copy_out(f, 200, 262144, out.data(), reinterpret_cast<hipStream_t>(&s));
    } catch (const std::runtime_error&) {
      threw = true;
    }
    CHECK(threw);
  }
  CHECK(one(37, 262144, 5));
  vb::staging_user(-1);
  CHECK(g_blocks == 0 && g_events == 0);
}

// no pinned memory: nothing is launched, the caller goes its own way
static void no_pinned() {
  vb::staging_user(1);
  g_no_pinned = true;
  for (long long items : {4, 200}) {
    Stream s;
    Fill f(s, 262144, 3);
    std::vector<unsigned> out((size_t)items * 65536, 7u);
    CHECK(!vb::staging_copy_out(f, items, 262144, out.data(), reinterpret_cast<hipStream_t>(&s)));
    CHECK(f.calls == 0 && out[0] == 7u && out.back() == 7u);
  }
  g_no_pinned = false;
  CHECK(one(37, 262144, 5));
  vb::staging_user(-1);
  CHECK(g_blocks == 0 && g_events == 0);
}

// a block is made when it pays, over all solvers there are; an idle one serves
// every reader
static void make() {
  const size_t M = (size_t)1 << 20;
  vb::staging_user(1);
  CHECK(!one(16, M / 64, 1) && g_mallocs == 0);   // 256 KB: the first read
  CHECK(one(16, M / 64, 1) && g_mallocs == 1);    // and the second
  CHECK(one(16, M / 8, 2) && g_mallocs == 1);     // 2 MB: the idle one
  CHECK(!one(40, M / 8, 3) && g_mallocs == 1);    // the other kind
  vb::staging_user(1);
  CHECK(one(32, M, 3) && g_mallocs == 2);
  CHECK(one(40, M / 8, 3) && g_mallocs == 2);
  vb::staging_user(-1);
  CHECK(g_blocks == 2);
  vb::staging_user(-1);
  CHECK(g_blocks == 0);
  vb::staging_user(1);   // counted from the first solver again
  CHECK(!one(40, M / 8, 3) && g_mallocs == 2);
  vb::staging_user(-1);
  CHECK(!vb::staging_pays(0, M / 4) && vb::staging_pays(M / 4, M / 4));
  CHECK(!vb::staging_pays(0, 2 * M) && !vb::staging_pays(28 * M, 2 * M) && vb::staging_pays(30 * M, 2 * M));
  CHECK(!vb::staging_pays(0, 16 * M) && vb::staging_pays(16 * M, 16 * M) && vb::staging_pays(0, 54 * M));
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "sizes") sizes();
  else if (what == "threads") threads();
  else if (what == "pool") pool();
  else if (what == "launch_failure") launch_failure();
  else if (what == "no_pinned") no_pinned();
  else if (what == "make") make();
  else return 2;
  std::printf("ok\n");
  return 0;
}
