// vb_staging.cpp -- see vb_staging.hpp.
#include "vb_staging.hpp"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace vb {

namespace {
struct Block {
  static constexpr int kSlots = 8;
  unsigned char* mem = nullptr;   // pinned
  size_t slot = 0;                // bytes per slot
  int device = 0;                 // the events' device
  hipEvent_t ev[kSlots] = {};
};

constexpr size_t kSmall = (size_t)2 << 20, kLarge = (size_t)4 << 20;   // slot bytes
constexpr int kThreads = 6, kKeep = 2;

std::mutex g_mu;
std::vector<Block*> g_idle;
int g_users = 0;
size_t g_read = 0;   // bytes that copies were asked for since the first solver

void destroy(Block* s) {
  for (auto e : s->ev)
    if (e) (void)hipEventDestroy(e);
  if (s->mem) (void)hipHostFree(s->mem);
  delete s;
}

// a block for a field of that size, nullptr where there is none to be had
Block* acquire(size_t field_bytes) {
  const size_t slot = field_bytes <= kSmall ? kSmall : kLarge;
  int dev = 0;
  VB_HIP(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> l(g_mu);
    for (size_t i = 0; i < g_idle.size(); ++i)
      if (g_idle[i]->slot == slot && g_idle[i]->device == dev) {
        Block* s = g_idle[i];
        g_idle.erase(g_idle.begin() + (long)i);
        g_read += field_bytes;
        return s;
      }
    const bool pays = staging_pays(g_read, field_bytes);
    g_read += field_bytes;
    if (!pays) return nullptr;
  }
  Block* s = new Block;
  s->slot = slot;
  s->device = dev;
  hipError_t e = hipHostMalloc((void**)&s->mem, slot == kSmall ? slot : slot * Block::kSlots, hipHostMallocDefault);
  if (e != hipSuccess) s->mem = nullptr;
  for (auto& v : s->ev)
    if (e == hipSuccess && (e = hipEventCreateWithFlags(&v, hipEventDisableTiming)) != hipSuccess) v = nullptr;
  if (e == hipSuccess) return s;
  (void)hipGetLastError();   // not the next call's error
  destroy(s);
  return nullptr;
}

void release(Block* s) {
  {
    std::lock_guard<std::mutex> l(g_mu);
    int same = 0;
    for (auto* i : g_idle) same += i->slot == s->slot && i->device == s->device;
    if (g_users > 0 && same < kKeep) {
      try {
        g_idle.push_back(s);
        return;
      } catch (const std::bad_alloc&) {
      }
    }
  }
  destroy(s);
}

void copy_out(Block* s, StagingJob& job, long long items, size_t item_bytes, void* dst, hipStream_t st);
}  // namespace

void staging_user(int d) {
  std::vector<Block*> drop;
  {
    std::lock_guard<std::mutex> l(g_mu);
    g_users += d;
    if (g_users <= 0) {
      drop.swap(g_idle);
      g_read = 0;
    }
  }
  for (auto* s : drop) destroy(s);
}

bool staging_copy_out(StagingJob& job, long long items, size_t item_bytes, void* dst, hipStream_t st) {
  Block* const s = acquire((size_t)items * item_bytes);
  if (!s) return false;
  try {
    copy_out(s, job, items, item_bytes, dst, st);
  } catch (...) {
    (void)hipStreamSynchronize(st);   // the kernels launched write to the block
    release(s);
    throw;
  }
  release(s);
  return true;
}

namespace {
void copy_out(Block* s, StagingJob& job, long long items, size_t item_bytes, void* dst, hipStream_t st) {
  const long long per = std::max<long long>(1, (long long)(s->slot / item_bytes));
  const long long chunks = (items + per - 1) / per;
  unsigned char* const out = static_cast<unsigned char*>(dst);
  auto count = [&](long long c) { return std::min(per, items - c * per); };
  auto copy = [&](long long c) {
    std::memcpy(out + (size_t)(c * per) * item_bytes, s->mem + (size_t)(c % Block::kSlots) * s->slot,
                (size_t)count(c) * item_bytes);
  };
  if (chunks == 1) {
    job.produce(0, items, s->mem);
    VB_HIP(hipStreamSynchronize(st));
    copy(0);
    return;
  }
  // This thread launches and waits for the events in order; the workers copy
  // the chunks it has seen complete and free their slots.
  std::mutex mu;
  std::condition_variable cv;
  long long ready = 0, next = 0;
  bool stop = false;
  std::vector<char> done((size_t)chunks, 0);
  auto work = [&] {
    for (;;) {
      long long c;
      {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return stop || next < ready; });
        if (next >= ready) return;   // stop, nothing left
        c = next++;
      }
      copy(c);
      {
        std::lock_guard<std::mutex> l(mu);
        done[(size_t)c] = 1;
      }
      cv.notify_all();
    }
  };
  std::vector<std::thread> th;
  th.reserve(kThreads);
  try {
    for (int i = 0; i < kThreads && i < chunks; ++i) th.emplace_back(work);
  } catch (const std::system_error&) {
    // fewer workers, or none: this thread copies then
  }
  auto join = [&] {
    {
      std::lock_guard<std::mutex> l(mu);
      stop = true;
    }
    cv.notify_all();
    for (auto& t : th) t.join();
  };
  try {
    long long issued = 0;
    for (long long c = 0; c < chunks; ++c) {
      for (; issued < chunks && issued < c + Block::kSlots; ++issued) {
        if (issued >= Block::kSlots) {
          std::unique_lock<std::mutex> l(mu);
          const size_t prev = (size_t)(issued - Block::kSlots);
          // the slot's last chunk: wait for it only where nothing else is in flight
          if (!done[prev] && issued > c) break;
          cv.wait(l, [&] { return done[prev] != 0; });
        }
        job.produce(issued * per, count(issued), s->mem + (size_t)(issued % Block::kSlots) * s->slot);
        VB_HIP(hipEventRecord(s->ev[issued % Block::kSlots], st));
      }
      VB_HIP(hipEventSynchronize(s->ev[c % Block::kSlots]));
      if (th.empty()) {
        copy(c);
        done[(size_t)c] = 1;
        continue;
      }
      {
        std::lock_guard<std::mutex> l(mu);
        ready = c + 1;
      }
      cv.notify_all();
    }
  } catch (...) {
    join();
    throw;
  }
  join();   // the workers finish what is ready
}
}  // namespace

}  // namespace vb
