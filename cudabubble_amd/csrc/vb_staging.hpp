// vb_staging.hpp -- pinned host blocks that a field passes through on its way to
// the caller's (pageable) memory.
//
// The x kernel that ends a field's inverse transform writes its rows straight
// into a pinned block, a chunk of planes per slot, and the chunks are copied on
// by a few host threads as their events complete, so the transfer, the copies
// and the page faults of a fresh destination overlap.  (A copy from device
// memory into pageable memory went through the runtime's own staging in 1 MB
// pieces on one thread.)  vb_get_phi, ms: 32^3 0.15 -> 0.04, 128^3 1.20 -> 0.75,
// 256^3 13.0 -> 3.3, 384^3 43.9 -> 10.7.
#pragma once
#include <cstddef>

#include "vb_host.hpp"

namespace vb {

struct Staging {
  static constexpr int kSlots = 8;
  unsigned char* mem = nullptr;   // pinned
  size_t slot = 0;                // bytes per slot
  int device = 0;                 // the events' device
  hipEvent_t ev[kSlots] = {};
};

// A block of one of two slot sizes (fields of up to 2 MB take the small one, a
// single slot) for the current device; held by the caller until released.
// Blocks are kept for reuse, at most two of each kind, and freed when the last
// solver goes.
Staging* staging_acquire(size_t field_bytes);
void staging_release(Staging* s);
void staging_user(int d);   // +1 / -1: a solver was created / destroyed

// Copies a field of `items` items (planes) of item_bytes to dst.  produce(first,
// count, p) launches on st the kernels that write items [first, first + count)
// to pinned memory p.  Returns when dst is complete.
struct StagingJob {
  virtual void produce(long long first, long long count, void* p) = 0;
  virtual ~StagingJob() = default;
};
void staging_copy_out(Staging* s, StagingJob& job, long long items, size_t item_bytes, void* dst, hipStream_t st);

}  // namespace vb
