// vb_staging.hpp -- pinned host blocks that a field passes through on its way to
// the caller's (pageable) memory.
//
// The x kernel that ends a field's inverse transform writes its rows straight
// into a pinned block, a chunk of planes per slot, and the chunks are copied on
// by a few host threads as their events complete, so the transfer, the copies
// and the page faults of a fresh destination overlap.  (A copy from device
// memory into pageable memory went through the runtime's own staging in 1 MB
// pieces on one thread.)  vb_get_phi, ms, once a block is there: 32^3 0.046 -> 0.036,
// 128^3 1.22 -> 0.75, 256^3 12.8 -> 3.3, 384^3 43.6 -> 10.3.
#pragma once
#include <cstddef>

#include "vb_hip.hpp"

namespace vb {

void staging_user(int d);   // +1 / -1: a solver was created / destroyed

// Copies a field of `items` items (planes) of item_bytes to dst.  produce(first,
// count, p) launches on st the kernels that write items [first, first + count)
// to pinned memory p.  Returns true when dst is complete, or false, with nothing
// launched, where there is no pinned block for it: none is idle, and a new one
// does not pay yet (staging_pays) or cannot be had.
// A call holds one block, of one of two slot sizes (fields of up to 2 MB take the
// small one, a single slot), on the current device.  Blocks are kept for reuse,
// at most two of each kind, and freed when the last solver goes.
struct StagingJob {
  virtual void produce(long long first, long long count, void* p) = 0;
  virtual ~StagingJob() = default;
};
bool staging_copy_out(StagingJob& job, long long items, size_t item_bytes, void* dst, hipStream_t st);

// A new block costs its allocation and the page faults of its first pass: 0.02 ms
// for a 32^3 field, 0.75 at 64^3, up to 2 at 96^3 and 128^3, 3.5 at 256 x 64 and
// 192^3 (much less where the runtime still has the memory of a freed one), where a
// read saves 0.01, 0.02, 0.13, 0.45, 2.0, 3.8.  So one is made when the reads since
// the first solver have come to about that: `before` bytes, and this one of `bytes`.
inline bool staging_pays(size_t before, size_t bytes) {
  return bytes <= (size_t)1 << 20 ? before > 0 : before + bytes >= (size_t)32 << 20;
}

}  // namespace vb
