// Library-wide runtime state: the stream used by the drop-in calls and
// device workspaces reused across calls.
#pragma once

#include "mitos_common.h"

namespace mitos {

// Stream of the drop-in (reference-named) entry points.  Every drop-in call
// is host-synchronous, as the reference's CPU functions are.
hipStream_t api_stream();
int api_sync();

// Per-device scratch buffer of at least `bytes`, grown on demand and kept
// until mitos_release_workspace().  Where there is no room, cached free blocks (below)
// go first.
void* workspace(int slot, size_t bytes);

// Held from workspace() to the last launch that uses the block (recursive).  The calls
// of all host threads issue on one stream per device, so what one thread issued under
// the lock is done before another's launches touch the block, and workspace() waits
// for the device before it frees.  Transforms, k-space tables, Poisson and the CIC
// deposit take it: calls of several threads on a device do not disturb each other.
class ScratchLock {
  public:
    ScratchLock();
    ~ScratchLock();
    ScratchLock(const ScratchLock&) = delete;
};
// Slots that are in use only under the lock; an allocation of the library that finds no
// room takes their memory back.
enum { SLOT_FFT = 0, SLOT_APPLY_TABLE = 9, SLOT_CIC_SORT = 10 };

// Device blocks of the drop-in grids and temporaries, cached by exact size:
// pool_free keeps a block for the next pool_alloc of that size on the same
// device (the reference's call order allocates and frees the same grid
// sizes again and again; hipMalloc/hipFree of multi-GB blocks cost far more
// than the kernels).  pool_free waits for the device first, so work queued
// on any stream has finished with the block.  mitos_release_workspace()
// returns the cached blocks; an allocation that fails releases them, then the
// slots above, and tries again.
void* pool_alloc(size_t bytes);
void pool_free(void* p);
// return the cached free blocks (before the large allocations of a fused
// pipeline or an ensemble)
void pool_trim();

}  // namespace mitos
