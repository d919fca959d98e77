// Device memory of datasets and their bricking.
//
// Memory that hipFree gave back has to be cleared by the driver before it can be
// handed out again, at about 35 GB/s: a process that bricks a 1024^3 volume anew
// in a loop (a 4.5 GB pool each time) waits 140 ms per hipMalloc once it has
// been through the card's memory, 20 times what the bricking takes.  The blocks of
// bricking (pool, linear volume, temporaries, cell grid) are therefore kept, once
// released, for the next request of about their size; pools that are filled brick by
// brick (tvk_set_bricks) and the slots of budgeted pools are allocated and freed.
//
// What is kept is bounded (1/16 of the device's memory, 16 blocks per device,
// the longest kept go first) and given back: when an allocation fails
// (device_alloc frees what is kept and tries again), when the program asks for it
// (tvk_release_memory: another allocator may need the memory) and when the device's
// last context is destroyed.  A block is kept only after hipDeviceSynchronize, which
// hipFree implies too, so no queued work still uses it, whatever the stream; a
// caller that has waited for the only stream that used it says so (device_idle).
// All calls are safe from several threads.
#pragma once
#include <hip/hip_runtime.h>
#include <memory>

namespace tvk {

// hipMalloc on the current device; out of memory, once more without the kept blocks
hipError_t device_alloc_bytes(void** p, size_t bytes);
template <typename T>
hipError_t device_alloc(T** p, size_t bytes) { return device_alloc_bytes(reinterpret_cast<void**>(p), bytes); }

// A block of at least `bytes` on the current device, a kept one or a new one; it
// goes back with its last reference.  Contents are undefined.  spare: a block the
// caller can do without; it is given up (left null) where there is no room else.
hipError_t device_block(std::shared_ptr<void>* out, size_t bytes, std::shared_ptr<void>* spare = nullptr);

// Says that no queued work uses the block any more (its stream was waited for, and
// no other saw it): it goes back without a wait for the whole device.
void device_idle(const std::shared_ptr<void>& block);

// contexts of a device: the last one to go gives back what is kept
void device_hold(int device);
void device_drop(int device);
// gives back what is kept now
void device_release(int device);

}  // namespace tvk
