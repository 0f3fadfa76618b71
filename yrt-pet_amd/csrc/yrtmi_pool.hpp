// Device memory of plans and of the library's own scratch, kept for reuse.
//
// Plans hold gigabytes and are made and dropped by the dozen (one per
// sensitivity subset, four per autotune, one per data subset).  The driver
// clears freed memory before it hands it out again, in the background at a
// few tens of GB/s: a loop that makes and drops a 4 GB plan each 13 ms of
// GPU work ran at 100 ms a round once clean memory had run out.  Blocks given
// back here are handed out again instead.
//
// Per device: at most kPoolBytes are kept (the longest unused go first); all
// of them return to the driver with the device's last context, with
// yrtmi_mem_trim, and when an allocation of the library fails.  Other
// allocators of the process do not see them.  A block is kept once the device
// has finished with it (poolQuiesce, or the stream that used it waited for),
// so it may be handed to any stream.  Any thread may call; the mutex covers the
// lists only.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace yrtmi
{

constexpr size_t kPoolBytes = size_t(16) << 30;

// Context count of a device (create / destroy).
void poolRetain(int device);
void poolRelease(int device);
// *out = at least `bytes` (> 0) bytes on `device`, which is current: a kept
// block of up to a quarter (and 1 MiB) more than that, or, with `exact`, of no
// more than the pool's rounding, else new memory.
hipError_t poolAlloc(int device, void** out, size_t bytes, bool exact = false);
template <class T>
hipError_t poolAlloc(int device, T** out, size_t bytes, bool exact = false)
{
	return poolAlloc(device, reinterpret_cast<void**>(out), bytes, exact);
}
// hipMalloc, once more with the kept blocks returned where it fails: for
// memory that is not given back through the pool.
hipError_t poolMalloc(int device, void** out, size_t bytes);
template <class T>
hipError_t poolMalloc(int device, T** out, size_t bytes)
{
	return poolMalloc(device, reinterpret_cast<void**>(out), bytes);
}
// Gives p (null: nothing) back.  idle: the device has finished with it (the
// caller has waited for every stream that used it); else it goes to hipFree,
// which waits itself.
void poolFree(int device, void* p, bool idle);
// Waits for the device, as hipFree would.  False where it cannot (an error,
// or the thread is recording a graph).
bool poolQuiesce(int device);
// The kept blocks of `device` return to the driver.
void poolTrim(int device);
// Bytes of them.
size_t poolKept(int device);

}  // namespace yrtmi
