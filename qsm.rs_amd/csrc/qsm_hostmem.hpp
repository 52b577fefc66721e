// Host-side memory services of the library: device workspaces, streams and
// pinned blocks kept between calls, and copies between pageable host arrays
// and the device.  Everything here is thread-safe, per device, bounded, and
// lives until the process ends.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace qsm {

// Device memory.  A freed block is kept (at most kWorkspaceKept bytes over all
// devices, the least recently freed go back first) and handed to a later
// request of about its size on the same device.  The caller frees a block
// only after it has waited for the work that uses it, so a kept block is idle
// and any stream or thread may have it.
constexpr size_t kWorkspaceKept = (size_t)2 << 30;
hipError_t workspace_alloc(void** p, size_t bytes);
void workspace_free(void* p);
// Gives every kept block, stream and pinned block back.
void workspace_trim();

// Runs a call that takes device or pinned memory.  Where it finds none left,
// everything kept is given back and the call made once more, so that no call
// of this library fails for want of memory that the library itself holds idle.
// A failure that remains is the returned one only: HIP's last error, which the
// next launch check would read, is cleared.
template <class F>
hipError_t with_trim(F&& call) {
    hipError_t e = call();
    if (e != hipErrorOutOfMemory) return e;
    (void)hipGetLastError();
    workspace_trim();
    if ((e = call()) != hipSuccess) (void)hipGetLastError();
    return e;
}

// A non-blocking stream of default priority, and back once it is idle.
hipError_t stream_take(hipStream_t* s);
void stream_give(hipStream_t s);

// Mapped, coherent pinned host memory (at most kPinnedBlock bytes).
constexpr size_t kPinnedBlock = 4096;
hipError_t pinned_take(void** p);
void pinned_give(void* p);

// Blocking copies between a pageable host array and the device, through two
// pinned chunks: one is filled (or drained) while the other is in flight.  Not ordered with
// any stream: the source is complete and the destination idle when the caller
// calls.
hipError_t copy_to_device(void* dst, const void* src, size_t bytes);
hipError_t copy_to_host(void* dst, const void* src, size_t bytes);
// n values, f64 on the host and f32 on the device (rounded to nearest, widened
// exactly).
hipError_t copy_to_device_f32(float* dst, const double* src, size_t n);
hipError_t copy_to_host_f32(double* dst, const float* src, size_t n);
// Has the system back a host array that a download will fill with memory now,
// while the device works (what the array holds stays as it is): of a 38 MB
// download into a fresh array, 1.0 ms for the page faults in one call here
// against 1.6-2.4 ms one by one in the copy, which then takes 1.3 ms.
void prefault(void* p, size_t bytes);

}  // namespace qsm
