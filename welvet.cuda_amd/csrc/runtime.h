// Device runtime (device 0, identity) and an owning stream handle.
#pragma once

#include <functional>
#include <string>

#include "common.h"

namespace wv {

Status init_device();
bool device_available();
std::string identity();
int cu_count();

// Copies between pageable host memory and device memory through pinned
// staging buffers the library allocates once (hipHostMalloc). The runtime
// is never handed a pageable buffer, so it never pins the caller's pages in
// place for a large transfer (host memory registration is refused on some
// systems, and the failed pin surfaces in a later call).
// copy_h2d returns once `src` has been read; the device writes are ordered
// on `st`. copy_d2h returns once `dst` holds the data (work queued on `st`
// before it is complete). Calls from different threads serialize.
Status copy_h2d(void* dst, const void* src, size_t n, hipStream_t st);
Status copy_d2h(void* dst, const void* src, size_t n, hipStream_t st);

// Held by a session whose calls may go through host_call: the pinned blocks
// that calls in flight at once needed are freed with the last one.
struct HostSession {
  HostSession();
  ~HostSession();
  HostSession(const HostSession&) = delete;
  HostSession& operator=(const HostSession&) = delete;
};

// One forward call on host buffers: x (xb bytes) to dx, `run` queued on `st`,
// then pre and post (yb and zb bytes) from dpre and dpost; complete on return.
// Device buffers are 16-byte aligned and sizes are whole floats. Calls of
// different threads overlap.
Status host_call(const void* x, void* dx, size_t xb, void* pre, const void* dpre, size_t yb,
                 void* post, const void* dpost, size_t zb, hipStream_t st,
                 const std::function<Status()>& run);

// Owning HIP stream at the default priority.
struct Stream {
  hipStream_t s = nullptr;
  Stream() = default;
  Stream(const Stream&) = delete;
  Stream& operator=(const Stream&) = delete;
  ~Stream();
  Status create();
};

}  // namespace wv
