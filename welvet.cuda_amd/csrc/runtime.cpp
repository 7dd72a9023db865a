// Device runtime: one process-wide GPU (device 0), initialized once under a
// mutex, and its identity string. Mirrors src/cuda/device.cpp:40-92 of the
// reference (init_default_device / available / runtime_identity).
#include "runtime.h"

#include "kernels.h"

#include <cstring>
#include <mutex>
#include <sstream>

namespace wv {
namespace {
std::mutex g_mu;
bool g_ready = false;
hipDeviceProp_t g_prop;

// Device name for the identity: the runtime's marketing name, else the
// name hipDeviceGetName reports, else one built from what the properties
// always carry (architecture, compute units, peak engine clock).
std::string device_name() {
  std::string name(g_prop.name, strnlen(g_prop.name, sizeof(g_prop.name)));
  if (name.empty()) {
    char buf[256] = {0};
    if (hipDeviceGetName(buf, sizeof(buf) - 1, 0) == hipSuccess) name = buf;
    else (void)hipGetLastError();
  }
  if (name.empty()) {
    std::string arch(g_prop.gcnArchName);
    arch = arch.substr(0, arch.find(':'));
    std::ostringstream os;
    os << "AMD " << arch << " " << g_prop.multiProcessorCount << "CU "
       << g_prop.clockRate / 1000 << "MHz";
    name = os.str();
  }
  return name;
}

// Pinned staging: two buffers, so the host copy of one chunk overlaps the
// DMA of the other.
constexpr size_t kStageBytes = 8u << 20;
std::mutex g_stage_mu;
void* g_stage[2] = {nullptr, nullptr};
hipEvent_t g_stage_ev[2] = {nullptr, nullptr};

Status stage_ready() {
  for (int i = 0; i < 2; ++i) {
    if (!g_stage[i]) WV_HIP(hipHostMalloc(&g_stage[i], kStageBytes, hipHostMallocDefault));
    if (!g_stage_ev[i])
      WV_HIP(hipEventCreateWithFlags(&g_stage_ev[i], hipEventDisableTiming));
  }
  return Status::ok();
}

// Pinned blocks of host_call, one per call in flight, allocated when first
// needed and grown to the largest call that used them: at most 16 MiB each. The
// first stays for the next session, as the staging buffers do; the others are
// freed with the last session. Calls beyond kHostBlocks take staged copies.
constexpr size_t kHostCallBytes = 8u << 20;  // x; and pre with post
constexpr int kHostBlocks = 4;
struct HostBlock {
  void* p = nullptr;
  size_t bytes = 0;
  bool used = false;
};
std::mutex g_host_mu;
HostBlock g_host[kHostBlocks];
int g_host_sessions = 0;

// A block of at least n bytes for the holder's lifetime; p is null when all are
// in use or the memory cannot be had. The lock covers the choice alone.
struct HostLoan {
  void* p = nullptr;
  explicit HostLoan(size_t n) {
    {
      std::lock_guard<std::mutex> lock(g_host_mu);
      for (HostBlock& b : g_host)
        if (!b.used) {
          block_ = &b;
          b.used = true;
          break;
        }
    }
    if (!block_) return;
    if (block_->bytes < n) {
      size_t size = 64u << 10;
      while (size < n) size *= 2;
      free_block(block_);
      if (hipHostMalloc(&block_->p, size, hipHostMallocDefault) == hipSuccess) {
        block_->bytes = size;
      } else {
        (void)hipGetLastError();
        block_->p = nullptr;
      }
    }
    p = block_->p;
  }
  ~HostLoan() {
    if (!block_) return;
    std::lock_guard<std::mutex> lock(g_host_mu);
    block_->used = false;
  }
  HostLoan(const HostLoan&) = delete;
  HostLoan& operator=(const HostLoan&) = delete;
  static void free_block(HostBlock* b) {
    if (b->p && hipHostFree(b->p) != hipSuccess) (void)hipGetLastError();
    b->p = nullptr, b->bytes = 0;
  }

 private:
  HostBlock* block_ = nullptr;
};
}  // namespace

HostSession::HostSession() {
  std::lock_guard<std::mutex> lock(g_host_mu);
  ++g_host_sessions;
}

HostSession::~HostSession() {
  std::lock_guard<std::mutex> lock(g_host_mu);
  if (--g_host_sessions > 0) return;
  for (int i = 1; i < kHostBlocks; ++i)
    if (!g_host[i].used) HostLoan::free_block(&g_host[i]);
}

Status init_device() {
  std::lock_guard<std::mutex> lock(g_mu);
  if (g_ready) return hip_status(hipSetDevice(0), "hipSetDevice");
  int n = 0;
  const hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess || n <= 0) {
    (void)hipGetLastError();
    return Status::err(kUnsupported, "no HIP device visible");
  }
  WV_HIP(hipSetDevice(0));
  WV_HIP(hipGetDeviceProperties(&g_prop, 0));
  g_ready = true;
  return Status::ok();
}

bool device_available() {
  int n = 0;
  const hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) (void)hipGetLastError();
  return e == hipSuccess && n > 0;
}

std::string identity() {
  if (!init_device()) return "hip:unavailable";
  std::lock_guard<std::mutex> lock(g_mu);
  std::ostringstream os;
  os << "hip:" << device_name() << ":idx=0:arch=" << g_prop.gcnArchName
     << ":cu=" << g_prop.multiProcessorCount << ":mem=" << (g_prop.totalGlobalMem >> 20) << "MiB";
  return os.str();
}

int cu_count() {
  if (!init_device()) return 0;
  return g_prop.multiProcessorCount;
}

Status copy_h2d(void* dst, const void* src, size_t n, hipStream_t st) {
  if (n == 0) return Status::ok();
  if (!dst || !src) return Status::err(kInvalid, "copy_h2d: null buffer");
  std::lock_guard<std::mutex> lock(g_stage_mu);
  WV_TRY(stage_ready());
  bool used[2] = {false, false};
  // The next caller refills the buffers, so every DMA queued here must have
  // read its buffer before this returns, on the error paths too. A failed
  // copy or record leaves an earlier event that may still be pending; the
  // whole stream is drained then, since that event no longer marks the last
  // use of its buffer.
  auto fail = [&](Status s) {
    if (hipStreamSynchronize(st) != hipSuccess) (void)hipGetLastError();
    return s;
  };
  int i = 0;
  for (size_t off = 0; off < n; off += kStageBytes, i ^= 1) {
    const size_t len = n - off < kStageBytes ? n - off : kStageBytes;
    // the DMA that last read this buffer must be done before it is refilled
    if (used[i]) {
      Status s = hip_status(hipEventSynchronize(g_stage_ev[i]), "copy_h2d: stage wait");
      if (!s) return fail(s);
    }
    std::memcpy(g_stage[i], static_cast<const char*>(src) + off, len);
    used[i] = true;
    Status s = hip_status(hipMemcpyAsync(static_cast<char*>(dst) + off, g_stage[i], len,
                                         hipMemcpyHostToDevice, st),
                          "copy_h2d: hipMemcpyAsync");
    if (s) s = hip_status(hipEventRecord(g_stage_ev[i], st), "copy_h2d: hipEventRecord");
    if (!s) return fail(s);
  }
  for (int k = 0; k < 2; ++k)
    if (used[k]) {
      Status s = hip_status(hipEventSynchronize(g_stage_ev[k]), "copy_h2d: stage wait");
      if (!s) return fail(s);
    }
  return Status::ok();
}

Status copy_d2h(void* dst, const void* src, size_t n, hipStream_t st) {
  if (n == 0) return Status::ok();
  if (!dst || !src) return Status::err(kInvalid, "copy_d2h: null buffer");
  std::lock_guard<std::mutex> lock(g_stage_mu);
  WV_TRY(stage_ready());
  bool pend[2] = {false, false};
  size_t pend_off[2] = {0, 0}, pend_len[2] = {0, 0};
  // as in copy_h2d: no DMA into a staging buffer may still be running when
  // this returns, on the error paths too
  auto fail = [&](Status s) {
    if (hipStreamSynchronize(st) != hipSuccess) (void)hipGetLastError();
    return s;
  };
  auto drain = [&](int k) -> Status {
    WV_HIP(hipEventSynchronize(g_stage_ev[k]));
    std::memcpy(static_cast<char*>(dst) + pend_off[k], g_stage[k], pend_len[k]);
    pend[k] = false;
    return Status::ok();
  };
  int i = 0;
  for (size_t off = 0; off < n; off += kStageBytes, i ^= 1) {
    const size_t len = n - off < kStageBytes ? n - off : kStageBytes;
    if (pend[i]) {
      Status s = drain(i);
      if (!s) return fail(s);
    }
    Status s = hip_status(hipMemcpyAsync(g_stage[i], static_cast<const char*>(src) + off, len,
                                         hipMemcpyDeviceToHost, st),
                          "copy_d2h: hipMemcpyAsync");
    if (s) s = hip_status(hipEventRecord(g_stage_ev[i], st), "copy_d2h: hipEventRecord");
    if (!s) return fail(s);
    pend[i] = true, pend_off[i] = off, pend_len[i] = len;
  }
  for (int k = 0; k < 2; ++k)
    if (pend[i ^ k]) {
      Status s = drain(i ^ k);
      if (!s) return fail(s);
    }
  return Status::ok();
}

Status host_call(const void* x, void* dx, size_t xb, void* pre, const void* dpre, size_t yb,
                 void* post, const void* dpost, size_t zb, hipStream_t st,
                 const std::function<Status()>& run) {
  // Small calls: x and the outputs go through a pinned block by kernels on the
  // call's own stream, and the host waits once, at the end, under no lock. A
  // copy_h2d and two copy_d2h wait three times more and pass from the copy
  // engine to the kernels and back.
  const size_t pre_at = (size_t)round_up((int64_t)xb, 256);
  const size_t post_at = pre_at + (size_t)round_up((int64_t)yb, 256);
  if (xb <= kHostCallBytes && post_at - pre_at + zb <= kHostCallBytes) {
    HostLoan loan(post_at + zb);
    if (loan.p) {
      char* buf = static_cast<char*>(loan.p);
      // the block's next user refills it: the stream is drained on every way
      // out of here
      struct Drain {
        hipStream_t st;
        bool done = false;
        ~Drain() {
          if (!done && hipStreamSynchronize(st) != hipSuccess) (void)hipGetLastError();
        }
      } drain{st};
      std::memcpy(buf, x, xb);
      WV_TRY(launch_copy({dx, buf, xb}, {}, st));
      WV_TRY(run());
      WV_TRY(launch_copy({buf + pre_at, dpre, yb}, {buf + post_at, dpost, zb}, st));
      drain.done = true;
      WV_HIP(hipStreamSynchronize(st));
      std::memcpy(pre, buf + pre_at, yb);
      std::memcpy(post, buf + post_at, zb);
      return Status::ok();
    }
  }
  WV_TRY(copy_h2d(dx, x, xb, st));
  WV_TRY(run());
  WV_TRY(copy_d2h(pre, dpre, yb, st));
  WV_TRY(copy_d2h(post, dpost, zb, st));
  return hip_status(hipStreamSynchronize(st), "host call");
}

Status Stream::create() {
  if (s) return Status::ok();
  WV_TRY(init_device());
  WV_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  return Status::ok();
}

Stream::~Stream() {
  if (s) (void)hipStreamDestroy(s);
}

}  // namespace wv
