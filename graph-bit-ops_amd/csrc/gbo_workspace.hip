// Device scratch of synchronous calls, kept between calls.
//
// Every driver and two-phase operation needs a few buffers and waits for its
// stream before it returns.  From the runtime's stream-ordered pool they cost
// 10 to 100 us each (an allocation of 64 MB 30 us, its release 9, and the next
// synchronization gives the memory back: 31 us for 4 x 1 MB, 0.8 ms for 4 x
// 64 MB), several times the kernels of a small call.  Here a block goes back
// to a list when its call is over and is handed out again:
//   - a block enters the list only after the stream that used it has been
//     waited for, so whichever thread or stream takes it next finds it idle;
//   - the list holds at most kKeepBytes and kKeepBlocks per device, the
//     longest unused go first, and a block of more than half of that is not kept
//     (it would send all others off); all of it goes back to the runtime when an
//     allocation fails and when the last matrix that the library allocated or
//     planned is freed.
#include <algorithm>
#include <cstring>
#include <mutex>

#include "gbo_device.hpp"
#include "gbo_ops.hpp"

namespace gbo {
namespace {

constexpr int kKeepBlocks = 128;
constexpr int kDevices = 64;

struct Block {
  void* p;
  size_t bytes;
};

// Arrays of fixed length: no call into the pool can throw.  Never destroyed (at
// exit the runtime may be gone before it).
struct Idle {
  Block blocks[kKeepBlocks];  // the longest unused first
  int n;
  size_t bytes;
  void remove(int i) {
    bytes -= blocks[i].bytes;
    std::copy(blocks + i + 1, blocks + n, blocks + i);
    --n;
  }
};
std::mutex pool_mu;
Idle pool_idle[kDevices];
int64_t pool_live = 0;  // matrices and plans the library allocated

// Sizes in steps of an eighth of a power of two (512 bytes at least), so that
// calls of about the same size find each other's blocks.
size_t rounded(size_t bytes) {
  size_t step = 512;
  while (step * 16 < bytes) step *= 2;
  return (std::max<size_t>(bytes, 1) + step - 1) / step * step;
}

}  // namespace

void workspace_release(int dev) {
  for (int d = dev < 0 ? 0 : dev; d < (dev < 0 ? kDevices : std::min(dev + 1, kDevices)); ++d) {
    Block out[kKeepBlocks];
    int n = 0;
    {
      std::lock_guard<std::mutex> lk(pool_mu);
      Idle& v = pool_idle[d];
      n = v.n;
      std::copy(v.blocks, v.blocks + n, out);
      v.n = 0;
      v.bytes = 0;
    }
    for (int i = 0; i < n; ++i) (void)hipFree(out[i].p);
  }
}

void workspace_live(int delta) {
  bool last = false;
  {
    std::lock_guard<std::mutex> lk(pool_mu);
    pool_live += delta;
    last = delta < 0 && pool_live <= 0;
  }
  if (last) workspace_release(-1);
}

namespace {

template <class Alloc>
hipError_t alloc_or_release(Alloc alloc) {
  hipError_t e = alloc();
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    int dev = 0;
    (void)hipGetDevice(&dev);
    workspace_release(dev);
    e = alloc();
  }
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

}  // namespace

hipError_t device_malloc(void** p, size_t bytes) {
  return alloc_or_release([&] { return hipMalloc(p, bytes); });
}

hipError_t device_malloc_async(void** p, size_t bytes, hipStream_t st) {
  return alloc_or_release([&] { return hipMallocAsync(p, bytes, st); });
}

Workspace::~Workspace() {
  if (n_ == 0) return;
  const bool idle = hipStreamSynchronize(st_) == hipSuccess && dev_ >= 0 && dev_ < kDevices;
  Block out[kMax + kKeepBlocks];
  int drop = 0;
  {
    std::lock_guard<std::mutex> lk(pool_mu);
    for (int i = 0; i < n_; ++i) {
      const Block b{ptrs_[i], bytes_[i]};
      if (!idle || b.bytes > kKeepBytes / 2) {
        out[drop++] = b;
        continue;
      }
      Idle& v = pool_idle[dev_];
      if (v.n == kKeepBlocks) {
        out[drop++] = v.blocks[0];
        v.remove(0);
      }
      v.blocks[v.n++] = b;
      v.bytes += b.bytes;
    }
    while (idle && pool_idle[dev_].bytes > kKeepBytes) {
      out[drop++] = pool_idle[dev_].blocks[0];
      pool_idle[dev_].remove(0);
    }
  }
  for (int i = 0; i < drop; ++i) (void)hipFree(out[i].p);
}

int Workspace::take(void** p, size_t bytes, const char* who) {
  *p = nullptr;
  const size_t want = rounded(bytes);
  int s = -1;  // the smallest dropped block that fits
  for (int i = 0; i < n_; ++i)
    if (spare_[i] && bytes_[i] >= want && (s < 0 || bytes_[i] < bytes_[s])) s = i;
  if (s >= 0) {
    spare_[s] = false;
    *p = ptrs_[s];
    return GBO_OK;
  }
  if (n_ == kMax) return set_error(GBO_EINVAL, "%s: too many scratch allocations", who);
  if (n_ == 0) GBO_HIP_CHECK(hipGetDevice(&dev_));
  void* q = nullptr;
  size_t got = want;
  if (dev_ >= 0 && dev_ < kDevices) {
    std::lock_guard<std::mutex> lk(pool_mu);
    Idle& v = pool_idle[dev_];
    int best = -1;
    for (int i = 0; i < v.n; ++i)  // the smallest that fits and is not twice too large
      if (v.blocks[i].bytes >= want && v.blocks[i].bytes <= 2 * want && (best < 0 || v.blocks[i].bytes < v.blocks[best].bytes))
        best = i;
    if (best >= 0) {
      q = v.blocks[best].p;
      got = v.blocks[best].bytes;
      v.remove(best);
    }
  }
  if (!q) {
    hipError_t e = device_malloc(&q, want);
    if (e == hipErrorOutOfMemory && free_dropped()) e = device_malloc(&q, want);
    if (e != hipSuccess)
      return set_error(GBO_ENOMEM, "%s: device allocation of %zu bytes failed: %s", who, bytes, hipGetErrorString(e));
  }
  ptrs_[n_] = q;
  spare_[n_] = false;
  bytes_[n_++] = got;
  *p = q;
  return GBO_OK;
}

// The dropped blocks back to the runtime; false if there are none.
bool Workspace::free_dropped() {
  int keep = 0;
  bool any = false;
  if (hipStreamSynchronize(st_) != hipSuccess) return false;
  for (int i = 0; i < n_; ++i) {
    if (spare_[i]) {
      any = true;
      (void)hipFree(ptrs_[i]);
      continue;
    }
    ptrs_[keep] = ptrs_[i];
    bytes_[keep] = bytes_[i];
    spare_[keep++] = false;
  }
  n_ = keep;
  return any;
}

void Workspace::drop(const void* p) {
  for (int i = 0; i < n_; ++i)
    if (ptrs_[i] == p) spare_[i] = true;
}

// ---- small host reads.  A copy into ordinary host memory is staged by the
// runtime (20 us with the wait); into one of these pinned slots it is not
// (12 us).  With every slot taken the ordinary copy serves.
namespace {

constexpr size_t kSlotBytes = 16384;
constexpr int kSlots = 16;

struct Slots {
  std::mutex mu;
  char* base = nullptr;
  bool tried = false;
  uint32_t taken = 0;
};
Slots slots;

}  // namespace

int read_back(void* h, const void* d, size_t bytes, hipStream_t st) {
  Slots& S = slots;
  int k = -1;
  if (bytes <= kSlotBytes) {
    std::lock_guard<std::mutex> lk(S.mu);
    if (!S.tried) {
      S.tried = true;
      void* p = nullptr;
      if (hipHostMalloc(&p, kSlotBytes * kSlots, hipHostMallocPortable) == hipSuccess) S.base = (char*)p;
      else (void)hipGetLastError();
    }
    if (S.base)
      for (int i = 0; i < kSlots && k < 0; ++i)
        if (!(S.taken >> i & 1u)) k = i;
    if (k >= 0) S.taken |= 1u << k;
  }
  void* to = k >= 0 ? S.base + (size_t)k * kSlotBytes : h;
  hipError_t e = hipMemcpyAsync(to, d, bytes, hipMemcpyDeviceToHost, st);
  // waited for in any case: the slot must not be written once it is free again
  const hipError_t s = hipStreamSynchronize(st);
  if (e == hipSuccess) e = s;
  if (k >= 0) {
    if (e == hipSuccess) std::memcpy(h, to, bytes);
    std::lock_guard<std::mutex> lk(S.mu);
    S.taken &= ~(1u << k);
  }
  if (e != hipSuccess) return set_error(GBO_EDEVICE, "device to host copy: %s", hipGetErrorString(e));
  return GBO_OK;
}

}  // namespace gbo
