// hostio.hpp (part of runtime.cpp) — what the host-buffer entry points need beside the kernels:
// copies between the device and a caller's pageable memory, and device memory
// for the buffers of one call.
//
// Copies.  hipMemcpy moves pageable memory by one host thread; its memcpy,
// and the page faults of a destination the caller has just allocated, bound
// large copies (64 MB down into fresh pages 6.8 ms, up 2.5).  Copies from 32
// MB up and 8 MB down are cut into pieces that up to eight threads take in
// turn, each through its own pinned slot: the DMA of one piece runs during
// the memcpys and faults of the others (64 MB down 2.4 ms, up 1.9; 16 MB down
// 1.23 -> 0.86; below, starting the threads costs what they save: 4 MB down
// 0.37 either way, up 0.18 -> 0.30).  Pinned memory and smaller copies go to
// hipMemcpyAsync as they are.  The threads end with the copy; 16 slots (32
// MB) are kept and the rest freed.
//
// Device memory.  A call's hipMalloc and hipFree (which waits for the whole
// device) are a tenth of a one-shot call: 1024^2 Float16 b32 NormalBP 1308 ->
// 1145 us, forward 425 -> 359 with DevBuf's pool of freed blocks (at most 256
// MB in all, larger blocks are not kept; every device allocation of the
// library goes through dev_malloc, which gives all idle blocks back and tries
// again where memory runs out).  A block returns to the pool only after its stream has
// drained.  A resident store's mount allocates and frees its staging buffers
// outside the pool: a grid whose mounts kept them there paid for it in its
// first training step (32 layers of 1024^2: 1.5-2.0 ms -> 1.6-6.3), where the
// gradients are allocated.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <unordered_map>
#include <vector>

#include "runtime.hpp"

namespace wh {
namespace rt {

namespace {

constexpr size_t kSlotBytes = size_t(2) << 20;
constexpr size_t kUpFrom = size_t(32) << 20, kDownFrom = size_t(8) << 20;
constexpr int kMaxThreads = 8, kMaxSlots = 16;

struct Slot {
  void *mem = nullptr;
  hipEvent_t done = nullptr;
};

struct SlotPool {
  std::mutex mu;
  std::vector<Slot> idle;
};
SlotPool &slots() {
  static SlotPool *p = new SlotPool;  // never destroyed: the runtime may be gone by then
  return *p;
}

void free_slot(Slot s) {
  if (s.done) (void)hipEventDestroy(s.done);
  if (s.mem) (void)hipHostFree(s.mem);
}

hipError_t take_slot(Slot *s) {
  {
    std::lock_guard<std::mutex> lk(slots().mu);
    if (!slots().idle.empty()) {
      *s = slots().idle.back();
      slots().idle.pop_back();
      return hipSuccess;
    }
  }
  hipError_t e = hipHostMalloc(&s->mem, kSlotBytes, hipHostMallocDefault);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&s->done, hipEventDisableTiming);
  if (e != hipSuccess) {
    free_slot(*s);
    *s = Slot();
  }
  return e;
}

void give_slot(Slot s) {
  try {
    std::lock_guard<std::mutex> lk(slots().mu);
    if (slots().idle.size() < kMaxSlots) {
      slots().idle.push_back(s);
      return;
    }
  } catch (const std::bad_alloc &) {
  }
  free_slot(s);
}

// Pieces of a staged copy, taken in turn by every thread that works on it.  A
// thread that gets no slot takes none: what no thread took (`next`) is left to
// the caller.
struct Staged {
  char *host;
  char *dev;
  size_t bytes, piece;
  bool up;  // host -> device
  hipStream_t stream;
  int device;
  std::atomic<size_t> next{0};
  std::atomic<int> error{hipSuccess};

  void work() {
    hipError_t e = hipSetDevice(device);
    Slot s;
    if (e != hipSuccess) {
      error = e;
      return;
    }
    if (take_slot(&s) != hipSuccess) {
      (void)hipGetLastError();  // no pinned memory must not read as a failed launch
      return;
    }
    for (size_t at = next.fetch_add(piece); at < bytes && error == hipSuccess; at = next.fetch_add(piece)) {
      const size_t n = std::min(piece, bytes - at);
      if (up) std::memcpy(s.mem, host + at, n);
      e = up ? hipMemcpyAsync(dev + at, s.mem, n, hipMemcpyHostToDevice, stream)
             : hipMemcpyAsync(s.mem, dev + at, n, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipEventRecord(s.done, stream);
      if (e == hipSuccess) e = hipEventSynchronize(s.done);
      if (e != hipSuccess) {
        error = e;
        break;
      }
      if (!up) std::memcpy(host + at, s.mem, n);
    }
    if (error != hipSuccess) (void)hipStreamSynchronize(stream);  // a slot goes back with no copy on it
    give_slot(s);
  }
};

// A pinned (or managed) pointer needs no staging.
bool pageable(const void *p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();  // an unknown pointer must not read as a failed launch
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

hipError_t staged_copy(void *host, void *dev, size_t bytes, bool up, hipStream_t s) {
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  const unsigned cores = std::max(2u, std::thread::hardware_concurrency());
  const int threads = (int)std::min<size_t>(kMaxThreads, cores / 2 + 1);
  Staged c;
  c.host = (char *)host;
  c.dev = (char *)dev;
  c.bytes = bytes;
  // two pieces per thread at least, so the DMA of one overlaps another's memcpy
  c.piece = std::min(kSlotBytes, std::max(size_t(256) << 10, (bytes / (2 * threads) + 4095) / 4096 * 4096));
  c.up = up;
  c.stream = s;
  c.device = device;
  std::thread team[kMaxThreads];
  int started = 0;
  try {
    for (; started < threads - 1; ++started) team[started] = std::thread([&c] { c.work(); });
  } catch (const std::exception &) {  // no more threads (or memory for one): those there are do it
  }
  c.work();
  for (int i = 0; i < started; ++i) team[i].join();
  if (c.error != hipSuccess) return (hipError_t)c.error.load();
  const size_t at = c.next;
  if (at >= bytes) return hipSuccess;
  return up ? hipMemcpyAsync(c.dev + at, c.host + at, bytes - at, hipMemcpyHostToDevice, s)
            : hipMemcpyAsync(c.host + at, c.dev + at, bytes - at, hipMemcpyDeviceToHost, s);
}

}  // namespace

hipError_t copy_to_device(void *dst, const void *src, size_t bytes, hipStream_t s) {
  if (bytes < kUpFrom || !pageable(src)) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
  return staged_copy(const_cast<void *>(src), dst, bytes, true, s);
}

hipError_t copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t s) {
  if (bytes < kDownFrom || !pageable(dst)) return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
  return staged_copy(dst, const_cast<void *>(src), bytes, false, s);
}

// ------------------------------------------------------------ device memory
namespace {

constexpr size_t kPoolBytes = size_t(256) << 20;

struct Block {
  void *p;
  size_t bytes;
  int device;
};
struct DevPool {
  std::mutex mu;
  std::vector<Block> idle;
  std::unordered_map<void *, Block> out;  // blocks handed out
  size_t kept = 0;
};
DevPool &pool() {
  static DevPool *p = new DevPool;
  return *p;
}

}  // namespace

hipError_t dev_malloc_bytes(void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();  // must not read as a failed launch
    dev_trim();
    e = hipMalloc(p, bytes);
  }
  return e;
}

hipError_t dev_alloc(void **p, size_t bytes) try {
  DevPool &d = pool();
  bytes = (std::max<size_t>(bytes, 1) + 4095) / 4096 * 4096;
  *p = nullptr;
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  {
    std::lock_guard<std::mutex> lk(d.mu);
    size_t best = d.idle.size();  // the smallest block that fits without wasting half of itself
    for (size_t i = 0; i < d.idle.size(); ++i)
      if (d.idle[i].device == device && d.idle[i].bytes >= bytes && d.idle[i].bytes <= 2 * bytes &&
          (best == d.idle.size() || d.idle[i].bytes < d.idle[best].bytes))
        best = i;
    if (best < d.idle.size()) {
      const Block b = d.idle[best];
      d.out[b.p] = b;
      d.idle[best] = d.idle.back();
      d.idle.pop_back();
      d.kept -= b.bytes;
      *p = b.p;
      return hipSuccess;
    }
  }
  e = dev_malloc(p, bytes);
  if (e != hipSuccess) return e;
  try {
    std::lock_guard<std::mutex> lk(d.mu);
    d.out[*p] = Block{*p, bytes, device};
  } catch (const std::bad_alloc &) {
    (void)hipFree(*p);
    *p = nullptr;
    return hipErrorOutOfMemory;
  }
  return hipSuccess;
} catch (const std::bad_alloc &) {
  return hipErrorOutOfMemory;
}

void dev_free(void *p) {
  if (p == nullptr) return;
  DevPool &d = pool();
  try {
    std::lock_guard<std::mutex> lk(d.mu);
    const auto it = d.out.find(p);
    if (it != d.out.end()) {
      const Block b = it->second;
      d.out.erase(it);
      if (d.kept + b.bytes <= kPoolBytes) {
        d.idle.push_back(b);
        d.kept += b.bytes;
        return;
      }
    }
  } catch (const std::bad_alloc &) {
  }
  (void)hipFree(p);
}

void dev_trim() {
  DevPool &d = pool();
  std::vector<Block> idle;
  {
    std::lock_guard<std::mutex> lk(d.mu);
    idle.swap(d.idle);
    d.kept = 0;
  }
  for (const Block &b : idle) (void)hipFree(b.p);
}

DevBuf::~DevBuf() {
  if (p == nullptr) return;
  (void)hipStreamSynchronize(stream);
  if (pooled) dev_free(p);
  else (void)hipFree(p);
}

}  // namespace rt
}  // namespace wh
