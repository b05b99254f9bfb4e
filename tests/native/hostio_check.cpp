// hostio.hpp's allocation and copy paths against a fake HIP runtime (host
// memory, a settable limit of device bytes and of pinned slots), on the CPU:
// the definitions here take the place of the runtime library's.
//
//   hostio_check     prints "hostio_check: ok" or the first failed check
#include <cstdio>
#include <cstdlib>

#include "../../welvet.metal_amd/csrc/hostio.hpp"

namespace {
std::mutex mu;
std::unordered_map<void *, size_t> device;
size_t used = 0, limit = ~size_t(0);
int slots_left = 1 << 30;
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  *p = nullptr;
  if (used + n > limit) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  device[*p] = n;
  used += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lk(mu);
  used -= device.at(p);
  device.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned int) {
  std::lock_guard<std::mutex> lk(mu);
  if (slots_left-- <= 0) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
  a->type = hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
}

#define CHECK(c)                                                     \
  do {                                                               \
    if (!(c)) {                                                      \
      std::printf("hostio_check: line %d: %s\n", __LINE__, #c);      \
      return 1;                                                      \
    }                                                                \
  } while (0)

int main() {
  using namespace wh::rt;
  constexpr size_t MB = size_t(1) << 20;
  // a call leaves its blocks idle in the pool; an allocation that needs their
  // memory gets it, one that fits beside them leaves them
  {
    void *a = nullptr, *b = nullptr, *c = nullptr;
    CHECK(dev_alloc(&a, 60 * MB) == hipSuccess && dev_alloc(&b, 100 * MB) == hipSuccess);
    dev_free(a);
    dev_free(b);
    CHECK(used == 160 * MB);
    limit = 200 * MB;
    CHECK(dev_malloc(&c, 40 * MB) == hipSuccess && used == 200 * MB);
    CHECK(hipFree(c) == hipSuccess);
    CHECK(dev_malloc(&c, 150 * MB) == hipSuccess && used == 150 * MB);
    CHECK(hipFree(c) == hipSuccess && used == 0);
    CHECK(dev_malloc(&c, 201 * MB) == hipErrorOutOfMemory && c == nullptr && used == 0);
    // an unpooled and a pooled buffer the same way
    for (bool pooled : {false, true}) {
      CHECK(dev_alloc(&a, 90 * MB) == hipSuccess);
      dev_free(a);
      DevBuf d(nullptr, pooled);
      CHECK(d.alloc(190 * MB) == hipSuccess && used == 190 * MB);
    }
    dev_trim();
    CHECK(used == 0);
    limit = ~size_t(0);
  }
  // copies in pieces: every byte, both ways, from several threads at once, and
  // with some and then all of the pinned slots refused
  for (int slots : {1 << 30, 3, 0}) {
    slots_left = slots;
    std::atomic<int> bad{0};
    std::thread team[4];
    for (int t = 0; t < 4; ++t)
      team[t] = std::thread([t, &bad] {
        const size_t n = 40 * MB + 4097 * t;
        std::vector<unsigned char> src(n), dst(n);
        for (size_t i = 0; i < n; ++i) src[i] = (unsigned char)(i * 2654435761u >> 7 ^ t);
        void *d = nullptr;
        if (dev_alloc(&d, n) != hipSuccess || copy_to_device(d, src.data(), n, nullptr) != hipSuccess ||
            copy_to_host(dst.data(), d, n, nullptr) != hipSuccess || src != dst)
          ++bad;
        dev_free(d);
      });
    for (std::thread &t : team) t.join();
    CHECK(bad == 0);
  }
  std::printf("hostio_check: ok\n");
  return 0;
}
