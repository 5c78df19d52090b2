// The pinned host page through which kernels hand small results to the host.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <mutex>
#include <type_traits>

namespace oc {

// A pinned host page that kernels write small results to (k_publish): word
// 0 is the flag, the data start at word 16.
// A handle takes its page on its first run and gives it back when it is
// destroyed, with no work in flight; up to kIdle pages wait for the next
// handles (allocating and freeing one costs about 100 us).
// The host reads a page while the kernel that writes it may still run, so the
// memory has to be coherent: with neither coherence flag the environment
// (HIP_HOST_COHERENT) decides, and non-coherent memory orders a kernel's
// stores only at a synchronisation.
struct HostPage {
  static constexpr uint32_t kWords = 24 * 1024, kData = 16, kIdle = 16;
  static constexpr unsigned kFlags =
      hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent;
  uint32_t *p = nullptr, seq = 0;
  // Never destroyed, and without the heap: give() runs in destructors.
  struct Idle {
    std::mutex mu;
    uint32_t *pages[kIdle], n = 0;
  };
  static Idle &idle() {
    static_assert(std::is_trivially_destructible<Idle>::value, "outlives every handle");
    static Idle i;
    return i;
  }
  hipError_t take() {
    if (p) return hipSuccess;
    {
      Idle &i = idle();
      std::lock_guard<std::mutex> lk(i.mu);
      if (i.n) p = i.pages[--i.n];
    }
    if (!p) {
      const hipError_t e = hipHostMalloc((void **)&p, kWords * 4, kFlags);
      if (e != hipSuccess) {
        p = nullptr;
        return e;
      }
    }
    p[0] = seq = 0;
    return hipSuccess;
  }
  void give() {
    if (!p) return;
    {
      Idle &i = idle();
      std::lock_guard<std::mutex> lk(i.mu);
      if (i.n < kIdle) {
        i.pages[i.n++] = p;
        p = nullptr;
      }
    }
    if (p) (void)hipHostFree(p);
    p = nullptr;
  }
};

}  // namespace oc
