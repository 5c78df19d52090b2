// The CSR entries a lane or a wave takes, in 32-bit indices up to the last
// that an offset can hold.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace oc {

// The entries s + first, s + first + step, ... below e.  An index stepped
// past e wraps to a small one where e is within a step of 2^32, and then
// passes a test against e, so the walk counts what is left instead; `at` is
// an entry only while `left` is not zero.
struct EntryWalk {
  uint32_t at, left;
  __host__ __device__ EntryWalk(uint32_t s, uint32_t e, uint32_t first)
      : at(s + first), left(e - s > first ? e - s - first : 0u) {}
  // whether at + n is below e too
  __host__ __device__ bool has(uint32_t n) const { return left > n; }
  __host__ __device__ void skip(uint32_t n) {
    at += n;
    left = left > n ? left - n : 0u;
  }
};

}  // namespace oc
