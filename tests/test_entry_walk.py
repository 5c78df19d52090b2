"""The 32-bit walk over CSR entries (research_amd/csrc/entry_walk.hpp), on the
CPU: compiled for the host and compared with a walk in 64 bits, for rows in
the middle of the index range and rows that end at, or a few entries before,
2^32 - 1, with every step the kernels take.  A walk that tests a stepped index
against the row's end instead wraps there and never ends; the program shows
that the comparison tells the two apart."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "research_amd", "csrc")
ROCM = "/opt/rocm"

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "entry_walk.hpp"

typedef std::vector<uint32_t> Seq;
static const size_t kMost = 20000;  // more entries than any row here has

// one lane's entries, `unroll` at a time and then one by one
static Seq by_walk(uint32_t s, uint32_t e, uint32_t first, uint32_t step, uint32_t unroll) {
  Seq out;
  oc::EntryWalk w(s, e, first);
  for (; w.has((unroll - 1) * step) && out.size() < kMost; w.skip(unroll * step))
    for (uint32_t u = 0; u < unroll; ++u) out.push_back(w.at + u * step);
  for (; w.has(0) && out.size() < kMost; w.skip(step)) out.push_back(w.at);
  return out;
}
// the same, a masked batch at a time
static Seq by_batch(uint32_t s, uint32_t e, uint32_t first, uint32_t step, uint32_t unroll) {
  Seq out;
  for (oc::EntryWalk w(s, e, first); w.has(0) && out.size() < kMost; w.skip(unroll * step))
    for (uint32_t u = 0; u < unroll; ++u)
      if (w.has(u * step)) out.push_back(w.at + u * step);
  return out;
}
static Seq by_index(uint32_t s, uint32_t e, uint32_t first, uint32_t step, uint32_t unroll) {
  Seq out;
  uint32_t j = s + first;
  for (; j < e && e - j > (unroll - 1) * step && out.size() < kMost; j += unroll * step)
    for (uint32_t u = 0; u < unroll; ++u) out.push_back(j + u * step);
  for (; j < e && out.size() < kMost; j += step) out.push_back(j);
  return out;
}
static Seq in_64(uint64_t s, uint64_t e, uint64_t first, uint64_t step) {
  Seq out;
  for (uint64_t j = s + first; j < e; j += step) out.push_back((uint32_t)j);
  return out;
}

int main() {
  const uint32_t top = 0xFFFFFFFFu;
  const uint32_t ends[] = {5000, top - 5000, top - 300, top - 64, top - 15, top - 1, top};
  const uint32_t lens[] = {0, 1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 300, 1000, 4096, 5000};
  const uint32_t steps[] = {1, 4, 8, 16, 32, 64, 128, 256, 512, 1024};
  unsigned cases = 0, wrong = 0, index_wrong = 0;
  for (uint32_t e : ends)
    for (uint32_t n : lens)
      for (uint32_t step : steps)
        for (uint32_t unroll : {1u, 4u, 8u})
          for (uint32_t first : {0u, 1u, step / 2, step - 1}) {
            if (first >= step) continue;
            const Seq want = in_64(e - n, e, first, step);
            ++cases;
            wrong += by_walk(e - n, e, first, step, unroll) != want;
            wrong += by_batch(e - n, e, first, step, unroll) != want;
            index_wrong += by_index(e - n, e, first, step, unroll) != want;
          }
  std::printf("%u %u %u\n", cases, wrong, index_wrong);
  return 0;
}
"""


def test_walk_to_the_last_index(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include", f"-I{CSRC}",
                    "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=100).stdout
    cases, wrong, index_wrong = (int(x) for x in out.split())
    assert cases > 5000
    assert wrong == 0
    assert index_wrong > 0


@pytest.mark.parametrize("source,names", [
    ("k_prep.hip", ["k_analysis", "k_analysis_long", "hll_entries", "hll_merge_range"]),
    ("k_accum.hip", ["for_products", "list_longer"]),
])
def test_kernels_step_by_the_walk(source, names):
    """These loops step by up to 4096 entries at once."""
    text = open(os.path.join(CSRC, source)).read()
    for name in names:
        body = text[text.index(f" {name}("):]
        body = body[:body.index("\n}\n")]
        assert "EntryWalk" in body, name
