"""The pinned page on which the host spins while kernels are still running
(research_amd/csrc/host_page.hpp), on the CPU: the header is compiled against
stand-ins for hipHostMalloc and hipHostFree that record how they are called.

The host trusts "flag == sequence number" without a synchronisation and sizes
C from the words beside the flag.  HIP guarantees that a kernel's system-scope
release is seen in order before the kernel ends only for coherent host memory,
and leaves the choice to the environment when an allocation names neither
coherence flag, so the page has to ask for it."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "research_amd", "csrc")
ROCM = "/opt/rocm"

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>
#include "host_page.hpp"

static unsigned news = 0;  // heap allocations by C++ code
void *operator new(std::size_t n) {
  ++news;
  return std::malloc(n);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

static std::vector<unsigned> flags;
static unsigned mallocs = 0, frees = 0;

extern "C" hipError_t hipHostMalloc(void **p, size_t bytes, unsigned f) {
  ++mallocs;
  flags.push_back(f);
  *p = std::malloc(bytes);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
extern "C" hipError_t hipHostFree(void *p) {
  ++frees;
  std::free(p);
  return hipSuccess;
}

int main() {
  const unsigned kept = oc::HostPage::kIdle, n = kept + 3;
  unsigned allocations = 0;
  flags.reserve(3 * n);
  for (int round = 0; round < 2; ++round) {
    std::vector<oc::HostPage> pages(n);
    const unsigned before = news;
    for (auto &p : pages) {
      if (p.take() != hipSuccess || !p.p || p.p[0] != 0 || p.seq != 0) return 1;
      uint32_t *first = p.p;
      if (p.take() != hipSuccess || p.p != first) return 2;  // a second run: the same page
      p.p[0] = p.seq = 7;
    }
    for (auto &p : pages) p.give();
    allocations += news - before;
  }
  for (unsigned f : flags) std::printf("%x ", f);
  std::printf("\n%u %u %u %u\n", mallocs, frees, kept, allocations);
  return 0;
}
"""


def build(tmp_path):
    src, exe = tmp_path / "page.cpp", tmp_path / "page"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include", f"-I{CSRC}",
                    "-o", str(exe), str(src), "-pthread"], check=True)
    return str(exe)


def test_page_is_coherent_and_pool_bounded(tmp_path):
    out = subprocess.run([build(tmp_path)], check=True, capture_output=True, text=True).stdout
    flags, counts = out.splitlines()
    portable, mapped, coherent, non_coherent = 0x1, 0x2, 0x40000000, 0x80000000
    assert flags.split()
    for f in (int(x, 16) for x in flags.split()):
        assert f & coherent and not f & non_coherent, hex(f)
        assert f & mapped and f & portable, hex(f)
    # 19 pages, 3 of them freed; then 16 from the pool and 3 new ones
    mallocs, frees, kept, allocations = (int(x) for x in counts.split())
    assert (mallocs, frees, kept) == (22, 6, 16)
    # pages come and go without the heap: give() runs in a handle's destructor,
    # where an allocation that fails would end the process
    assert allocations == 0
