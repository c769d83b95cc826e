"""Device allocations kept between the handles of a batched call (csrc/dev_mem.hpp), compiled
for the host against a counting stand-in for the allocator."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = "/opt/rocm/include"
CXX = shutil.which("g++") or shutil.which("c++")
pytestmark = pytest.mark.skipif(CXX is None or not os.path.isdir(HIP), reason="no host compiler or HIP headers")

# an allocator of `limit` bytes; addresses are made up, nothing is read or written there
PROGRAM = r"""
#include <cstdio>
#include <map>
#include "dev_mem.hpp"
static size_t limit = size_t(-1), used = 0, next = 4096;
static int mallocs = 0;
static std::map<void*, size_t> live;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (n > limit - used) return hipErrorOutOfMemory;
  ++mallocs;
  *p = reinterpret_cast<void*>(next);
  next += n + 4096;
  live[*p] = n;
  used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  used -= live.at(p);
  live.erase(p);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}
#define CHECK(c) if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; }
using omx::DevCache;
using omx::DevMem;
constexpr size_t MB = size_t(1) << 20;
int main() {
  {
    DevCache cache;
    { DevMem a(1024 * MB), b(40 * MB); }      // both kept
    CHECK(mallocs == 2 && used == 1064 * MB);
    DevMem small(1024), big, half;
    CHECK(mallocs == 2);                      // from the 40 MB block, not the large one
    DevMem small2(1024);
    CHECK(mallocs == 3);                      // not from the large one either
    half.alloc(300 * MB);
    CHECK(mallocs == 3);
    half.release();
    limit = 1200 * MB;                        // no room beside the large block
    big.alloc(1000 * MB);
    CHECK(mallocs == 3);
    big.release();
    big.alloc(1100 * MB);                     // none fits: the kept blocks make room
    CHECK(mallocs == 4);
  }
  CHECK(used == 0 && live.empty());           // everything goes back with the scope
  DevMem plain(5);
  { DevMem other(std::move(plain)); CHECK(other.size() == 5 && plain.size() == 0); }
  CHECK(used == 0);
  for (size_t cap : {size_t(1), 256 * MB, 256 * MB + 1, 1000 * MB})
    for (size_t n : {size_t(1), size_t(1000), 16 * MB, 64 * MB, 250 * MB, 1000 * MB})
      CHECK(DevCache::serves(cap, n) == (cap >= n && (cap <= 256 * MB || cap < 8 * n + 8)));
  return 0;
}
"""


def test_kept_blocks(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    r = subprocess.run([CXX, "-O1", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I", HIP,
                        "-I", os.path.join(ROOT, "optimode.jl_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                        str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
