"""What is noted about a device buffer ends when the buffer is allocated again,
also where the allocator hands the old address out once more.  The host-only
header is compiled against an allocator that always returns one address."""
import os
import subprocess

from plumed2_amd import build_lib

MAIN = r"""
#include "dbuf.h"
#include <cstdio>
static char pool[1 << 16];
static bool full = false;
extern "C" hipError_t hipMalloc(void** p, size_t) { *p = pool; return full ? hipErrorOutOfMemory : hipSuccess; }
extern "C" hipError_t hipFree(void*) { return hipSuccess; }
namespace p2a { int fail(int code, const std::string&) { return code; } }
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
  p2a::DBuf<int> b;
  p2a::Held h;
  CHECK(!h.of(b));
  CHECK(b.reserve(9) == P2A_OK);
  const int* first = b.p;
  h.note(b);
  CHECK(h.of(b));
  CHECK(b.reserve(8) == P2A_OK && h.of(b));      // as large as asked for: the same memory
  CHECK(b.reserve(12) == P2A_OK && b.p == first);
  CHECK(!h.of(b));                               // other memory at the old address
  h.note(b);
  CHECK(h.of(b));
  h.drop();
  CHECK(!h.of(b));
  h.note(b);
  full = true;
  CHECK(b.reserve(100) != P2A_OK && !b.p && !h.of(b));
  h.note(b);
  CHECK(!h.of(b));
  full = false;
  CHECK(b.reserve(12) == P2A_OK && !h.of(b));
  return 0;
}
"""


def test_a_note_ends_with_the_allocation(tmp_path):
    src, exe = tmp_path / "main.cpp", tmp_path / "main"
    src.write_text(MAIN)
    rocm = os.path.dirname(os.path.dirname(build_lib.HIPCC))
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", os.path.join(build_lib.ROOT, "include"), "-I", build_lib.CSRC, str(src), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
