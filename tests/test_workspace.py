"""The context's device scratch after an allocation that fails: a slot that was
to grow holds nothing, so a later, smaller request gets memory of its own rather
than the address it had before with the capacity of then.  Runs on the CPU:
splotch_amd/csrc/workspace.hpp is compiled against a stand-in for the HIP
allocator that fails past a limit.  Buffers that a pass can do without are taken
only where they leave half of the free memory.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <cstdlib>
#include <cstddef>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
inline size_t &limit() { static size_t v = 0; return v; }
inline hipError_t &last() { static hipError_t e = hipSuccess; return e; }
inline hipError_t hipMalloc(void **p, size_t n) {
  if (n > limit()) return last() = hipErrorOutOfMemory;
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { return hipSuccess; }
inline hipError_t hipGetLastError() { hipError_t e = last(); last() = hipSuccess; return e; }
inline hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = limit(); return hipSuccess; }
"""

MAIN = r"""
#include "workspace.hpp"
#include <cstdio>
using namespace splhip;
int main() {
  Workspace w;
  limit() = 4 << 20;
  if (!w.get(S_REC, 1 << 20)) return 1;
  bool failed = false;
  try {
    w.get(S_REC, 64 << 20);
  } catch (const HipError &e) {
    failed = e.code == hipErrorOutOfMemory;
  }
  if (!failed) return 2;
  char *p = static_cast<char *>(w.get(S_REC, 1 << 19));  // less than the slot once held
  if (!p) return 3;
  p[0] = p[(1 << 19) - 1] = 1;
  if (w.total_bytes() < (1 << 19) || w.total_bytes() > (1 << 20)) return 4;
  return 0;
}
"""


OPTIONAL = r"""
#include "workspace.hpp"
using namespace splhip;
int main() {
  Workspace w;
  limit() = 16 << 20;  // free
  if (w.optional({{S_REC, 5 << 20}, {S_ACT, 4 << 20}})) return 1;  // more than half
  if (w.total_bytes() != 0) return 2;
  if (!w.optional({{S_REC, 5 << 20}, {S_ACT, 2 << 20}})) return 3;
  const size_t held = w.total_bytes();
  if (held < (7 << 20) || held > (8 << 20)) return 4;
  limit() = 0;  // held already: nothing more is needed
  if (!w.optional({{S_REC, 5 << 20}, {S_ACT, 1 << 20}})) return 5;
  limit() = 4 << 20;  // growth beyond what is held counts
  if (w.optional({{S_REC, 5 << 20}, {S_ACT, 5 << 20}})) return 6;
  if (w.total_bytes() != held) return 7;
  return 0;
}
"""


def compiled(tmp_path, main):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(main)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-I", str(tmp_path), "-I",
                    os.path.join(ROOT, "splotch_amd", "csrc"), str(tmp_path / "main.cpp"),
                    "-o", exe], check=True)
    return subprocess.run([exe]).returncode


def test_slot_after_failed_growth(tmp_path):
    rc = compiled(tmp_path, MAIN)
    assert rc == 0, {3: "a null pointer for a slot that failed to grow"}.get(rc, rc)


def test_optional_buffers(tmp_path):
    assert compiled(tmp_path, OPTIONAL) == 0
