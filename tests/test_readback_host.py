"""The readers' copies (mpm_readback.h), compiled for the host against a stand-in
for the few HIP calls they make: what arrives is what was sent, for one slot and
many, host and device segments in any order, with movers and without; and where
pinned memory, an event, a thread or host memory is refused, the copies are plain
ones, as before there were slots."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <cstdlib>
#include <cstring>
typedef int hipError_t;
typedef void* hipStream_t;
typedef void* hipEvent_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipMemcpyDeviceToHost = 2, hipEventDisableTiming = 2 };
extern bool no_pinned, no_events, bad_copy;
inline hipError_t hipGetLastError() { return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return 0; }
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return 0; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  if (bad_copy) return 1;
  memcpy(d, s, n);
  return 0;
}
inline hipError_t hipHostMalloc(void** p, size_t n) {
  *p = nullptr;
  return no_pinned || !(*p = malloc(n)) ? hipErrorOutOfMemory : 0;
}
inline hipError_t hipHostFree(void* p) { free(p); return 0; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) {
  *e = nullptr;
  return no_events || !(*e = malloc(1)) ? hipErrorOutOfMemory : 0;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { free(e); return 0; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return 0; }
"""

MAIN = r"""
#include "mpm_readback.h"
#include <cstdio>
#include <new>
bool no_pinned = false, no_events = false, bad_copy = false;
static bool no_memory = false;
void* operator new(size_t n) {
  void* p = no_memory ? nullptr : malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
static int read(mpm::Readback& r, size_t n, int seed) {
  std::vector<char> a(n), b(n / 2 + 1), x(n), y(n / 2 + 1);
  for (size_t i = 0; i < n; i++) a[i] = (char)(i * 7 + seed);
  for (size_t i = 0; i < b.size(); i++) b[i] = (char)(i * 3 + seed);
  int e = 5 + seed, f = 0;
  const std::vector<mpm::Readback::Segment> s = {{a.data(), x.data(), n, false},
                                                 {nullptr, nullptr, 0, false},
                                                 {b.data(), y.data(), b.size(), true},
                                                 {&e, &f, sizeof(int), false}};
  const bool refuse = no_memory;
  const int rc = r.copy(s, nullptr);
  no_memory = false;
  const bool same = a == x && b == y && e == f;
  no_memory = refuse;
  return rc ? rc : same ? 0 : -1;
}
#define EXPECT(c) if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; }
int main() {
  const size_t sizes[] = {0, 1, (2u << 20) - 4, (2u << 20) - 3, 2u << 20, 9000001, 40000007};
  mpm::Readback r;
  for (size_t n : sizes)
    for (int k = 0; k < 3; k++) EXPECT(read(r, n, k) == 0);
  bad_copy = true;  // an error of the copies is the caller's, and ends every thread
  EXPECT(read(r, 40000007, 1) == 1);
  EXPECT(read(r, 5000, 1) == 1);
  bad_copy = false;
  EXPECT(read(r, 40000007, 1) == 0);
  r.release();
  mpm::Readback p;
  no_pinned = true;
  for (size_t n : sizes)
    for (int k = 0; k < 2; k++) EXPECT(read(p, n, k) == 0);
  no_pinned = false;
  no_events = true;
  for (size_t n : sizes) EXPECT(read(p, n, 3) == 0);
  no_events = false;
  for (size_t n : sizes) EXPECT(read(p, n, 4) == 0);
  const size_t n = 9000001;  // host memory refused inside copy alone
  std::vector<char> a(n, 'a'), x(n);
  const std::vector<mpm::Readback::Segment> s = {{a.data(), x.data(), n, false}};
  no_memory = true;
  const int rc = p.copy(s, nullptr);
  no_memory = false;
  EXPECT(rc == 0 && a == x);
  p.release();
  puts("ok");
}
"""


def test_copies_and_refusals(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("needs g++")
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "readback")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", str(tmp_path), "-I",
                    os.path.join(ROOT, "taichi_elements_amd", "csrc"),
                    str(tmp_path / "main.cpp"), "-o", exe, "-lpthread"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.endswith("ok\n"), out.stdout + out.stderr
