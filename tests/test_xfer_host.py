"""The transfers through pinned chunks (nc_xfer.hip), compiled against a
stand-in for the HIP runtime in which the device is host memory, streams run at
once and any call or allocation can be made to fail."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <stdlib.h>
#include <string.h>
#include <atomic>
typedef int hipError_t;
struct ihipStream_t { int live; };
struct ihipEvent_t { int live; };
typedef ihipStream_t* hipStream_t;
typedef ihipEvent_t* hipEvent_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum { hipMemcpyDeviceToHost = 2, hipMemcpyHostToDevice = 1 };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2, hipStreamNonBlocking = 1 };
inline std::atomic<int> h_pinned{0}, h_streams{0}, h_events{0}, h_pin_calls{0}, h_last{0};
inline int h_no_pinned = 0, h_no_events = 0;  // such calls fail
inline hipError_t h_ret(hipError_t e) { if (e) h_last = e; return e; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return h_last.exchange(0); }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ++h_pin_calls;
  if (h_no_pinned) return h_ret(hipErrorOutOfMemory);
  *p = malloc(n);
  ++h_pinned;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { free(p); --h_pinned; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  if (h_no_events) return h_ret(hipErrorOutOfMemory);
  *e = (hipEvent_t)malloc(sizeof(ihipEvent_t));
  ++h_events;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { free(e); --h_events; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)malloc(sizeof(ihipStream_t));
  ++h_streams;
  return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) { free(s); --h_streams; return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  memcpy(d, s, n);
  return hipSuccess;
}
"""

COMMON = r"""
#include <stdio.h>
#include <new>
#include <thread>
#include <vector>
#include <hip/hip_runtime.h>
static thread_local long t_left = -1;  // this thread's allocations until one fails (negative: none does)
void* operator new(size_t n) {
  if (t_left >= 0 && t_left-- == 0) throw std::bad_alloc();
  void* p = malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
#include "nc_internal.h"
using namespace nc;
static std::vector<char> pattern(size_t n, int k) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)(i * 7 + k);
  return v;
}
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
"""


def run(tmp_path, body):
    os.makedirs(str(tmp_path / "hip"))
    with open(str(tmp_path / "hip" / "hip_runtime.h"), "w") as f:
        f.write(HIP)
    with open(str(tmp_path / "t.cpp"), "w") as f:
        f.write(COMMON + body)
    exe = str(tmp_path / "t")
    csrc = os.path.join(ROOT, "neurocorrelation_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIP__", "-I", str(tmp_path), "-I", csrc, "-x", "c++",
                    str(tmp_path / "t.cpp"), os.path.join(csrc, "nc_xfer.hip"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


# two arrays: a piece, one chunk (2 MiB) in all, one more than that, several
@pytest.mark.parametrize("a,b", [(100, 0), (1 << 20, 1 << 20), ((2 << 20) + 1, 3), (9 << 20, 5)])
def test_transfers_when_memory_runs_out(tmp_path, a, b):
    run(tmp_path, r"""
int main() {
  const size_t n[2] = {%d, %d};
  for (long k = -1; k < 24; ++k)
    for (int down = 0; down < 2; ++down) {
      std::vector<char> host[2], dev[2];
      Segment seg[2];
      for (int i = 0; i < 2; ++i) {
        host[i] = pattern(n[i], down ? 0 : i + 1), dev[i] = pattern(n[i], down ? i + 1 : 0);
        seg[i] = Segment{host[i].data(), dev[i].data(), n[i]};
      }
      t_left = k;
      bool thrown = false;
      hipError_t e = hipSuccess;
      try {
        e = down ? download(0, nullptr, seg, 2) : upload(0, nullptr, seg, 2);
      } catch (const std::bad_alloc&) {
        thrown = true;
      }
      t_left = -1;
      CHECK(e == hipSuccess);
      CHECK(!thrown || k >= 0);
      if (!thrown)
        for (int i = 0; i < 2; ++i) CHECK(host[i] == pattern(n[i], i + 1) && dev[i] == host[i]);
    }
  return 0;
}
""" % (a, b))


@pytest.mark.parametrize("what", ["h_no_pinned", "h_no_events"])
def test_transfers_without_memory_to_pin(tmp_path, what):
    run(tmp_path, r"""
int main() {
  %s = 1;
  const size_t n[3] = {5u << 20, 0, 77};
  for (int down = 0; down < 2; ++down) {
    std::vector<char> host[3], dev[3];
    Segment seg[3];
    for (int i = 0; i < 3; ++i) {
      host[i] = pattern(n[i], down ? 0 : i + 1), dev[i] = pattern(n[i], down ? i + 1 : 0);
      seg[i] = Segment{host[i].data(), dev[i].data(), n[i]};
    }
    CHECK((down ? download(0, nullptr, seg, 3) : upload(0, nullptr, seg, 3)) == hipSuccess);
    for (int i = 0; i < 3; ++i) CHECK(host[i] == pattern(n[i], i + 1) && dev[i] == host[i]);
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(h_pinned == 0 && h_events == 0);
  }
  return 0;
}
""" % what)


def test_what_is_kept_between_calls(tmp_path):
    # several threads wire at once, with and without a simulation alive
    run(tmp_path, r"""
static void wire() {
  hipStream_t st = nullptr;
  if (stream_take(0, &st) != hipSuccess) abort();
  std::vector<char> host(5 << 20), dev = pattern(5 << 20, 3);
  const Segment seg{host.data(), dev.data(), host.size()};
  if (download(0, st, &seg, 1) != hipSuccess || host != dev) abort();
  stream_give(0, st);
}
static void wires(int n) {
  std::vector<std::thread> th;
  for (int i = 0; i < n; ++i) th.emplace_back([] { for (int k = 0; k < 5; ++k) wire(); });
  for (auto& t : th) t.join();
}
int main() {
  wires(8);
  CHECK(h_pinned <= 1 && h_streams <= 1 && h_events <= 4);
  const int calls = h_pin_calls;
  for (int i = 0; i < 5; ++i) wire();
  CHECK(h_pin_calls <= calls + 1);  // (one kept is used again)
  xfer_user(1);
  wires(8);
  CHECK(h_pinned <= 6 && h_streams <= 6);
  xfer_user(1), xfer_user(-1);
  CHECK(h_pinned >= 1 && h_streams >= 1);
  hipStream_t st = nullptr;
  CHECK(stream_take(0, &st) == hipSuccess);
  xfer_user(-1);
  CHECK(h_pinned == 0 && h_events == 0 && h_streams == 1);
  stream_give(0, st);  // after the last simulation went
  wires(8);
  CHECK(h_pinned <= 1 && h_streams <= 1);
  // another device's are not handed out
  hipStream_t a = nullptr, b = nullptr;
  CHECK(stream_take(1, &a) == hipSuccess && stream_take(0, &b) == hipSuccess && a != b);
  stream_give(1, a), stream_give(0, b);
  CHECK(h_streams <= 1);
  xfer_user(1), xfer_user(-1);
  CHECK(h_pinned == 0 && h_events == 0 && h_streams == 0);
  // and keeping one allocates nothing
  xfer_user(1);
  wire();
  CHECK(stream_take(0, &a) == hipSuccess && stream_take(0, &b) == hipSuccess);
  t_left = 0;
  stream_give(0, a), stream_give(0, b);
  t_left = -1;
  xfer_user(-1);
  CHECK(h_pinned == 0 && h_streams == 0);
  return 0;
}
""")
