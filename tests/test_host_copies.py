"""Large host copies by several threads (nc_hostmem.h) when memory runs out at
any of their allocations: the copy is whole, or std::bad_alloc is thrown; the
process is not ended by threads left unjoined."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <stdio.h>
#include <new>
#include "nc_hostmem.h"

static long g_left = -1;  // allocations until one fails (negative: none does)
void* operator new(size_t n) {
  if (g_left >= 0 && g_left-- == 0) throw std::bad_alloc();
  void* p = malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

int main() {
  const size_t bytes = 9u << 20;  // several threads' work
  char *a = (char*)malloc(bytes), *b = (char*)malloc(bytes);
  int whole = 0, thrown = 0;
  for (long k = 0; k < 24; ++k) {
    for (size_t i = 0; i < bytes; ++i) a[i] = (char)(i * 31 + k), b[i] = 0;
    g_left = k;
    try {
      nc::copy_bytes(b, a, bytes);
      g_left = -1;
      if (memcmp(a, b, bytes)) return 1;
      ++whole;
    } catch (const std::bad_alloc&) {
      g_left = -1;
      ++thrown;
    }
  }
  printf("%d whole, %d thrown\n", whole, thrown);
  return thrown <= 2 && whole >= 22 ? 0 : 2;
}
"""


def test_copies_when_memory_runs_out(tmp_path):
    src, exe = str(tmp_path / "copies.cpp"), str(tmp_path / "copies")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "neurocorrelation_amd", "csrc"),
                    src, "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
