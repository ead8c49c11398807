"""mcr_run_noalloc's host side: no operator new from the library's own code, from
the first call of each kernel on (the HIP runtime's own allocations are its own)."""
from __future__ import annotations

import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# The program's operator new replaces the library's, too; it counts the calls that
# return into the library.
PROGRAM = r"""
#include <dlfcn.h>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>
#include "mcr_hip.h"
static bool counting = false;
static long counted = 0;
static void* take(std::size_t n, void* from) {
  Dl_info d;
  if (counting && dladdr(from, &d) && d.dli_fname && std::strstr(d.dli_fname, "libmcr_hip")) ++counted;
  void* p = std::malloc(n ? n : 1);
  if (!p) std::abort();
  return p;
}
void* operator new(std::size_t n) { return take(n, __builtin_return_address(0)); }
void* operator new[](std::size_t n) { return take(n, __builtin_return_address(0)); }
void* operator new(std::size_t n, const std::nothrow_t&) noexcept { return take(n, __builtin_return_address(0)); }
void operator delete(void* p, const std::nothrow_t&) noexcept { std::free(p); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete[](void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
void operator delete[](void* p, std::size_t) noexcept { std::free(p); }

static int run(int n, int precision, int kernel, unsigned flags) {
  std::vector<double> mu(n, 0.0), sigma((size_t)n * n, 0.0);
  for (int i = 0; i < n; ++i) sigma[(size_t)i * n + i] = 1e-4;
  std::vector<int32_t> S(1000);
  std::vector<int64_t> hist(n + 1);
  mcr_query q = {};
  q.n = n;
  q.mu = mu.data();
  q.sigma = sigma.data();
  q.ld_sigma = n;
  q.x = 0.02;
  q.k = 1;
  q.paths = 1000;
  q.precision = precision;
  q.kernel = kernel;
  q.flags = MCR_F_VAR | MCR_F_SHIST | flags;
  q.n_alpha = 1;
  q.alpha[0] = 0.9;
  q.S_out = S.data();
  q.s_hist = hist.data();
  mcr_result r;
  counted = 0;
  counting = true;
  const int e = mcr_run_noalloc(&q, &r);
  counting = false;
  std::printf("n %d precision %d kernel %d flags %u: code %d, %ld allocations\n", n, precision, kernel, flags, e, counted);
  return e != MCR_OK || counted != 0;
}

int main() {
  if (mcr_init(0) != MCR_OK) return 2;
  int bad = 0;
  for (int n : {20, 70, 100, 127, 200, 608}) bad |= run(n, MCR_PREC_FP32, 0, 0);
  for (int n : {20, 100, 200, 400, 600}) bad |= run(n, MCR_PREC_BF16X3, 0, 0);
  bad |= run(40, MCR_PREC_BF16X3, MCR_KERNEL_MFMA_LDS, 0);
  bad |= run(40, MCR_PREC_FP32, MCR_KERNEL_VALU_TILE, MCR_F_TEST_NARROW);
  bad |= run(40, MCR_PREC_FP32, MCR_KERNEL_VALU_CHUNK, MCR_F_TEST_WIDE);
  mcr_shutdown();
  return bad;
}
"""


def test_noalloc_takes_nothing_from_the_heap(mcr, tmp_path):
    src, exe = tmp_path / "heap.cpp", tmp_path / "heap"
    src.write_text(PROGRAM)
    lib = os.path.dirname(mcr.LIB_PATH)
    subprocess.run(["g++", "-std=c++17", "-O1", str(src), "-o", str(exe), f"-I{ROOT}/include", f"-L{lib}", "-lmcr_hip",
                    f"-Wl,-rpath,{lib}", "-rdynamic", "-ldl"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
