"""HostIo (csrc/hostio.h) on the CPU: the header compiled with g++ against a stand-in of the few runtime calls it makes
(copies and the gather kernel run at once), so that the bookkeeping of a call's inputs and results is checked without a
GPU: what is refused, what falls back to a plain copy, and what is left behind by a call that failed."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lastro-rust_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <cstdint>
#include <cstdlib>
#include <cstring>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorLaunchFailure = 719 };
typedef int* hipStream_t;
enum { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipHostMallocMapped };
struct dim3 { unsigned x, y, z; dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {} };
struct uint4 { unsigned x, y, z, w; };
static dim3 blockIdx, threadIdx, gridDim;
static int copies = 0, launches = 0;  // plain copies and gather launches so far
#define __global__
#define __launch_bounds__(n)
static hipError_t hipHostMalloc(void** p, size_t n, int) { *p = aligned_alloc(64, (n + 63) / 64 * 64); return hipSuccess; }
static hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
static hipError_t hipHostGetDevicePointer(void** d, void* p, int) { *d = p; return hipSuccess; }
static hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
static hipError_t hipGetLastError() { return hipSuccess; }
static hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  copies++;
  if (n) memcpy(d, s, n);
  return hipSuccess;
}
template <class K, class... A>
static void hipLaunchKernelGGL(K k, dim3 g, int threads, int, hipStream_t, A... a) {
  launches++;
  gridDim = g;
  for (blockIdx.y = 0; blockIdx.y < g.y; blockIdx.y++)
    for (blockIdx.x = 0; blockIdx.x < g.x; blockIdx.x++)
      for (threadIdx.x = 0; threadIdx.x < (unsigned)threads; threadIdx.x++) k(a...);
}
"""

MAIN = r"""
#include "hostio.h"
#include <cstdio>
#include <new>
static int news = 0;  // allocations so far
void* operator new(size_t n) { news++; return malloc(n); }
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
#define NEED(c) do { if (!(c)) { std::printf("failed: %s (line %d)\n", #c, __LINE__); return 1; } } while (0)
using namespace moert;
int main(int, char** argv) {
  const char* name = argv[1];
  alignas(16) static uint32_t dev[24100];
  for (unsigned i = 0; i < 24100; i++) dev[i] = i * 2654435761u;
  HostIo io;
  NEED(io.create(4096) == hipSuccess);
  CASES
  std::printf("no such case\n");
  return 1;
}
"""

CASES = {
    # a null output or input of any size is refused, as the runtime's own copy refuses it; nothing is registered
    "null": r"""
      uint32_t got[4] = {};
      NEED(io.out(0, nullptr, dev, 16) == hipErrorInvalidValue);
      NEED(io.in(0, dev, nullptr, 16) == hipErrorInvalidValue);
      NEED(io.out(0, got, dev + 1, 16) == hipSuccess);
      NEED(io.out(0, nullptr, dev, 0) == hipSuccess && io.in(0, dev, nullptr, 0) == hipSuccess);
      NEED(io.flush(0) == hipSuccess);
      io.finish(true);
      NEED(!memcmp(got, dev + 1, 16));""",
    # every size and alignment of a source, more results than one launch gathers, and results past the buffer
    "results": r"""
      static uint32_t got[40][600];
      for (int round = 0; round < 3; round++) {
        memset(got, 0, sizeof got);
        for (int i = 0; i < 40; i++) NEED(io.out(0, got[i], dev + 600 * i + i % 5, 4 * (i * 13 % 600)) == hipSuccess);
        NEED(io.out(0, (char*)got[39] + 2300, (char*)dev + 2, 3) == hipSuccess);  // not whole words: a plain copy
        NEED(io.flush(0) == hipSuccess);
        io.finish(true);
        for (int i = 0; i < 40; i++) NEED(!memcmp(got[i], dev + 600 * i + i % 5, 4 * (i * 13 % 600)));
        NEED(!memcmp((char*)got[39] + 2300, (char*)dev + 2, 3));
      }""",
    # more results than the table holds: the rest are plain copies, and no call allocates (an allocation that fails
    # would leave the C entry point as an exception)
    "many": r"""
      static uint32_t got[100][2];
      HostIo big;
      NEED(big.create(1 << 16) == hipSuccess);
      news = 0;
      for (int i = 0; i < 100; i++) NEED(big.out(0, got[i], dev + 2 * i, 8) == hipSuccess);
      NEED(copies == 36 && big.flush(0) == hipSuccess);
      big.finish(true);
      NEED(news == 0 && !memcmp(got, dev, sizeof got));""",
    # a call that failed between registering and the wait leaves nothing for the next one
    "restart": r"""
      uint32_t gone[4] = {7, 7, 7, 7};  // the caller's memory, its own again when the call has failed
      NEED(io.out(0, gone, dev, 16) == hipSuccess);
      NEED(io.restart(0) == hipSuccess);
      uint32_t got[4];
      NEED(io.out(0, got, dev + 4, 16) == hipSuccess && io.flush(0) == hipSuccess);
      io.finish(true);
      NEED(!memcmp(got, dev + 4, 16));
      for (uint32_t g : gone) NEED(g == 7);""",
}


@pytest.fixture(scope="session")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("hostio")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    body = "".join(f'if (!strcmp(name, "{n}")) {{{c}\n      return 0;\n  }}\n' for n, c in CASES.items())
    (d / "main.cpp").write_text(MAIN.replace("CASES", body))
    exe = d / "hostio"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", str(d), "-I", CSRC, "-o", str(exe), str(d / "main.cpp")],
                   check=True)
    return exe


@pytest.mark.parametrize("name", CASES)
def test_host_io(program, name):
    r = subprocess.run([str(program), name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_no_model_call_returns_between_registering_a_result_and_the_wait():
    """A result registered with the model (model_copy_out) keeps the caller's pointer until model_sync has filled it or
    a failure handled by MTRY has dropped it. A plain return in between would leave the pointer for a later call."""
    src = open(os.path.join(CSRC, "engine.hip")).read()
    src = re.sub(r"//[^\n]*", "", src)
    seen = 0
    for body in re.findall(r"^(?:static )?int \w+\([^;{]*\) \{\n(.*?)^\}", src, re.M | re.S):
        open_at = None
        for line in body.split("\n"):
            if "model_copy_out(m" in line:
                open_at, seen = line, seen + 1
            if open_at:
                assert not re.search(r"\b(CHECK_HIP|CHECK_CFG|TRY|return)\b", line.replace("MTRY", "")), (open_at, line)
            if "model_sync(m)" in line:
                open_at = None
        assert open_at is None, open_at
    assert seen > 10
