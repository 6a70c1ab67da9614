"""The host side of the field transfers (lh_xfer.hpp) compiled for the CPU, with the HIP calls it
makes taken from a stub: a transfer that waits for its device holds up neither the handles that other
threads create and destroy nor another device's transfers, concurrent ones get their own bytes, and
the pinned memory is given back with the last handle."""
import os
import shutil
import subprocess

import pytest

from littleharsh_amd.build import HERE

STUB = r"""
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <mutex>
#define __global__
#define __shared__ static
#define __launch_bounds__(n)
#define __syncthreads()
struct Idx { unsigned x, y, z; };
static Idx blockIdx, threadIdx;
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum { hipHostMallocPortable = 1, hipHostMallocMapped = 2, hipEventDisableTiming = 2 };
typedef int* hipEvent_t;
typedef void* hipStream_t;
static std::atomic<int> live{0}, at_gate{0};
static std::mutex gate_mu;
static std::condition_variable gate_cv;
static bool gate_shut = false;               // device 0's copies do not end
static thread_local int cur_dev = 0;
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::malloc(n); ++live; return hipSuccess; }
inline hipError_t hipHostFree(void* p) { std::free(p); --live; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { cur_dev = d; return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = cur_dev; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new int(0); return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) {
  std::unique_lock<std::mutex> g(gate_mu);
  if (cur_dev == 0 && gate_shut) ++at_gate;
  gate_cv.wait(g, [] { return cur_dev != 0 || !gate_shut; });
  return hipSuccess;
}
"""

MAIN = r"""
#include "lh_xfer.hpp"
#include <chrono>
#include <cstdio>
#include <future>
#include <unistd.h>

using namespace lh;
static void need(bool ok, const char* what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::fflush(stdout);
  _exit(1);
}
// up and down again through a "device" buffer of its own: two fields, a null one between them
static void round_trip(int dev, int ncol, int n, unsigned seed) {
  const size_t el = 16, bytes = (size_t)n * ncol * el;
  std::vector<char> stage(2 * bytes), a(bytes), b(bytes), a2(bytes), b2(bytes);
  for (size_t i = 0; i < bytes; ++i) {
    a[i] = (char)(seed = seed * 1664525u + 1013904223u, seed >> 24);
    b[i] = (char)(seed >> 16);
  }
  XferFields fs{};
  fs.f[0] = XferField{nullptr, a.data(), 0, n, 0, n};
  fs.f[1] = XferField{nullptr, nullptr, bytes, 0, 0, 0};
  fs.f[2] = XferField{nullptr, b.data(), bytes, n, 0, n};
  need(xfer_bytes(true, dev, nullptr, stage.data(), fs, 3, ncol, el) == hipSuccess, "up");
  fs.f[0].host = a2.data();
  fs.f[2].host = b2.data();
  need(xfer_bytes(false, dev, nullptr, stage.data(), fs, 3, ncol, el) == hipSuccess, "down");
  need(a == a2 && b == b2, "bytes of a transfer");
}

int main() {
  double* const slot = host_stage().retain();
  need(slot != nullptr, "slot");
  round_trip(1, 33, 17, 1);                          // a part of a chunk
  round_trip(1, 1, (int)(HostStage::kChunk / 16), 2);     // whole chunks
  round_trip(1, 1201, 409, 3);                       // several, the last in part
  gate_shut = true;
  auto held = std::async(std::launch::async, [] { round_trip(0, 1201, 409, 4); });
  while (at_gate == 0) usleep(1000);
  auto other = std::async(std::launch::async, [] {
    double* const s = host_stage().retain();
    need(s != nullptr, "slot beside a transfer");
    host_stage().release(s);
    round_trip(1, 1201, 409, 5);
  });
  need(other.wait_for(std::chrono::seconds(20)) == std::future_status::ready,
       "a handle and another device beside a transfer that waits");
  other.get();
  {
    std::lock_guard<std::mutex> g(gate_mu);
    gate_shut = false;
  }
  gate_cv.notify_all();
  held.get();
  std::vector<std::future<void>> many;
  for (unsigned i = 0; i < 6; ++i)
    many.push_back(std::async(std::launch::async, [i] { round_trip((int)(i % 2), 401 + (int)i, 409, 6 + i); }));
  for (auto& f : many) f.get();
  host_stage().release(slot);
  need(live == 0, "pinned memory given back");
  std::puts("ok");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_transfers_wait_for_nothing_else(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "t"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-pthread", "-I", str(tmp_path), "-I", os.path.join(HERE, "csrc"),
                        str(tmp_path / "main.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert (r.returncode, r.stdout) == (0, "ok\n"), r.stdout + r.stderr
