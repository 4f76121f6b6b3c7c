"""The download pool (atus2_amd/csrc/staging.hpp) on the CPU, over a stand-in
for the runtime's calls that copies at once and counts: downloads alternating
between devices reuse their slots, several devices download at once, and the
memory goes with each device's last context."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = """
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>
enum hipError_t { hipSuccess = 0, hipErrorNotReady = 600 };
enum hipMemcpyKind { hipMemcpyDeviceToHost };
struct Event { int device; };
typedef Event* hipEvent_t;
typedef void* hipStream_t;
constexpr unsigned hipEventDisableTiming = 2, hipHostMallocDefault = 0;
inline std::atomic<int> mallocs{0}, live{0}, events{0}, wrong{0};
inline thread_local int current = 0;
inline hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
template <class T>
hipError_t hipHostMalloc(T** p, size_t n, unsigned) { ++mallocs; ++live; *p = static_cast<T*>(malloc(n)); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { --live; free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { ++events; *e = new Event{current}; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { --events; delete e; return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
// an event belongs to the device it was made on
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { if (e->device != current) ++wrong; return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
"""

MAIN = """
#include "staging.hpp"
#include <cstdio>
using namespace atus_host;
static bool ok = true;
static void check(bool b, const char* what) { if (!b) { ok = false; printf("%s\\n", what); } }
static std::vector<char> image(size_t n, int seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)((i * 2654435761u >> 7) + seed);
  return v;
}
static void download(int d, const std::vector<char>& src) {
  hipSetDevice(d);
  std::vector<char> dst(src.size());
  const hipError_t e = staging(d)->to_host(dst.data(), src.data(), src.size(), nullptr);
  check(e == hipSuccess, "download");
  check(dst == src, "bytes");
}
int main() {
  const std::vector<char> small = image(3 << 20, 1), large = image((41 << 20) + 24, 2);
  for (int d : {0, 1}) staging(d)->ref();
  staging(1)->ref();
  for (int d : {0, 1}) download(d, large);
  const int first = mallocs;
  for (int k = 0; k < 10; ++k)
    for (int d : {0, 1}) download(d, k & 1 ? small : large);
  check(mallocs == first, "slots reused");
  std::vector<std::thread> t;
  for (int d : {0, 1}) t.emplace_back([&, d] { for (int k = 0; k < 20; ++k) download(d, large); });
  for (std::thread& th : t) th.join();
  check(mallocs == first, "slots reused by several devices at once");
  std::vector<char> dst(1000);
  check(staging(0)->to_host(dst.data(), small.data(), 1000, nullptr) == hipErrorNotReady, "short copies are refused");
  check(staging(-1) == nullptr && staging(64) == nullptr, "device range");
  staging(0)->unref();
  staging(1)->unref();
  check(live > 0, "a context is left");
  download(1, small);
  staging(1)->unref();
  check(live == 0 && events == 0, "memory given back");
  check(wrong == 0, "events on their device");
  return ok ? 0 : 1;
}
"""


def test_one_pool_per_device(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(tmp_path), "-I",
                    os.path.join(ROOT, "atus2_amd", "csrc"), str(tmp_path / "main.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
