"""The pipelined host copies (csrc/transfer.cpp) compiled for the host against a few
stand-ins for the runtime's calls (copies done at once): arrays of every piece count
come through, also when the memory for a thread cannot be had -- then the threads that
did start and the caller do the work, and nothing is thrown or ended.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "distributed-cfd-solver_amd")

HIP = r"""
#pragma once
#include <cstddef>
#include <cstdlib>
#include <cstring>
typedef int hipError_t;
typedef void* hipStream_t;
typedef void* hipEvent_t;
enum { hipSuccess = 0, hipEventDisableTiming = 2, hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
inline const char* hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipEventDestroy(hipEvent_t) { return 0; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = e; return 0; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return 0; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return 0; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return 0; }
inline hipError_t hipSetDevice(int) { return 0; }
inline bool no_pinned = false;
inline int last_error = 0;
inline hipError_t hipHostMalloc(void** p, std::size_t n) {
    if (no_pinned) return last_error = 2;
    *p = std::malloc(n);
    return 0;
}
inline hipError_t hipGetLastError() { const int e = last_error; last_error = 0; return e; }
inline hipError_t hipHostFree(void* p) { std::free(p); return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return 0; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, std::size_t n, int, hipStream_t) { std::memcpy(d, s, n); return 0; }
"""

MAIN = r"""
#include <atomic>
#include <cstdio>
#include <new>
#include <vector>
#include "transfer.hpp"

static std::atomic<int> countdown{0};  // the allocation that fails, 0 for none
void* operator new(std::size_t n) {
    int left = countdown.load();
    while (left > 0 && !countdown.compare_exchange_weak(left, left - 1)) {}
    if (left == 1) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main() {
    const std::size_t mib = 1u << 20;
    int failed = 0;
    for (std::size_t bytes : {mib / 2, 2 * mib, 5 * mib + 8, 16 * mib, 37 * mib + 123}) {
      for (const bool pinned : {true, false}) {
        no_pinned = !pinned;
        cfdg::HostPipe pipe;
        pipe.reserve(bytes);
        if (last_error != 0) failed = 1;
        std::vector<char> src(bytes), dev(bytes), back(bytes);
        for (std::size_t i = 0; i < bytes; ++i) src[i] = static_cast<char>(i * 2654435761u >> 13);
        // the first allocation of a copy is its list of threads, the others one per thread
        for (int at : {0, 2, 3, 5, 8}) {
            std::memset(dev.data(), 0, bytes);
            std::memset(back.data(), 0, bytes);
            countdown = at;
            pipe.to_device(dev.data(), src.data(), bytes, nullptr);
            countdown = at;
            pipe.to_host(back.data(), dev.data(), bytes, nullptr);
            countdown = 0;
            if (dev != src || back != src) {
                std::printf("wrong copy: %zu bytes, allocation %d\n", bytes, at);
                failed = 1;
            }
        }
      }
    }
    return failed;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_copies_without_memory_for_threads(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "transfer"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{tmp_path}", f"-I{PKG}/csrc", f"-I{ROOT}/include",
                    str(tmp_path / "main.cpp"), f"{PKG}/csrc/transfer.cpp", "-o", str(exe)], check=True, timeout=120)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, (out.returncode, out.stdout, out.stderr)
