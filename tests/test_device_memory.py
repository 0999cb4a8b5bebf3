"""The bookkeeping of kept device memory where the host itself runs out of memory, on the CPU: glide_amd/csrc/device_memory.hpp
over a stand-in for the HIP runtime that counts what is allocated, with each allocation of the bookkeeping failing in turn."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "glide_amd", "csrc")
STUB = r"""
#pragma once
#include <cstddef>
#include <cstdint>
typedef void* hipStream_t;
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
hipError_t hipGetDevice(int*);
hipError_t hipMalloc(void**, size_t);
hipError_t hipFree(void*);
hipError_t hipDeviceSynchronize();
hipError_t hipGetLastError();
"""
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <new>
#include <set>
static long fails_in = -1;      // the how manieth allocation from now fails
void* operator new(size_t n) {
    if (fails_in >= 0 && fails_in-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
#include "device_memory.hpp"
static char device[64];
static bool used[64];
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t) {
    for (int i = 0; i < 64; i++) if (!used[i]) { used[i] = true; *p = device + i; return hipSuccess; }
    return hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
    const long i = static_cast<char*>(p) - device;
    if (i < 0 || i >= 64 || !used[i]) std::abort();      // freed twice
    used[i] = false;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }

int main() {
    const size_t gib = size_t{1} << 30;
    long failed = 0;
    for (long at = 0; at < 40; at++) {
        glide::DeviceMemory memory;
        void* p[12] = {};
        fails_in = at;
        for (int i = 0; i < 12; i++) {
            try {
                if (memory.allocate(&p[i], gib / 2 + i * gib / 16) != 0) std::abort();
            } catch (const std::bad_alloc&) { p[i] = nullptr; failed++; }
        }
        for (int i = 0; i < 12; i++) {      // more than is held: the oldest go
            if (!p[i]) continue;
            try {
                if (memory.free(p[i]) != 0) std::abort();
            } catch (const std::bad_alloc&) { failed++; }
        }
        fails_in = -1;
        long held = 0;
        for (bool u : used) held += u;
        if (held > 4 || memory.held() > 2 * gib) { std::printf("%ld blocks held\n", held); return 1; }
        memory.release();
        for (bool u : used) if (u) { std::printf("a block is lost (failure %ld)\n", at); return 1; }
    }
    std::printf("ok\n");
    return failed > 0 ? 0 : 1;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_no_block_is_lost_and_nothing_hangs_without_host_memory(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", str(tmp_path), "-I", CSRC, str(tmp_path / "main.cpp"), "-o", str(tmp_path / "main")], check=True)
    r = subprocess.run([str(tmp_path / "main")], capture_output=True, text=True, timeout=20)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
