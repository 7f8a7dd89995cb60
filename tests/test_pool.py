"""The cache of freed device blocks, on the CPU: pool.cpp compiled over a counting stand-in for the HIP runtime
(tests/cpp/pool_harness.cpp), so that its bound, the order in which blocks leave it, blocks past it, memory that runs out
on the device or the host, a failed wait, two devices and eight threads are each seen exactly."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = """#pragma once
#include <cstddef>
#include <cstdint>
#define __host__
#define __device__
struct alignas(16) float4 { float x, y, z, w; };
struct alignas(16) uint4 { unsigned x, y, z, w; };
struct uint2 { unsigned x, y; };
struct alignas(32) double4 { double x, y, z, w; };
typedef struct ihipStream_t* hipStream_t;
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
hipError_t hipGetDevice(int*);
hipError_t hipSetDevice(int);
hipError_t hipMemGetInfo(size_t*, size_t*);
hipError_t hipGetLastError();
hipError_t hipDeviceSynchronize();
hipError_t hipMalloc(void**, size_t);
hipError_t hipFree(void*);
"""


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(STUB)
    exe = d / "pool"
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-I", str(d), "-I", ROOT,
                    os.path.join(ROOT, "tests", "cpp", "pool_harness.cpp"), "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("what", ["reuse", "bound_and_order", "large_blocks", "out_of_memory", "failed_wait", "two_devices",
                                  "host_memory_fails", "threads"])
def test_pool(harness, what):
    r = subprocess.run([harness, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
