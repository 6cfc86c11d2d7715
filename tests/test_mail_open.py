"""Opening a context's message slots, compiled for the host against stand-ins
for the HIP calls: a failure at either call leaves the box closed, so that the
next run tries again instead of handing kernels a null address."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = """
#pragma once
#include <cstdlib>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
typedef void *hipStream_t;
enum { hipHostMallocMapped = 1, hipHostMallocCoherent = 2 };
#define __device__
#define __forceinline__ inline
#define __HIP_MEMORY_SCOPE_SYSTEM 0
template <class T> void __hip_atomic_store(T *p, T v, int, int) { *p = v; }
inline void __threadfence_system() {}
static int fail_malloc, fail_map, live;
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (fail_malloc)
        return hipErrorOutOfMemory;
    ++live;
    *p = std::malloc(n);
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p) { --live; std::free(p); return hipSuccess; }
inline hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned)
{
    if (fail_map)
        return hipErrorUnknown;
    *d = h;
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
"""

MAIN = """
#include "bx_mail.h"
int main()
{
    bx::MailBox b;
    fail_malloc = 1;
    if (b.open() == hipSuccess || b.slots || b.dev || live != 0)
        return 1;
    fail_malloc = 0;
    fail_map    = 1;
    if (b.open() == hipSuccess || b.slots || b.dev || live != 0)
        return 2;
    fail_map = 0;
    if (b.open() != hipSuccess || !b.slots || !b.dev || live != 1)
        return 3;
    bx::mail_post(b.dev, 5, 2.5, 1.0);
    if (!b.arrived(5) || b.wait(5, nullptr) != hipSuccess || b[5].v[0] != 2.5)
        return 4;
    b.close();
    return b.slots || b.dev || live != 0 ? 5 : 0;
}
"""


def test_a_failed_open_leaves_the_box_closed(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", str(tmp_path), "-I",
                    os.path.join(ROOT, "bamrex_amd", "csrc"), "-o", exe,
                    str(tmp_path / "main.cpp")], check=True)
    assert subprocess.run([exe]).returncode == 0
