"""The pinned rings of large field downloads (cf_copy.hip), on the CPU: the
file is compiled against a stand-in for the HIP runtime whose copies are
memcpys and which counts its pinned allocations.

Rings that two overlapping copies of one device left idle do not keep
another device from having one: its later copies take the ring of its first.
The rings kept are at most two, and none is left with the last run.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "ubiquitous-spoon_amd")

STUB = r"""
#pragma once
#include <cstdlib>
#include <cstring>
#include <atomic>
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorUnknown = 1 };
typedef void *hipStream_t;
typedef void *hipEvent_t;
enum { hipMemcpyDeviceToHost, hipHostMallocDefault, hipEventDisableTiming };
enum { hipMemoryTypeUnregistered = 0 };
struct hipPointerAttribute_t { int type; };
extern std::atomic<int> pinned, made;
extern void (*on_sync)();
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) { a->type = hipMemoryTypeUnregistered; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char *hipGetErrorString(hipError_t) { return ""; }
inline hipError_t hipHostMalloc(void **p, size_t n, int) { pinned++; made++; *p = malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void *p) { pinned--; free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, int) { *e = malloc(1); return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { if (on_sync) { void (*f)() = on_sync; on_sync = nullptr; f(); } return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
"""

MAIN = r"""
#include "chanflow.h"
#include "cf_internal_host.h"
#include <hip/hip_runtime.h>
#include <cstdarg>
#include <cstdio>
#include <vector>
std::atomic<int> pinned{ 0 }, made{ 0 };
void (*on_sync)() = nullptr;
extern "C" void cf_set_error(const char *, ...) {}
static const size_t N = ((size_t) 33 << 20) + 123;
static std::vector<char> src(N), dst(N);
static void copy(int device)
{
    std::fill(dst.begin(), dst.end(), 0);
    if (cf_copy_to_host(dst.data(), src.data(), N, device, nullptr) != CF_OK || dst != src) { puts("bad copy"); exit(1); }
}
int main()
{
    for (size_t i = 0; i < N; i++) src[i] = (char) (i * 2654435761u >> 13);
    if (cf_copy_users(1) != 1) return 2;
    on_sync = [] { std::vector<char> d(N); (void) cf_copy_to_host(d.data(), src.data(), N, 0, nullptr); };
    copy(0);                                    /* holds a ring while another copy takes one */
    printf("overlapping %d\n", made.load());
    copy(1);
    made = 0;
    for (int q = 0; q < 3; q++) copy(1);
    printf("again %d kept %d\n", made.load(), pinned.load());
    copy(0);
    printf("first device again %d\n", made.load());
    if (cf_copy_users(-1) != 0) return 2;
    printf("left %d\n", pinned.load());
    return 0;
}
"""


def test_rings_of_two_devices(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(tmp_path), "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(PKG, "host"), "-x", "c++", os.path.join(PKG, "csrc", "cf_copy.hip"), str(tmp_path / "main.cpp"),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.splitlines()
    assert out == ["overlapping 2", "again 0 kept 2", "first device again 0", "left 0"], out
