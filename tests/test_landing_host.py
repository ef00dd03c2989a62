"""The download path of snac_amd/csrc/snh_landing.h compiled for the host, its
HIP calls replaced by ones that copy at once, count and fail when told to:
every byte lands, for all sizes around a chunk and around the part of a
thread; the chunks are pinned for every device; a download for which events or
pinned memory are refused takes the plain copy and leaves no error behind for
the next launch to find; chunks are allocated, bounded and given back as the
header says; a download without a copy waits for the stream."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <stdio.h>
#include <atomic>
#include <vector>
typedef int hipError_t;
typedef void* hipStream_t;
typedef int* hipEvent_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipMemcpyDeviceToHost = 2, hipEventDisableTiming = 2,
       hipHostMallocDefault = 0, hipHostMallocPortable = 1 };
static std::atomic<int> mallocs{0}, frees{0}, not_portable{0}, events{0}, copies{0}, waits{0};
static int fail_malloc_at = -1, fail_event_at = -1;
static thread_local hipError_t last = hipSuccess;
static hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
static hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    if (mallocs++ == fail_malloc_at) return last = hipErrorOutOfMemory;
    if (!(flags & hipHostMallocPortable)) not_portable++;
    return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory;
}
static hipError_t hipHostFree(void* p) { frees++; free(p); return hipSuccess; }
static hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (events++ == fail_event_at) return last = hipErrorOutOfMemory;
    *e = new int(0);
    return hipSuccess;
}
static hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
static hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
static hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
static hipError_t hipStreamSynchronize(hipStream_t) { waits++; return hipSuccess; }
static hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
    copies++;
    memcpy(d, s, n);
    return hipSuccess;
}
#include "snh_landing.h"
"""

MAIN = r"""
static int bad = 0;
#define WANT(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); bad++; } } while (0)
static std::vector<char> src, dst;
static bool land(size_t bytes, size_t shift, size_t total) {
    Landing l(nullptr, total);
    memset(dst.data(), 0, bytes + shift + 64);
    const bool ok = l.push(dst.data() + shift, src.data(), bytes) == hipSuccess && l.finish() == hipSuccess;
    for (size_t k = 0; k < 64; k++)
        if (dst[bytes + shift + k]) return false;
    return ok && !memcmp(dst.data() + shift, src.data(), bytes) && hipGetLastError() == hipSuccess;
}
int main() {
    const size_t MB = (size_t)1 << 20, C = LAND_CHUNK;
    src.resize(48 * MB);
    dst.resize(49 * MB);
    for (size_t k = 0; k < src.size(); k++) src[k] = (char)(1 + (k * 2654435761u >> 13) % 250);
    land_context_made();
    /* a refused event: the plain copy, no error left */
    fail_event_at = 1;
    WANT(land(41 * MB, 8, 41 * MB));
    fail_event_at = -1;
    land_context_gone();
    WANT(frees == mallocs);
    /* refused pinned memory, the third chunk */
    land_context_made();
    fail_malloc_at = mallocs + 2;
    WANT(land(41 * MB, 8, 41 * MB));
    fail_malloc_at = -1;
    /* sizes around chunks and parts, odd destinations */
    for (size_t n : {C - 8, C, C + 8, 2 * C + 8, 5 * C, 5 * C + 4096, (size_t)8, (size_t)4096, (size_t)40000, 9 * C - 8})
        for (size_t s : {(size_t)0, (size_t)8, (size_t)16, (size_t)4088})
            WANT(land(n, s, 48 * MB));
    WANT(mallocs - frees <= LAND_CHUNKS + 1);   /* one was refused */
    land_context_gone();
    WANT(not_portable == 0);
    /* chunks only when downloads are worth them */
    land_context_made();
    const int m0 = mallocs;
    for (int k = 0; k < 6; k++) WANT(land(13 * MB, 8, 13 * MB));
    WANT(mallocs == m0);
    WANT(land(13 * MB, 8, 13 * MB) && mallocs == m0 + LAND_SLOTS);
    land_context_gone();
    land_context_made();
    for (int k = 0; k < 3; k++) WANT(land(13 * MB, 8, 13 * MB));
    WANT(mallocs == m0 + LAND_SLOTS);
    WANT(land(40 * MB, 8, 40 * MB) && mallocs == m0 + 2 * LAND_SLOTS);
    land_context_gone();
    /* nothing pushed: the stream is waited for */
    {
        Landing l(nullptr, 0);
        const int w = waits;
        WANT(l.finish() == hipSuccess && waits == w + 1);
    }
    /* the threads' parts cover a chunk once and part it at page boundaries */
    for (size_t n : {(size_t)4, (size_t)8, (size_t)4095, (size_t)4096, (size_t)70000, C - 8, C})
        for (uintptr_t d : {(uintptr_t)0x7f0000000000, (uintptr_t)0x7f0000000010, (uintptr_t)0x7f0000000ff8})
            for (size_t T : {1, 3, 8}) {
                size_t at = 0;
                for (size_t t = 0; t < T; t++) {
                    size_t a, b;
                    land_part((char*)d, n, T, t, &a, &b);
                    WANT(a == at && b >= a && b <= n);
                    WANT(b == n || (d + b) % 4096 == 0);
                    at = b;
                }
                WANT(at == n);
            }
    printf("bad %d\n", bad);
    return bad != 0;
}
"""


def test_landing_on_the_host(tmp_path):
    src, exe = tmp_path / "landing.cpp", tmp_path / "landing"
    src.write_text(HIP + MAIN)
    subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "snac_amd", "csrc"),
                           "-o", str(exe), str(src)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "bad 0" in r.stdout, r.stdout + r.stderr
