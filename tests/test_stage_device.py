"""Field transfers of owners on different devices (csrc/transfer.hip), on the CPU:
the host code of Stage runs against a stand-in for the HIP calls it makes, which
refuses an event on another device's stream, as HIP does.  The kernels' moves are
not run."""
import pathlib
import subprocess

CSRC = pathlib.Path(__file__).resolve().parents[1] / "cloverleaf3d_ref_amd" / "csrc"

HIP = r"""
#pragma once
#include <cstdlib>
#define __host__
#define __device__
#define __global__
#define __launch_bounds__(n)
struct dim3 { unsigned x, y, z; dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {} };
inline dim3 threadIdx, blockIdx, gridDim;
enum hipError_t { hipSuccess = 0, hipErrorInvalidHandle = 400, hipErrorOutOfMemory = 2, hipErrorNotReady = 600 };
struct ihipStream { int device; };
struct ihipEvent { int device; };
typedef ihipStream *hipStream_t;
typedef ihipEvent *hipEvent_t;
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
inline int g_device = 0, g_events = 0;
inline const char *hipGetErrorString(hipError_t) { return "refused"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { *d = g_device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { g_device = d; return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, int *d) { *d = s->device; return hipSuccess; }
inline hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
enum hipDeviceAttribute_t { hipDeviceAttributeMultiprocessorCount };
inline hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = calloc(n, 1); return hipSuccess; }
inline hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
inline hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new ihipEvent{g_device}; g_events++; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; g_events--; return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return e->device == s->device ? hipSuccess : hipErrorInvalidHandle; }
#define hipLaunchKernelGGL(...) ((void)0)
"""

DRIVER = r"""
#include <cstdio>
#include <vector>
#include "transfer.hip"
using namespace clover;
int main()
{
    ihipStream streams[2] = {{0}, {1}};
    const Lay g = make_lay(1, 7, 1, 5, 1, 3);
    std::vector<double> host(12 * 10 * 8), dev((size_t)lay_elems(g));
    int bad = 0;
    for (int owner = 0; owner < 2; owner++)
        for (int current = 0; current < 2; current++)
            for (int up = 0; up < 2; up++) {
                Stage stage;
                hipSetDevice(current);
                try {
                    if (up) stage.upload(g, AC_CELL, host.data(), dev.data(), &streams[owner]);
                    else stage.download(g, AC_VERT, dev.data(), 8, host.data(), &streams[owner]);
                } catch (const Error &e) {
                    printf("owner on %d, device %d current, %s: %s\n", owner, current, up ? "upload" : "download", e.what());
                    bad++;
                }
                if (g_device != current) { printf("current device changed\n"); bad++; }
                stage.release();
                if (g_events) { printf("%d events left\n", g_events); bad++; }
            }
    return bad != 0;
}
"""


def test_transfers_use_the_streams_device(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    src, exe = tmp_path / "stage.cpp", tmp_path / "stage"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", f"-I{tmp_path}", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
