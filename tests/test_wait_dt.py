"""The host's wait for a step's dt (csrc/runtime.h wait_dt), on the CPU against a
stand-in for the HIP calls: on one core it leaves the core to the thread that has
to run next instead of polling through its time slice, and it ends with an error
when the stream ends or fails without a dt."""
import os
import pathlib
import subprocess

from test_stage_device import HIP

CSRC = pathlib.Path(__file__).resolve().parents[1] / "cloverleaf3d_ref_amd" / "csrc"

DRIVER = r"""
#include <cstdio>
#include <ctime>
#include <thread>
#include "runtime.h"
using namespace clover;
static double cpu_s()
{
    timespec t;
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
    return t.tv_sec + 1e-9 * t.tv_nsec;
}
int main()
{
    const int n = 200;
    DtSlot a{}, b{};  // two threads hand a tag back and forth
    ihipStream st{0};
    const double t0 = cpu_s();
    std::thread other([&] {
        for (int q = 1; q <= n; q++) {
            const double x = wait_dt(&a, q, &st);
            b.dtlp = x + 1.0;
            __atomic_store_n(&b.seq, q, __ATOMIC_RELEASE);
        }
    });
    int bad = 0;
    for (int q = 1; q <= n; q++) {
        a.dtlp = q;
        __atomic_store_n(&a.seq, q, __ATOMIC_RELEASE);
        bad += wait_dt(&b, q, &st) != q + 1.0;
    }
    other.join();
    printf("cpu_s %.6f bad %d\n", cpu_s() - t0, bad);
    int errors = 0;
    for (hipError_t r : {hipSuccess, hipErrorInvalidHandle}) {
        g_query = r;
        try {
            wait_dt(&a, n + 1, &st);
        } catch (const Error &) {
            errors++;
        }
    }
    printf("errors %d\n", errors);
    return 0;
}
"""


def test_one_core(tmp_path):
    (tmp_path / "hip").mkdir()
    query = "inline hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }"
    assert query in HIP
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP.replace(
        query, "inline hipError_t g_query = hipErrorNotReady;\n"
               "inline hipError_t hipStreamQuery(hipStream_t) { return g_query; }"))
    src, exe = tmp_path / "wait.cpp", tmp_path / "wait"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-pthread", f"-I{tmp_path}", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    core = {min(os.sched_getaffinity(0))}
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120, check=True,
                       preexec_fn=lambda: os.sched_setaffinity(0, core))
    words = r.stdout.split()
    # 400 hand-overs, each some 20 us of polls: 8 ms of CPU time.  Polling through a time
    # slice (1 ms at the least) takes 400 ms.
    assert float(words[1]) < 0.1 and words[3] == "0", r.stdout
    assert words[5] == "2", r.stdout
