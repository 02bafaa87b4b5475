"""The launch shapes a mesh starts with follow the device's CUs (a partition has a
fraction of a whole GPU's), on the CPU: the rule is host code."""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parents[1]
PKG = ROOT / "cloverleaf3d_ref_amd"

DRIVER = r"""
#include <cstdio>
#include "fast.h"
using namespace clover;
int main()
{
    for (int n : {16, 64})
        for (int cus : {256, 128, 32}) {
            Lay g = make_lay(1, n, 1, n, 1, n);
            g.mirror = 63;
            printf("%d %d %d\n", n, cus, size_shapes(ST_F64, &g, 1, cus).k[SK_ACCEL_PDV].planes);
        }
}
"""


def test_fewer_cus_march_longer(tmp_path):
    src, exe = tmp_path / "shapes.cpp", tmp_path / "shapes"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{PKG / 'csrc'}", str(src), f"-L{PKG}", "-lclover_hip", f"-Wl,-rpath,{PKG}",
                    "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-lamdhip64", "-o", str(exe)], check=True)
    rows = [tuple(map(int, line.split())) for line in
            subprocess.run([str(exe)], capture_output=True, text=True, timeout=60, check=True).stdout.splitlines()]
    planes = {(n, cus): p for n, cus, p in rows}
    # 64 cells: 2 x 7 tiles of 61 columns and 10 rows, 65 planes; one workgroup per CU:
    # 17 chunks of 4 planes are 238 workgroups, one round of 256 CUs
    assert planes[64, 256] == 4
    for n in (16, 64):
        assert planes[n, 256] <= planes[n, 128] <= planes[n, 32], rows
    assert planes[64, 256] < planes[64, 32]
