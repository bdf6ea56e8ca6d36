"""csrc/launch.hpp on the host: a small program that includes it, with the HIP
runtime calls it makes replaced by ones that record their arguments."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bare-metal-bard_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include <stdio.h>
#include "launch.hpp"
static int device = 0;
extern "C" hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int v) {
    printf("%d %d %d\n", device, (int)(size_t)f, v);
    return hipSuccess;
}
namespace bmb { void note_launch_status(hipError_t) {} }
int main() {
    typedef void (*kernel)(float *);
    const kernel a = (kernel)1, b = (kernel)2;
    bmb::allow_smem(a, 65536);
    bmb::allow_smem(a, 98304);   // set
    bmb::allow_smem(a, 98304);
    bmb::allow_smem(a, 131072);  // set: more than before
    bmb::allow_smem(a, 70000);
    bmb::allow_smem(b, 70000);   // set: another kernel
    device = 1;
    bmb::allow_smem(a, 70000);   // set: another device
    bmb::allow_smem(a, 163840);  // set
}
"""


def test_lds_limit_is_raised_for_every_larger_request(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    src, obj, exe = (str(tmp_path / n) for n in ("p.cpp", "p.o", "p"))
    with open(src, "w") as f:
        f.write(PROGRAM)
    for cmd in ([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-fPIC",
                 "-I" + CSRC, "-c", src, "-o", obj], ["g++", obj, "-o", exe]):
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split("\n")[:-1] == ["0 1 98304", "0 1 131072", "0 2 70000", "1 1 70000",
                                         "1 1 163840"]
