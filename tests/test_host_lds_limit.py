"""Dynamic LDS above the default is a property of a kernel on one device: the host helper that asks for it, compiled against a
stand-in for the three runtime calls it makes (no GPU)."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "machx_inference_engine_amd", "csrc")

PROGRAM = r"""
#include "mxq_host.h"
#include <assert.h>
namespace mxq { thread_local int g_last_hip_error = 0; }
static int device = 0, asked = 0, refused = 0, pending = 0;
extern "C" hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) {
    ++asked;
    if (refused) pending = hipErrorInvalidValue;
    return refused ? hipErrorInvalidValue : hipSuccess;
}
extern "C" hipError_t hipGetLastError() { const int e = pending; pending = 0; return (hipError_t)e; }
int main() {
    static mxq::LdsLimit a, b;
    assert(mxq::raise_lds_limit(&a, a, 100000) == MX_OK && asked == 1);
    assert(mxq::raise_lds_limit(&a, a, 100000) == MX_OK && asked == 1);      // once per device
    device = 1;
    assert(mxq::raise_lds_limit(&a, a, 100000) == MX_OK && asked == 2);      // the second device is asked too
    assert(mxq::raise_lds_limit(&b, b, 100000) == MX_OK && asked == 3);      // and every kernel by itself
    device = 2;
    refused = 1;
    assert(mxq::raise_lds_limit(&a, a, 100000) == MX_ERR_LAUNCH && pending == 0);   // no error left for the launch that follows
    refused = 0;
    assert(mxq::raise_lds_limit(&a, a, 100000) == MX_OK && asked == 5);
    device = mxq::kMaxDevices;
    assert(mxq::raise_lds_limit(&a, a, 100000) == MX_ERR_LAUNCH && asked == 5);
    return 0;
}
"""


def test_limit_is_asked_for_once_per_kernel_and_device(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-x", "c++", "-D__HIP_PLATFORM_AMD__", "-std=c++17", "-I", CSRC,
                    "-I", "/opt/rocm/include", str(src), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)


def test_every_opt_in_goes_through_the_helper():
    users = [f for f in sorted(os.listdir(CSRC)) if f.endswith((".hip", ".cpp", ".h")) and re.search(r"hipFuncSetAttribute\(", open(os.path.join(CSRC, f)).read())]
    assert users == ["mxq_host.h"]
