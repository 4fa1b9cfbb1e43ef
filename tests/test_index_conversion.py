"""The sample index of a t/dt that no int holds.  A trace's traveltime may be a NaN, an
infinity or far past the trace (negative radicands, candidates with c = inf); the window test
must then come out of the device's own conversion, not of what the compiler makes of an
undefined one.  Compiled for the device with such values as constants, a defined conversion
stays in the code; an undefined one is folded away, and with it the test."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "highperformanceseismicstacking_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SOURCE = """
#include "kernels/device_common.hpp"
using namespace hss;
extern "C" __global__ void probe(int *out, IndexBounds ib) {
    int k;
    float f;
    const float t = VALUE;
    out[0] = CALL;
    out[1] = k;
}
"""
CALLS = {"window_k": "window_k<true>(t, 1.0f, 1.0f, ib, &k, &f)",
         "window_index": "window_index<true>(t, 1.0f, 1.0f, ib, ib.tau, &k, &f)"}


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("call", list(CALLS))
@pytest.mark.parametrize("value", ["__builtin_nanf(\"\")", "3e9f", "-3e9f"])
def test_the_conversion_is_the_devices(call, value, tmp_path):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(SOURCE.replace("VALUE", value).replace("CALL", CALLS[call]))
    subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "--cuda-device-only", "-S", f"-I{CSRC}", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    assert re.search(r"^\s+v_cvt_i32_f32", out.read_text(), re.M)
