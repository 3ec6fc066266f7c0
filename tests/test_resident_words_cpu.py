"""What the words of the resident decode kernels rest on (decode_resident_order.h), in the instructions they become: near stores stay in the
XCD's L2 (no sc1), far ones go to the memory side, polls pass the L1, all of them eight bytes at once, and a poll waits for everything its wave has
asked for and stored before."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zig_gpt2_amd", "csrc")

SOURCE = r"""
#include "decode_resident_parts.h"
using namespace zg::resident;
extern "C" __global__ void near_store(u64* p, unsigned t, float v) { put_near(p, threadIdx.x, tagged(t, v)); }
extern "C" __global__ void far_store(u64* p, unsigned t, float v) { put_far(p, threadIdx.x, tagged(t, v)); }
extern "C" __global__ void poll(u64* p, float* q, float* row, unsigned t, unsigned limit) {
    __shared__ unsigned f;
    Waiter w{limit, &f};
    row[threadIdx.x] = 1.0f;
    q[threadIdx.x] = w.get(p, threadIdx.x, t);
}
"""


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    d = tmp_path_factory.mktemp("words")
    (d / "w.hip").write_text(SOURCE)
    subprocess.run(["/opt/rocm/bin/hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{CSRC}", "-o", str(d / "w.s"), str(d / "w.hip")], check=True, stderr=subprocess.DEVNULL)
    text = (d / "w.s").read_text()
    return {k: [ln.split(";")[0].strip() for ln in re.search(rf"^{k}:.*?s_endpgm", text, re.M | re.S).group(0).splitlines()] for k in ("near_store", "far_store", "poll")}


def memory(lines):
    return [ln for ln in lines if re.match(r"(global|flat|buffer)_", ln)]


def test_stores(kernels):
    near, = memory(kernels["near_store"])
    far, = memory(kernels["far_store"])
    assert near.startswith("global_store_dwordx2") and "sc1" not in near.split(), near
    assert far.startswith("global_store_dwordx2") and "sc1" in far.split(), far


def test_polls(kernels):
    lines = [ln for ln in kernels["poll"] if ln]
    loads = [i for i, ln in enumerate(lines) if "_load_" in ln and ln.startswith(("global", "flat", "buffer"))]
    first_store = next(i for i, ln in enumerate(lines) if "global_store_dword " in ln)
    assert loads and first_store < loads[0]
    for i in loads:
        assert lines[i].startswith("global_load_dwordx2") and "sc1" in lines[i].split(), lines[i]
        wait = next(ln for ln in lines[i:] if ln.startswith("s_waitcnt") and "vmcnt" in ln)
        assert "vmcnt(0)" in wait, wait
