"""Handles of the layered tier are per device: nothing its library holds may be done once per process for whichever device came first."""
import pathlib
import re
import subprocess

CSRC = pathlib.Path(__file__).resolve().parents[1] / "zig_gpt2_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include "zg_once.h"
int main() {
    static zg::OncePerDevice once;
    int calls[4] = {0, 0, 0, 0};
    const int order[] = {0, 0, 3, 0, 3, 1, 1};
    for (int d : order) if (once.run(d, [&] { ++calls[d]; return 0; }) != 0) return 1;
    int failed = 0;                                   // a failure is not kept
    for (int i = 0; i < 2; ++i) if (once.run(2, [&] { ++failed; return 7; }) != 7) return 2;
    if (once.run(2, [&] { ++calls[2]; return 0; }) != 0) return 3;
    int far = 0;                                      // devices it has no bit for: every time
    for (int i = 0; i < 3; ++i) once.run(64, [&] { ++far; return 0; });
    std::printf("%d %d %d %d %d %d\n", calls[0], calls[1], calls[2], calls[3], failed, far);
}
"""


def test_once_per_device(tmp_path):
    src = tmp_path / "once.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "once"
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)]).split() == b"1 1 1 1 2 3".split()


def test_the_layered_library_keeps_no_flag_per_process():
    objects = re.search(r"^LM_OBJS := (.*)$", (CSRC / "Makefile").read_text(), re.M).group(1)
    for name in re.findall(r"build/(\w+)\.o", objects):
        assert not re.search(r"\bstatic (thread_local )?bool\b", (CSRC / f"{name}.hip").read_text()), name
