"""Many values divided by one (zig_gpt2_amd/csrc/lm_quotient.h, the last step of the latent attention of bf16 portions): the bits of the
division operator for sums of 1 to some thousand keys.  A multiplication with the reciprocal, which this replaced there, is a last bit away
for a quarter of them."""
import os
import subprocess

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zig_gpt2_amd", "csrc")

SOURCE = r"""
#include "lm_quotient.h"
extern "C" void quotients(const float* v, const float* by, float* corrected, float* plain, long n) {
    for (long i = 0; i < n; ++i) {
        const float inv = 1.0f / by[i];
        corrected[i] = zg::quotient(v[i], by[i], inv);
        plain[i] = v[i] * inv;
    }
}
"""


def test_bits_of_the_division(tmp_path):
    import ctypes as C

    src, lib = tmp_path / "q.cpp", tmp_path / "q.so"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", f"-I{CSRC}", "-o", str(lib), str(src)])
    f = C.CDLL(str(lib)).quotients
    rng = np.random.default_rng(5)
    n = 1 << 20
    v = np.concatenate([(rng.standard_normal(n) * 2.0 ** rng.integers(-20, 20, n)).astype(np.float32), np.arange(n, dtype=np.float32)])
    by = np.concatenate([rng.uniform(1, 2100, n).astype(np.float32), rng.integers(1, 2100, n).astype(np.float32)])
    odd = np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 1.0, -3.0e38], np.float32)
    vs, bs = np.meshgrid(odd, np.array([1.0, 3.0, np.inf, np.nan, 0.0, 2047.9999], np.float32))
    v, by = np.ascontiguousarray(np.concatenate([v, vs.ravel()])), np.ascontiguousarray(np.concatenate([by, bs.ravel()]))
    got, plain = np.empty_like(v), np.empty_like(v)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    f(p(v), p(by), p(got), p(plain), C.c_long(v.size))
    with np.errstate(all="ignore"):
        want = v / by
    assert np.array_equal(got, want, equal_nan=True)
    assert np.mean(plain[:2 * n] != want[:2 * n]) > 0.1  # (what the test would have said of the multiplication)
