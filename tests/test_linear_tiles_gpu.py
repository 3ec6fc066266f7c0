"""fp32 Linears of few rows and of a medium number of rows (linear_tiles.hip): rows and columns around the edges of its tiles, one slice of K and several,
the fewest and the most steps a slice has, sizes on both sides of the rule that leaves a Linear to the other kernels, values that are
not finite."""
import ctypes as C

import numpy as np
import pytest

import oracle
from golden_io import assert_ref_close
from zig_gpt2_amd import _lib, ops, synth

pytestmark = pytest.mark.gpu


def run(m, k, n, bias=True, x=None):
    w = synth.fill_normal(100 + n, n * k, 0, 0.05).reshape(n, k)
    b = synth.fill_normal(200 + n, n, 0, 0.05) if bias else None
    x = synth.fill_normal(300 + m, m * k, 0, 1.0).reshape(m, k) if x is None else x
    y = np.full((m, n), 7.0, np.float32)
    ops.Linear(k, n, w, b).forward(x, y)
    return w, b, x, y


@pytest.mark.parametrize("m", [9, 15, 16, 63, 64, 65, 130])
@pytest.mark.parametrize("k,n", [(128, 1), (128, 64), (192, 65), (384, 63), (768, 260), (3072, 129), (6400, 66), (8192, 8)])
def test_tile_edges(zg, m, k, n):
    w, b, x, y = run(m, k, n, bias=n % 2 == 0)
    assert_ref_close(oracle.linear_forward(k, n, w, b, x), y, f"Linear {m}x{k}x{n}", scale_floor=2e-6)


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 7, 8])
@pytest.mark.parametrize("k,n", [(64, 1), (512, 9), (520, 16), (768, 1031), (1032, 65), (1528, 8), (1536, 3), (2056, 130), (8192, 5), (128, 6200), (60, 9), (100, 7)])
def test_few_rows(zg, m, k, n):
    w, b, x, y = run(m, k, n, bias=n % 2 == 1)
    assert_ref_close(oracle.linear_forward(k, n, w, b, x), y, f"Linear {m}x{k}x{n}", scale_floor=2e-6)


@pytest.mark.parametrize("m,k,n,kernel", [(5, 6400, 70, "linear_few"), (8, 8192, 40, "linear_few"), (8, 128, 6144, "linear_few"), (8, 128, 6152, "gemv"),
                                          (4, 128, 6152, "linear_few"), (1500, 128, 3072, "linear_tiles"), (1856, 128, 3072, "linear_tiles"),
                                          (1857, 128, 3072, "gemm_s4"), (2000, 128, 3072, "gemm_s4"), (4100, 128, 1600, "gemm_s4"), (20, 16448, 24, "linear_tiles"),
                                          (40, 100, 37, "gemv"), (12, 64, 9, "gemv"), (1, 768, 768, "gemv")])
def test_both_sides_of_the_rule(zg, m, k, n, kernel):
    run(1, 768, 768)  # (a general kernel; the ragged ones among them leave the note as it is)
    w, b, x, y = run(m, k, n)
    name = C.create_string_buffer(160)
    _lib.check(zg.zg_debug_last_kernel(name, 160))
    assert name.value.decode().startswith(kernel)
    assert_ref_close(oracle.linear_forward(k, n, w, b, x), y, f"Linear {m}x{k}x{n}", scale_floor=2e-6)


@pytest.mark.parametrize("m,k,n,kernel", [
    (4, 512, 15, "linear_few"), (5, 512, 15, "matrix cores"), (15, 512, 64, "matrix cores"), (16, 512, 64, "linear_tiles"),
    # five to eight rows: 512 columns, 1024 of more than 2048 outputs, 1536 to 1792 of more than 1024
    (8, 248, 6144, "matrix cores"), (8, 248, 6145, "gemv"), (8, 256, 6145, "matrix cores"), (8, 520, 33, "linear_few"),
    (8, 520, 2048, "linear_few"), (8, 520, 2049, "matrix cores"), (8, 1024, 2049, "matrix cores"), (8, 1032, 2049, "linear_few"),
    (8, 1528, 1025, "linear_few"), (8, 1536, 1024, "linear_few"), (8, 1536, 1025, "matrix cores"),
    (5, 1792, 1025, "matrix cores"), (5, 1800, 1025, "linear_few"),
    # nine to fifteen: 128 to 1024 columns, to 1792 of up to 4096 outputs
    (9, 120, 40, "gemv"), (9, 128, 40, "matrix cores"), (9, 1024, 4097, "matrix cores"), (9, 1088, 4096, "matrix cores"),
    (9, 1088, 4097, "linear_tiles"), (15, 1792, 4096, "matrix cores"), (15, 1856, 40, "linear_tiles"), (15, 1800, 40, "gemv")])
def test_which_kernel_takes_few_rows(zg, m, k, n, kernel):
    run(1, 768, 768)  # (a general kernel; the ragged ones among them leave the note as it is)
    before = zg.zg_debug_linear_few_mfma_launches()
    w, b, x, y = run(m, k, n)
    name = C.create_string_buffer(160)
    _lib.check(zg.zg_debug_last_kernel(name, 160))
    assert zg.zg_debug_linear_few_mfma_launches() - before == (kernel == "matrix cores")
    assert name.value.decode().startswith("linear_few" if kernel == "matrix cores" else kernel), name.value
    assert_ref_close(oracle.linear_forward(k, n, w, b, x), y, f"Linear {m}x{k}x{n}", scale_floor=2e-6)


@pytest.mark.parametrize("m", [5, 8, 9, 15])
@pytest.mark.parametrize("k,n", [(64, 1), (120, 40), (136, 1), (136, 6145), (256, 16), (264, 17), (512, 15), (520, 33), (768, 2049), (1024, 2048), (1032, 31),
                                 (1536, 1025), (1792, 4096), (1784, 4097), (1800, 40)])
def test_few_rows_on_the_matrix_cores(zg, m, k, n):
    """Five to fifteen rows: the last columns of a piece, weight rows around the tile's sixteen, one piece of a wave to seven; those of them that the
    rule gives to other kernels are held to the same.  A row that is not finite stays by itself."""
    w, b, x, y = run(m, k, n, bias=n % 2 == 1)
    assert_ref_close(oracle.linear_forward(k, n, w, b, x), y, f"Linear {m}x{k}x{n}", scale_floor=2e-6)
    xs = x.copy()
    xs[m - 1, k - 1], xs[m - 2, k - 8] = np.inf, np.nan
    ys = run(m, k, n, bias=n % 2 == 1, x=xs)[3]
    with np.errstate(all="ignore"):
        assert_same_class(oracle.linear_forward(k, n, w, b, xs)[m - 2:], ys[m - 2:], "not finite")
    assert np.array_equal(ys[:m - 2], y[:m - 2])


@pytest.mark.parametrize("m", [0, 1, 2, 8, 9, 16, 70])
@pytest.mark.parametrize("k", [100, 128, 768, 8200, 16384])
def test_no_outputs(zg, m, k):
    """No output columns, or no rows: nothing to do, whichever kernel's rule would have been asked."""
    x = synth.fill_normal(1, m * k, 0, 1.0).reshape(m, k)
    ops.Linear(k, 0, np.zeros((1, k), np.float32), None).forward(x, np.zeros((m, 0), np.float32))
    ops.Linear(k, 0, np.zeros((1, k), np.float32), np.zeros(1, np.float32)).forward(x, np.zeros(0, np.float32))
    y = np.full((1, 3), 7.0, np.float32)
    ops.Linear(k, 3, synth.fill_normal(2, 3 * k, 0, 1.0).reshape(3, k), None).forward(x[:0], y)
    assert (y == 7.0).all()


def assert_same_class(want, y, what):
    """Infinities and NaN where the oracle has them, of its sign; the rest close to it (row by row: their sizes differ)."""
    assert np.array_equal(np.isnan(y), np.isnan(want)), what
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(y), inf) and np.array_equal(y[inf], want[inf]), what
    for w, v in zip(want, y):
        ok = np.isfinite(w)
        assert_ref_close(w[ok], v[ok], what, scale_floor=2e-6)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("m,k", [(70, 768), (8, 520), (3, 2056)])
def test_values_that_are_not_finite(zg, bad, m, k):
    n, at = 96, m - 2
    x = synth.fill_normal(1, m * k, 0, 1.0).reshape(m, k).copy()
    clean = run(m, k, n, x=x)[3]
    x[at, k - 1] = bad  # (what a lane beyond the row's end loads again)
    run_w, run_b, _, y = run(m, k, n, x=x)
    with np.errstate(all="ignore"):
        assert_same_class(oracle.linear_forward(k, n, run_w, run_b, x)[at:at + 1], y[at:at + 1], f"{bad}")
    keep = np.arange(m) != at
    assert np.array_equal(y[keep], clean[keep])


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 3.4e38, -3.4e38])
@pytest.mark.parametrize("m,k,n", [(9, 128, 96), (12, 768, 130), (15, 3072, 65), (70, 768, 96), (9, 128, 33000), (130, 192, 8300)])
def test_what_an_fp32_sum_keeps(zg, bad, m, k, n):
    """An infinity times a number is an infinity, times zero NaN; a number beyond the largest bf16 is a number: in a row of inputs, and in
    a row of weights (one slice of K and several).  Some of what they meet has one bf16 term only, whose other terms are zero."""
    x = synth.fill_normal(1, m * k, 0, 1.0).reshape(m, k).copy()
    w = synth.fill_normal(2, n * k, 0, 0.05).reshape(n, k).copy()
    b = synth.fill_normal(3, n, 0, 0.05)
    row, at = m - 2, k - 3
    w[: n // 2, at] = np.resize(np.array([1.0, -2.0, 0.5, 0.0, 1e-30, -1e-30, 2.0 ** -130], np.float32), n // 2)
    xs, ws = x.copy(), w.copy()
    xs[row, at] = bad
    with np.errstate(all="ignore"):
        want = oracle.linear_forward(k, n, w, b, xs)
        y = np.full((m, n), 7.0, np.float32)
        ops.Linear(k, n, w, b).forward(xs, y)
        assert_same_class(want, y, f"input {bad}")
        col = n - 1
        x[: m // 2, at] = np.resize(np.array([1.0, -2.0, 0.0, 1e-30], np.float32), m // 2)
        ws[col, at] = bad
        want = oracle.linear_forward(k, n, ws, b, x)
        ops.Linear(k, n, ws, b).forward(x, y)
        assert_same_class(want[:, :col], y[:, :col], f"beside weight {bad}")
        assert_same_class(want[:, col:], y[:, col:], f"weight {bad}")


@pytest.mark.parametrize("m,k,n", [(9, 128, 96), (12, 768, 130), (70, 3072, 96)])
@pytest.mark.parametrize("size", [1e-37, 2e-38, 1e-30])
def test_small_numbers(zg, size, m, k, n):
    """Inputs whose second and third terms are below the smallest normal number (their products are normal numbers again)."""
    x = (synth.fill_normal(1, m * k, 0, 1.0) * np.float32(size)).reshape(m, k)
    w = (synth.fill_normal(2, n * k, 0, 1.0) * np.float32(1e30)).reshape(n, k)
    y = np.full((m, n), 7.0, np.float32)
    ops.Linear(k, n, w, None).forward(x, y)
    assert_ref_close(oracle.linear_forward(k, n, w, None, x), y, f"Linear {m}x{k}x{n} at {size}", scale_floor=2e-6)
