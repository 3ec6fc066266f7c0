"""fp32 Linears of few rows and of a medium number of rows (linear_tiles.hip): rows and columns around the edges of its tiles, one slice of K and several,
the fewest and the most steps a slice has, sizes on both sides of the rule that leaves a Linear to the other kernels, values that are
not finite."""
import numpy as np
import pytest

import oracle
from golden_io import assert_ref_close
from zig_gpt2_amd import ops, synth

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


@pytest.mark.parametrize("m,k,n", [(5, 6400, 70), (8, 8192, 40), (1500, 128, 3072), (2000, 128, 3072), (4100, 128, 1600), (20, 16448, 24), (40, 100, 37), (12, 64, 9)])
def test_both_sides_of_the_rule(zg, m, k, n):
    w, b, x, y = run(m, k, n)
    assert_ref_close(oracle.linear_forward(k, n, w, b, x), y, f"Linear {m}x{k}x{n}", scale_floor=2e-6)


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


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("m,k", [(70, 768), (8, 520), (3, 2056)])
def test_values_that_are_not_finite(zg, bad, m, k):
    n, at = 96, m - 2
    x = synth.fill_normal(1, m * k, 0, 1.0).reshape(m, k).copy()
    clean = run(m, k, n, x=x)[3]
    x[at, k - 1] = bad  # (what a lane beyond the row's end loads again)
    y = run(m, k, n, x=x)[3]
    assert not np.isfinite(y[at]).any()
    keep = np.arange(m) != at
    assert np.array_equal(y[keep], clean[keep])
