"""fp32 Linears of many rows and 640 columns or more, and of some hundred rows and 1536 columns or more: three products of two-term fp16 planes on the
persistent GEMM (gemm_s4.hip) and on prefill_ring_kernel, whose rows carry exponents of their own.  Tile edges, ragged widths, one and several tiles a workgroup, both sides of the column rule, rows of very different
sizes, rows of zeros, of the smallest and of the largest values, values that are not finite.

Rows that two terms do not hold, few and many, are worked out another way.

The bound, element by element, is what three products of such terms can be off: 2^-21 of the sum of |x w| for the terms (2^-23 each and 2^-22
for the product that is left out), as much for what values far below their row's largest lose in the rows that are taken so, and 2^-24 of it for each of the
K / 8 additions of the matrix cores.  Nothing depends on a row's largest value: exact planes are inside it with any rows."""
import ctypes as C

import numpy as np
import pytest
import torch

from zig_gpt2_amd import _lib, ops

pytestmark = pytest.mark.gpu


def last_kernel(zg):
    name = C.create_string_buffer(160)
    _lib.check(zg.zg_debug_last_kernel(name, 160))
    return name.value.decode()


def draw(m, k, n, spread=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(m + 3 * n + 7 * k)
    x, w, b = (torch.randn(*s, generator=g, device="cuda") for s in ((m, k), (n, k), (n,)))
    if spread:
        x *= torch.exp2(torch.randint(-spread, spread, (m, 1), generator=g, device="cuda").float())
        w *= torch.exp2(torch.randint(-spread, spread, (n, 1), generator=g, device="cuda").float())
    return x, w, b


def forward(x, w, b):
    y = torch.full((x.shape[0], w.shape[0]), 7.0, device="cuda")
    torch.cuda.synchronize()  # (the library launches on a stream of its own)
    ops.Linear(x.shape[1], w.shape[0], w, b).forward(x, y)
    torch.cuda.synchronize()
    return y


def check(x, w, b, y):
    k = x.shape[1]
    ref = x.double() @ w.double().T
    size = x.abs().double() @ w.abs().double().T
    bound = (2.0 ** -20 + k / 8 * 2.0 ** -24) * size + 2.0 ** -149
    if b is not None:
        ref, bound = ref + b.double(), bound + 2.0 ** -23 * b.abs().double()
    over = ((y.double() - ref).abs() / bound).max().item()
    assert over <= 1.0, over
    return ((y.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("m,k,n", [(4096, 512, 3072), (4097, 576, 3071), (1537, 768, 3073), (8191, 640, 1601), (4501, 1600, 1601), (6401, 3072, 769), (12300, 512, 1029)])
def test_tile_edges(zg, m, k, n):
    x, w, b = draw(m, k, n)
    b = None if n % 2 else b
    before = zg.zg_debug_gemm_launches()
    y = forward(x, w, b)
    assert zg.zg_debug_gemm_launches() == before + 1 and last_kernel(zg) == "gemm_s4_kernel"
    # (2-norm: what a chain of K products in two halves and the terms leave, each seen in the comments of the kernels, and a third more)
    assert check(x, w, b, y) <= 1.33 * ((1.2e-7 * (k / 768) ** 0.5) ** 2 + 0.75e-7 ** 2) ** 0.5


@pytest.mark.parametrize("m,k,n,ring", [(700, 1600, 1600, 1), (700, 1600, 1603, 1), (321, 1600, 4800, 1), (1023, 3072, 769, 1), (700, 3072, 768, 1), (300, 2048, 8193, 1),
                                        (450, 6400, 1600, 1), (2049, 1536, 1031, 1), (1501, 1600, 1600, 1), (1409, 1600, 1667, 1), (1500, 3072, 768, 1),
                                        (2047, 6400, 1600, 1), (700, 1472, 1600, 0), (128, 1600, 1600, 0), (3000, 1600, 4800, 0),
                                        (65, 6400, 9601, 0), (128, 4800, 5120, 0), (192, 6400, 6400, 0), (478, 4096, 1024, 0), (420, 6400, 9601, 0)])  # (the weight's split pass would be most of the call)
def test_some_hundred_rows(zg, m, k, n, ring):
    """Tiles of 64 and 128 rows, of 64 and 128 columns, one slice of K and several, widths in no whole tiles and no whole fours, both sides of the rule."""
    x, w, b = draw(m, k, n, spread=9)
    b = None if n % 2 else b * 0.125
    before = zg.zg_debug_linear_ring_launches()
    y = forward(x, w, b)
    assert zg.zg_debug_linear_ring_launches() == before + ring
    check(x, w, b, y)


@pytest.mark.parametrize("m,k,n", [(700, 1600, 1600), (700, 3072, 769), (1501, 1600, 1600)])  # one slice, several; tiles of 128 columns
def test_values_that_are_not_finite_among_some_hundred_rows(zg, m, k, n):
    """Outputs are what a plain sum makes of them: infinities stay infinities of their sign."""
    x, w, b = draw(m, k, n)
    clean = forward(x, w, b)
    x[3, 100], x[300, 5], x[m - 1, k - 1] = float("nan"), float("inf"), -float("inf")
    w[11, 5] = 0.0  # (times infinity)
    before = zg.zg_debug_linear_ring_launches()
    y = forward(x, w, b)
    assert zg.zg_debug_linear_ring_launches() == before + 1
    bad = torch.zeros(m, dtype=torch.bool, device="cuda")
    bad[[3, 300, m - 1]] = True
    keep = torch.ones(n, dtype=torch.bool, device="cuda")
    keep[11] = False  # (its weight changed)
    assert torch.equal(y[~bad][:, keep], clean[~bad][:, keep])
    assert torch.isnan(y[3]).all() and torch.isnan(y[300, 11])
    assert torch.equal(y[300][keep], torch.copysign(torch.full((n,), float("inf"), device="cuda"), w[:, 5])[keep])
    assert torch.equal(y[m - 1], torch.copysign(torch.full((n,), float("inf"), device="cuda"), -w[:, k - 1]))


@pytest.mark.parametrize("wgs", ["3", "16"])
def test_many_tiles_a_workgroup(zg, monkeypatch, wgs):
    monkeypatch.setenv("ZGPT2_GEMM_WGS", wgs)  # the ring of exponents goes round several times
    x, w, b = draw(2100, 768, 2400, spread=12)
    check(x, w, b * 0, forward(x, w, b * 0))


def test_rows_of_any_size(zg):
    x, w, _ = draw(2048, 768, 3072, spread=40)
    x[5] = 0.0
    w[7] = 0.0
    x[9] *= 2.0 ** -100  # subnormal products and results
    x[11, 3] = 3.0e38
    x[13] = 1e-40
    w[15] = 1e-41
    y = forward(x, w, None)
    assert torch.equal(y[5], torch.zeros_like(y[5])) and torch.equal(y[:, 7], torch.zeros_like(y[:, 7]))
    finite = (x.double() @ w.double().T).abs().amax(1) < 3e38
    check(x[finite], w, None, y[finite])


def test_values_that_are_not_finite_stay_in_their_row(zg):
    x, w, b = draw(2048, 768, 3072)
    clean = forward(x, w, b)
    x[3, 100], x[700, 5], x[2047, 767] = float("nan"), float("inf"), -float("inf")
    y = forward(x, w, b)
    bad = torch.zeros(2048, dtype=torch.bool, device="cuda")
    bad[[3, 700, 2047]] = True
    assert torch.equal(y[~bad], clean[~bad]) and not torch.isfinite(y[bad]).any()


@pytest.mark.parametrize("k,err", [(512, 1.27e-7), (576, 1.353e-7), (640, 1.433e-7), (704, 1.511e-7), (1536, 2.32e-7)])
def test_no_further_from_64_bits_than_exact_planes(zg, k, err):
    """err: of three exact bf16 terms (4096 x k x 3072, the mean of three draws, which lie within 0.2 % of it)"""
    x, w, _ = draw(4096, k, 3072)
    assert check(x, w, None, forward(x, w, None)) <= 1.01 * err


def test_column_rule(zg):
    for k, err in ((448, 1.33 * 1.58e-7 * (448 / 768) ** 0.5), (512, 1.33 * 1.25e-7)):  # three exact terms below 512 columns
        x, w, b = draw(4096, k, 3072)
        y = forward(x, w, None)
        assert last_kernel(zg) == "gemm_s4_kernel"
        assert check(x, w, None, y) <= err


SHAPES = [(2048, 768, 3072, "s4"), (1500, 768, 3073, "s4"), (700, 1600, 1600, "ring"), (700, 3072, 769, "ring")]  # (the last in slices of K)


def launches(zg):
    return zg.zg_debug_gemm_launches() + zg.zg_debug_linear_ring_launches()


@pytest.mark.parametrize("m,k,n,path", SHAPES)
@pytest.mark.parametrize("top", [1e3, 1e6, 1e9, 1e12, 1e30])
def test_a_row_with_one_value_far_above_the_rest_that_meets_zeros(zg, m, k, n, path, top):
    """As one bf16 split after the other had it: the others' sum is as exact as without it."""
    for of_w in (False, True):
        x, w, b = draw(m, k, n)
        if of_w:
            w[n - 2, 11], x[:, 11] = top, 0.0
        else:
            x[m - 2, 11], w[:, 11] = top, 0.0
        check(x, w, b, forward(x, w, b))


@pytest.mark.parametrize("m,k,n,path", SHAPES)
@pytest.mark.parametrize("kind", ["spread within rows", "softmax rows", "identity", "half zeros", "sparse weights", "powers of two"])
def test_rows_of_all_kinds(zg, m, k, n, path, kind):
    g = torch.Generator(device="cuda")
    g.manual_seed(m + k)
    x, w, b = draw(m, k, n)
    b = None
    if kind == "spread within rows":
        x *= torch.exp2(torch.randint(-50, 50, x.shape, generator=g, device="cuda").float())
        w *= torch.exp2(torch.randint(-50, 50, w.shape, generator=g, device="cuda").float())
    elif kind == "softmax rows":
        x = torch.softmax(20 * x, -1)
    elif kind == "identity":
        x *= torch.exp2(torch.randint(-30, 30, x.shape, generator=g, device="cuda").float())
        w = torch.zeros_like(w)
        at = torch.arange(n, device="cuda")
        w[at, at % k] = 1.0
    elif kind == "half zeros":
        x = torch.relu(x)
    elif kind == "sparse weights":
        w *= torch.rand(w.shape, generator=g, device="cuda") < 0.05
    else:
        x = torch.exp2(torch.randint(-14, 15, x.shape, generator=g, device="cuda").float())
        w = torch.exp2(torch.randint(-14, 15, w.shape, generator=g, device="cuda").float())
    check(x, w, b, forward(x, w, b))


def test_ordinary_rows_are_taken_as_two_terms(zg):
    """One launch of the planes' kernel and none of another: normal values, ReLU outputs, weights with rows of zeros, with large values in some rows."""
    for m, k, n, path in SHAPES:
        x, w, b = draw(m, k, n)
        for change in (lambda: None, lambda: x.relu_(), lambda: w[5].zero_(), lambda: w[::7, 3].mul_(8.0), lambda: x[9].zero_()):
            change()
            before = launches(zg)
            y = forward(x, w, b)
            assert launches(zg) == before + 1 and last_kernel(zg).startswith("gemm_s4_kernel" if path == "s4" else "prefill_ring_kernel")
            check(x, w, b, y)


@pytest.mark.parametrize("m,k,n,path", SHAPES)
def test_outputs_that_are_not_finite(zg, m, k, n, path):
    """Infinities of their sign where a plain sum has them, in the buffers of a host caller as well."""
    x, w, b = draw(m, k, n)
    clean = forward(x, w, b)
    x[3, 100], x[300, 5], x[m - 1, k - 1] = float("nan"), float("inf"), -float("inf")
    w[n - 1, 7] = float("inf")
    y = forward(x, w, b)
    rows = torch.ones(m, dtype=torch.bool, device="cuda")
    rows[[3, 300, m - 1]] = False
    assert torch.equal(y[rows][:, :-1], clean[rows][:, :-1])
    inf = torch.full((), float("inf"), device="cuda")
    assert torch.isnan(y[3]).all()
    assert torch.equal(y[300, :-1], torch.copysign(inf, w[:-1, 5])) and torch.equal(y[m - 1, :-1], torch.copysign(inf, -w[:-1, k - 1]))
    assert torch.equal(y[rows][:, -1], torch.copysign(inf, x[rows][:, 7]))
    host = np.full((m, n), 7.0, np.float32)
    ops.Linear(k, n, w.cpu().numpy(), b.cpu().numpy()).forward(x.cpu().numpy(), host)
    assert np.array_equal(host, y.cpu().numpy(), equal_nan=True)


def test_host_buffers_and_rows_far_apart(zg):
    x, w, b = draw(2048, 768, 3072)
    x[7, 11], w[:, 11] = 1e12, 0.0
    y = forward(x, w, b)
    host = np.full((2048, 3072), 7.0, np.float32)
    ops.Linear(768, 3072, w.cpu().numpy(), b.cpu().numpy()).forward(x.cpu().numpy(), host)
    assert np.array_equal(host, y.cpu().numpy())
    check(x, w, b, y)


@pytest.mark.parametrize("m,k,n,path", SHAPES)
@pytest.mark.parametrize("rows", [1, 5, 300])
def test_rows_beside_rows_of_another_kind(zg, m, k, n, path, rows):
    """A few rows that two terms do not hold leave the others as they are, bit for bit; more of them and the call takes exact planes."""
    x, w, b = draw(m, k, n)
    clean = forward(x, w, b)
    at = torch.arange(rows, device="cuda") * 2 + 1
    for of_w in (False, True):
        x1, w1 = x.clone(), w.clone()
        (w1 if of_w else x1)[at, 3] = 1e12
        (x1 if of_w else w1)[:, 3] = 0.0  # (they meet zeros)
        reference = clean if rows == 300 else forward(x if not of_w else x1, w if of_w else w1, b)
        y = forward(x1, w1, b)
        check(x1, w1, b, y)
        if rows < 300:
            keep = torch.ones(n if of_w else m, dtype=torch.bool, device="cuda")
            keep[at] = False
            assert torch.equal(y[:, keep], reference[:, keep]) if of_w else torch.equal(y[keep], reference[keep])
