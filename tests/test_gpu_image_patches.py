"""Large 3x3 layers through reef_ops_conv2d (reef_conv2d_x9_g*): sizes that end inside a tile, a step of channels and a
group of output channels, a residual, and values that have no parts in bf16."""
import ctypes
import time

import numpy as np
import pytest

from oracle import oracle as O
from reef_amd import binding as B

pytestmark = pytest.mark.gpu


def run(x, w, b, res, act):
    cin, H, W = x.shape
    cout = w.shape[0]
    d = B.Conv2dDesc(cin, H, W, cout, 3, 3, 1, 1, 1, 1, act)
    bufs = [B.DeviceBuffer.from_array(a) if a is not None else None for a in (x, w, b, res)]
    out = B.DeviceBuffer(cout * H * W * 4)
    out.fill(0xFF)
    assert B.ops_conv2d(d, bufs[0], bufs[1], bufs[2], bufs[3], out) == 0, B.last_error()
    return out.to_array().reshape(cout, H, W)


# cin, H, W, cout, image rows: whole tiles; every edge ragged; few channels in; one column behind a segment; the same of four
# rows a tile: every edge ragged; whole rows of tiles; one column and one output channel behind the last tile
CASES = [(256, 112, 112, 256, 7), (252, 113, 83, 270, 7), (44, 139, 111, 326, 7), (84, 95, 97, 348, 7),
         (120, 86, 56, 292, 4), (580, 12, 79, 717, 4), (192, 98, 29, 369, 4), (276, 23, 129, 257, 4)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("residual", [False, True])
def test_against_64_bits(case, residual):
    B.ops_init()
    cin, H, W, cout, _ = case
    rng = np.random.default_rng(11)
    x = rng.standard_normal((cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((cout, cin, 3, 3)) * np.sqrt(2.0 / (cin * 9))).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32)
    res = rng.standard_normal((cout, H, W)).astype(np.float32) if residual else None
    got = run(x, w, b, res, 1)
    # some output channels, everywhere: the first and last of a wavefront and of the layer
    rows = sorted({0, 15, 16, 63, cout // 64 * 64 % cout, cout - 1})
    xp = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1)))
    ab = np.abs(xp)
    for m in rows:
        want, mag = np.full((H, W), float(b[m])), np.full((H, W), abs(float(b[m])))
        for i in range(3):
            for j in range(3):
                want += np.tensordot(w[m, :, i, j].astype(np.float64), xp[:, i:i + H, j:j + W], 1)
                mag += np.tensordot(np.abs(w[m, :, i, j]).astype(np.float64), ab[:, i:i + H, j:j + W], 1)
        if res is not None:
            want += res[m]
            mag += np.abs(res[m])
        # a rounding of at most 2^-24 of the sum of magnitudes per product and one each for the epilogue's terms
        assert (np.abs(got[m] - np.maximum(want, 0.0)) <= (9 * cin + 4) * 2.0 ** -24 * mag).all(), m


def test_values_without_parts():
    B.ops_init()
    cin, H, W, cout = 256, 112, 112, 256
    rng = np.random.default_rng(12)
    x = rng.standard_normal((cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((cout, cin, 3, 3)) * 0.02).astype(np.float32)
    plain = run(x, w, None, None, 0)
    x[3, 10, 20], x[5, 50, 60], x[255, 111, 111], x[0, 0, 0], x[17, 80, 30] = np.inf, np.nan, -np.inf, 3.4e38, -3.4e38
    got = run(x, w, None, None, 0)
    touched = np.zeros((H, W), bool)
    for y, z in ((10, 20), (50, 60), (111, 111), (0, 0), (80, 30)):
        touched[max(0, y - 1):y + 2, max(0, z - 1):z + 2] = True
    np.testing.assert_array_equal(got[:, ~touched], plain[:, ~touched])
    with np.errstate(all="ignore"):
        want = O.conv2d(x, w, np.zeros(cout, np.float32), None, None, None, (1, 1), (1, 1), 1, 0, 6.0, False).reshape(cout, H, W)[:, touched]
    got = got[:, touched]
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    ok = np.isfinite(want)
    # a value of 3.4e38 in the sum: its product decides
    np.testing.assert_allclose(got[ok], want[ok], rtol=1e-5, atol=1e-3)


@pytest.mark.parametrize("case", [CASES[1], CASES[4]])
def test_values_without_parts_cost_one_more_pass_over_the_channels(case):
    """NaN all over: an element at a time it took eighty times as long."""
    B.ops_init()
    cin, H, W, cout, _ = case
    rng = np.random.default_rng(13)
    x = rng.standard_normal((cin, H, W)).astype(np.float32)
    w = B.DeviceBuffer.from_array((rng.standard_normal((cout, cin, 3, 3)) * 0.02).astype(np.float32))
    d, out = B.Conv2dDesc(cin, H, W, cout, 3, 3, 1, 1, 1, 1, 0), B.DeviceBuffer(cout * H * W * 4)
    best = []
    for data in (x, np.full_like(x, np.nan)):
        inp, times = B.DeviceBuffer.from_array(data), []
        for _ in range(8):
            t0 = time.perf_counter()
            assert B.ops_conv2d(d, inp, w, None, None, out) == 0, B.last_error()
            times.append(time.perf_counter() - t0)
        best.append(min(times))
    assert np.isnan(out.to_array()).all() and best[1] < 5 * best[0], best


@pytest.mark.parametrize("case", [CASES[5], CASES[7]])
def test_values_without_parts_at_the_edges(case):
    """Infinities and NaN in the corners, in the last channel and in filters: the oracle's classes, everywhere."""
    B.ops_init()
    cin, H, W, cout, _ = case
    rng = np.random.default_rng(14)
    x = rng.standard_normal((cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((cout, cin, 3, 3)) * 0.02).astype(np.float32)
    x[0] = np.clip(x[0], -0.9, 0.9)      # (times 3.4e38 below the largest value: beside an infinity no sum depends on its order)
    x[cin - 1, H - 1, W - 1], x[0, 0, 0], x[cin // 2, 0, W - 1], x[5, H - 1, 0], x[3, H // 2, 16] = np.inf, np.nan, -np.inf, 3.4e38, np.inf
    # (filters in the middle tap: the pixels around the image are zeros that every kernel here multiplies, and the oracle leaves out)
    w[cout - 1, cin - 1, 1, 1], w[17, 2, 1, 1], w[33, 0, 2, 0] = np.inf, np.nan, 3.4e38
    got = run(x, w, None, None, 0)
    with np.errstate(all="ignore"):
        want = O.conv2d(x, w, np.zeros(cout, np.float32), None, None, None, (1, 1), (1, 1), 1, 0, 6.0, False).reshape(cout, H, W)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    ok = np.isfinite(want)
    np.testing.assert_allclose(got[ok], want[ok], rtol=1e-5, atol=1e-3)


# pixels, filters, both
@pytest.mark.parametrize("scales", [(1e-33, 1.0), (1e-35, 1.0), (1e-37, 1.0), (1.0, 1e-35), (1e-18, 1e-17), (1e-36, 1e-1)])
@pytest.mark.parametrize("case", [CASES[1], CASES[7]])
def test_small_operands_are_as_exact_as_others(case, scales):
    """(At 1e-36 the parts of a value keep 15 bits of it.)  Against the same layer on ordinary values; the errors are thousands of alike
    and independent ones: 1.1 for what their root mean square is known to, and a rounding to 2^-149 for each of the sums that an
    output goes through, three for nine channels' worth of 32-bit products."""
    B.ops_init()
    cin, H, W, cout, _ = case
    rng = np.random.default_rng(15)
    x0 = rng.standard_normal((cin, H, W)).astype(np.float32)
    w0 = (rng.standard_normal((cout, cin, 3, 3)) * 0.02).astype(np.float32)
    rows, errs = [0, 16, cout - 1], []
    for a, b in ((1.0, 1.0), scales):
        x, w = (x0 * np.float64(a)).astype(np.float32), (w0 * np.float64(b)).astype(np.float32)
        got = run(x, w, None, None, 0)[rows]
        xp = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1)))
        want = np.stack([sum(np.tensordot(w[m, :, i, j].astype(np.float64), xp[:, i:i + H, j:j + W], 1) for i in range(3) for j in range(3))
                         for m in rows])
        errs.append(np.linalg.norm(got - want) / np.linalg.norm(want))
    small = 2.0 ** -149 / 12 ** 0.5 * (3 * cin) ** 0.5 / np.sqrt((want ** 2).mean())
    assert errs[1] <= 1.1 * errs[0] + small, (errs, small)


def test_a_small_pixel_among_others_changes_nothing_else():
    B.ops_init()
    cin, H, W, cout, _ = CASES[4]
    rng = np.random.default_rng(16)
    x = rng.standard_normal((cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((cout, cin, 3, 3)) * 0.02).astype(np.float32)
    x[7, 40, 20] = 0.0
    plain = run(x, w, None, None, 0)
    x[7, 40, 20] = 1.0000001e-38
    np.testing.assert_array_equal(run(x, w, None, None, 0), plain)      # (far below a rounding of every sum)
    # alone in its surroundings it is all there is
    x[:, 38:43, 18:23] = 0.0
    x[7, 40, 20] = 1.0000001e-36
    got = run(x, w, None, None, 0)[:, 39:42, 19:22]
    want = w[:, 7, ::-1, ::-1].astype(np.float64) * x[7, 40, 20].astype(np.float64)
    assert (np.abs(got - want) <= 2.0 ** -22 * np.abs(want) + 3 * 2.0 ** -149).all()


def exact(x, w, rows):
    cin, H, W = x.shape
    xp = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1)))
    return np.stack([sum(np.tensordot(w[m, :, i, j].astype(np.float64), xp[:, i:i + H, j:j + W], 1) for i in range(3) for j in range(3)) for m in rows])


# (wide layers and deep ones; sums of the image-row kernels are split over four wavefronts and, for the last, over workgroups)
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("relu", [False, True])
def test_no_further_off_than_the_image_row_kernels(case, relu):
    """The same layer with a channel of zeros more runs on 32-bit products.  The errors are thousands of alike and independent ones:
    1.1 for what their root mean square is known to."""
    B.ops_init()
    cin, H, W, cout, rows = case
    rng = np.random.default_rng(17)
    x = rng.standard_normal((cin, H, W)).astype(np.float32)
    x = np.maximum(x, 0) if relu else x
    w = (rng.standard_normal((cout, cin, 3, 3)) * np.sqrt(2.0 / (cin * 9))).astype(np.float32)
    some = [0, 16, cout // 2, cout - 1]
    want, errs = exact(x, w, some), []
    for more in (1, 0):
        xm, wm = np.pad(x, ((0, more), (0, 0), (0, 0))), np.pad(w, ((0, 0), (0, more), (0, 0), (0, 0)))
        name = B.ops_conv2d_kernel(B.Conv2dDesc(cin + more, H, W, cout, 3, 3, 1, 1, 1, 1, 0))[0]
        assert ("_x9_" in name) == (not more), name
        errs.append(np.linalg.norm(run(xm, wm, None, None, 0)[some] - want) / np.linalg.norm(want))
    assert errs[1] <= 1.1 * errs[0], errs


@pytest.mark.parametrize("case", [CASES[1], CASES[4], CASES[7]])
def test_every_product_of_parts_is_there(case):
    """Filters with one weight each, all 24 bits in use: an output is one product, whose parts leave out at most 2^-23 of it, and
    is rounded when its sums meet, twice; without any of the six products four fifths of them are further off, up to 2^-16."""
    B.ops_init()
    cin, H, W, cout, _ = case
    rng = np.random.default_rng(18)
    x = np.ldexp(rng.integers(2 ** 23, 2 ** 24, (cin, H, W)) | 1, -23).astype(np.float32) * rng.choice((-1, 1), (cin, H, W)).astype(np.float32)
    some = list(range(0, cout, 5))
    for turn in range(2):
        w = np.zeros((cout, cin, 3, 3), np.float32)
        tap, ch = (np.arange(cout) + turn) % 9, (np.arange(cout) * 7 + 3 * turn) % cin       # every tap of every lane and k slot
        w[np.arange(cout), ch, tap // 3, tap % 3] = np.ldexp(rng.integers(2 ** 23, 2 ** 24, cout) | 1, -23)
        got, want = run(x, w, None, None, 0)[some], exact(x, w, some)
        assert (np.abs(got - want) <= 2.0 ** -22 * np.abs(want)).all()


def test_operands_that_lie_on_four_bytes():
    """A caller's tensors may start at any float; the filters are loaded sixteen bytes at a time."""
    B.ops_init()
    cin, H, W, cout, _ = CASES[7]
    rng = np.random.default_rng(19)
    x = rng.standard_normal((cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((cout, cin, 3, 3)) * 0.02).astype(np.float32)
    b, res = rng.standard_normal(cout).astype(np.float32), rng.standard_normal((cout, H, W)).astype(np.float32)
    want = run(x, w, b, res, 1)

    class At:
        def __init__(self, arr, skip):
            self.buf = B.DeviceBuffer.from_array(np.concatenate([np.zeros(skip, np.float32), arr.reshape(-1)]))
            self.ptr = ctypes.c_void_p(self.buf.ptr.value + 4 * skip)
    for skip in (1, 2, 3):
        ops = [At(a, skip) for a in (x, w, b, res, np.zeros_like(want))]
        d = B.Conv2dDesc(cin, H, W, cout, 3, 3, 1, 1, 1, 1, 1)
        assert B.ops_conv2d(d, *ops) == 0, B.last_error()
        np.testing.assert_array_equal(ops[4].buf.to_array()[skip:].reshape(want.shape), want)
