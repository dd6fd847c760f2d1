"""reef_ops_conv2d: one fused convolution on plain device pointers (the call a kernel of the
reference's fused_nn_conv2d_* family serves, resource/resnet152/resnet152.cu:35,376) against the
CPU oracle, through the C-ABI.  Tolerance: 1e-4 of the output's largest magnitude (fp32)."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from reef_amd import binding as B
from tests.helpers import max_rel_err, REL_TOL

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(11)

# cin, H, W, cout, k, stride, pad, act, bias, residual
CASES = [
    (256, 14, 14, 256, 3, 1, 1, 1, True, False),     # row form, split folded inside the launch
    (64, 56, 56, 64, 3, 1, 1, 1, True, True),        # row form, single pass
    (1024, 14, 14, 256, 1, 1, 0, 1, True, False),    # 1x1 direct, split
    (256, 14, 14, 1024, 1, 1, 0, 0, False, True),    # 1x1 + residual
    (256, 56, 56, 128, 1, 2, 0, 1, True, False),     # strided 1x1
    (3, 64, 64, 64, 7, 2, 3, 1, True, False),        # 7x7 stem: K = 147, unaligned loader
    (24, 9, 11, 40, (1, 7), 1, (0, 3), 2, True, False),
    (16, 17, 17, 24, 5, 1, 2, 0, True, True),        # 25 taps: staged tile
    (40, 15, 15, 136, 3, 2, 1, 1, True, False),      # 3x3 stride 2: tap form
    (20, 5, 5, 8, 1, 1, 0, 0, False, False),         # 1x1 with Cin % 8 != 0: staged tile
]


def run_case(case, noalloc=False):
    cin, H, W, cout, k, s, p, act, has_bias, has_res = case
    kh, kw = (k, k) if isinstance(k, int) else k
    ph, pw = (p, p) if isinstance(p, int) else p
    Ho, Wo = (H + 2 * ph - kh) // s + 1, (W + 2 * pw - kw) // s + 1
    x = RNG.standard_normal((cin, H, W)).astype(np.float32)
    w = (RNG.standard_normal((cout, cin, kh, kw)) * np.sqrt(2.0 / (cin * kh * kw))).astype(np.float32)
    bias = RNG.standard_normal(cout).astype(np.float32) if has_bias else None
    res = RNG.standard_normal((cout, Ho, Wo)).astype(np.float32) if has_res else None
    ref = O.conv2d(x, w, bias, res, None, None, (s, s), (ph, pw), 1, act, 6.0, False)
    d = B.Conv2dDesc(cin, H, W, cout, kh, kw, s, s, ph, pw, act)
    bx, bw = B.DeviceBuffer.from_array(x), B.DeviceBuffer.from_array(w)
    bb = B.DeviceBuffer.from_array(bias) if has_bias else None
    br = B.DeviceBuffer.from_array(res) if has_res else None
    out = B.DeviceBuffer(cout * Ho * Wo * 4)
    out.fill(0xFF)
    st = B.ops_conv2d(d, bx, bw, bb, br, out, noalloc=noalloc)
    return st, out.to_array().reshape(cout, Ho, Wo), ref


@pytest.mark.parametrize("case", CASES)
def test_conv2d_op_matches_oracle(case):
    B.ops_init()
    st, got, ref = run_case(case)
    assert st == 0, B.last_error()
    assert np.isfinite(got).all()
    assert max_rel_err(got, ref) <= REL_TOL


def test_conv2d_op_rejects_bad_arguments():
    B.ops_init()
    buf = B.DeviceBuffer(1024)
    assert B.ops_conv2d(B.Conv2dDesc(0, 4, 4, 4, 1, 1, 1, 1, 0, 0, 0), buf, buf, None, None, buf) == 1
    assert "bad shape" in B.last_error()
    assert B.ops_conv2d(B.Conv2dDesc(4, 2, 2, 4, 5, 5, 1, 1, 0, 0, 0), buf, buf, None, None, buf) == 1
    assert B.ops_conv2d(B.Conv2dDesc(4, 4, 4, 4, 1, 1, 1, 1, 0, 0, 9), buf, buf, None, None, buf) == 1


def device_layer(case, seed):
    """A layer of CASES' form with operands in device memory."""
    cin, H, W, cout, k, s, p, act, has_bias, has_res = case
    rng = np.random.default_rng(seed)
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    arrays = [rng.standard_normal((cin, H, W)), rng.standard_normal((cout, cin, k, k)) * np.sqrt(2.0 / (cin * k * k)),
              rng.standard_normal(cout) if has_bias else None, rng.standard_normal((cout, Ho, Wo)) if has_res else None]
    arrays = [a if a is None else a.astype(np.float32) for a in arrays]
    bufs = [a if a is None else B.DeviceBuffer.from_array(a) for a in arrays]
    return B.Conv2dDesc(cin, H, W, cout, k, k, s, s, p, p, act), arrays, bufs, (cout, Ho, Wo)


@pytest.mark.parametrize("noalloc", [False, True])
def test_a_call_runs_with_its_own_arguments_whatever_came_before(noalloc):
    """Hundreds of calls in turn that differ in a pointer or two: each writes where it was told to, from what it was given."""
    B.ops_init()
    d, _, (x, w, _, _), shape = device_layer((64, 14, 14, 64, 1, 1, 0, 1, False, False), 1)
    _, _, (x2, w2, _, _), _ = device_layer((64, 14, 14, 64, 1, 1, 0, 1, False, False), 2)
    want = {}
    for i, a in enumerate((x, x2)):
        for j, b in enumerate((w, w2)):
            o = B.DeviceBuffer(4 * int(np.prod(shape)))
            assert B.ops_conv2d(d, a, b, None, None, o) == 0, B.last_error()
            want[i, j] = o.to_array()
    outs = [B.DeviceBuffer(4 * int(np.prod(shape))) for _ in range(70)]
    for rep in range(4):
        for o in outs:
            o.fill(0xFF)
        for n, o in enumerate(outs):
            i, j = (n + rep) % 2, (n // 2 + rep) % 2
            for _ in range(1 + n % 3):
                assert B.ops_conv2d(d, (x, x2)[i], (w, w2)[j], None, None, o, noalloc=noalloc) == 0, B.last_error()
        for n, o in enumerate(outs):
            np.testing.assert_array_equal(o.to_array(), want[(n + rep) % 2, (n // 2 + rep) % 2])


@pytest.mark.parametrize("case", [(64, 14, 14, 64, 1, 1, 0, 1, True, True), (1024, 14, 14, 256, 1, 1, 0, 1, True, False),
                                  (64, 112, 112, 64, 3, 1, 1, 0, True, True)])
def test_a_call_sees_what_the_caller_has_uploaded_since_the_last(case):
    """Operands that earlier calls have left in the caches are replaced by copies of up to 3 MiB, one at a time."""
    B.ops_init()
    d, _, first, shape = device_layer(case, 1)
    sets = [device_layer(case, seed)[1:3] for seed in (1, 2)]
    n = 4 * int(np.prod(shape))

    def call(bufs, out, noalloc=False):
        assert B.ops_conv2d(d, *bufs, out, noalloc=noalloc) == 0, B.last_error()
        return out.to_array()

    state = [0, 0, 0, 0]
    out = B.DeviceBuffer(n)
    for step in range(24):
        operand = step % 4
        if first[operand] is None:
            continue
        call(first, out, step % 3 == 0)
        state[operand] ^= 1
        a = sets[state[operand]][0][operand]
        assert B.lib().reef_hal_memcpy_h2d(first[operand].ptr, a.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(a.nbytes)) == 0
        mixed = [sets[s][1][k] for k, s in enumerate(state)]
        np.testing.assert_array_equal(call(first, out, step % 3 == 0), call(mixed, B.DeviceBuffer(n)))


@pytest.mark.parametrize("case", [(64, 14, 14, 64, 1, 1, 0, 1, True, True), (1024, 14, 14, 256, 1, 1, 0, 1, True, False)])
def test_a_waited_call_follows_the_default_stream_and_no_other(case):
    B.ops_init()
    L, size_t = B.lib(), ctypes.c_size_t
    d, _, bufs, shape = device_layer(case, 3)
    x, out = bufs[0], B.DeviceBuffer(4 * int(np.prod(shape)))
    x.fill(0)
    assert B.ops_conv2d(d, *bufs, out) == 0, B.last_error()
    want = out.to_array()
    x.fill(0xFF)
    big, side, idle = B.DeviceBuffer(1 << 30), ctypes.c_void_p(), ctypes.c_int()
    assert L.reef_hal_stream_create(0, ctypes.byref(side)) == 0      # a non-blocking one
    assert L.reef_hal_device_sync() == 0
    for _ in range(200):                                   # 1 GiB each: 30 ms and more
        assert L.reef_hal_memset_async(big.ptr, 0, size_t(big.nbytes), side) == 0
    for byte in (0xFF,) * 20 + (0,):                       # the default stream's last launch stores the input
        assert L.reef_hal_memset_async(x.ptr, byte, size_t(x.nbytes), None) == 0
    assert B.ops_conv2d(d, *bufs, out) == 0, B.last_error()
    assert L.reef_hal_stream_query(side, ctypes.byref(idle)) == 0
    np.testing.assert_array_equal(out.to_array(), want)
    assert not idle.value
    assert L.reef_hal_stream_destroy(side) == 0
