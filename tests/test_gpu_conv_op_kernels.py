"""The kernels behind reef_ops_conv2d where they can go wrong: filters by rows (any height, few and many
channels, rows outside the image), 1x1 filters on channel counts that fill no load, image rows and
staged tiles at ragged sizes, splits of K -- against the oracle; and the argument copies and
workspaces that calls share."""
import threading

import numpy as np
import pytest

from oracle import oracle as O
from reef_amd import binding as B
from tests.helpers import max_rel_err, REL_TOL

pytestmark = pytest.mark.gpu

# cin, H, W, cout, (kh, kw), stride, (ph, pw)
CASES = [(1, 9, 9, 1, (3, 3), 1, (1, 1)), (3, 30, 31, 33, (7, 7), 2, (3, 3)), (37, 12, 50, 9, (7, 7), 1, (3, 3)),
         (210, 9, 20, 14, (7, 7), 2, (3, 3)), (5, 17, 19, 40, (5, 5), 2, (2, 2)), (130, 11, 12, 70, (5, 5), 1, (2, 2)),
         (19, 14, 13, 21, (5, 3), 1, (2, 1)), (19, 14, 13, 21, (3, 5), 2, (0, 0)), (6, 20, 9, 17, (11, 3), 1, (5, 1)),
         (33, 8, 40, 18, (1, 5), 1, (0, 2)), (33, 40, 8, 18, (7, 1), 1, (3, 0)), (33, 40, 8, 18, (3, 1), 2, (1, 0)),
         (2, 6, 6, 65, (1, 1), 1, (0, 0)), (63, 7, 9, 31, (1, 1), 1, (0, 0)), (257, 5, 5, 20, (1, 1), 1, (0, 0)),
         (129, 13, 11, 16, (1, 1), 2, (0, 0)), (4, 5, 5, 8, (1, 1), 1, (1, 1)), (300, 15, 29, 17, (3, 3), 1, (1, 1)),
         (9, 13, 15, 10, (2, 2), 1, (0, 0)), (12, 16, 16, 24, (4, 4), 2, (1, 1)), (700, 4, 4, 33, (3, 3), 2, (1, 1)),
         (64, 61, 43, 150, (3, 3), 1, (1, 1))]


def make(case, seed=0):
    cin, H, W, cout, (kh, kw), s, (ph, pw) = case
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((cin, H, W)).astype(np.float32)
    w = (rng.standard_normal((cout, cin, kh, kw)) * np.sqrt(2.0 / (cin * kh * kw))).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32)
    ref = O.conv2d(x, w, b, None, None, None, (s, s), (ph, pw), 1, 1, 6.0, False)
    d = B.Conv2dDesc(cin, H, W, cout, kh, kw, s, s, ph, pw, 1)
    return d, [B.DeviceBuffer.from_array(a) for a in (x, w, b)], B.DeviceBuffer(ref.size * 4), ref


@pytest.mark.parametrize("case", CASES)
def test_matches_oracle_call_after_call(case):
    B.ops_init()
    d, (x, w, b), out, ref = make(case)
    got = []
    for noalloc in (False, False, True, True):      # pool, then fixed array; each again with what the last left
        out.fill(0xFF)
        assert B.ops_conv2d(d, x, w, b, None, out, noalloc=noalloc) == 0, B.last_error()
        got.append(out.to_array())
    assert max_rel_err(got[0].reshape(ref.shape), ref) <= REL_TOL
    for g in got[1:]:
        np.testing.assert_array_equal(got[0], g)


def test_calls_of_several_threads():
    B.ops_init()
    jobs = [make(c, i) for i, c in enumerate((CASES[3], CASES[5], CASES[17], CASES[14], CASES[12], CASES[21]))]
    bad = []

    def work(job):
        d, (x, w, b), out, ref = job
        for _ in range(20):
            if B.ops_conv2d(d, x, w, b, None, out) or max_rel_err(out.to_array().reshape(ref.shape), ref) > REL_TOL:
                bad.append(B.last_error())
    ts = [threading.Thread(target=work, args=(j,)) for j in jobs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    assert B.lib().reef_ops_release() == 0
    work(jobs[0])                                   # a workspace is made again
    assert not bad
