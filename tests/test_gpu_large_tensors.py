"""Elementwise and copy launches on tensors of more than 4 GiB: the first and last elements and those around the four."""
import os

import numpy as np
import pytest

from reef_amd import binding as B
from reef_amd.modelgen import builder as MB

pytestmark = pytest.mark.gpu


def test_copy_and_eltwise_beyond_4_gib(tmp_path):
    n, part = 2 ** 30 + 8192, 4096
    g = MB.GraphBuilder("large")
    big = [g.temp((4, n // 4, 1)) for _ in range(3)]
    at = (0, 2 ** 30 - 2048, n - part)
    marks = [g.input("m%d" % i, (part,)) for i in range(3)]
    for m, off in zip(marks, at):
        g.copy_into(m, big[0], off)
    g.copy_into(big[0], big[1], 0)
    shift = g.param((4,), 1.0)
    g.eltwise(big[1], shift=True, shift_t=shift, out=big[2])
    seen = []
    for t in big[1:]:
        for off in at:
            seen.append(g.temp((part,)))
            g.copy_into(seen[-1], seen[-1], 0)
            g.kernels[-1]["args"][0], g.kernels[-1]["arg_offsets"] = t.idx, [4 * off, 0]
    g.mark_output(seen[-1])
    g.write(os.path.join(str(tmp_path), "large"))
    exe = B.Executor.from_dir(os.path.join(str(tmp_path), "large"), "large", B.BASE)
    rng = np.random.default_rng(1)
    data = [rng.standard_normal(part).astype(np.float32) for _ in marks]
    for i, d in enumerate(data):
        exe.set_input_checked("m%d" % i, d)
    exe.execute()
    got = [exe.get_data(t.idx, part) for t in seen]
    exe.close()
    add = g.param_array(shift)
    for i, off in enumerate(at):
        np.testing.assert_array_equal(got[i], data[i], "copy at %d" % off)
        np.testing.assert_array_equal(got[3 + i], data[i] + add[(off + np.arange(part)) // (n // 4)], "eltwise at %d" % off)
