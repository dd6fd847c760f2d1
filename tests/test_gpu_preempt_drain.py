"""Launches that start under a raised preemption flag leave without multiplying first."""
import os
import time

import pytest

from reef_amd import binding as B
from reef_amd.modelgen import builder as MB

pytestmark = pytest.mark.gpu


# layers whose K is deep enough that a round of it is a good part of a launch: a pass under a raised flag took 0.97 and 0.73 of
# an uninterrupted one where every wavefront ran its first round, and takes 0.82 and 0.61
@pytest.mark.parametrize("cin,k,most", [(256, 3, 0.9), (1024, 1, 0.67)])
def test_a_pass_under_a_raised_flag(tmp_path, cin, k, most):
    g = MB.GraphBuilder("chain", under_load=True)
    x = g.input("x", (cin, 14, 14))
    for _ in range(64):
        x = g.conv2d(x, cin, k, 1, k // 2)
    g.mark_output(x)
    assert {c["name"].split("#")[0] for c in g.kernels} == {"reef_conv2d_v9_g1" if k == 3 else "reef_conv2d_v1_32x32d4"}
    g.write(os.path.join(str(tmp_path), "chain"))
    exe = B.Executor.from_dir(os.path.join(str(tmp_path), "chain"), "chain", B.HYBRID)
    exe.execute_preemptable()
    best = []
    for flag in (0, 1):
        exe.poke_preempt_flag(flag)
        times = []
        for _ in range(30):
            t0 = time.perf_counter()
            exe.execute_preemptable()
            times.append(time.perf_counter() - t0)
        best.append(min(times))
    exe.poke_preempt_flag(0)
    exe.close()
    assert best[1] < most * best[0], best
