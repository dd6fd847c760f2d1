"""Kernels on packed weights against 64 bits: no further off than the kernels whose place they take."""
import os

import numpy as np
import pytest

from reef_amd import binding as B
from reef_amd.modelgen import builder as MB, tiling

pytestmark = pytest.mark.gpu

# A result is a few thousand values whose errors are alike and independent, so the root mean square of them is known to
# about 2 %; twice as long a chain of sums has 1.4 times the error.
SAME = 1.1


def off(g, d, x, outs, wants):
    """Distance of each storage from its 64-bit values, relative to them."""
    g.write(os.path.join(str(d), g.name))
    exe = B.Executor.from_dir(os.path.join(str(d), g.name), g.name, B.BASE)
    exe.set_input_checked("x", x)
    exe.execute()
    return [float(np.linalg.norm(exe.get_data(t.idx, y.size).astype(np.float64) - y.reshape(-1)) / np.linalg.norm(y))
            for t, y in zip(outs, wants)]


@pytest.mark.parametrize("tile", list(tiling.GEMM_DIRECT_TILES) + list(tiling.GEMM_WIDE_TILES))
def test_product_on_packed_weights(tmp_path, tile):
    m, n, k = 64, 256, 3072
    x = np.random.default_rng(41).standard_normal((m, k)).astype(np.float32)
    errs = []
    for packed in (False, True):
        g = MB.GraphBuilder("packed" if packed else "plain")
        g.pack_weights = packed
        w = g.param((n, k), 0.5)
        out = g.gemm(g.input("x", (m, k)), w, m, n, k, force_tile=tile, split_k=1)
        g.mark_output(out)
        assert (g.kernels[0]["attrs"][12] == 0) == packed
        errs += off(g, tmp_path, x, [out], [x.astype(np.float64) @ g.param_array(w).reshape(n, k).T.astype(np.float64)])
    assert errs[1] <= SAME * errs[0], errs


@pytest.mark.parametrize("tile,taps,pre", [("g1", 9, False), ("16x16k4", 1, False), ("16x16k4", 1, True)])
def test_unsplit_convolution_in_place_of_a_split_in_two(tmp_path, tile, taps, pre):
    cin, cout, side = 256 if taps == 9 else 1024, 64, 14
    edge = 1 if taps == 9 else 0
    x = np.random.default_rng(43).standard_normal((cin, side, side)).astype(np.float32)
    g = MB.GraphBuilder("conv")
    t = g.input("x", x.shape)
    outs, wants = [], []
    for split in (2, 1):
        f = (tiling.forced_rows(tile, cout, side, side, cin * 9, split) if taps == 9 else
             tiling.forced(tile, cout, side * side, cin, split, 1))
        assert f["split_k"] == split
        first = len(g.params)
        outs.append(g.conv2d(t, cout, 1 + 2 * edge, 1, edge, bias=False, force=f, fused_reduce=True, pre_act=pre))
        own = [a.astype(np.float64) for k, a in g.params[first:] if not k.endswith("k")]      # weights, scale, shift
        v = np.maximum(x * own[1][:, None, None] + own[2][:, None, None], 0.0) if pre else x.astype(np.float64)
        v = np.pad(v, ((0, 0), (edge, edge), (edge, edge)))
        w = own[0].reshape(cout, cin, 1 + 2 * edge, 1 + 2 * edge)
        wants.append(sum(w[:, :, i, j] @ v[:, i:i + side, j:j + side].reshape(cin, -1)
                         for i in range(1 + 2 * edge) for j in range(1 + 2 * edge)))
    g.mark_output(outs[-1])
    errs = off(g, tmp_path, x, outs, wants)
    assert errs[1] <= SAME * errs[0], errs
