"""Convolutions on packed weights that take whole cache lines (reef_conv2d_v1_*, reef_conv2d_v9_*):
every storage against the oracle, and the three flavours bit for bit."""
import os

import numpy as np
import pytest

from reef_amd import binding as B
from reef_amd.modelgen import builder as MB, tiling
from tests.helpers import compare_storages, run_both

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(17)


def rnd(*shape):
    return RNG.standard_normal(shape).astype(np.float32)


def flavours_agree(exe, g, d, inputs):
    """The padding and the best-effort flavour hold the plain one's bits in every storage."""
    hyb = B.Executor.from_dir(os.path.join(str(d), g.name), g.name, B.HYBRID)
    for k, v in inputs.items():
        hyb.set_input_checked(k, v)
    for go in (hyb.execute, hyb.execute_preemptable):
        go()
        for k in g.kernels:
            idx = k["args"][2]
            n = g.storage[idx]["size"]
            if g.storage[idx]["stype"] == "float32":
                np.testing.assert_array_equal(hyb.get_data(idx, n), exe.get_data(idx, n))


# Cin of fewer channels than a step, of half a group of 16 at the end and of several steps; images of one piece of
# four pixels, of a ragged last tile and of several; Cout that fills no row tile
V1_SHAPES = [(8, 2, 2, 8), (72, 6, 6, 88), (200, 14, 14, 40), (648, 10, 18, 24)]


@pytest.mark.parametrize("split,fused", [(1, False), (2, False), (2, True), (3, True)])
@pytest.mark.parametrize("shape", V1_SHAPES)
@pytest.mark.parametrize("tile", list(tiling.DIRECT_TILES))
def test_pointwise_on_packed_weights(tmp_path, monkeypatch, tile, shape, split, fused):
    monkeypatch.setattr(tiling, "V1_MIN_CIN", {})
    cin, H, W, cout = shape
    f = tiling.forced(tile, cout, H * W, cin, split, 1)
    if f["split_k"] != split:
        pytest.skip("too few channels for this split")
    g = MB.GraphBuilder("v1")
    x = g.input("data", (cin, H, W))
    res = g.input("res", (cout, H, W))
    for pre in (False, True) if tile in tiling.PRE_ACT_TILES else (False,):
        kw = dict(force=f, fused_reduce=fused, pre_act=pre)
        g.conv2d(x, cout, 1, 1, 0, bias=True, act=MB.ACT_RELU, **kw)
        g.conv2d(x, cout, 1, 1, 0, bias=False, act=MB.ACT_NONE, residual=res, **kw)
        g.conv2d(x, cout, 1, 1, 0, bias=False, act=MB.ACT_RELU6, residual=res, affine=not pre, **kw)
        cat = g.temp((cout + 4, H, W))
        y = g.conv2d(x, cout, 1, 1, 0, out=cat, out_channel=4, **kw)
    g.mark_output(y)
    syms = {k["name"].split("#")[0] for k in g.kernels if k["op"] == "conv2d"}
    assert syms == {"reef_conv2d_v1_" + tile} | ({"reef_conv2d_p1_v_" + tile} if tile in tiling.PRE_ACT_TILES else set())
    inputs = {"data": rnd(cin, H, W), "res": rnd(cout, H, W)}
    exe, orc, model = run_both(g, tmp_path, inputs)
    compare_storages(exe, orc, model, what="v1 %s %s x%d%s" % (tile, shape, split, " fused" if fused else ""))
    flavours_agree(exe, g, tmp_path, inputs)


# images of one row, narrower than a segment, of exactly one and of several with a ragged last; heights that are no
# multiple of the tile's; channels below a step, half a group at the end, several steps
V9_SHAPES = [(16, 1, 14, 16), (24, 5, 3, 8), (136, 9, 29, 17), (272, 3, 15, 32)]


@pytest.mark.parametrize("split,fused", [(1, False), (2, False), (2, True), (3, True)])
@pytest.mark.parametrize("shape", V9_SHAPES)
@pytest.mark.parametrize("tile", list(tiling.V9_TILES))
def test_3x3_on_weights_packed_by_channels(tmp_path, tile, shape, split, fused):
    cin, H, W, cout = shape
    f = tiling.forced_rows(tile, cout, H, W, cin * 9, split)
    if f["split_k"] != split:
        pytest.skip("too few channels for this split")
    g = MB.GraphBuilder("v9")
    x = g.input("data", (cin, H, W))
    res = g.input("res", (cout, H, W))
    kw = dict(force=f, fused_reduce=fused)
    g.conv2d(x, cout, 3, 1, 1, bias=True, act=MB.ACT_RELU, **kw)
    g.conv2d(x, cout, 3, 1, 1, bias=False, act=MB.ACT_NONE, residual=res, dual_act=MB.ACT_RELU, **kw)
    cat = g.temp((cout + 4, H, W))
    y = g.conv2d(x, cout, 3, 1, 1, out=cat, out_channel=4, **kw)
    g.mark_output(y)
    assert all(k["name"].startswith("reef_conv2d_v9_" + tile) for k in g.kernels if k["op"] == "conv2d")
    inputs = {"data": rnd(cin, H, W), "res": rnd(cout, H, W)}
    exe, orc, model = run_both(g, tmp_path, inputs)
    compare_storages(exe, orc, model, what="v9 %s %s x%d%s" % (tile, shape, split, " fused" if fused else ""))
    flavours_agree(exe, g, tmp_path, inputs)


def test_the_bit_of_a_retired_mode_changes_nothing(tmp_path):
    """Model files may carry flag 8192 on splits of two (reef_kernels.h): with and without it the same bits, in all
    flavours, also where ten operands leave no slot for a prefetch record."""
    shape = (256, 14, 14)
    inputs = {"data": rnd(*shape), "res": rnd(*shape)}
    held = []
    for bit in (0, 8192):
        g = MB.GraphBuilder("bit")
        x, r = g.input("data", shape), g.input("res", shape)
        rows = dict(force=tiling.forced_rows("g1", 256, 14, 14, 256 * 9, 2), fused_reduce=True)
        y, z = g.conv2d(x, 256, 3, 1, 1, bias=True, residual=r, dual_act=MB.ACT_RELU, **rows)
        one = dict(force=tiling.forced("16x16k4", 256, 196, 1024, 2, 1), fused_reduce=True)
        cat = g.temp((1024, 14, 14))
        g.conv2d(z, 1024, 1, 1, 0, out=cat)
        g.mark_output(g.conv2d(cat, 256, 1, 1, 0, residual=y, **one))
        split = [k for k in g.kernels if k["attrs"][12] & 64]
        assert len(split) == 2 and len(split[0]["args"]) == 10
        for k in split:
            k["attrs"][12] |= bit
        exe, orc, model = run_both(g, tmp_path / str(bit), inputs)
        compare_storages(exe, orc, model, what="flag %d" % bit)
        flavours_agree(exe, g, tmp_path / str(bit), inputs)
        held.append([exe.get_data(k["args"][2], g.storage[k["args"][2]]["size"]) for k in g.kernels])
    for a, b in zip(*held):
        np.testing.assert_array_equal(a, b)
