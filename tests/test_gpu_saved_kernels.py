"""Kernels that the generator no longer names and saved model files may: the row form on weights packed by taps
(reef_conv2d_r9k_*), and the 1-tap kernels on weights as OIHW has them (reef_conv2d_d1_*, reef_conv2d_p1_* with no packed
copy).  Every storage against the oracle, and the three flavours bit for bit."""
import numpy as np
import pytest

from reef_amd.modelgen import builder as MB, tiling
from tests.helpers import compare_storages, run_both
from tests.test_gpu_packed_convs import V9_SHAPES, flavours_agree

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(29)
SPLITS = [(1, False), (2, False), (2, True), (3, True)]
# Cin below a step, no multiple of 16 at the end, several steps; an odd image, ragged last tiles; Cout that fills no row tile
ONE_TAP_SHAPES = [(8, 2, 2, 8), (72, 7, 7, 88), (200, 14, 14, 40), (648, 9, 17, 24)]


def rnd(*shape):
    return RNG.standard_normal(shape).astype(np.float32)


def check(g, tmp_path, cin, cout, H, W, what):
    inputs = {"data": rnd(cin, H, W), "res": rnd(cout, H, W)}
    exe, orc, model = run_both(g, tmp_path, inputs)
    compare_storages(exe, orc, model, what=what)
    flavours_agree(exe, g, tmp_path, inputs)


@pytest.mark.parametrize("split,fused", SPLITS)
@pytest.mark.parametrize("shape", V9_SHAPES)
@pytest.mark.parametrize("tile", list(tiling.V9_TILES))
def test_rows_on_weights_packed_by_taps(tmp_path, monkeypatch, tile, shape, split, fused):
    cin, H, W, cout = shape
    f = tiling.forced_rows(tile, cout, H, W, cin * 9, split)
    if f["split_k"] != split:
        pytest.skip("too few channels for this split")
    monkeypatch.setattr(tiling, "V9_TILES", ())
    g = MB.GraphBuilder("r9k")
    x, res = g.input("data", (cin, H, W)), g.input("res", (cout, H, W))
    kw = dict(force=f, fused_reduce=fused)
    g.conv2d(x, cout, 3, 1, 1, bias=True, act=MB.ACT_RELU, **kw)
    g.conv2d(x, cout, 3, 1, 1, bias=False, act=MB.ACT_NONE, residual=res, dual_act=MB.ACT_RELU, **kw)
    cat = g.temp((cout + 4, H, W))
    g.mark_output(g.conv2d(x, cout, 3, 1, 1, out=cat, out_channel=4, **kw))
    convs = [k for k in g.kernels if k["op"] == "conv2d"]
    assert all(k["name"].startswith("reef_conv2d_r9k_" + tile) and k["attrs"][23] for k in convs)
    check(g, tmp_path, cin, cout, H, W, "r9k %s %s x%d%s" % (tile, shape, split, " fused" if fused else ""))


@pytest.mark.parametrize("split,fused", SPLITS)
@pytest.mark.parametrize("shape", ONE_TAP_SHAPES)
@pytest.mark.parametrize("tile", list(tiling.DIRECT_TILES))
def test_pointwise_on_unpacked_weights(tmp_path, tile, shape, split, fused):
    cin, H, W, cout = shape
    f = tiling.forced(tile, cout, H * W, cin, split, 1)
    if f["split_k"] != split:
        pytest.skip("too few channels for this split")
    g = MB.GraphBuilder("d1")
    g.pack_weights = False
    x, res = g.input("data", (cin, H, W)), g.input("res", (cout, H, W))
    for pre in (False, True) if tile in tiling.PRE_ACT_TILES else (False,):
        kw = dict(force=f, fused_reduce=fused, pre_act=pre)
        g.conv2d(x, cout, 1, 1, 0, bias=True, act=MB.ACT_RELU, **kw)
        g.conv2d(x, cout, 1, 1, 0, bias=False, act=MB.ACT_RELU6, residual=res, affine=not pre, **kw)
        cat = g.temp((cout + 4, H, W))
        y = g.conv2d(x, cout, 1, 1, 0, out=cat, out_channel=4, **kw)
    g.mark_output(y)
    convs = [k for k in g.kernels if k["op"] == "conv2d"]
    assert {k["name"].split("#")[0] for k in convs} == {"reef_conv2d_d1_" + tile} | (
        {"reef_conv2d_p1_" + tile} if tile in tiling.PRE_ACT_TILES else set())
    assert not any(k["attrs"][23] for k in convs)
    check(g, tmp_path, cin, cout, H, W, "d1 %s %s x%d%s" % (tile, shape, split, " fused" if fused else ""))
