"""Kernels that the generator no longer names and saved model files may: the row form on weights packed by taps
(reef_conv2d_r9k_*), the 1-tap kernels on weights as OIHW has them (reef_conv2d_d1_*, reef_conv2d_p1_* with no packed
copy), and matrix products of 32 rows and more on weights packed as 32-bit values.  Every storage against the oracle, and the
three flavours bit for bit."""
import numpy as np
import pytest

from reef_amd.modelgen import builder as MB, tiling
from tests.helpers import compare_storages, run_both
from tests.test_gpu_packed_convs import V9_SHAPES, flavours_agree
from tests.test_gpu_packed_products import SHAPES as PRODUCT_SHAPES

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


@pytest.mark.parametrize("split", [1, 2, 3])
@pytest.mark.parametrize("shape", PRODUCT_SHAPES)
@pytest.mark.parametrize("tile", list(tiling.GEMM_SPLIT_TILES))
def test_product_on_weights_packed_as_32_bit_values(tmp_path, monkeypatch, tile, shape, split):
    m, n, k = shape
    if split > 1 and tiling.forced(tile, m, n, k, split)["split_k"] != split:
        pytest.skip("too little depth for this split")
    monkeypatch.setattr(tiling, "GEMM_SPLIT_TILES", ())
    g = MB.GraphBuilder("pk32")
    x, r = g.input("data", (m, k)), g.input("res", (m, n))
    w, bias = g.param((n, k), 0.5), g.param((n,), 0.5)
    g.gemm(x, w, m, n, k, bias=bias, act=MB.ACT_GELU, res=r, force_tile=tile, split_k=split)
    plain = g.gemm(x, w, m, n, k, alpha=0.5, force_tile=tile, split_k=split)
    if split == 1 and tile in g.LN_GEMM_TILES:
        ln = dict(gamma=g.param((k,), 0.5), beta=g.param((k,), 0.5))
        g.gemm(x, w, m, n, k, bias=bias, force_tile=tile, ln=dict(ln, out=g.temp((m, k))))
        g.gemm(x, w, m, n, k, res=r, force_tile=tile, ln=ln)
    g.mark_output(plain)
    products = [c for c in g.kernels if c["op"] == "gemm"]
    assert all(c["attrs"][12] == 0 and not c["attrs"][5] & 32 and c["name"].split("#")[0].endswith(tile) for c in products)
    inputs = {"data": rnd(m, k), "res": rnd(m, n)}
    exe, orc, model = run_both(g, tmp_path, inputs)
    compare_storages(exe, orc, model, what="pk32 %s %s x%d" % (tile, shape, split))
    flavours_agree(exe, g, tmp_path, inputs)
