"""Matrix products on packed weights (reef_gemm_ntd_* and reef_gemm_ntl_* with ldb = 0): every storage against the
oracle, and the three flavours bit for bit."""
import numpy as np
import pytest

from reef_amd.modelgen import builder as MB, tiling
from tests.helpers import compare_storages, run_both
from tests.test_gpu_packed_convs import flavours_agree

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(23)


def rnd(*shape):
    return RNG.standard_normal(shape).astype(np.float32)


# (rows, columns, depth): below a tile and a step of K, half a group of 16 at the end of either, several tiles and steps
SHAPES = [(1, 4, 8), (37, 72, 40), (65, 100, 328), (130, 68, 776)]


@pytest.mark.parametrize("split", [1, 2, 3])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("tile", list(tiling.GEMM_DIRECT_TILES) + list(tiling.GEMM_WIDE_TILES))
def test_product_on_packed_weights(tmp_path, tile, shape, split):
    m, n, k = shape
    if split > 1 and tiling.forced(tile, m, n, k, split)["split_k"] != split:
        pytest.skip("too little depth for this split")
    g = MB.GraphBuilder("pk")
    x, r = g.input("x", (m, k)), g.input("r", (m, n))
    w, bias = g.param((n, k), 0.5), g.param((n,), 0.5)
    g.gemm(x, w, m, n, k, bias=bias, act=MB.ACT_GELU, res=r, force_tile=tile, split_k=split)
    plain = g.gemm(x, w, m, n, k, alpha=0.5, force_tile=tile, split_k=split)
    if split == 1 and tile in g.LN_GEMM_TILES:
        ln = dict(gamma=g.param((k,), 0.5), beta=g.param((k,), 0.5))
        g.gemm(x, w, m, n, k, bias=bias, force_tile=tile, ln=dict(ln, out=g.temp((m, k))))
        g.gemm(x, w, m, n, k, res=r, force_tile=tile, ln=ln)
    g.mark_output(plain)
    products = [c for c in g.kernels if c["op"] == "gemm"]
    assert all(c["attrs"][12] == 0 and g.storage[c["args"][1]]["name"].endswith("pk") for c in products)
    inputs = {"x": rnd(m, k), "r": rnd(m, n)}
    exe, orc, model = run_both(g, tmp_path, inputs)
    compare_storages(exe, orc, model, what="%s %s x%d" % (tile, shape, split))
    flavours_agree(exe, g, tmp_path, inputs)
