"""The wide direct tiles of the matrix products and the attention on the matrix cores, at the edges of their tiles."""
import numpy as np
import pytest

from reef_amd.modelgen import builder as MB
from reef_amd.modelgen import tiling
from tests.helpers import compare_storages, run_both

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(29)


def rnd(*shape):
    return RNG.standard_normal(shape).astype(np.float32)


@pytest.mark.parametrize("tile", list(tiling.GEMM_WIDE_TILES))
@pytest.mark.parametrize("edge,depth", [(-1, 8), (0, 256), (1, 328)])
def test_wide_direct_tiles(tmp_path, tile, edge, depth):
    """One row and column less than two tiles, exactly two, one more; a depth of less than a step, of whole
    steps, and with a remainder; bias, activation, residual and alpha; whole, and split in two and three."""
    _, bm, bn = tiling.GEMM_WIDE_TILES[tile]
    m, n = 2 * bm + edge, 2 * bn + edge
    g = MB.GraphBuilder("wt", weight_std=0.05)
    x, r = g.input("x", (m, depth)), g.input("r", (m, n))
    w, bias = g.param((n, depth), 0.05), g.param((n,), 0.02)
    g.gemm(x, w, m, n, depth, trans_b=True, bias=bias, act=MB.ACT_GELU, res=r, force_tile=tile)
    for split in (1, 2, 3) if depth > 256 else (1,):
        out = g.gemm(x, w, m, n, depth, trans_b=True, alpha=0.5, force_tile=tile, split_k=split)
    g.mark_output(out)
    exe, orc, model = run_both(g, tmp_path, {"x": rnd(m, depth), "r": rnd(m, n)})
    compare_storages(exe, orc, model, what="wide gemm " + tile)


@pytest.mark.parametrize("seq,hd,masked", [(1, 64, False), (15, 4, True), (16, 20, False), (17, 64, True), (63, 32, False),
                                           (65, 16, True), (129, 48, True), (257, 64, False), (509, 64, True), (512, 8, False)])
def test_attention_on_the_matrix_cores(tmp_path, seq, hd, masked):
    """One query row, ragged and whole blocks of 16 rows and of keys, the longest sequence; head sizes from
    4 to 64; padding at the end.  Against the oracle and numpy on the same tensor."""
    heads = 3
    hid = heads * hd
    g = MB.GraphBuilder("am", weight_std=0.05)
    qkv = g.input("x", (seq, 3 * hid))
    mask = g.input("attention_mask", (seq,), "uint1") if masked else None
    ctx = g.attention(qkv, seq, heads, hd, 3 * hid, 0, hid, 2 * hid, 1.0 / np.sqrt(hd), mask=mask, mma=True)
    g.mark_output(ctx)
    pad = np.zeros(seq, np.uint8)
    pad[seq - seq // 4:] = 1
    x = 2.0 * rnd(seq, 3 * hid)
    exe, orc, model = run_both(g, tmp_path, dict({"x": x}, **({"attention_mask": pad} if masked else {})))
    compare_storages(exe, orc, model, what="attention")
    m = x.reshape(seq, 3, heads, hd).astype(np.float64)
    sc = np.einsum("shd,thd->hst", m[:, 0], m[:, 1]) / np.sqrt(hd)
    if masked:
        sc[:, :, pad != 0] = -np.inf
    pr = np.exp(sc - sc.max(-1, keepdims=True))
    pr /= pr.sum(-1, keepdims=True)
    want = np.einsum("hst,thd->shd", pr, m[:, 2]).reshape(seq, hid)
    got = exe.get_data(ctx.idx, seq * hid).reshape(seq, hid)
    assert np.isfinite(got).all() and np.abs(got - want).max() <= 2e-5 * np.abs(want).max()
