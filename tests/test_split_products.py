"""Matrix products on split weights (REEF_GEMM_F_SPLIT): the parts are the weight, and what has no parts in bf16 -- infinities,
NaN, values that round to infinity -- comes out as it does on the weights themselves."""
import json
import os
import time

import numpy as np
import pytest

from reef_amd import binding as B
from reef_amd.modelgen import builder as MB, tiling
from tests.test_gpu_packed_convs import flavours_agree


def bf16(u):
    return (u.astype(np.uint32) << np.uint32(16)).view(np.float32)


def test_parts_of_a_weight_add_up_to_it():
    rng = np.random.default_rng(3)
    n, k = 21, 72
    w = rng.integers(0, 2 ** 32, (n, k), dtype=np.uint32).view(np.float32)
    w[np.abs(w) < 2.0 ** -100] = 1.5        # (below 2^-110 the third part falls under the smallest bf16)
    w[0, :8] = [np.inf, -np.inf, np.nan, 3.4028235e38, -3.4028235e38, 0.0, -0.0, 1 + 2.0 ** -23]
    p = MB.split_matrix(w).view(np.uint16).reshape(2, 3, 3, 4, 16, 2, 4)     # tile, group of 32, part, slot, column, half, k
    h, m, l = (bf16(p[:, :, i]) for i in range(3))
    with np.errstate(invalid="ignore"):
        back = (h + m) + l
    back = back.transpose(0, 3, 1, 4, 2, 5).reshape(32, 96)
    assert np.array_equal(back[:n, :k], w, equal_nan=True) and not back[n:].any() and not back[:, k:].any()
    assert np.isfinite(h[np.isfinite(back).reshape(2, 16, 3, 2, 4, 4).transpose(0, 2, 4, 1, 3, 5)]).all()


def test_parts_of_a_matrix_with_and_without_values_that_have_none():
    rng = np.random.default_rng(4)
    for n, k in ((48, 96), (17, 40)):
        w = rng.standard_normal((n, k)).astype(np.float32)
        w[3, 5], w[4, 7] = 3.37e38, -3.37e38
        plain = MB.split_matrix(w)
        for bad in (np.inf, -np.inf, np.nan, 3.4028235e38):
            v = w.copy()
            v[n - 1, k - 1] = bad
            differ = np.flatnonzero(MB.split_matrix(v).view(np.uint16) != plain.view(np.uint16))
            col, at = (n - 1) % 16, (k - 1) % 32                 # where the value's parts lie, by the layout's definition
            first = ((n - 1) // 16 * -(-k // 32) + (k - 1) // 32) * 1536 + (at % 16 // 4 * 16 + col) * 8 + at // 16 * 4 + at % 4
            assert differ.size and set(differ) <= {first, first + 512, first + 1024}


def product(d, name, tile, a, w, split, packed):
    (m, k), n = a.shape, w.shape[0]
    g = MB.GraphBuilder(name)
    g.pack_weights = packed
    wt = g.param((n, k), 0.5)
    g.params[g._param_pos[wt.idx]][1][:] = w.reshape(-1)
    out = g.gemm(g.input("a", (m, k)), wt, m, n, k, force_tile=tile, split_k=split)
    g.mark_output(out)
    assert bool(g.kernels[0]["attrs"][5] & 32) == packed
    g.write(os.path.join(str(d), name))
    exe = B.Executor.from_dir(os.path.join(str(d), name), name, B.BASE)
    exe.set_input_checked("a", a)
    exe.execute()
    y = exe.get_data(out.idx, m * n).reshape(m, n).copy()
    exe.close()
    return y


# column tiles that are a multiple of the XCDs and that are not, a split that ends inside a step, the smallest
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 4, 8, 1), (33, 17 * 48 + 4, 264, 1), (70, 8 * 48, 520, 3), (49, 100, 392, 2)])
@pytest.mark.parametrize("tile", tiling.GEMM_SPLIT_TILES)
def test_product_of_split_operands(tmp_path, tile, shape):
    m, n, k, split = shape
    if split > 1 and tiling.forced(tile, m, n, k, split)["split_k"] != split:
        pytest.skip("too little depth for this split")
    rng = np.random.default_rng(5)
    a, w = rng.standard_normal((m, k)).astype(np.float32), (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    # k + 1 roundings of at most 2^-24 of the sum of magnitudes, and the terms left out: at most 2^-23 of each product
    bound = (k + 3) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(w).T.astype(np.float64))
    y = product(tmp_path, "split", tile, a, w, split, True)
    assert (np.abs(y - a.astype(np.float64) @ w.T.astype(np.float64)) <= bound).all()
    # rows and columns with values that have no parts: one each, so that no sum depends on its order
    a[m // 2, k // 2], w[n // 2, 3] = 3.4e38, np.inf
    if m > 4:
        a[0, 1], a[1, 2], a[2, k - 1], a[3, 0] = np.inf, np.nan, -np.inf, -3.4e38
    if n > 4:
        w[1, k - 2], w[2, 5] = np.nan, 3.4e38
        w[2, :5] = w[2, 6:] = 0.0          # (its only product with the huge values is with itself)
        a[:, 5] = np.clip(a[:, 5], -0.5, 0.5)
    with np.errstate(all="ignore"):
        want = product(tmp_path, "plain", tile, a, w, split, False)
        y = product(tmp_path, "split2", tile, a, w, split, True)
        same = np.isfinite(want)
        assert np.array_equal(np.isnan(want), np.isnan(y)) and np.array_equal(want[np.isinf(want)], y[np.isinf(want)])
        bound = 2 * (k + 2) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(w).T.astype(np.float64))
        assert (np.abs(y[same].astype(np.float64) - want[same]) <= bound[same]).all()


def loaded(d, tile, a, w, kind):
    (m, k), n = a.shape, w.shape[0]
    g = MB.GraphBuilder("nan")
    wt = g.param((n, k), 0.5)
    g.params[g._param_pos[wt.idx]][1][:] = w.reshape(-1)
    out = g.gemm(g.input("a", (m, k)), wt, m, n, k, force_tile=tile, split_k=1)
    g.mark_output(out)
    assert g.kernels[0]["attrs"][5] & 32
    g.write(os.path.join(str(d), "nan"))
    exe = B.Executor.from_dir(os.path.join(str(d), "nan"), "nan", kind)
    exe.set_input_checked("a", a)
    return g, exe, out


@pytest.mark.gpu
@pytest.mark.parametrize("tile", tiling.GEMM_SPLIT_TILES)
def test_flavours_agree_on_values_without_parts(tmp_path, tile):
    m, n, k = 70, 100, 392
    rng = np.random.default_rng(6)
    a, w = rng.standard_normal((m, k)).astype(np.float32), (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    a[0, 1], a[1, 2], a[2, k - 1], a[40, 200], w[n // 2, 3] = np.inf, np.nan, -np.inf, 3.4e38, np.inf
    g, exe, out = loaded(tmp_path, tile, a, w, B.BASE)
    exe.execute()
    assert not np.isfinite(exe.get_data(out.idx, m * n)).all()
    flavours_agree(exe, g, tmp_path, {"a": a})


@pytest.mark.gpu
@pytest.mark.parametrize("tile", ["32x48d4", "64x64d4"])
def test_values_without_parts_cost_one_more_pass_over_the_depth(tmp_path, tile):
    """A best-effort launch whose data holds NaN must not keep the device to itself (an element at a time it took a hundred
    times as long)."""
    m, n, k = 128, 768, 3072
    rng = np.random.default_rng(7)
    a, w = rng.standard_normal((m, k)).astype(np.float32), (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    _, exe, _ = loaded(tmp_path, tile, a, w, B.HYBRID)
    best = []
    for x in (a, np.full_like(a, np.nan)):
        exe.set_input_checked("a", x)
        times = []
        for _ in range(8):
            t0 = time.perf_counter()
            exe.execute_preemptable()
            times.append(time.perf_counter() - t0)
        best.append(min(times))
    exe.close()
    assert best[1] < 5 * best[0], best


@pytest.mark.gpu
@pytest.mark.parametrize("tile", tiling.GEMM_SPLIT_TILES)
def test_every_product_of_parts_is_there(tmp_path, tile):
    """Columns with one weight each, all 24 bits in use, a column for every k: an output is one product, whose parts leave out at
    most 2^-23 of it, and is rounded when its sums meet, twice; without any of the six products four fifths of them are further
    off, up to 2^-16."""
    m, k = 49, 264
    rng = np.random.default_rng(10)
    a = (np.ldexp(rng.integers(2 ** 23, 2 ** 24, (m, k)) | 1, -23) * rng.choice((-1, 1), (m, k))).astype(np.float32)
    w = np.diag(np.ldexp(rng.integers(2 ** 23, 2 ** 24, k) | 1, -23)).astype(np.float32)
    want = a.astype(np.float64) * np.diag(w).astype(np.float64)
    assert (np.abs(product(tmp_path, "one", tile, a, w, 1, True) - want) <= 2.0 ** -22 * np.abs(want)).all()


def test_weights_that_are_not_the_sum_of_their_parts_are_not_split():
    w = np.full((20, 40), 0.5, np.float32)
    for x, exact in ((2.0 ** -110 * (1 + 2.0 ** -23), True), (2.0 ** -111 * (1 + 2.0 ** -23), False), (2.0 ** -111 * (1 + 2.0 ** -22), True),
                     (2.0 ** -133, True), (2.0 ** -134, False), (-1e-40, False), (2.0 ** -149, False)):
        w[7, 11] = x
        assert (MB.split_matrix(w) is not None) == exact, x
        g = MB.GraphBuilder("tiny")
        wt, gamma = g.param(w.shape, 0.5), g.param((40,), 0.5)
        g.params[g._param_pos[wt.idx]][1][:] = w.reshape(-1)
        g.params[g._param_pos[gamma.idx]][1][:] = 1.0
        a = g.input("a", (33, 40))
        for ln in (None, dict(gamma=gamma, beta=gamma)):
            g.gemm(a, wt, 33, 20, 40, force_tile="32x48d4", ln=ln)
            g.gemm(a, wt, 33, 20, 40, force_tile="16x32k4", ln=ln)
        names = [g.storage[k["args"][1]]["name"] for k in g.kernels]
        p = g.storage[wt.idx]["name"]
        assert names == [p + s for s in (("xpk", "pk", "gkxpk", "gkpk") if exact else ("pk", "pk", "gkpk", "gkpk"))]
        assert [bool(k["attrs"][5] & 32) for k in g.kernels] == [exact, False] * 2


def test_split_weights_whose_offsets_need_more_than_32_bits(tmp_path, monkeypatch):
    """131072 x 5461 are 4 GiB as parts and 2.7 as 32-bit values: the generator keeps the latter, and a model that names the former
    is refused (its kernel would read the weights modulo 4 GiB)."""
    assert tiling.takes_split("32x48d4", 131072, 5440) and not tiling.takes_split("32x48d4", 131072, 5464)
    assert tiling.takes_split("64x64d4", 4096, 4096) and not tiling.takes_split("16x32k4", 64, 64)

    def model(name):
        g = MB.GraphBuilder(name)
        w = g.param((96, 72), 0.5)
        g.mark_output(g.gemm(g.input("a", (40, 72)), w, 40, 96, 72, force_tile="32x48d4"))
        return g, json.load(open(g.write(str(tmp_path / name), link_code_objects=False) + ".json"))
    g, m = model("fits")
    assert g.kernels[0]["attrs"][5] == 32
    monkeypatch.setattr(tiling, "GEMM_SPLIT_BYTES", 6 * 3 * 3072)
    assert model("large")[0].kernels[0]["attrs"][5] == 0
    k, N, K = m["kernels"][0], 131072, 5464
    k["attrs"][2:4], k["attrs"][10], k["attrs"][11], k["attrs"][13] = [N, K], N // 48 + 1, K, N
    k["launch_params"][0] = 2 * k["attrs"][10]
    for i, n in zip(k["args"], (40 * K, N // 16 * 171 * 768, 40 * N)):
        m["storage"][i]["size"] = n
    for bad in (True, False):
        if not bad:
            k["attrs"][3] = k["attrs"][11] = 5440
        json.dump(m, open(str(tmp_path / "m.json"), "w"))
        ok, why = B.check_model(str(tmp_path / "m.json"))
        assert ok != bad and ("4 GiB" in why) == bad, why


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-28, 1e-30, 1e-32, 1e-34, 1e-36, 1e-38])
@pytest.mark.parametrize("tile", tiling.GEMM_SPLIT_TILES)
def test_small_operands_are_as_exact_as_in_32_bits(tmp_path, tile, scale):
    """(At 1e-36 the parts of a value keep 15 bits of it.)  The errors are thousands of alike and independent ones: 1.1 for what their
    root mean square is known to.  Beside it the roundings of sums near the smallest normal value, to 2^-149: a standard deviation
    of 2^-149 / 12^0.5 each, a quarter, six and a quarter again for every four and 32 values of k in 32 bits, in parts and for
    what these leave."""
    m, n, k = 64, 256, 768
    rng = np.random.default_rng(8)
    a = (rng.standard_normal((m, k)) * scale).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    want = a.astype(np.float64) @ w.T.astype(np.float64)
    errs = [np.linalg.norm(product(tmp_path, "p%d" % packed, tile, a, w, 1, packed).astype(np.float64) - want) / np.linalg.norm(want)
            for packed in (False, True)]
    small = 2.0 ** -149 / 12 ** 0.5 * (k / 4 + 6 * k / 32) ** 0.5 / np.sqrt((want ** 2).mean())
    assert errs[1] <= 1.1 * errs[0] + small, (errs, small)
    if scale > 1e-37:
        assert errs[1] <= 0.8 * errs[0], errs      # (in parts the sums have a quarter of the roundings)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", tiling.GEMM_SPLIT_TILES)
def test_a_row_of_small_values_leaves_the_other_rows_alone(tmp_path, tile):
    m, n, k = 70, 100, 392
    rng = np.random.default_rng(9)
    a, w = rng.standard_normal((m, k)).astype(np.float32), (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    whole = product(tmp_path, "whole", tile, a, w, 1, True)
    small = [0, 15, 16, 37, m - 1]
    a[small] *= np.float32(1e-36)
    y = product(tmp_path, "small", tile, a, w, 1, True)
    others = np.setdiff1d(np.arange(m), small)
    np.testing.assert_array_equal(y[others], whole[others])
    bound = (k + 2) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(w).T.astype(np.float64))
    assert (np.abs(y - a.astype(np.float64) @ w.T.astype(np.float64)) <= bound)[small].all()
    g, exe, _ = loaded(tmp_path, tile, a, w, B.BASE)
    exe.execute()
    flavours_agree(exe, g, tmp_path, {"a": a})
