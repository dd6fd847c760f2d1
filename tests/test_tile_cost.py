"""Tile choice by the measured cost of every tile (tiling.CONV_COST), for layers the measured table
does not hold: the choice is a kernel that exists for the filter, and on the GPU it computes the
convolution (split folded inside the launch, ragged last tiles, row form, strides)."""
import json
import os

import numpy as np
import pytest

from reef_amd.modelgen import tiling
from reef_amd.modelgen.builder import GraphBuilder, ACT_RELU
from tests.helpers import max_rel_err, REL_TOL

# cin, H, W, cout, k, stride, pad: one workgroup's worth, a split, just past a round of workgroups,
# many rounds; a filter no direct tile has; channels and pixels that fill no tile
LAYERS = [(8, 5, 5, 12, 1, 1, 0), (520, 9, 9, 130, 1, 1, 0), (36, 31, 33, 70, 1, 1, 0), (64, 57, 57, 250, 1, 2, 0),
          (128, 13, 13, 200, 3, 1, 1), (96, 45, 43, 100, 3, 1, 1), (72, 63, 61, 130, 3, 1, 1), (256, 15, 15, 96, 3, 2, 1),
          (40, 23, 23, 48, 5, 1, 2), (12, 21, 21, 20, (1, 7), 1, (0, 3)), (16, 20, 20, 24, 4, 2, 1)]


def build(layer):
    cin, H, W, cout, k, s, p = layer
    g = GraphBuilder("layer", seed=3)
    x = g.input("data", (cin, H, W))
    g.mark_output(g.conv2d(x, cout, k, s, p, bias=True, act=ACT_RELU))
    return g


@pytest.mark.parametrize("layer", LAYERS)
def test_choice_has_a_kernel_and_covers_the_layer(layer):
    g = build(layer)
    assert len(g.kernels) == 1                      # a split of K is folded inside the launch
    a = g.kernels[0]["attrs"]
    assert a[15] * a[16] >= a[0] * a[6] * a[7]      # split_k * k_chunk covers K
    assert g.kernels[0]["launch_params"][0] == a[15] * a[17] * a[18]


@pytest.mark.gpu
@pytest.mark.parametrize("layer", LAYERS)
def test_choice_computes_the_layer(layer, tmp_path):
    from oracle import oracle as O
    from reef_amd import binding as B
    g = build(layer)
    g.write(str(tmp_path))
    x = np.random.default_rng(5).standard_normal(layer[:3]).astype(np.float32)
    exe = B.Executor.from_dir(str(tmp_path), g.name, B.BASE)
    exe.set_input_checked("data", x)
    for _ in range(2):                              # the counters of a fold are ready for the next run
        exe.execute()
        got = exe.get_output()
        orc = O.GraphOracle(json.load(open(os.path.join(str(tmp_path), g.name + ".json"))), os.path.join(str(tmp_path), g.name + ".param"))
        orc.set_input("data", x)
        assert max_rel_err(got, orc.run()) <= REL_TOL
    exe.close()


def test_cost_table_names_tiles_and_kinds():
    for tile, kind in tiling.CONV_COST:
        assert tile in tiling.TILES and kind in "1s9npq"


# (cout, cin, taps, image side, under load): split entry and row form; the same for 1x1; an odd image, whose 1x1 layers have
# no kernel on whole lines; tap-form entries, unsplit and split, whose cost is near the row form's and above it; a staged entry; a split of
# two of the same tile, alone and under load
@pytest.mark.parametrize("cout,cin,taps,side,loaded,replaced", [
    (256, 256, 9, 14, False, True), (256, 1024, 1, 14, False, True), (512, 2048, 1, 7, False, False), (96, 96, 9, 35, False, False),
    (32, 128, 9, 56, False, True), (384, 448, 9, 8, False, False), (512, 512, 9, 7, False, True), (320, 64, 1, 56, False, False), (32, 128, 9, 14, False, False), (32, 128, 9, 14, True, True)])
def test_a_packed_layer_and_the_entry_of_its_shape(cout, cin, taps, side, loaded, replaced):
    M, N, K = cout, side * side, cin * taps
    kw = dict(fused=False, pointwise=taps == 1, taps=taps, direct=True, rows=taps == 9, image=(side, side), under_load=loaded)
    plain, packed = tiling.choose(M, N, K, **kw), tiling.choose(M, N, K, packed=True, **kw)
    key = (M, N, K, int(taps == 1))
    entry = tiling.TUNED_UNDER_LOAD[key] if loaded and key in tiling.TUNED_UNDER_LOAD else tiling.TUNED[key]
    assert (plain["tile"], plain["split_k"], plain["fused"]) == (entry[0], abs(entry[1]), entry[1] < 0)
    assert (packed != plain) == replaced
    if replaced:
        kind = tiling.conv_kind(packed["tile"], taps, 1, taps == 1, True, N, cin)
        assert kind in ("v", "w") and packed["split_k"] == 1 and not packed["fused"]
    else:
        assert packed == plain


def test_the_layers_of_the_image_patch_tests_run_on_image_patches():
    from reef_amd import binding as B
    from tests.test_gpu_image_patches import CASES
    assert {c[4] for c in CASES} == {4, 7}
    for cin, H, W, cout, rows in CASES:
        assert B.ops_conv2d_kernel(B.Conv2dDesc(cin, H, W, cout, 3, 3, 1, 1, 1, 1, 1)) == ("reef_conv2d_x9_g%d" % rows, 1)
    assert B.ops_conv2d_kernel(B.Conv2dDesc(254, 112, 112, 256, 3, 3, 1, 1, 1, 1, 1))[0].startswith("reef_conv2d_r9_")
    assert B.ops_conv2d_kernel(B.Conv2dDesc(4, 8, 8, 4, 3, 3, 0, 1, 1, 1, 0)) is None
