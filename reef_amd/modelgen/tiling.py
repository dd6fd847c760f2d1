"""Tile and split-K choice for the implicit-GEMM convolution / GEMM kernels.

The reference takes grid and block sizes from TVM's tuned schedules
(script/generate_final_schedule.py:98: launch_params come from the raw
schedule).  Here the generator picks, per layer, one of the compiled tile
configurations and a split-K factor from a small analytic cost model of a
256-CU part: batch-1 layers are tiny (49..3136 output pixels), so most need
split-K to put a workgroup on every CU.
"""
import math

from .tuned import TUNED, TUNED_UNDER_LOAD, GEMM_UNDER_LOAD

# name -> (id, BM, BN, relative MFMA efficiency of the inner loop, workgroups per CU)
TILES = {
    "128x128": (0, 128, 128, 1.00, 2),
    "128x64": (1, 128, 64, 0.85, 2),
    "64x64": (2, 64, 64, 0.60, 4),
    "128x32": (3, 128, 32, 0.60, 3),
    "32x128": (4, 32, 128, 0.60, 3),
    "64x128": (5, 64, 128, 0.85, 2),
    # k<n>: the workgroup's four wavefronts split K n ways on one small tile
    "32x32k4": (6, 32, 32, 0.50, 2),
    "64x32k2": (7, 64, 32, 0.55, 3),
    "32x64k2": (8, 32, 64, 0.55, 3),
    # direct family (reef_conv2d_d<taps>_16x16k4): picked through the measured table, an explicit
    # request, or for a shape outside the table by the cost model direct_cost below
    "16x16k4": (9, 16, 16, 0.40, 2),
    "16x32k4": (10, 16, 32, 0.40, 2),
    "16x64k4": (11, 16, 64, 0.40, 2),
    "32x32d4": (12, 32, 32, 0.40, 2),   # direct; the name differs from the staged 32x32k4
    # row form of the direct 3x3 / stride 1 / padding 1 convolution (reef_conv2d_r9_<name>): BM output
    # channels x G image rows x one 14-column segment; BN here is the nominal 16 G lanes it computes
    "g1": (13, 16, 16, 0.40, 2),
    "g2": (14, 16, 32, 0.40, 2),
    "g4": (15, 16, 64, 0.40, 2),
    "g7": (16, 16, 112, 0.40, 2),
    "g2m2": (17, 32, 32, 0.40, 2),
    "g4m2": (18, 32, 64, 0.40, 2),
}
# matrix products only (reef_gemm_ntd_<tile>, reef_gemm_ntl_<tile>): name -> (id, BM, BN)
GEMM_WIDE_TILES = {"32x48d4": (19, 32, 48), "48x48d4": (20, 48, 48), "64x64d4": (21, 64, 64)}
GEMM_SPLIT_TILES = ("32x32d4",) + tuple(GEMM_WIDE_TILES)      # direct tiles that take packed weights as three bf16 parts
GEMM_SPLIT_BYTES = 1 << 32         # their offsets are 32 bits: larger copies stay 32-bit values, which are two thirds of that
V9_TILES = ("g1", "g2", "g4")      # row tiles that exist as reef_conv2d_v9_<tile>
# row form: image rows per tile
ROW_TILES = {"g1": 1, "g2": 2, "g4": 4, "g7": 7, "g2m2": 2, "g4m2": 4}
ROW_SEG = 14
DIRECT_TILE = "16x16k4"
DIRECT_TILES = ("16x16k4", "16x32k4", "16x64k4", "32x32d4")
# filter sizes kh*kw each direct tile is compiled for
PRE_ACT_TILES = ("16x16k4", "16x32k4", "32x32d4")   # tiles with a pre-activation 1x1 kernel (reef_conv2d_p1_*)
DIRECT_TAPS = {"16x16k4": (1, 3, 7, 9, 25), "16x32k4": (1, 3, 7, 9, 25), "16x64k4": (1, 9), "32x32d4": (1, 9)}
# wavefronts that share one output block and split K inside the workgroup
KW = {"32x32k4": 4, "64x32k2": 2, "32x64k2": 2}
GEMM_TILES = ("128x128", "64x64", "32x128", "32x32k4", "64x32k2")


GEMM_DIRECT_TILES = ("16x16k4", "16x32k4", "32x32d4")   # reef_gemm_ntd_<tile>


def choose_gemm(M, N, K, batch=1, direct_ok=False, under_load=False):
    """Tile of a GEMM, and for a direct tile whether K is split in two across workgroups.
    Without a measured table: the staged choice of the analytic model, against the direct tiles
    (both operands K-contiguous) scored by the rule the batch-1 convolutions were found to
    follow -- a workgroup's time grows with the cache lines it has to pull in, (BM + BN) K / 32
    of them, and workgroups beyond one per CU queue up.  A split of two (folded inside the
    launch through the pair slots) halves a workgroup's lines and doubles the workgroups, at a
    price measured on BERT-base's 128 x 768 x 3072 product (32x32d4: 25.8 us whole, 16.8 us
    split in two, against 19.4 us for 16x32k4 whole; splits of three and more meet on counters
    and were slower throughout).
    under_load: the product belongs to a model that shares the device with other streams; a
    choice measured for that case (tuned.GEMM_UNDER_LOAD) comes first."""
    if under_load and direct_ok and batch == 1 and (M, N, K) in GEMM_UNDER_LOAD:
        tile, split = GEMM_UNDER_LOAD[(M, N, K)]
        t = forced(tile, M, N, K, 1)
        t["gemm_split"] = split
        return t
    staged = choose(M, N, K, allow_split=False, tiles=GEMM_TILES)
    if not direct_ok:
        return staged

    def cost(bm, bn, split=1):
        wgs = batch * math.ceil(M / bm) * math.ceil(N / bn) * split
        return math.ceil(wgs / NUM_CUS) * (bm + bn) * (K / split) / 32.0 + (GEMM_PAIR_FOLD_LINES if split == 2 else 0)
    cands = [(t, 1) for t in GEMM_DIRECT_TILES]
    if batch == 1 and K >= 1024:
        cands += [(t, 2) for t in GEMM_DIRECT_TILES]
    best, split = min(cands, key=lambda c: (cost(TILES[c[0]][1], TILES[c[0]][2], c[1]), c[1],
                                            -TILES[c[0]][1] * TILES[c[0]][2]))
    _, bm, bn, _, _ = TILES[staged["tile"]]
    if cost(bm, bn) * GEMM_STAGED_BONUS <= cost(TILES[best][1], TILES[best][2], split):
        return staged
    t = forced(best, M, N, K, 1)
    t["gemm_split"] = split
    return t


# Microseconds of a product (tile, reads its rows through a LayerNorm), fitted as CONV_COST is, in the form
# of _cost with whole rounds of workgroups: 16 sequence lengths of 8 to 512 times 13 layer shapes of 256 to 4096 columns and
# a depth of 256 to 4096, splits of 1 to 6, 3100 launches on MI355X; it picks within 0.3 % of the fastest
# launch on average (worst 7 %).  Without the three wide direct tiles it would lose 4 to 5 %.
GEMM_COST = {
    ("16x16k4", False): (2.534, 0.3324, 2.843, 0.4488, 0.2743, 1.799, 1.127),
    ("16x16k4", True): (3.635, 0.17, 3.258, 0.04108, 0.4272, 0, 0),
    ("16x32k4", False): (2.691, 0.6074, 4.59, 0.2421, 0.4406, 1.636, 2.151),
    ("16x32k4", True): (3.518, 1.365, 4.748, 0, 0.5508, 0, 0),
    ("32x32d4", False): (2.801, 0, 5.975, 1.091, 1.507, 1.92, 1.86),
    ("32x48d4", False): (3.211, 0.1859, 8.06, 0.3396, 1.479, 2.465, 2.754),
    ("32x48d4", True): (4.578, 0.2621, 8.58, 0, 1.171, 0, 0),
    ("48x48d4", False): (3.424, 0.6952, 9.742, 0, 2.909, 2.943, 2.692),
    ("48x48d4", True): (5.234, 0, 11.05, 0, 1.908, 0, 0),
    ("64x64d4", False): (4.323, 0, 15.27, 0, 6.721, 2.321, 5.733),
    ("64x64d4", True): (6.322, 0, 18.41, 0, 2.093, 0, 0),
    ("32x32k4", False): (3.647, 2.504, 3.621, 0.3601, 0.5328, 0, 0),
    ("32x32k4", True): (5.233, 0.809, 4.395, 2.123, 0.502, 0, 0),
    ("64x32k2", False): (4.431, 12.06, 0, 0, 0.5025, 0, 0),
    ("64x32k2", True): (5.956, 3.589, 7.457, 1.34, 0.4235, 0, 0),
}
# The same for the direct kernels on packed weights (reef_kernels.h, ldb = 0; from 32x32 on split ones): 12 sequence lengths
# of 16 to 512 times 13 layer shapes of 256 to 4096 columns and depth, 2087 launches.  It picks within 1.5 % of the fastest
# launch on average, by the table of the same tiles on 32-bit weights 5.6 %.  The 16-row tiles that split K keep
# the coefficients of that table (all measured anew: 1.0 %), which split the products of 8 to 64 rows finer or alike: with the
# new ones a network of 24 rows is 7 % faster and its distance from 64 bits 3 % larger.
GEMM_COST_PACKED = {
    ("16x16k4", False): (3.735, 0, 0.1841, 1.183, 0.01631, 0, 3.281),
    ("16x16k4", True): (2.926, 0.7903, 1.179, 0.5716, 0.3408, 0, 0),
    ("16x32k4", False): (3.405, 0, 1.262, 0.9671, 0.2277, 0, 4.159),
    ("16x32k4", True): (3.315, 0.4111, 1.854, 0.8625, 0.5116, 0, 0),
    ("32x32d4", False): (2.774, 1.242, 1.86, 1.274, 0.8819, 0, 6.57),
    ("32x48d4", False): (2.977, 0.7474, 3.161, 0.8269, 1.442, 0, 8.945),
    ("32x48d4", True): (3.947, 0.9158, 2.47, 2.651, 1.316, 0, 0),
    ("48x48d4", False): (2.441, 0, 6.958, 0, 3.176, 0, 11.35),
    ("48x48d4", True): (3.385, 0, 8.917, 0, 2.992, 0, 0),
    ("64x64d4", False): (2.969, 0, 9.973, 0, 5.348, 0, 16.48),
    ("64x64d4", True): (3.781, 0, 14.86, 0, 3.562, 0, 0),
}
GEMM_COST_MIN, GEMM_COST_MAX_OUT = 256, 512 * 4096     # columns and depth from which, outputs up to which it was measured


def choose_product(M, N, K, batch=1, direct_ok=False, under_load=False, ln=False, packed=False):
    """Tile (and split of K, gemm_split) of a matrix product: inside the measured range by GEMM_COST, outside
    it by choose_gemm (behind a LayerNorm: the staged 32x32k4, which takes every shape).
    under_load: as in choose_gemm.  packed: the direct kernels will find packed weights (GEMM_COST_PACKED)."""
    if (under_load or packed) and direct_ok and not ln and batch == 1 and (M, N, K) in GEMM_UNDER_LOAD:
        return choose_gemm(M, N, K, batch, direct_ok, True)
    if batch == 1 and direct_ok and min(N, K) >= GEMM_COST_MIN and M * N <= GEMM_COST_MAX_OUT:
        best = None
        for (tile, through_ln), c in (GEMM_COST_PACKED if packed else GEMM_COST).items():
            if through_ln != ln:
                continue
            staged = tile not in DIRECT_TILES and tile not in GEMM_WIDE_TILES
            for s in (1,) if ln or staged else (1, 2, 3, 4, 6):
                t = forced(tile, M, N, K, s)
                if t["split_k"] == s:
                    us = _cost(c, t["k_chunk"] if s > 1 else K, t["tasks"], s, math.ceil(t["tasks"] / NUM_CUS))
                    if best is None or us < best[0]:
                        best = (us, dict(t, gemm_split=s, est_us=us))
        return best[1]
    if ln:
        return forced("32x32k4", M, N, K, 1)
    return choose_gemm(M, N, K, batch, direct_ok, under_load)


def takes_split(tile, N, K):
    """Whether the tile runs a product with [N][K] packed weights on three parts of each."""
    return tile in GEMM_SPLIT_TILES and math.ceil(N / 16) * math.ceil(K / 32) * 3072 < GEMM_SPLIT_BYTES


GEMM_PAIR_FOLD_LINES = 900.0    # what a split of two costs, in the cost rule's cache lines
GEMM_STAGED_BONUS = 1.0


def step_k(tile, taps=1):
    """Granularity of a split's share of K (taps = kh*kw, direct family only: 16 channels of a
    filter with taps > 1, one K step; 128 channels of a 1x1 filter, two of its 64-channel steps --
    rounding to 64 instead was measured on DenseNet-201 and changes nothing)."""
    if tile in DIRECT_TILES or tile in GEMM_WIDE_TILES:
        return 128 if taps == 1 else 16 * taps
    return BK * KW.get(tile, 1)


def direct_ok(cin, kh, kw, tile=DIRECT_TILE):
    """Whether the direct family has a kernel for this filter (and tile)."""
    taps = kh * kw
    if taps not in DIRECT_TAPS[tile]:
        return False
    return taps > 1 or cin % 8 == 0


def rows_ok(kh, kw, sh, sw, ph, pw):
    """Whether the row form has a kernel for this filter."""
    return (kh, kw, sh, sw, ph, pw) == (3, 3, 1, 1, 1, 1)


def forced_rows(tile, M, H, W, K, split=1):
    """Launch geometry of a row-form tile: spatial tiles are G image rows x one 14-column segment."""
    tid, bm, _, _, _ = TILES[tile]
    G = ROW_TILES[tile]
    bk = 16 * 9
    k_chunk = math.ceil(math.ceil(K / split) / bk) * bk
    s = math.ceil(K / k_chunk)
    mt = math.ceil(M / bm)
    nt = math.ceil(H / G) * math.ceil(W / ROW_SEG)
    return dict(tile=tile, tile_id=tid, BM=bm, BN=16 * G, split_k=s, k_chunk=k_chunk, m_tiles=mt,
                n_tiles=nt, tasks=s * mt * nt, est_us=1.0)


def forced(tile, M, N, K, split=1, taps=1):
    """The launch geometry of a given tile and split-K factor (no cost model)."""
    assert tile not in ROW_TILES, "row-form tiles take the image shape: forced_rows"
    tid, bm, bn = GEMM_WIDE_TILES[tile] if tile in GEMM_WIDE_TILES else TILES[tile][:3]
    bk = step_k(tile, taps)
    k_chunk = math.ceil(math.ceil(K / split) / bk) * bk
    s = math.ceil(K / k_chunk)
    mt, nt = math.ceil(M / bm), math.ceil(N / bn)
    return dict(tile=tile, tile_id=tid, BM=bm, BN=bn, split_k=s, k_chunk=k_chunk, m_tiles=mt,
                n_tiles=nt, tasks=s * mt * nt, est_us=1.0)

NUM_CUS = 256
BK = 32
# Cost model constants (microseconds); calibrated against measured kernels.
T_STEP_128x128 = 1.9     # one BK=32 step of a 128x128 tile on one CU at efficiency 1.0
T_FIXED = 2.0            # prologue + epilogue of a workgroup
T_REDUCE_LAUNCH = 3.0    # extra launch of the split-K reduce
T_FUSED_REDUCE = 1.0     # fence + last-arrival fold inside the conv kernel
HBM_BYTES_PER_US = 4.0e6
# The constants above describe a workgroup in a long, warm run; in a model (cold operands, one
# launch per layer) the staged tiles measure about three times that, on small and on
# device-filling layers alike (sweeps behind tuned.py; bench.py's steady_state_conv).  With the
# factor the estimate is in the same microseconds as direct_cost, and choosing between the two
# families by estimate loses 7 % against the measured best over the 181 shapes of the sweeps.
STAGED_SCALE = 3.0


def _steps_time(bm, bn, eff, steps):
    return steps * T_STEP_128x128 * (bm * bn) / (128.0 * 128.0) / eff


def choose(M, N, K, allow_split=True, tiles=None, max_split=32, fused=True, pointwise=False,
           taps=1, direct=False, rows=False, image=None, under_load=False, stride=1, pre_act=False, packed=False):
    """Returns dict(tile, tile_id, BM, BN, split_k, k_chunk, m_tiles, n_tiles, tasks).
    Measured choices (tuned.py) win over the analytic model for the shapes they cover; an entry
    that names the direct tile counts only if the caller says the filter qualifies.
    under_load: the layer belongs to a model that shares the device with other streams; the
    entries measured for that case (TUNED_UNDER_LOAD) come before those measured alone.
    packed: the layer's weights will be packed, so that it runs on the kernels that take whole cache lines
    (v1_ok, the row tiles' v9), which the entries were not measured with: see over_entry.
    image: output rows and columns of a convolution (with stride, pre_act: the input goes through an
    activation of its own); shapes outside the table are then chosen by the measured cost of every
    tile (CONV_COST), those of a bare matrix product by the analytic model."""
    if allow_split and tiles is None and not fused:
        key = (M, N, K, 1 if pointwise else 0)
        hit = TUNED.get(key)
        if under_load and key in TUNED_UNDER_LOAD:
            hit = TUNED_UNDER_LOAD[key] + (hit[2] if hit is not None else 0.0,)
        if hit is not None and hit[0] in ROW_TILES and not (rows and image is not None):
            hit = None
        if hit is not None and (hit[0] not in DIRECT_TILES or direct):
            # a negative split factor in the table: the split is folded inside the launch
            if hit[0] in ROW_TILES:
                t = forced_rows(hit[0], M, image[0], image[1], K, abs(hit[1]))
            else:
                t = forced(hit[0], M, N, K, abs(hit[1]), taps)
            t["est_us"] = hit[2]
            t["fused"] = hit[1] < 0
            if packed and image is not None:
                best = _choose_conv(M, N, K, taps, direct, rows, image, stride, pointwise, pre_act, True)
                if over_entry(best, t, taps, stride, pointwise, N, K, pre_act, under_load):
                    return best
            return t
    if allow_split and tiles is None and (image is not None or direct and M * N <= NUM_CUS * 4096):
        return _choose_conv(M, N, K, taps, direct, rows and image is not None, image, stride, pointwise, pre_act, packed)
    best = None
    for name in (tiles or [t for t in TILES if t not in DIRECT_TILES and t not in ROW_TILES]):
        tid, bm, bn, eff, occ = TILES[name]
        m_tiles, n_tiles = math.ceil(M / bm), math.ceil(N / bn)
        nt = m_tiles * n_tiles
        splits = [1]
        if allow_split:
            splits += [s for s in (2, 3, 4, 6, 8, 12, 16, 24, 32) if s <= max_split]
        bk = step_k(name)
        for s in splits:
            k_chunk = math.ceil(math.ceil(K / s) / bk) * bk
            s_eff = math.ceil(K / k_chunk)
            if s_eff != s and s != 1:
                continue
            wgs = nt * s_eff
            rounds = math.ceil(wgs / (NUM_CUS * occ))
            # co-resident workgroups share the CU's matrix pipe
            share = min(occ, math.ceil(wgs / NUM_CUS))
            t = rounds * (_steps_time(bm, bn, eff, k_chunk // bk) * share + T_FIXED)
            if s_eff > 1:
                t += (T_FUSED_REDUCE if fused else T_REDUCE_LAUNCH) + (s_eff + 1) * M * N * 4 / HBM_BYTES_PER_US
            t *= STAGED_SCALE
            cand = (t, name, s_eff, k_chunk, m_tiles, n_tiles)
            if best is None or cand[0] < best[0] - 1e-9:
                best = cand
    t, name, s, k_chunk, m_tiles, n_tiles = best
    tid, bm, bn, _, _ = TILES[name]
    return dict(tile=name, tile_id=tid, BM=bm, BN=bn, split_k=s, k_chunk=k_chunk,
                m_tiles=m_tiles, n_tiles=n_tiles, tasks=s * m_tiles * n_tiles, est_us=t)


# Cost of a convolution launch in microseconds, for shapes the measured table does not cover: per
# tile and kind of filter,
#     c0 + w (c1 + c2 (r + ceil(r)) / 2 + c3 max(1, r)) + c4 r   (+ c5 + c6 split / 10 where K is split)
# with w = a workgroup's share of K in thousands and r = workgroups per CU.  c1 is the serial chain
# of one workgroup, c2 and c3 what the CU's matrix pipes and loads need for all of its workgroups,
# c4 the start and end of each, c5 and c6 the fold of a split inside the launch.  Fitted (non-negative
# least squares on relative error, candidates near the best of their shape weighted up) to 21 600
# candidates over 782 layer shapes of the image networks at image sizes of 64 to 448 and twelve
# device-filling layers, timed as launches of one long model.  Choosing by it costs 5 % on average
# against the measured best of every shape (the linear model of the direct family alone with the
# staged tiles' estimate scaled by 3, which was fitted at 224: 18 %, and up to 3x on layers of more
# than 500 pixels, which it left to the staged tiles).
# Kinds: "1" 1x1 stride 1 and "s" 1x1 strided on the direct tiles; on the staged ones "p" the
# pointwise loader, "q" a 1x1 filter it cannot take, "s" strided; "9" 3x3; "n" any other filter.
CONV_COST = {
    ("16x16k4", "1"): (3.864, 0, 2.361, 0, 0.176, 0, 0.87),
    ("16x16k4", "s"): (3.929, 0, 2.743, 0.246, 0.445, 0, 0),
    ("16x16k4", "9"): (3.08, 1.304, 1.368, 0, 0.564, 0.17, 2.749),
    ("16x16k4", "n"): (3.329, 0.182, 1.761, 0.453, 0.274, 0, 2.575),
    ("16x32k4", "1"): (3.902, 0, 3.553, 0.038, 0.222, 0, 1.036),
    ("16x32k4", "s"): (3.863, 0, 4.739, 0, 0.57, 0, 0),
    ("16x32k4", "9"): (3.636, 2.107, 2.124, 0, 0.83, 0.389, 2.679),
    ("16x32k4", "n"): (2.934, 0.083, 3.144, 1.977, 0.306, 0.583, 2.758),
    ("16x64k4", "1"): (3.953, 0.388, 3.741, 2.128, 0.669, 0, 2.147),
    ("16x64k4", "s"): (4.082, 0, 8.982, 0, 1.094, 0, 0),
    ("16x64k4", "9"): (4.756, 3.955, 4.628, 0.196, 1.746, 0.241, 2.752),
    ("32x32d4", "1"): (3.907, 1.517, 4.385, 0.45, 0.818, 0, 3.727),
    ("32x32d4", "s"): (4.102, 0, 8.38, 0, 0.884, 0.202, 0.67),
    ("32x32d4", "9"): (4.484, 2.719, 3.542, 0.286, 1.081, 0.01, 4.04),
    ("g1", "9"): (3.549, 0.474, 1.311, 0, 0.248, 0.102, 2.009),
    ("g2", "9"): (3.727, 1.089, 1.993, 0, 0.351, 0.025, 2.573),
    ("g4", "9"): (4.29, 1.461, 2.599, 1.143, 0.715, 0.103, 3.085),
    ("64x64", "s"): (9.068, 14.79, 19.38, 5.296, 1.646, 6.436, 0),
    ("64x64", "9"): (9.626, 17.47, 18.78, 4.938, 0.945, 6.364, 0),
    ("64x64", "n"): (6.715, 32.23, 13.12, 0, 0.74, 6.959, 0),
    ("64x64", "p"): (6.828, 8.68, 7.25, 6.944, 1.996, 7.122, 0),
    ("64x64", "q"): (7.02, 30.34, 15.1, 0, 2.243, 6.398, 0),
    ("128x32", "s"): (8.123, 18.61, 10.09, 2.462, 2.242, 7.287, 0),
    ("128x32", "9"): (8.851, 11.91, 12.4, 8.535, 1.186, 5.927, 0),
    ("128x32", "n"): (7.783, 29.36, 1.753, 0, 0, 6.173, 0),
    ("128x32", "p"): (6.496, 10.34, 6.87, 6.631, 2.695, 6.766, 0),
    ("128x32", "q"): (6.557, 3.254, 2.007, 27.51, 3.213, 6.061, 0),
    ("64x32k2", "s"): (6.11, 5.167, 6.082, 8.086, 1.944, 3.971, 0),
    ("64x32k2", "9"): (6.353, 6.917, 6.546, 7.894, 1.763, 3.457, 0),
    ("64x32k2", "n"): (5.643, 19.9, 0, 0, 1.828, 4.177, 0),
    ("64x32k2", "p"): (4.947, 4.238, 5.818, 3.177, 1.217, 4.379, 0),
    ("64x32k2", "q"): (5.417, 0, 2.793, 18.77, 1.872, 3.878, 0),
    ("32x64k2", "s"): (7.462, 8.888, 17.1, 2.856, 0.841, 3.958, 0),
    ("32x64k2", "9"): (8.526, 12.45, 15.32, 2.858, 0.694, 3.183, 0),
    ("32x64k2", "n"): (5.941, 28.4, 0, 0, 1.546, 4.225, 0),
    ("32x64k2", "p"): (5.524, 1.379, 3.516, 6.325, 1.184, 4.288, 0),
    ("32x64k2", "q"): (6.407, 11.94, 2.272, 13.94, 2.239, 3.673, 0),
    ("32x32k4", "s"): (6.845, 0, 6.321, 5.181, 1.577, 1.65, 0),
    ("32x32k4", "9"): (6.803, 4.635, 1.99, 8.083, 1.942, 1.107, 0),
    ("32x32k4", "n"): (5.74, 0, 5.897, 11.65, 0.09, 1.704, 1.883),
    ("32x32k4", "p"): (4.406, 1, 2.163, 3.927, 1.29, 2.115, 0),
    ("32x32k4", "q"): (6.071, 2.839, 0, 10.58, 2.008, 1.917, 0),
}
# The same for the kernels on packed weights that take whole cache lines: "v" 1x1 (reef_conv2d_v1_*), "w" 3x3
# (reef_conv2d_v9_*).  340 layer shapes of the same networks at 64 to 448, 3700 candidates; choosing by it costs
# 5 % (1x1) and 2 % (3x3) on average against the measured best of a shape.
CONV_COST_PACKED = {
    ("16x16k4", "v"): (4.001, 0, 1.59, 0, 0.1832, 0, 1.203),
    ("16x32k4", "v"): (3.821, 0, 3.041, 0, 0.2629, 0, 1.921),
    ("16x64k4", "v"): (3.469, 0, 3.819, 2.785, 0.8784, 0, 3.612),
    ("32x32d4", "v"): (3.444, 1.303, 2.86, 1.301, 0.7217, 0, 4.165),
    ("g1", "w"): (3.502, 0.1328, 0.9924, 0.07493, 0.3518, 0, 2.982),
    ("g2", "w"): (3.258, 0.2351, 1.289, 0.7421, 0.7164, 0, 4.338),
    ("g4", "w"): (3.564, 0, 1.267, 2.714, 1.729, 0, 5.952),
}
PRE_ACT_LAUNCH_US = 6.0   # a pre-activation launch of its own, in front of a tile without the form


# Input channels from which a plain 1x1 layer of these tiles loads its input in 16-byte pieces; below, the kernel that
# loads single values starts sooner.  Device time of whole passes: MobileNet-v2 (16x16k4, 144 to 576 channels)
# 154.6 us with all of them in pieces, 153.4 from 256 channels, 152.5 from 512, 151.6 with none; ResNet-152 (16x32k4)
# 836 with all, 832 from 65, 829 from 129 or 192, 842 from 257; ResNet-50 at 448 656 and 645 from 256.  Layers with
# a pre-activation and 32x32d4 gain at every size (DenseNet-201's best-effort kernels 1037 us, 1041 from 512; ResNet-50 at
# 448 645, 647 from 129, 654 from 513).
V1_MIN_CIN = {"16x16k4": 640, "16x32k4": 256}


def v1_ok(kh, kw, sh, sw, ph, pw, n_pixels, tile, cin, pre):
    """Whether a 1x1 layer on packed weights loads its input in 16-byte pieces (reef_conv2d_v1_*)."""
    return (kh, kw, sh, sw, ph, pw) == (1, 1, 1, 1, 0, 0) and n_pixels % 4 == 0 and (
        pre or cin >= V1_MIN_CIN.get(tile, 0))


def conv_kind(tile, taps, stride=1, pointwise=True, packed=False, n_pixels=0, cin=0, pre=False):
    if taps != 1:
        return "w" if packed and tile in V9_TILES else "9" if taps == 9 else "n"
    if stride > 1:
        return "s"
    if tile in DIRECT_TILES:
        return "v" if packed and n_pixels % 4 == 0 and (pre or cin >= V1_MIN_CIN.get(tile, 0)) else "1"
    return "p" if pointwise else "q"


def direct_cost(tile, geom, fused=True, kind="1"):
    """Microseconds of a launch of this geometry (forced, forced_rows) by CONV_COST."""
    s = geom["split_k"]
    r = geom["tasks"] / NUM_CUS
    us = _cost((CONV_COST_PACKED if kind in "vw" else CONV_COST)[(tile, kind)], geom["k_chunk"], geom["tasks"], s, (r + math.ceil(r)) / 2)
    return us + T_REDUCE_LAUNCH if s > 1 and not fused else us


# Part of a tap-form entry's cost below which the row form on whole cache lines replaces it (over_entry).  Gain: 32 x 784 x 1152
# and 32 x 3136 x 1152 of DenseNet-201 (0.83, 0.72: as a best-effort model 1004 -> 986 us with the second), 512 x 49 x 4608 of
# ResNet-152 (0.86).  Lose: Inception-v3's 384 x 64 x 4032 (0.875: 456.0 -> 457.5 us; its rows of 8 pixels fill 8 of 14
# columns), 96 x 1225 x 576 and 864 (0.89, 0.93: 457.5 -> 461.2).
ROWS_OVER_TAPS = 0.87


def over_entry(best, entry, taps, stride, pointwise, n_pixels, K, pre, under_load):
    """Whether a layer on packed weights takes the cost rule's choice and not the measured entry of its shape: where
    the choice is an unsplit kernel on whole cache lines and the entry splits K, or is a tap-form 3x3 kernel of a
    higher cost.  The entries were measured before these kernels.  Their splits fill the device where a workgroup
    waited for its loads; the kernels on whole lines wait less, and an exchange between two workgroups is 2100
    cycles of 14 600.  (A split of two of the same tile stays where the model is alone, where it is one exchange: DenseNet-201
    885 us either way.  Under load it meets on counters: 996 -> 986.)  Device time of a pass, entries only and by
    this rule: ResNet-152 911 -> 820 us, ResNet-50 313 -> 302, ResNet-18 149.3 -> 145.7, DenseNet-201 902 -> 885 and 1110 ->
    986 as a best-effort model; with every entry replaced that way, split or not, ResNet-152 821, MobileNet-v2 149.4 ->
    152.6 and Inception-v3 456 -> 460.6."""
    kind, was = (conv_kind(t["tile"], taps, stride, pointwise, True, n_pixels, K // taps, pre) for t in (best, entry))
    if kind not in ("v", "w") or best["split_k"] > 1:
        return False
    if was == "9":
        return (entry["tile"], was) in CONV_COST and best["est_us"] < ROWS_OVER_TAPS * direct_cost(entry["tile"], entry, True, was)
    return entry["split_k"] > 1 and (under_load or entry["split_k"] > 2 or entry["tile"] != best["tile"])


def _cost(c, depth, tasks, split, rounds):
    """The fitted form of CONV_COST and GEMM_COST: `tasks` workgroups over `depth` values of K each."""
    w, r = depth / 1000.0, tasks / NUM_CUS
    t = c[0] + (c[1] + c[2] * rounds + c[3] * max(1.0, r)) * w + c[4] * r
    return t + c[5] + 0.1 * c[6] * split if split > 1 else t


def _choose_conv(M, N, K, taps, direct, rows, image, stride, pointwise, pre_act, packed=False):
    """Cheapest tile and split of a convolution by CONV_COST; a split is folded inside the launch."""
    best = None
    pointwise = pointwise and stride == 1 and N % 4 == 0 and K % 4 == 0
    for tile in TILES:
        if tile in ROW_TILES and not rows:
            continue
        if tile in DIRECT_TILES and not (direct and taps in DIRECT_TAPS[tile]):
            continue
        kind = conv_kind(tile, taps, stride, pointwise, packed and image is not None, N, K // taps, pre_act)
        if (tile, kind) not in CONV_COST and (tile, kind) not in CONV_COST_PACKED:
            continue
        for s in (1, 2, 3, 4, 6, 8):
            g = forced_rows(tile, M, image[0], image[1], K, s) if tile in ROW_TILES else forced(tile, M, N, K, s, taps)
            if g["split_k"] != s:
                continue
            t = direct_cost(tile, dict(g, k_chunk=min(g["k_chunk"], K)), True, kind)
            if pre_act and tile not in PRE_ACT_TILES:
                t += PRE_ACT_LAUNCH_US
            if image is None:
                t *= 1.0 + 0.04 * max(0.0, 1.0 - g["tasks"] / NUM_CUS)   # of two alike, the one that leaves fewer CUs idle
            if best is None or t < best[0] - 1e-9:
                g["est_us"] = t
                g["fused"] = s > 1
                best = (t, g)
    return best[1]


def lds_bytes(tile):
    if tile in GEMM_WIDE_TILES:
        return 4 * (GEMM_WIDE_TILES[tile][1] // 16) * (GEMM_WIDE_TILES[tile][2] // 16) * 320 * 4 + 16
    if tile in DIRECT_TILES or tile in ROW_TILES:
        # four wavefronts x (BM/16)(BN/16) partial 16x16 tiles (skewed rows) + leave / last-arrival flags
        return 4 * (TILES[tile][1] // 16) * (TILES[tile][2] // 16) * 320 * 4 + 16
    _, bm, bn, _, _ = TILES[tile]
    bk = step_k(tile)
    a = bm * (bk + 4)
    b = max(bk * bn, bn * (bk + 4))
    return 2 * (a + b) * 4 + 16
