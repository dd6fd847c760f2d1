"""x Phi(x) of the GELU epilogues against 64 bits: both pieces, where they meet, where the tail ends, and beyond."""
import os

import numpy as np
import pytest
from scipy.special import ndtr

from reef_amd import binding as B
from reef_amd.modelgen import builder as MB

pytestmark = pytest.mark.gpu


def test_gelu_against_64_bits(tmp_path):
    edges = [v for c in (0.0, 2.0 ** 0.5, 5.65, 1e-30, 1e-40, 1e30, 3.4e38) for e in (c, np.nextafter(np.float32(c), np.float32(9))) for v in (e, -e)]
    x = np.concatenate([np.linspace(-8, 8, 40000), edges, [np.inf, -np.inf, np.nan]]).astype(np.float32)
    x = np.concatenate([x, np.zeros(-x.size % 64, np.float32)])
    g = MB.GraphBuilder("gelu")
    out = g.bias_gelu(g.input("x", (x.size // 64, 64)), x.size // 64, 64, bias=False)
    g.mark_output(out)
    g.write(os.path.join(str(tmp_path), "gelu"))
    exe = B.Executor.from_dir(os.path.join(str(tmp_path), "gelu"), "gelu", B.BASE)
    exe.set_input_checked("x", x)
    exe.execute()
    y = exe.get_data(out.idx, x.size)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) * ndtr(x.astype(np.float64))
    ok = np.isfinite(x)
    assert (y[np.isposinf(x)] == np.inf).all() and np.isnan(y[np.isnan(x) | np.isneginf(x)]).all()
    # two roundings of Phi and of the product, and the tail behind 5.65: 5.65 Phi(-5.65)
    assert (np.abs(y[ok] - want[ok]) <= 2.0 ** -23 * np.abs(x[ok].astype(np.float64)) + 4.6e-8).all()
