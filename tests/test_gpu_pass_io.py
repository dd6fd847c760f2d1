"""Inputs stored straight into device memory and results mirrored to host memory by a recorded pass:
every order of inputs, passes, single launches and fetches sees what a run kernel by kernel sees."""
import ctypes

import numpy as np
import pytest

from reef_amd import binding as B
from reef_amd.modelgen import nets

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("pass_io"))
    g = nets.resnet(18, image=(3, 64, 64), classes=100, name="passio18")
    g.write(d)
    scores = g.kernels[-1]["args"][0]                      # what the softmax reads
    n_first = 64 * 16 * 16                                 # a storage in the middle, too large to be mirrored
    return d, g.name, scores, g.kernels[0]["args"][2], n_first, len(g.kernels)


def by_kernel(exe, x, n):
    exe.set_input_checked("data", x)
    for i in range(n):
        exe.execute_kernel(i)


@pytest.mark.parametrize("kind", [B.BASE, B.TRANS, B.HYBRID])
def test_every_order_sees_its_own_run(model, kind):
    d, name, scores, first, n_first, n = model
    exe, ref = B.Executor.from_dir(d, name, kind), B.Executor.from_dir(d, name, kind)
    run = {"pass": exe.execute}
    if kind == B.HYBRID:
        run["be"] = exe.execute_preemptable
    rng = np.random.default_rng(kind)
    order = ["pass"] * 4 + list(run) + ["kernels", "pass", "pass", "to", "kernels", "pass"] + list(run) * 2
    for step, how in enumerate(order):
        x = nets.image_input("passio", (3, 64, 64), 100 + step)
        by_kernel(ref, x, n)
        if how == "kernels":
            by_kernel(exe, x, n)
        elif how == "to":
            exe.set_input_checked("data", x)
            exe.execute_to(n - 1)
            exe.execute_kernel(n - 1)
        else:
            exe.set_input_checked("data", x)
            if step % 3 == 0:                              # what has just been stored can be fetched
                np.testing.assert_array_equal(exe.get_data(0, 3 * 64 * 64), x.reshape(-1))
            run[how]()
        for _ in range(int(rng.integers(1, 3))):
            np.testing.assert_array_equal(exe.get_output(), ref.get_output())
            np.testing.assert_array_equal(exe.get_data(scores, 100), ref.get_data(scores, 100))
            np.testing.assert_array_equal(exe.get_data(first, n_first), ref.get_data(first, n_first))
    # a fetch behind the next input still returns the last run's results
    want = exe.get_output()
    exe.set_input_checked("data", nets.image_input("passio", (3, 64, 64), 5))
    np.testing.assert_array_equal(exe.get_output(), want)
    exe.close()
    ref.close()


def test_a_mirrored_storage_that_is_written_is_read_back(model):
    d, name, scores, _, _, n = model
    exe = B.Executor.from_dir(d, name, B.BASE)
    for step in range(4):                                  # the scores join what the passes mirror
        exe.set_input_checked("data", nets.image_input("passio", (3, 64, 64), step))
        exe.execute()
        exe.get_data(scores, 100)
    v = np.arange(100, dtype=np.float32)
    assert B.lib().reef_executor_set_input_idx(exe.h, scores, ctypes.c_void_p(v.ctypes.data), ctypes.c_size_t(v.nbytes)) == 0
    np.testing.assert_array_equal(exe.get_data(scores, 100), v)
    exe.execute_kernel(n - 1)                              # softmax of what the host has written
    e = np.exp(v - v.max(), dtype=np.float32)
    np.testing.assert_allclose(exe.get_output(), e / e.sum(), rtol=1e-5, atol=1e-7)
    exe.close()


def test_parameters_loaded_again_between_passes(model, tmp_path):
    """The runtime's copies replace what the last pass has left in the caches: small parameters and ones of 2 MiB."""
    d, name, scores, _, _, _ = model
    g = nets.resnet(18, image=(3, 64, 64), classes=100, name=name)
    g.params = [(k, (a * np.float32(0.5)).astype(a.dtype) if a.dtype == np.float32 else a) for k, a in g.params]
    halved = str(tmp_path / "halved")
    g.write(halved)
    files = ["%s/%s.param" % (p, name) for p in (d, halved)]
    x = nets.image_input("passio", (3, 64, 64), 7)
    want = []
    for f in files:
        ref = B.Executor.from_dir(d, name, B.BASE)
        ref.load_param(f)
        by_kernel(ref, x, ref.num_kernels())
        want.append((ref.get_output(), ref.get_data(scores, 100)))
        ref.close()
    assert not np.array_equal(want[0][1], want[1][1])
    exe = B.Executor.from_dir(d, name, B.BASE)
    exe.set_input_checked("data", x)
    for step in range(8):
        exe.load_param(files[step % 2])
        for _ in range(1 + step // 4):
            exe.execute()
        np.testing.assert_array_equal(exe.get_output(), want[step % 2][0])
        np.testing.assert_array_equal(exe.get_data(scores, 100), want[step % 2][1])
    exe.close()
