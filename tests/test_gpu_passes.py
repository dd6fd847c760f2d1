"""A whole-model run is submitted as recorded packets whose launches carry a few more workgroups that
bring the next launch's parameters into L2: every run holds the bits of the same model launched kernel
by kernel, in each flavour, over enough runs for the packet ring to wrap."""
import threading
import time

import numpy as np
import pytest

from reef_amd import binding as B
from reef_amd.modelgen import nets
from tests.helpers import write_model
from tests.test_gpu_conv_op import device_layer

pytestmark = pytest.mark.gpu


def by_kernel(exe):
    for i in range(exe.num_kernels()):
        exe.execute_kernel(i)
    return exe.get_output()


@pytest.mark.parametrize("name,kind,preemptible", [("mocked", B.BASE, False), ("mobilenet_33", B.BASE, False), ("resnet_40", B.TRANS, False),
                                                   ("densenet_33", B.HYBRID, True), ("bert_9", B.HYBRID, True), ("bert_132", B.BASE, False)])
def test_recorded_pass_holds_the_bits_of_single_launches(tmp_path, name, kind, preemptible):
    net, _, size = name.partition("_")
    size = int(size or 0)
    g = {"mocked": nets.mocked_kernel, "mobilenet": lambda: nets.mobilenet_v2(image=(3, size, size), classes=10),
         "resnet": lambda: nets.resnet(50, image=(3, size, size), classes=10),
         "densenet": lambda: nets.densenet(blocks=(2, 3), image=(3, size, size), classes=10),
         "bert": lambda: nets.bert(layers=2, seq=size, vocab=64)}[net]()
    exe = B.Executor.from_dir(write_model(g, tmp_path), g.name, kind)
    rng = np.random.default_rng(3)
    for rep in range(2):
        if net == "mocked":
            for k in "abc":
                exe.set_input_checked(k, rng.standard_normal(8192).astype(np.float32))
        elif net == "bert":
            exe.set_input_checked("input0", rng.integers(0, 64, size))
        else:
            exe.set_input_checked("data", rng.standard_normal((3, size, size)).astype(np.float32))
        want = by_kernel(exe)
        assert np.isfinite(want).all() and want.any()
        for _ in range(1100 // exe.num_kernels() + 2):
            exe.execute_preemptable() if preemptible else exe.execute()
        np.testing.assert_array_equal(exe.get_output(), want)


def test_a_call_waits_for_no_pass_while_a_queue_is_free(tmp_path):
    """More models than there are queues, each run by another thread in turn: a single convolution beside it takes a small part
    of that model's pass."""
    g = nets.resnet(50, image=(3, 224, 224), classes=10)
    d = write_model(g, tmp_path)
    B.ops_init()
    layer, _, bufs, shape = device_layer((64, 14, 14, 64, 1, 1, 0, 1, True, True), 1)
    out = B.DeviceBuffer(4 * int(np.prod(shape)))

    def call():
        t = time.perf_counter()
        assert B.ops_conv2d(layer, *bufs, out, noalloc=True) == 0, B.last_error()
        return time.perf_counter() - t

    call()
    want = out.to_array()
    for _ in range(5):
        exe = B.Executor.from_dir(d, g.name, B.BASE)
        exe.set_input_checked("data", nets.image_input("passes", (3, 224, 224)))
        exe.execute()
        scores, passes, stop = exe.get_output(), [], threading.Event()

        def loop():
            while not stop.is_set():
                t = time.perf_counter()
                exe.execute()
                passes.append(time.perf_counter() - t)

        th = threading.Thread(target=loop)
        th.start()
        while len(passes) < 5:
            time.sleep(0.001)
        calls = [call() for _ in range(100)]
        stop.set()
        th.join()
        np.testing.assert_array_equal(exe.get_output(), scores)
        np.testing.assert_array_equal(out.to_array(), want)
        print("call %.0f us, pass %.0f us" % (1e6 * np.median(calls), 1e6 * np.median(passes)))
        assert np.median(calls) < 0.4 * np.median(passes)
        exe.close()
