"""A whole-model run is submitted as recorded packets whose launches carry a few more workgroups that
bring the next launch's parameters into L2: every run holds the bits of the same model launched kernel
by kernel, in each flavour, over enough runs for the packet ring to wrap."""
import numpy as np
import pytest

from reef_amd import binding as B
from reef_amd.modelgen import nets
from tests.helpers import write_model

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
