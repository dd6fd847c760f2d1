"""What a model keeps between a run and the fetches behind it -- the mirror of the last run, what a fetch has copied --
on the recording backend with passes switched on: a fetch returns what the storages hold, whenever it comes."""
import os
import time

import numpy as np
import pytest

from reef_amd import binding as B
from reef_amd.modelgen import builder as MB, nets
from tests.fakehal import FakeHal
from tests.helpers import write_model

N = 8192


@pytest.fixture()
def fake():
    f = FakeHal().install()
    f.set_passes()
    yield f
    f.remove()


@pytest.fixture(scope="module")
def mocked(tmp_path_factory):
    g = nets.mocked_kernel()
    return g.name, write_model(g, tmp_path_factory.mktemp("mocked"))


def set_inputs(set_input, v):
    for k in "abc":
        set_input(k, np.full(N, v, np.float32))


def wait_for(cond):
    end = time.time() + 20
    while not cond():
        assert time.time() < end
        time.sleep(0.001)


def test_a_fetch_during_a_best_effort_run_leaves_nothing_for_the_one_after_it(fake, mocked):
    name, d = mocked
    s = B.Scheduler(B.MODE_REEF)
    m = s.load_model(d, name)
    s.bind_model_queue(s.create_queue(B.QUEUE_BE), m)
    for v in (3.0, 4.0):
        set_inputs(lambda k, x: s.set_input(m, x, k), v)
        fake.lib.fake_hal_set_auto_progress(0)             # launched, and nothing ends
        launched = len(fake.log())
        t = s.new_task(m)
        if v == 3.0:
            s.run()
        wait_for(lambda: len(fake.log()) == launched + 2)
        early = s.get_output(m, N)
        assert not np.array_equal(early, np.full(N, 2 * v * v))
        fake.lib.fake_hal_set_auto_progress(1)
        s.wait_task(t)
        before = fake.pass_counts()["fetches"]
        for _ in range(3):
            np.testing.assert_array_equal(s.get_output(m, N), np.full(N, 2 * v * v, np.float32))
        assert fake.pass_counts()["fetches"] == before + 1     # and of a run that has ended one copy is enough
    s.shutdown()
    s.close()


@pytest.mark.parametrize("kind,pre", [(B.BASE, False), (B.HYBRID, True)])
def test_a_fetch_in_the_middle_of_a_pass_and_an_input_behind_its_last_launch(fake, mocked, kind, pre):
    name, d = mocked
    exe = B.Executor.from_dir(d, name, kind)
    run = exe.execute_preemptable if pre else exe.execute
    c, seen = 3, []                                        # c: index of the storage of that name
    for _ in range(3):                                     # c joins what a pass mirrors
        set_inputs(exe.set_input_checked, 3.0)
        run()
        np.testing.assert_array_equal(exe.get_data(c, N), np.full(N, 3, np.float32))

    def hook(where):
        if where == 0:
            seen.append(exe.get_output())
        else:
            exe.set_input_checked("c", np.full(N, 7, np.float32))

    fake.set_pass_hook(hook)
    set_inputs(exe.set_input_checked, 5.0)
    run()
    np.testing.assert_array_equal(seen, np.full((1, N), 18, np.float32))
    for _ in range(2):
        np.testing.assert_array_equal(exe.get_output(), np.full(N, 50, np.float32))
        np.testing.assert_array_equal(exe.get_data(c, N), np.full(N, 7, np.float32))
    exe.close()


@pytest.mark.parametrize("host_writes", [True, False])
def test_packets_run_behind_whatever_was_stored_past_the_caches(fake, tmp_path, host_writes):
    """Inputs, parameters that are loaded again and a pass's own argument blocks are stored by the host or the runtime's
    copies: the first packets behind them drop the caches, those behind a pass of the same model do not."""
    g = nets.resnet(18, image=(3, 32, 32), classes=16, name="tiny18")
    d = write_model(g, tmp_path)
    scores = g.kernels[-1]["args"][0]
    fake.set_passes(host_writes)
    exe = B.Executor.from_dir(d, g.name, B.BASE)
    assert not exe.get_output(16).any()                    # the arena's zeros
    for step in range(3):                                  # the scores join what the pass mirrors
        exe.set_input_checked("data", nets.image_input("t", (3, 32, 32), step))
        exe.execute()
        exe.get_output(), exe.get_data(scores, 16)
    exe.execute()
    exe.load_param(os.path.join(d, g.name + ".param"))
    exe.execute()
    exe.load_param(os.path.join(d, g.name + ".param"))
    exe.get_data(0, 3 * 32 * 32)
    exe.execute()
    assert fake.pass_counts()["stale"] == 0
    exe.close()


@pytest.mark.parametrize("kind", [B.BASE, B.TRANS, B.HYBRID])
def test_runs_record_and_allocate_nothing(fake, mocked, kind):
    """Passes are recorded at load; a storage that joins what they mirror is added by the fetch that finds it missing."""
    name, d = mocked
    exe = B.Executor.from_dir(d, name, kind)
    runs = [exe.execute] + ([exe.execute_preemptable] if kind == B.HYBRID else [])
    assert fake.pass_counts()["creates"] == len(runs)
    changing = ("creates", "mallocs", "frees", "mirrors")

    def run(run_one):
        before = fake.pass_counts()
        run_one()
        after = fake.pass_counts()
        assert after["runs"] == before["runs"] + 1 and all(after[k] == before[k] for k in changing)

    for step in range(12):
        v = 2.0 + step
        set_inputs(exe.set_input_checked, v)
        if step == 5:                                      # not in the middle of a run
            fake.set_pass_hook(lambda where: exe.get_data(2, N))
        run(runs[step % len(runs)])
        fake.set_pass_hook(lambda where: None)
        for idx, want in ((4, 2 * v * v), (3, v), (2, 2 * v))[:1 + step // 3]:
            np.testing.assert_array_equal(exe.get_data(idx, N), np.full(N, want, np.float32))
    end = fake.pass_counts()
    assert end["mirrors"] == 2 * len(runs) and end["stale"] == 0
    set_inputs(exe.set_input_checked, 1.0)
    run(runs[0])
    for idx, want in ((4, 2), (3, 1), (2, 2)):             # all from the mirror
        np.testing.assert_array_equal(exe.get_data(idx, N), np.full(N, want, np.float32))
    assert fake.pass_counts()["fetches"] == end["fetches"]
    exe.close()


def test_a_scheduled_real_time_request_records_and_allocates_nothing(fake, mocked):
    name, d = mocked
    s = B.Scheduler(B.MODE_REEF)
    m = s.load_model(d, name)
    s.bind_model_queue(s.create_queue(B.QUEUE_RT), m)
    s.run()
    set_inputs(lambda k, x: s.set_input(m, x, k), 3.0)
    before = fake.pass_counts()
    assert before["creates"] == 1
    s.wait_task(s.new_task(m))
    after = fake.pass_counts()
    assert after["runs"] == 1 and all(after[k] == before[k] for k in ("creates", "mallocs", "frees", "mirrors"))
    np.testing.assert_array_equal(s.get_output(m, N), np.full(N, 18, np.float32))
    s.shutdown()
    s.close()


@pytest.mark.parametrize("kind", [B.BASE, B.HYBRID])
def test_a_pass_that_cannot_be_recorded_at_load_is_reported_by_the_run(fake, mocked, kind):
    name, d = mocked
    fake.lib.fake_hal_set_pass_failures(3 if kind == B.HYBRID else 2)   # at load, and in the first run
    exe = B.Executor.from_dir(d, name, kind)
    set_inputs(exe.set_input_checked, 3.0)
    with pytest.raises(B.ReefError):
        exe.execute()
    exe.execute()
    np.testing.assert_array_equal(exe.get_output(), np.full(N, 18, np.float32))
    exe.close()


# columns of the second product, 768 deep: 0.84 and 1.27 MiB an XCD split, 1.31 and 1.69 MiB in 32 bits
@pytest.mark.parametrize("n,tile,fits", [(1536, "32x48d4", True), (2304, "32x48d4", False), (3584, "16x32k4", True), (4608, "16x32k4", False)])
def test_weights_that_the_launch_in_front_brings_in(fake, tmp_path, n, tile, fits):
    g = MB.GraphBuilder("prefetch")
    x = g.gemm(g.input("x", (16, 768)), g.param((768, 768), 0.03), 16, 768, 768, force_tile="16x32k4")
    g.mark_output(g.gemm(x, g.param((n, 768), 0.03), 16, n, 768, force_tile=tile))
    fake._run_desc = lambda *args: None                     # (only the launches matter)
    exe = B.Executor.from_dir(write_model(g, tmp_path), g.name, B.BASE)
    exe.set_input_checked("x", np.ones((16, 768), np.float32))
    exe.execute()
    workgroups = fake.events[-2][3] - g.kernels[0]["launch_params"][0]
    assert workgroups == 8 + (8 * 6 if fits else 0)        # one of each XCD's for small operands, six for its weights
    exe.close()
