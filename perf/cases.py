"""The work that this framework is timed on: single convolutions on device pointers, whole-model
requests through the executors, and a real-time request among best-effort ones through the
scheduler.

A case is a dict of plain values; its "path" says which of the three it is.

  conv   one fused convolution (B.ops_conv2d) on tensors that the caller holds in device memory.
  net    one request to a loaded model: input from host memory, execute, output to host memory.
         "kind" is the executor: "base" (a model that has the device to itself), "preemptible"
         (the kernels a best-effort model runs), "padded" (the dynamic-kernel-padding kernels).
  serve  one request to a real-time model and one to each best-effort client of a running
         scheduler: all submitted, all waited for, all outputs fetched.

The networks, their parameters and their inputs are the seeded synthetic ones of
reef_amd.modelgen; the seed of a state gives its input.  A loaded model is kept for all states of
its configuration, as a serving program keeps it for all requests.
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch

from reef_amd import binding as B
from reef_amd import profiler
from reef_amd.modelgen import nets

VOCAB = 8192


def listed():
    return [
        # -- one convolution: the call a serving loop with its own memory management makes per layer
        # a layer of a small head, a few microseconds of work: what one call costs
        dict(name="conv_1x1_small", path="conv", cin=64, h=14, w=14, cout=64, k=1, stride=1, pad=0, residual=0, noalloc=1),
        # a 5x5 branch layer on a ragged image
        dict(name="conv_5x5_branch", path="conv", cin=48, h=35, w=35, cout=64, k=5, stride=1, pad=2, residual=0, noalloc=0),
        # a down-sampling layer on an odd, wide image (detection backbones, strips of a larger picture)
        dict(name="conv_3x3_s2_ragged", path="conv", cin=96, h=57, w=75, cout=160, k=3, stride=2, pad=1, residual=0, noalloc=0),
        # a layer that fills the device
        dict(name="conv_3x3_large", path="conv", cin=256, h=112, w=112, cout=256, k=3, stride=1, pad=1, residual=1, noalloc=1),
        # -- whole models at the sizes the serving configurations run them
        # the smallest network: 35 launches of a few microseconds
        dict(name="mobilenetv2_224", path="net", net="mobilenetv2", size=224, depth=0, kind="base"),
        # the real-time model of the headline configuration
        dict(name="resnet152_224", path="net", net="resnet", size=224, depth=152, kind="base"),
        # a picture of four times the pixels: where the launches carry real work
        dict(name="resnet50_448", path="net", net="resnet", size=448, depth=50, kind="base"),
        dict(name="inceptionv3_299", path="net", net="inceptionv3", size=299, depth=0, kind="base"),
        # the best-effort model of the headline configuration, on the kernels it runs there
        dict(name="densenet201_224_preemptible", path="net", net="densenet201", size=224, depth=0, kind="preemptible"),
        # the encoder's layers at the sequence length of the serving configuration, and at a long one
        dict(name="bert_128_preemptible", path="net", net="bert", size=128, depth=6, kind="preemptible"),
        dict(name="bert_384", path="net", net="bert", size=384, depth=4, kind="base"),
        # -- the headline configuration: one real-time request among four best-effort clients
        dict(name="serve_resnet152_4x_densenet201", path="serve", net="resnet", size=224, depth=152, be="densenet201", be_size=224,
             clients=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("conv", "conv", "net", "net", "net", "serve"))
    if kind == "conv":
        while True:
            k = rng.choice((1, 1, 3, 3, 3, 5, 7))
            c = dict(path="conv", cin=_log_int(rng, 3, 768), h=_log_int(rng, 7, 160), w=_log_int(rng, 7, 160),
                     cout=_log_int(rng, 8, 768), k=k, stride=rng.choice((1, 1, 2)), pad=k // 2, residual=rng.choice((0, 1)),
                     noalloc=rng.choice((0, 1)))
            if k == 1 and rng.random() < 0.75:
                c["cin"] = max(8, c["cin"] // 8 * 8)
            f = work(c)["flops"]
            if 1e6 < f < 1.2e10:
                return c
    if kind == "serve":
        net, depth = rng.choice((("mobilenetv2", 0), ("resnet", 18), ("resnet", 50)))
        return dict(path="serve", net=net, size=rng.randrange(160, 289), depth=depth, be=rng.choice(("mobilenetv2", "densenet201")),
                    be_size=rng.randrange(160, 257), clients=rng.randrange(1, 5))
    net = rng.choice(("mobilenetv2", "resnet", "resnet", "densenet201", "inceptionv3", "bert", "bert"))
    kind = rng.choice(("base", "base", "preemptible", "padded"))
    if net == "bert":
        # up to 128 tokens of any number, longer sequences in fours
        seq = _log_int(rng, 8, 512)
        return dict(path="net", net=net, size=seq if seq <= 128 else seq // 4 * 4, depth=rng.randrange(2, 5), kind=kind)
    depth = rng.choice((18, 50, 50)) if net == "resnet" else 0
    lo, hi = (139, 340) if net == "inceptionv3" else (64, 400)
    return dict(path="net", net=net, size=_log_int(rng, lo, hi), depth=depth, kind=kind)


# ---- models ------------------------------------------------------------------------------------
def _graph(net, size, depth, best_effort):
    image = (3, size, size)
    if net == "mobilenetv2":
        return nets.mobilenet_v2(image=image)
    if net == "resnet":
        return nets.resnet(depth, image=image)
    if net == "densenet201":
        return nets.densenet(image=image, under_load=best_effort)
    if net == "inceptionv3":
        return nets.inception_v3(image=image)
    return nets.bert(layers=depth, seq=size, vocab=VOCAB, under_load=best_effort)


_work = {}      # configuration -> (bytes, flops) of one pass
_loaded = {}    # configuration -> what a program keeps: an executor, or a running scheduler


def _totals(net, size, depth, best_effort, g=None):
    """Bytes (every parameter, the input and the output once) and multiply-add FLOPs of one inference."""
    key = (net, size, depth, best_effort)
    if key not in _work:
        g = g or _graph(*key)
        own = sum(a.size for k, a in g.params if not k.endswith("k"))       # without derived copies
        if net == "bert":
            own -= (VOCAB - size) * 768                                     # rows of the embedding that are not read
            io = size * 768 + 2 * size
        else:
            io = 3 * size * size + 2 * 1000
        _work[key] = (4 * (own + io), g.flops)
    return _work[key]


def _write(net, size, depth, best_effort, root):
    """Model directory, model name, and the storage that holds the scores in front of an image network's
    softmax (a random network's probabilities are nearly all 0 and 1)."""
    g = _graph(net, size, depth, best_effort)
    _totals(net, size, depth, best_effort, g)
    d = os.path.dirname(g.write(os.path.join(root, "%s_%d_%d" % (g.name, size, best_effort))))
    return d, g.name, None if net == "bert" else g.kernels[-1]["args"][0]


def _input(net, size, seed):
    if net == "bert":
        return "input0", nets.token_input("bert_base", size, VOCAB, seed)
    return "data", nets.image_input(net, (3, size, size), seed)


def _executor(c):
    key = (c["net"], c["size"], c["depth"], c["kind"])
    if key not in _loaded:
        for k in [k for k in _loaded if k[0] == "serve"]:       # no scheduler runs beside a model that is alone
            s = _loaded.pop(k)[0]
            s.shutdown()
            s.close()
        with tempfile.TemporaryDirectory() as root:
            d, name, scores = _write(c["net"], c["size"], c["depth"], c["kind"] == "preemptible", root)
            kind = {"base": B.BASE, "preemptible": B.HYBRID, "padded": B.TRANS}[c["kind"]]
            _loaded[key] = (B.Executor.from_dir(d, name, kind), scores)
    return _loaded[key]


def _scheduler(c):
    key = ("serve", c["net"], c["size"], c["depth"], c["be"], c["be_size"], c["clients"])
    if key not in _loaded:
        s = B.Scheduler(B.MODE_REEF)
        with tempfile.TemporaryDirectory() as root:
            models = [_write(c["net"], c["size"], c["depth"], False, root), _write(c["be"], c["be_size"], 0, True, root)]
            for m in models:
                profiler.write_profile(m[0], m[1], iters=5, warmup=1)
            rt, rt_scores = s.load_model(*models[0][:2]), models[0][2]
            bes = [s.load_model(*models[1][:2]) for _ in range(c["clients"])]
        s.bind_model_queue(s.create_queue(B.QUEUE_RT), rt)
        for m in bes:
            s.bind_model_queue(s.create_queue(B.QUEUE_BE), m)
        s.run()
        _loaded[key] = (s, [(rt, rt_scores)] + [(m, models[1][2]) for m in bes])
    return _loaded[key]


class _Dev:
    """A tensor of the caller's as the device pointer that the convolution takes."""

    def __init__(self, t):
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


def _conv_out(c):
    return ((c["h"] + 2 * c["pad"] - c["k"]) // c["stride"] + 1, (c["w"] + 2 * c["pad"] - c["k"]) // c["stride"] + 1)


def prepare(case, seed):
    if case["path"] == "conv":
        c, gen = case, torch.Generator(device="cuda").manual_seed(int(seed))

        def normal(*shape):
            return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)

        ho, wo = _conv_out(c)
        B.ops_init()
        x = _Dev(normal(c["cin"], c["h"], c["w"]).relu_())              # what a layer in front leaves
        w = _Dev(normal(c["cout"], c["cin"], c["k"], c["k"]) * math.sqrt(2.0 / (c["cin"] * c["k"] ** 2)))
        bias = _Dev(normal(c["cout"]) * 0.1)
        res = _Dev(normal(c["cout"], ho, wo)) if c["residual"] else None
        out = _Dev(torch.empty(c["cout"], ho, wo, device="cuda"))
        desc = B.Conv2dDesc(c["cin"], c["h"], c["w"], c["cout"], c["k"], c["k"], c["stride"], c["stride"], c["pad"], c["pad"], 1)
        torch.cuda.synchronize()
        return ("conv", desc, x, w, bias, res, out, bool(c["noalloc"]))
    if case["path"] == "net":
        key, x = _input(case["net"], case["size"], seed)
        return ("net",) + _executor(case) + (key, x, case["kind"] == "preemptible")
    s, models = _scheduler(case)
    inputs = [_input(case["net"], case["size"], seed)]
    inputs += [_input(case["be"], case["be_size"], seed + 7919 * i) for i in range(1, len(models))]
    return ("serve", s, [m + i for m, i in zip(models, inputs)])


def run(state):
    if state[0] == "conv":
        _, desc, x, w, bias, res, out, noalloc = state
        if B.ops_conv2d(desc, x, w, bias, res, out, noalloc=noalloc):
            raise RuntimeError(B.last_error())
        return out.t
    if state[0] == "net":
        _, exe, scores, key, x, preemptible = state
        exe.set_input_checked(key, x)
        if preemptible:
            exe.execute_preemptable()
        else:
            exe.execute()
        return [exe.get_output()] + ([exe.get_data(scores, 1000)] if scores is not None else [])
    _, s, inputs = state
    for m, _, key, x in inputs:
        if s.set_input(m, x, key):
            raise RuntimeError(B.last_error())
    # the clients' requests are under way when the real-time one arrives
    tasks = [s.new_task(m[0]) for m in inputs[1:]] + [s.new_task(inputs[0][0])]
    for t in reversed(tasks):
        s.wait_task(t)
    return [[s.get_output(m, 1000), s.get_data(m, scores, 1000)] for m, scores, _, _ in inputs]


def work(case):
    if case["path"] == "conv":
        c = case
        ho, wo = _conv_out(c)
        k = c["cin"] * c["k"] ** 2
        n = c["cin"] * c["h"] * c["w"] + c["cout"] * (k + 1) + (2 if c["residual"] else 1) * c["cout"] * ho * wo
        return {"bytes": 4 * n, "flops": 2 * c["cout"] * ho * wo * k}
    b, f = _totals(case["net"], case["size"], case["depth"], case.get("kind") == "preemptible")
    if case["path"] == "serve":
        b2, f2 = _totals(case["be"], case["be_size"], 0, True)
        b, f = b + case["clients"] * b2, f + case["clients"] * f2
    return {"bytes": b, "flops": f}


def tolerance(case):
    # fp32 throughout: sums of up to a few thousand products, in another order; through up to 154
    # layers for a network
    return {"rel": 1e-5 if case["path"] == "conv" else 1e-4}
