"""The work whose time this library is judged by: what a program does with it through the public entry points.

A case names a topology with its activations, the weight format, the number of samples and which entry point is called:

  forward    DeviceNet.forward_device: a batch that is on the device already, the result stays there
  one        forward(): one host sample in, every layer's activations out in net->neurons
  batch      forward_batch(): host arrays in and out
  evaluate   evaluate_batch(): host samples and targets in, the loss and the predictions out
  train      train() on host arrays, the full batch or one sample after the other: weights, moments and gradients out
  steps      DeviceNet.train_step over the mini-batches of a program's own data loader, then the weights out
  files      save_spingalett() and load_spingalett(): a net into its file and back

Sizes are those of the benchmark's workloads, of the reference's two examples (the 784-512-1000-10 training benchmark
and the 2-8-1 exclusive-or) and generic ones between and around them.
"""
import ctypes
import math
import os
import tempfile
import types

import numpy as np
import torch

import spingalett_amd as S

FORMATS = {"fp32": S.PRECISION_FLOAT32, "fp16": S.PRECISION_FP16, "bf16": S.PRECISION_BFLOAT16,
           "int8": S.PRECISION_INT8, "int4": S.PRECISION_INT4, "int2": S.PRECISION_INT2}
BITS = {"fp32": 32, "fp16": 16, "bf16": 16, "int8": 8, "int4": 4, "int2": 2}
ACTS = {"sigmoid": S.ACT_SIGMOID, "relu": S.ACT_RELU, "tanh": S.ACT_TANH, "leaky": S.ACT_LEAKY_RELU,
        "foo52": S.ACT_FOO52, "softmax": S.ACT_SOFTMAX, "none": S.ACT_NONE}
OPTIMIZERS = {"sgd": S.OPTIMIZER_SGD, "momentum": S.OPTIMIZER_MOMENTUM, "rmsprop": S.OPTIMIZER_RMSPROP,
              "adam": S.OPTIMIZER_ADAM, "adamw": S.OPTIMIZER_ADAMW}
LOSSES = {"mse": S.LOSS_MSE, "ce": S.LOSS_CROSS_ENTROPY}

MNIST_LIKE = dict(topo="784-512-1000-10", acts="relu-relu-softmax")
DEEP8192 = dict(topo="8192-" * 9 + "1000", acts="leaky-foo52-" * 4 + "softmax")
INT2_NET = dict(topo="2048-8192-8192-8192-8192-1000", acts="sigmoid-relu-relu-tanh-softmax")


def listed():
    return [
        # an interactive program asks a small quantized classifier about one sample: latency and launches are all there is
        dict(name="one_int8", kind="one", format="int8", inputs="u01", batch=1, **MNIST_LIKE),
        # a service answers a single request with a wide net: every packed weight is read once for one sample
        dict(name="wide_int4_b1", kind="forward", topo="4096-16384-16384-4096", acts="relu-tanh-none", format="int4",
             inputs="n01", batch=1, split=False),
        # requests collected over a short time: more samples than the vector path takes, fewer than a tile of the matrix path
        dict(name="int2_b50", kind="forward", format="int2", inputs="u11", batch=50, split=False, **INT2_NET),
        # the ordinary batch of the small classifier: four short dependent layers
        dict(name="int8_b256", kind="forward", format="int8", inputs="u01", batch=256, split=False, **MNIST_LIKE),
        # bulk scoring with a deep wide net, the largest product: the matrix cores decide
        dict(name="bf16_b8192", kind="forward", format="bf16", inputs="n01", batch=8192, split=False, **DEEP8192),
        # FP32 weights with the setting that keeps FP32-grade results on the 16-bit matrix cores
        dict(name="fp32_split_b2000", kind="forward", topo="4096-4096-4096-4096-1000", acts="relu-tanh-relu-softmax",
             format="fp32", inputs="n01", batch=2000, split=True),
        # rows that are not whole 16-byte units, host arrays in and out, as a program without device memory has them
        dict(name="fp16_ragged_host", kind="batch", topo="1030-1531-777-33", acts="leaky-tanh-none", format="fp16",
             inputs="n01", batch=1333),
        # the loss and accuracy on a test set of 10,000 images
        dict(name="evaluate_fp32", kind="evaluate", format="fp32", inputs="u01", batch=10000, loss="ce", **MNIST_LIKE),
        # the reference's published benchmark: full batch of 20,000 samples, five epochs, Adam
        dict(name="train_full", kind="train", strategy="full", inputs="u01", batch=20000, epochs=5, optimizer="adam",
             loss="ce", rate=0.001, decay=0.0, **MNIST_LIKE),
        # the reference's first example: exclusive-or, full batch of four, AdamW (500 of its 10,000 epochs; tanh instead of
        # its piecewise linear FOO52, so that no rounding decides on which side of a bend a neuron is)
        dict(name="train_xor", kind="train", strategy="full", topo="2-8-1", acts="tanh-sigmoid", inputs="xor", batch=4,
             epochs=500, optimizer="adamw", loss="mse", rate=0.01, decay=0.0001),
        # mini-batches of 64 from a program's own loader
        dict(name="steps_b64", kind="steps", inputs="u01", batch=64, epochs=16, optimizer="adam", loss="ce", rate=0.001,
             decay=0.0, **MNIST_LIKE),
        # a trained net into a quantized file and back
        dict(name="files_int8", kind="files", format="int8", optimizer_block=False, **MNIST_LIKE),
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """Half of the widths as they fall, half whole multiples of 16."""
    w = _log_int(rng, lo, hi)
    return max(16, w // 16 * 16) if lo >= 16 and rng.random() < 0.5 else w


def _net(rng, depth, lo, hi, head, hidden=("sigmoid", "relu", "tanh", "leaky", "foo52")):
    topo = [_width(rng, lo, hi) for _ in range(rng.randint(*depth))] + [_log_int(rng, *head)]
    acts = [rng.choice(hidden) for _ in topo[2:]] + [rng.choice(["softmax", "softmax", "none", "sigmoid"])]
    return dict(topo="-".join(map(str, topo)), acts="-".join(acts))


# most multiply-adds (times two) and weights of a drawn case of each kind
LIMITS = {"forward": (4e12, 3.0e8), "one": (1e9, 2e7), "batch": (4e11, 2e7), "evaluate": (4e11, 8e6),
          "train": (4e11, 4e6), "steps": (4e11, 4e6), "files": (1e12, 8e6)}


def draw(rng):
    kind = rng.choice(["forward"] * 6 + ["one", "batch", "evaluate", "train", "tiny", "steps", "files"])
    inputs = rng.choice(["u01", "n01", "u11"])
    fmt = rng.choice(sorted(FORMATS))
    while True:
        if kind == "forward":
            batch = _log_int(rng, 1, 16384)
            c = dict(kind=kind, format=fmt, inputs=inputs, batch=batch, split=batch > 4 and rng.random() < 0.15,
                     **_net(rng, (2, 5), 64, 12288, (10, 4096)))
        elif kind == "one":
            c = dict(kind=kind, format=fmt, inputs=inputs, batch=1, **_net(rng, (2, 5), 16, 4096, (1, 1000)))
        elif kind == "batch":
            c = dict(kind=kind, format=fmt, inputs=inputs, batch=_log_int(rng, 1, 8192), **_net(rng, (2, 4), 64, 4096, (1, 1000)))
        elif kind == "evaluate":
            c = dict(kind=kind, format=fmt, inputs=inputs, batch=_log_int(rng, 100, 20000), loss=rng.choice(["ce", "mse"]),
                     **_net(rng, (2, 4), 64, 2048, (2, 100)))
        elif kind == "train":
            c = dict(kind=kind, strategy="full", inputs=inputs, batch=_log_int(rng, 256, 20000), epochs=rng.randint(2, 6),
                     optimizer=rng.choice(sorted(OPTIMIZERS)), loss=rng.choice(["ce", "mse"]), rate=0.001,
                     decay=rng.choice([0.0, 0.0001]), **_net(rng, (2, 4), 32, 2048, (2, 100)))
        elif kind == "tiny":
            # small problems: the full batch, or one update per sample
            strategy = rng.choice(["full", "sample"])
            c = dict(kind="train", strategy=strategy, inputs=inputs, batch=_log_int(rng, 4, 200),
                     epochs=rng.randint(2, 4) if strategy == "sample" else _log_int(rng, 20, 200),
                     optimizer=rng.choice(["sgd", "adam", "adamw"]), loss=rng.choice(["ce", "mse"]), rate=0.001,
                     decay=rng.choice([0.0, 0.0001]), **_net(rng, (2, 3), 2, 48, (1, 10), ("tanh", "sigmoid")))
        elif kind == "steps":
            c = dict(kind=kind, inputs=inputs, batch=_log_int(rng, 8, 512), epochs=16, optimizer=rng.choice(sorted(OPTIMIZERS)),
                     loss=rng.choice(["ce", "mse"]), rate=0.001, decay=rng.choice([0.0, 0.0001]),
                     **_net(rng, (2, 4), 32, 2048, (2, 100)))
        else:
            c = dict(kind=kind, format=fmt, optimizer_block=rng.random() < 0.25, **_net(rng, (2, 5), 16, 4096, (1, 1000)))
        if c.get("loss") == "ce" and c["acts"].endswith("none"):
            c["loss"] = "mse"                                     # a cross-entropy wants outputs between 0 and 1
        most_flops, most_weights = LIMITS[c["kind"]]
        if _macs(c) <= most_weights and work(c)["flops"] <= most_flops:
            return c


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------
def _topo(case):
    return [int(w) for w in case["topo"].split("-")]


def _acts(case):
    return [ACTS[a] for a in case["acts"].split("-")]


def _macs(case):
    t = _topo(case)
    return sum(a * b for a, b in zip(t, t[1:]))


def _params(case):
    return _macs(case) + sum(_topo(case)[1:])


def work(case):
    t, macs, params = _topo(case), _macs(case), _params(case)
    kind, n = case["kind"], case.get("batch", 0)
    if kind == "files":
        # FP32 arrays read, the file written, the file read, FP32 arrays written
        arrays = 3 if case["optimizer_block"] else 1
        return {"bytes": arrays * params * (8 + 2 * BITS[case["format"]] / 8), "flops": 0}
    if kind in ("train", "steps"):
        steps = case["epochs"] * (n if case.get("strategy") == "sample" else 1)
        rows = n * (case["epochs"] if kind == "steps" else 1)
        # forward, weight gradients, hidden deltas; the samples in, weights, gradients and two moments in and out
        per_sample = 2 * (2 * macs + sum(a * b for a, b in zip(t[1:], t[2:])))
        return {"bytes": 4 * rows * (t[0] + t[-1]) + 28 * params,
                "flops": per_sample * steps * (1 if case.get("strategy") == "sample" else n)}
    out = sum(t) if kind == "one" else n if kind == "evaluate" else n * t[-1]
    more_in = n * t[-1] if kind == "evaluate" else 0
    return {"bytes": params * BITS[case["format"]] / 8 + 4 * (n * t[0] + out + more_in), "flops": 2.0 * n * macs}


def tolerance(case):
    kind = case["kind"]
    if kind == "files":
        return "exact"
    if kind in ("train", "steps"):
        # sums of 32 bits, each step's error carried through the next ones; an update divided by the root of its own
        # second moment follows the sign of a gradient that is nearly zero, so single values may move by a few steps
        return {"rel": 1e-4, "max": 0.1}
    if kind == "one" or case["batch"] <= 4 or (case["format"] == "fp32" and not case.get("split")):
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-3}         # FP32 arithmetic
    if case.get("split"):
        return {"rel": 2e-5, "max": 1e-3}                          # 22 bits between the layers, sums of 32 bits
    # 11 bits between the layers; a softmax turns the error of a logit into a relative one of its output
    return {"rel": 5e-3, "max": 0.2, "differ": 1e-2}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _std(case, l):
    return math.sqrt((2.0 if case["acts"].split("-")[l] in ("relu", "leaky", "foo52") else 1.0) / _topo(case)[l])


def _samples(gen, kind, n, width):
    if kind == "n01":
        return torch.randn((n, width), generator=gen, device="cuda")
    u = torch.rand((n, width), generator=gen, device="cuda")
    return u if kind == "u01" else u * 2 - 1


def _targets(gen, case, n):
    """One class of the head per sample, or values between 0 and 1 where the head is a single output."""
    width = _topo(case)[-1]
    if width == 1:
        return torch.rand((n, 1), generator=gen, device="cuda")
    cls = torch.randint(width, (n,), generator=gen, device="cuda")
    return torch.nn.functional.one_hot(cls, width).to(torch.float32)


def _serialized(w, fmt):
    """An array as the library's writer leaves it in a file: (codes as bytes on the host, scale)."""
    if fmt == "fp32":
        return w.cpu().numpy().view(np.uint8), 0.0
    if fmt == "fp16":
        return w.to(torch.float16).view(torch.uint8).cpu().numpy(), 0.0
    if fmt == "bf16":
        return w.to(torch.bfloat16).view(torch.uint8).cpu().numpy(), 0.0
    top = float(w.abs().max())
    ratio = w / top
    if fmt == "int8":
        return torch.round(ratio * 127).to(torch.int8).view(torch.uint8).cpu().numpy(), top
    per = 2 if fmt == "int4" else 4
    q = torch.round(ratio * 7) if fmt == "int4" else (ratio > 0.5).float() - (ratio < -0.5).float()
    q = torch.nn.functional.pad(q.to(torch.int8), (0, -q.numel() % per)).view(torch.uint8).view(-1, per)
    codes = torch.zeros(q.shape[0], dtype=torch.uint8, device="cuda")
    for i in range(per):
        codes |= (q[:, i] & (15 if fmt == "int4" else 3)) << (i * (8 // per))
    return codes.cpu().numpy(), top


def _device_net(gen, case, fmt):
    topo = _topo(case)
    net = S.DeviceNet(topo, _acts(case), FORMATS[fmt])
    for l in range(len(topo) - 1):
        w = torch.randn(topo[l] * topo[l + 1], generator=gen, device="cuda") * _std(case, l)
        b = torch.randn(topo[l + 1], generator=gen, device="cuda") * 0.05
        for which, a in ((0, w), (1, b)):
            codes, top = _serialized(a, fmt)
            net.upload(l, which, codes, top)
    return net


class _HostNet:
    """A net of the public interface, freed with the state that holds it."""

    def __init__(self, gen, case):
        topo = _topo(case)
        self.net = S.new_spingalett(LOSSES[case.get("loss", "ce")])
        S.layer(self.net, topo[0])
        for l, act in enumerate(_acts(case)):
            S.layer(self.net, topo[l + 1], act, S.WEIGHT_INITIALIZATION_NONE)
        for l in range(len(topo) - 1):
            S.weights_view(self.net, l)[:] = (torch.randn((topo[l + 1], topo[l]), generator=gen, device="cuda") * _std(case, l)).cpu().numpy()
            if case["kind"] != "train":
                S.biases_view(self.net, l)[:] = (torch.randn(topo[l + 1], generator=gen, device="cuda") * 0.05).cpu().numpy()

    def quantize(self, fmt):
        """Through the library's file format, as a quantized net comes to a program."""
        path = _scratch_file()
        S.save_spingalett(self.net, path, FORMATS[fmt], do_not_save_optimizer=True)
        S.free_network(self.net)
        self.net = S.load_spingalett(path)
        os.remove(path)
        if self.net is None:
            raise RuntimeError("load_spingalett: %s" % (S.last_error(),))

    def __del__(self):
        S.free_network(self.net)


def _scratch_file():
    fd, path = tempfile.mkstemp(suffix=".nn")
    os.close(fd)
    return path


class _Checkpoint:
    """The file of a net and the net that was read back from it last."""

    def __init__(self):
        self.path, self.net = _scratch_file(), None

    def close(self):
        if self.net is not None:
            S.free_network(self.net)
            self.net = None

    def __del__(self):
        self.close()
        os.remove(self.path)


def _host_array(pointer, count, owner):
    """A net's host array; the owner of the net lives as long as the view does."""
    buf = (ctypes.c_float * int(count)).from_address(ctypes.addressof(pointer.contents))
    buf.owner = owner
    return np.frombuffer(buf, dtype=np.float32)


def prepare(case, seed):
    S.set_verbose(False)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, topo = case["kind"], _topo(case)
    s = types.SimpleNamespace(case=case)
    if kind == "forward":
        s.net = _device_net(gen, case, case["format"])
        s.x = _samples(gen, case["inputs"], case["batch"], topo[0])
        s.y = torch.empty((case["batch"], topo[-1]), device="cuda")
        s.d_x = types.SimpleNamespace(ptr=ctypes.c_void_p(s.x.data_ptr()))
        s.d_y = types.SimpleNamespace(ptr=ctypes.c_void_p(s.y.data_ptr()))
        s.flags = S.SPHIP_SPLIT_ACTIVATIONS if case["split"] else 0
        return s
    if kind == "steps":
        s.net = _device_net(gen, case, "fp32")
        s.net.train_begin()
        s.x = [_samples(gen, case["inputs"], case["batch"], topo[0]).cpu().numpy() for _ in range(case["epochs"])]
        s.t = [_targets(gen, case, case["batch"]).cpu().numpy() for _ in range(case["epochs"])]
        s.done = 0
        return s
    s.host = _HostNet(gen, case)
    if kind == "files":
        s.file = _Checkpoint()
        for name in ("opt_m_weights", "opt_v_weights"):
            if case["optimizer_block"]:
                count = s.host.net.contents.total_weights
                _host_array(getattr(s.host.net.contents, name), count, s.host)[:] = (torch.rand(int(count), generator=gen, device="cuda") * 1e-3).cpu().numpy()
        return s
    if case.get("format", "fp32") != "fp32":
        s.host.quantize(case["format"])
    if case["inputs"] == "xor":
        s.x = np.float32([[0, 0], [0, 1], [1, 0], [1, 1]])
        s.t = np.float32([[0], [1], [1], [0]])
        return s
    s.x = _samples(gen, case["inputs"], case["batch"], topo[0]).cpu().numpy()
    if kind in ("evaluate", "train"):
        s.t = _targets(gen, case, case["batch"]).cpu().numpy()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "forward":
        s.net.forward_device(s.d_x, case["batch"], s.d_y, s.flags)
        return s.y
    if kind == "one":
        S.forward(s.host.net, s.x[0])
        return _host_array(s.host.net.contents.neurons, s.host.net.contents.total_neurons, s.host)
    if kind == "batch":
        return S.forward_batch(s.host.net, s.x)
    if kind == "evaluate":
        loss, predictions, _ = S.evaluate_batch(s.host.net, s.x, s.t)   # (the hits follow from the predictions)
        return {"loss": loss, "predictions": predictions}
    if kind == "train":
        S.train(s.host.net, s.x, s.t, case["epochs"], S.STRATEGY_FULL_BATCH if case["strategy"] == "full" else S.STRATEGY_SAMPLE,
                OPTIMIZERS[case["optimizer"]], learning_rate=case["rate"], weight_decay=case["decay"])
        net = s.host.net.contents
        weights = {k: _host_array(getattr(net, k), net.total_weights, s.host) for k in ("weights", "grad_weights", "opt_m_weights", "opt_v_weights")}
        biases = {k: _host_array(getattr(net, k), net.total_biases, s.host) for k in ("biases", "grad_biases", "opt_m_biases", "opt_v_biases")}
        return {**weights, **biases}
    if kind == "steps":
        for x, t in zip(s.x, s.t):
            s.done += 1
            args = S.SphipTrainArgs(OPTIMIZERS[case["optimizer"]], LOSSES[case["loss"]], case["rate"], case["decay"], 0.9, 0.9,
                                    0.999, 1e-8, 0.0, 0.9 ** s.done, 0.999 ** s.done)
            s.net.train_step(x, t, args)
        return [s.net.train_get(which, l) for l in range(len(s.net.acts)) for which in (S.SPHIP_TRAIN_W, S.SPHIP_TRAIN_B)]
    # files
    S.save_spingalett(s.host.net, s.file.path, FORMATS[case["format"]], do_not_save_optimizer=not case["optimizer_block"])
    s.file.close()
    s.file.net = S.load_spingalett(s.file.path)
    net = s.file.net.contents
    out = [_host_array(net.weights, net.total_weights, s.file), _host_array(net.biases, net.total_biases, s.file)]
    if case["optimizer_block"]:
        out += [_host_array(net.opt_m_weights, net.total_weights, s.file), _host_array(net.opt_v_weights, net.total_weights, s.file)]
    return out
