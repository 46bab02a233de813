"""Forward parity of the HIP path against the CPU oracle, through the C-ABI.

Tolerances (relative max-abs = max|gpu - ref| / max|ref|):
  FP32 weights (any n), and every format at n <= 4 (vector path) ... 1e-4
  16-bit matrix-core paths (n >= 5, 16-bit or integer weights) ...... 2e-2
The vector kernels accept up to 64 samples (SPHIP_FORCE_GEMV) and are held to
1e-4 there too.

Argmax agreement with the FP32 reference on the matrix-core path: at least
99.9 % of the samples (`raw`), asserted at 4096 samples and more in
test_argmax_agreement_with_the_fp32_reference; the cases that do not reach it
on random nets are marked xfail there with the measured figure, never given a
lower bar.  Everywhere, `decided` (rows whose reference top-2 gap exceeds
twice the largest deviation of the run: a flip there cannot be rounding) must
agree 100 %.
"""
import ctypes as C
import os
import tempfile
import threading
import time

import numpy as np
import pytest

from helpers import ALL_ACTS, FORMATS, argmax_agreement, make_oracle_net, quantized_pair, rel_max_abs

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden")
E = np.load(os.path.join(GOLD, "expected.npz"))
F32 = np.float32
TOL_VEC, TOL_MFMA = 1e-4, 2e-2


def tol_for(fmt, n):
    return TOL_VEC if fmt == "f32" or n <= 4 else TOL_MFMA


def sphip_forward(S, net, X, flags):
    """sphip_forward on the net's device handle (to pick the path regardless of n)."""
    h = S.lib().spingalett_hip_handle(net)
    assert h, S.last_error()
    nc = net.contents
    X = np.ascontiguousarray(X, dtype=F32)
    out = np.empty((X.shape[0], nc.topology[nc.layers - 1]), dtype=F32)
    rc = S.lib().sphip_forward(h, X.ctypes.data, X.shape[0], out.ctypes.data, flags)
    assert rc == 0, S.lib().sphip_last_error_string()
    return out


@pytest.mark.parametrize("fmt", FORMATS)
def test_golden_nets(S, fmt):
    net = S.load_spingalett(os.path.join(GOLD, f"tiny_{fmt}.nn"))
    X, want = E["tiny_X"], E[f"tiny_{fmt}_Y"]
    for i in range(X.shape[0]):                                   # public forward(), one sample
        y = S.forward(net, X[i])
        assert y is not None, S.last_error()
        assert rel_max_abs(y, want[i]) <= TOL_VEC
    assert rel_max_abs(S.forward_batch(net, X), want) <= tol_for(fmt, X.shape[0])   # batched entry
    assert rel_max_abs(S.forward_batch(net, X[:4]), want[:4]) <= TOL_VEC
    assert rel_max_abs(sphip_forward(S, net, X, S.SPHIP_FORCE_GEMV), want) <= TOL_VEC   # vector kernels
    got = sphip_forward(S, net, X, S.SPHIP_FORCE_GEMM)            # matrix-core path on the same inputs
    assert rel_max_abs(got, want) <= (TOL_VEC if fmt == "f32" else TOL_MFMA)
    S.free_network(net)


@pytest.mark.parametrize("fmt", ["bf16", "i4"])
def test_golden_softmax_net(S, fmt):
    net = S.load_spingalett(os.path.join(GOLD, f"soft_{fmt}.nn"))
    X, want = E["soft_X"], E[f"soft_{fmt}_Y"]
    assert rel_max_abs(S.forward_batch(net, X), want) <= tol_for(fmt, X.shape[0])
    assert rel_max_abs(sphip_forward(S, net, X, S.SPHIP_FORCE_GEMV), want) <= TOL_VEC
    got = sphip_forward(S, net, X, S.SPHIP_FORCE_GEMM)
    assert rel_max_abs(got, want) <= TOL_MFMA
    assert np.allclose(got.sum(axis=1), 1.0, atol=1e-5)
    S.free_network(net)


def test_forward_leaves_every_layer_in_neurons(S, O):
    """forward() mirrors all activations into net->neurons and returns a pointer
    into it (Network.c:214-250)."""
    with open(os.path.join(GOLD, "tiny_i8.nn"), "rb") as f:
        ref = O.Net.parse(f.read())
    net = S.load_spingalett(os.path.join(GOLD, "tiny_i8.nn"))
    x = E["tiny_X"][2]
    y = S.forward(net, x)
    nc = net.contents
    neurons = S.neurons_view(net)
    assert y.ctypes.data == C.addressof(nc.neurons.contents) + 4 * nc.neuron_offsets[3]
    assert np.array_equal(neurons[:37], x)
    # layer by layer against the oracle
    a = x.astype(np.float64)
    off = 37
    for l, act in enumerate(ref.act):
        pre = ref.W(l).astype(np.float64) @ a + ref.b(l)
        a = O.activate(pre.astype(F32), act).astype(np.float64)
        w = ref.topology[l + 1]
        assert rel_max_abs(neurons[off:off + w], a) <= TOL_VEC
        off += w
    S.free_network(net)


@pytest.mark.parametrize("fmt,acts", [("i4", ["foo52", "tanh", "softmax"]), ("bf16", ["leaky_relu", "sigmoid", "none"]),
                                      ("f32", ["relu", "tanh", "softmax"]), ("i2", ["sigmoid", "relu", "none"])])
def test_repeated_forward_calls_between_other_work_and_reuploads(S, O, fmt, acts):
    """forward() keeps device buffers, pinned staging and per-layer slots between calls: every one of a series of calls
    is checked against the oracle, with batched launches on the same stream and a change of the net's arrays in between."""
    topo = [96, 160, 64, 10]
    src = make_oracle_net(O, topo, acts, seed=21)
    _, ref, net = quantized_pair(O, S, src, fmt)
    rng = np.random.default_rng(8)
    X = rng.standard_normal((12, topo[0])).astype(F32)
    want = ref.forward_batch(X)
    for i in range(8):
        y = S.forward(net, X[i])
        assert y is not None, S.last_error()
        assert rel_max_abs(y, want[i]) <= TOL_VEC, (fmt, i)
        assert np.array_equal(S.neurons_view(net)[:topo[0]], X[i])
        if i in (3, 5):                                   # launches of another shape in between
            yb = S.forward_batch(net, X)
            assert rel_max_abs(yb, want) <= tol_for(fmt, 12)
    # new weights (FP32 host arrays, packed arrays dropped): the next call must use the re-uploaded arrays
    for l in range(3):
        S.weights_view(net, l)[:] = -S.weights_view(net, l)
        ref.W(l)[:] = -ref.W(l)
    S.lib().spingalett_hip_invalidate(net)
    want2 = ref.forward_batch(X)
    for i in range(5):
        y = S.forward(net, X[i])
        assert rel_max_abs(y, want2[i]) <= TOL_VEC, (fmt, "after invalidate", i)
    S.free_network(net)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("act", ALL_ACTS)
def test_every_activation_every_format(S, O, fmt, act):
    # hidden layer carries the activation under test (softmax included), aligned and odd widths
    for topo in ([64, 96, 32], [45, 77, 13]):
        src = make_oracle_net(O, topo, [act, "none"], seed=11)
        _, ref, net = quantized_pair(O, S, src, fmt)
        rng = np.random.default_rng(12)
        X = (rng.standard_normal((9, topo[0])) * 1.5).astype(F32)
        want = ref.forward_batch_f64(X)
        assert rel_max_abs(S.forward_batch(net, X), want) <= tol_for(fmt, 9), (topo, "default")
        assert rel_max_abs(S.forward_batch(net, X[:3]), want[:3]) <= TOL_VEC, (topo, "n=3")
        assert rel_max_abs(sphip_forward(S, net, X, S.SPHIP_FORCE_GEMV), want) <= TOL_VEC, (topo, "gemv")
        got = sphip_forward(S, net, X, S.SPHIP_FORCE_GEMM)
        assert rel_max_abs(got, want) <= (TOL_VEC if fmt == "f32" else TOL_MFMA), (topo, "gemm")
        S.free_network(net)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 7, 8, 9, 33, 64])
def test_vector_path_batch_sizes(S, O, n):
    src = make_oracle_net(O, [256, 512, 128, 10], ["relu", "tanh", "softmax"], seed=2)
    _, ref, net = quantized_pair(O, S, src, "i4")
    X = np.random.default_rng(n).standard_normal((n, 256)).astype(F32)
    want = ref.forward_batch_f64(X)
    assert rel_max_abs(S.forward_batch(net, X), want) <= tol_for("i4", n)
    got = sphip_forward(S, net, X, S.SPHIP_FORCE_GEMV)
    assert rel_max_abs(got, want) <= TOL_VEC
    # every row equals the single-sample forward of that row
    y0 = S.forward(net, X[n // 2]).copy()
    assert rel_max_abs(got[n // 2], y0) <= 2e-6
    S.free_network(net)


@pytest.mark.parametrize("fmt", ["f16", "bf16", "i8", "i4", "i2"])
def test_crossover_agreement(S, O, fmt):
    """n = 4 runs the vector path, n = 5 and up the matrix-core paths: same net, same rows."""
    src = make_oracle_net(O, [128, 256, 192, 16], ["leaky_relu", "foo52", "softmax"], seed=4)
    _, ref, net = quantized_pair(O, S, src, fmt)
    X = np.random.default_rng(5).standard_normal((65, 128)).astype(F32)
    lo = S.forward_batch(net, X[:4])
    mid = S.forward_batch(net, X[:5])
    hi = S.forward_batch(net, X)
    want = ref.forward_batch_f64(X)
    assert rel_max_abs(lo, want[:4]) <= TOL_VEC
    assert rel_max_abs(mid, want[:5]) <= TOL_MFMA
    assert rel_max_abs(hi, want) <= TOL_MFMA
    assert rel_max_abs(hi[:4], lo) <= TOL_MFMA
    S.free_network(net)


@pytest.mark.parametrize("n", [1, 256, 4096])
def test_config2_int8(S, O, n):
    """784->512->1000->10, INT8 through the serializer, inputs U[0,1)."""
    src = make_oracle_net(O, [784, 512, 1000, 10], ["relu", "relu", "softmax"], seed=42, bias_std=0.05)
    _, ref, net = quantized_pair(O, S, src, "i8")
    X = np.random.default_rng(7).random((n, 784), dtype=F32)
    want = ref.forward_batch(X)
    got = S.forward_batch(net, X)
    if n <= 4:
        assert rel_max_abs(got, want) <= TOL_VEC
    else:
        assert rel_max_abs(got, want) <= TOL_MFMA
        raw, decided = argmax_agreement(got, want)
        # 256 samples cannot resolve 99.9 % (one flip is 0.4 %): two flips allowed there
        assert decided == 1.0 and raw >= (0.999 if n >= 4096 else 0.992), (raw, decided)
    assert np.allclose(got.sum(axis=1), 1.0, atol=1e-4)
    S.free_network(net)


@pytest.mark.parametrize("fmt,topo,acts,n", [
    # classifier heads of at most 16 outputs: one streaming launch with the K split inside the workgroup; a softmax
    # is normalised in that kernel's epilogue when K is short enough to need no split across workgroups
    ("i8", [320, 10], ["softmax"], 5), ("i8", [1000, 10], ["softmax"], 33), ("i4", [1000, 16], ["softmax"], 300),
    ("bf16", [1000, 9], ["softmax"], 4096), ("f16", [72, 3], ["softmax"], 100), ("i2", [2048, 13], ["softmax"], 64),
    ("i8", [4096, 12], ["softmax"], 40),                      # more than 32 chunks: K split, reduce, softmax kernel
    ("i4", [512, 16], ["tanh"], 200), ("bf16", [256, 11], ["none"], 31),                  # heads without softmax
    ("i8", [256, 12, 64], ["softmax", "relu"], 128), ("bf16", [256, 8, 32], ["softmax", "none"], 77),  # softmax inside the net
    ("f16", [1000, 17], ["softmax"], 300),                    # 17 outputs: the wide thin kernel, separate softmax
])
def test_classifier_heads(S, O, fmt, topo, acts, n):
    src = make_oracle_net(O, topo, acts, seed=len(topo) * 100 + topo[-1], bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    X = np.random.default_rng(n).standard_normal((n, topo[0])).astype(F32)
    want = ref.forward_batch_f64(X)
    got = S.forward_batch(net, X)
    assert rel_max_abs(got, want) <= TOL_MFMA
    if acts[-1] == "softmax":
        assert np.allclose(got.sum(axis=1), 1.0, atol=1e-4)
    S.free_network(net)


def test_config1_fp32_batch256(S, O):
    """FP32 weights, batch 256: FP32 arithmetic end to end, 1e-4."""
    src = make_oracle_net(O, [784, 512, 1000, 10], ["relu", "relu", "softmax"], seed=42, bias_std=0.05)
    net = S.new_spingalett(S.LOSS_CROSS_ENTROPY)
    S.layer(net, 784)
    S.layer(net, 512, S.ACT_RELU, S.WEIGHT_INITIALIZATION_NONE)
    S.layer(net, 1000, S.ACT_RELU, S.WEIGHT_INITIALIZATION_NONE)
    S.layer(net, 10, S.ACT_SOFTMAX, S.WEIGHT_INITIALIZATION_NONE)
    for l in range(3):                                   # weights written straight into the public arrays
        S.weights_view(net, l)[:] = src.W(l)
        S.biases_view(net, l)[:] = src.b(l)
    X = np.random.default_rng(8).random((256, 784), dtype=F32)
    want = src.forward_batch(X)
    got = S.forward_batch(net, X)
    assert rel_max_abs(got, want) <= TOL_VEC
    assert np.array_equal(got.argmax(1), want.argmax(1))
    assert rel_max_abs(S.forward_batch(net, X[:3]), want[:3]) <= TOL_VEC
    S.free_network(net)


@pytest.mark.parametrize("topo,n", [([200, 3], 100), ([1000, 64], 300), ([520, 65], 257), ([96, 10, 40], 1000),
                                    ([64, 10], 4096)])
def test_fp32_softmax_heads(S, O, topo, n):
    """FP32 weights beyond 64 samples: a softmax layer of at most 64 outputs whose K is split is normalised by the
    reduction kernel (one thread per sample), wider ones and unsplit ones by the row kernel; 1e-4 either way."""
    acts = ["softmax"] + ["tanh"] * (len(topo) - 2)
    src = make_oracle_net(O, topo, acts, seed=topo[0] + n, bias_std=0.2)
    net = S.new_spingalett(S.LOSS_CROSS_ENTROPY)
    S.layer(net, topo[0])
    for l, width in enumerate(topo[1:]):
        S.layer(net, width, S.ACT_SOFTMAX if l == 0 else S.ACT_TANH, S.WEIGHT_INITIALIZATION_NONE)
        S.weights_view(net, l)[:] = src.W(l)
        S.biases_view(net, l)[:] = src.b(l)
    X = np.random.default_rng(n).standard_normal((n, topo[0])).astype(F32)
    want = src.forward_batch(X)
    got = S.forward_batch(net, X)
    assert rel_max_abs(got, want) <= TOL_VEC
    S.free_network(net)


@pytest.mark.parametrize("fmt,topo,acts,n", [
    ("i4", [1024, 2048, 2048, 512], ["relu", "tanh", "none"], 8),            # config 3 scaled down
    ("i4", [1024, 2048, 2048, 512], ["relu", "tanh", "none"], 64),
    ("bf16", [1024, 1024, 1024, 1024, 1000], ["leaky_relu", "foo52", "leaky_relu", "softmax"], 1024),  # config 4 scaled
    ("i2", [512, 1024, 1024, 1000], ["sigmoid", "relu", "softmax"], 1),       # config 5 scaled
    ("i2", [512, 1024, 1024, 1000], ["sigmoid", "relu", "softmax"], 2048),
    ("f16", [512, 768, 300], ["tanh", "none"], 300),
])
def test_scaled_configs(S, O, fmt, topo, acts, n):
    init = "xavier" if fmt == "i4" else "he"
    src = make_oracle_net(O, topo, acts, seed=21, init=init)
    _, ref, net = quantized_pair(O, S, src, fmt)
    rng = np.random.default_rng(22)
    X = (rng.random((n, topo[0]), dtype=F32) * 2 - 1) if fmt == "i2" else rng.standard_normal((n, topo[0])).astype(F32)
    fn, _, setter = O.find_sgemm()
    _, want = ref.time_forward_batch(X, 1, fn, 8)        # threaded BLAS leg of the oracle (same call sequence)
    got = S.forward_batch(net, X)
    assert rel_max_abs(got, want) <= tol_for(fmt, n)
    if acts[-1] == "softmax" and n > 64:
        _, decided = argmax_agreement(got, want)
        assert decided == 1.0
    S.free_network(net)


_C4S = ([1024] * 9, ["leaky_relu", "foo52"] * 4)             # configuration 4 scaled to 1024-wide layers
_C5S = ([512, 1024, 1024, 1024, 1024], ["sigmoid", "relu", "relu", "tanh"])
_C2S = ([784, 512, 1000], ["relu", "relu"])                  # configuration 2

# (format, hidden topology, hidden activations, classes, inputs).  "+bf16act": BF16 weights with
# spingalett_set_bf16_activations(BF16), i.e. BF16 activations on the BF16 matrix cores.
_ARGMAX_CASES = [
    ("i8", *_C2S, 10, "u01"), ("f16", *_C2S, 10, "u01"), ("i4", *_C2S, 10, "u01"), ("i2", *_C2S, 10, "u01"),
    ("bf16", *_C2S, 10, "u01"),
    ("f16", *_C4S, 10, "n01"), ("i8", *_C4S, 10, "n01"), ("bf16", *_C4S, 10, "n01"),
    ("bf16", *_C4S, 1000, "n01"), ("f16", *_C4S, 1000, "n01"), ("i8", *_C4S, 1000, "n01"),   # configuration 4's own head
    ("i2", *_C5S, 10, "u11"), ("i4", *_C5S, 10, "u11"), ("bf16", *_C5S, 10, "u11"),
    ("i2", *_C5S, 1000, "u11"), ("i4", *_C5S, 1000, "u11"), ("bf16", *_C5S, 1000, "u11"),   # configuration 5's own head
    ("bf16+bf16act", *_C2S, 10, "u01"), ("bf16+bf16act", *_C4S, 10, "n01"), ("bf16+bf16act", *_C4S, 1000, "n01"),
]
# Raw argmax agreement known to miss 99.9 %, with the floor each case must still hold (a regression guard: the miss
# is a property of 16-bit activations, not a licence for anything worse).  Measured at 8192 samples: FP16
# activations (11 significant bits) on random 1000-class heads 99.82-99.94 %; BF16 activations (8 bits) 99.0-99.3 %
# on 1000 classes and 99.6-99.96 % on 10.
_ARGMAX_KNOWN_MISS = {
    ("bf16", 1024, 1000): 0.9975, ("f16", 1024, 1000): 0.9975,
    ("i8", 1024, 1000): 0.9975,            # 99.94 % measured: passes today, five misses from the bar
    ("i2", 512, 1000): 0.9975, ("i4", 512, 1000): 0.9975, ("bf16", 512, 1000): 0.9975,
    ("bf16+bf16act", 784, 10): 0.994, ("bf16+bf16act", 1024, 10): 0.997, ("bf16+bf16act", 1024, 1000): 0.988,
}
_argmax_cache = {}


def _argmax_case(S, O, fmt, topo, acts, classes, inp, flags_setter=None, tag=""):
    """GPU outputs and the FP32 reference's (Training.c:313-345: the oracle's sgemm leg on the same decoded weights)
    for 8192 samples of one case; computed once per case and setting."""
    key = (fmt, tuple(topo), classes, inp, tag)
    if key in _argmax_cache:
        return _argmax_cache[key]
    topo = list(topo) + [classes]
    acts = list(acts) + ["softmax"]
    src = make_oracle_net(O, topo, acts, seed=42, bias_std=0.05)
    bf16act = fmt.endswith("+bf16act")
    _, ref, net = quantized_pair(O, S, src, fmt.split("+")[0])
    rng = np.random.default_rng(7)
    n = 8192
    X = {"u01": lambda: rng.random((n, topo[0]), dtype=F32), "u11": lambda: rng.random((n, topo[0]), dtype=F32) * 2 - 1,
         "n01": lambda: rng.standard_normal((n, topo[0])).astype(F32)}[inp]()
    fn, _, _ = O.find_sgemm()
    _, want = ref.time_forward_batch(X, 1, fn, 8)
    S.lib().spingalett_set_bf16_activations(1 if bf16act else 0)
    if flags_setter:
        flags_setter(True)
    try:
        got = S.forward_batch(net, X)
    finally:
        S.lib().spingalett_set_bf16_activations(0)
        if flags_setter:
            flags_setter(False)
    S.free_network(net)
    _argmax_cache[key] = (got, want)
    return got, want


@pytest.mark.parametrize("fmt,topo,acts,classes,inp", _ARGMAX_CASES)
def test_matrix_core_outputs_within_tolerance_of_the_fp32_reference(S, O, fmt, topo, acts, classes, inp):
    """Every case of the argmax test below, the known misses included: outputs within 2e-2 (relative max-abs) of the
    reference's FP32 batch_forward, and every decided sample (reference top-2 gap above twice the largest deviation)
    has the reference's argmax.  No case is excused from these two."""
    got, want = _argmax_case(S, O, fmt, topo, acts, classes, inp)
    assert rel_max_abs(got, want) <= TOL_MFMA
    _, decided = argmax_agreement(got, want)
    assert decided == 1.0, decided


@pytest.mark.parametrize("fmt,topo,acts,classes,inp", _ARGMAX_CASES)
def test_argmax_agreement_with_the_fp32_reference(S, O, fmt, topo, acts, classes, inp):
    """At least 99.9 % of 8192 samples must have the argmax of the reference's FP32 batch_forward.  The cases known to
    miss it must hold their floor and are then reported as expected failures with the measured figure; only this one
    comparison is excused for them."""
    got, want = _argmax_case(S, O, fmt, topo, acts, classes, inp)
    raw, _ = argmax_agreement(got, want)
    floor = _ARGMAX_KNOWN_MISS.get((fmt, topo[0], classes))
    if floor is None:
        assert raw >= 0.999, raw
        return
    assert raw >= floor, raw
    if raw < 0.999:
        pytest.xfail(f"raw argmax agreement {raw:.4%} of 8192 samples (needs more significant bits than a 16-bit "
                     "activation type has)")


# Split activations (SPHIP_SPLIT_ACTIVATIONS / spingalett_set_net_activations(SPLIT)): the mode that is meant to reach
# 99.9 % on the 1000-class heads, at FP32-grade distance from the reference.
_SPLIT_CASES = [c for c in _ARGMAX_CASES if c[3] == 1000 and "+" not in c[0]] + [("i8", *_C2S, 10, "u01"), ("bf16", *_C4S, 10, "n01")]


@pytest.mark.parametrize("fmt,topo,acts,classes,inp", _SPLIT_CASES)
def test_split_activations_reach_the_argmax_bar_on_every_head(S, O, fmt, topo, acts, classes, inp):
    """With every activation carried as two FP16 numbers (about 22 significant bits) the outputs are within 1e-4 of the
    reference's FP32 batch_forward (Training.c:313-345) instead of 2e-2, every decided sample agrees, and at least
    99.9 % of 8192 samples have its argmax: on the 1000-class heads of configurations 4 and 5, in every weight format,
    where plain FP16 activations reach 99.82-99.94 %."""
    src = make_oracle_net(O, list(topo) + [classes], list(acts) + ["softmax"], seed=42, bias_std=0.05)
    _, ref, net = quantized_pair(O, S, src, fmt)
    rng = np.random.default_rng(7)
    n = 8192
    X = {"u01": lambda: rng.random((n, topo[0]), dtype=F32), "u11": lambda: rng.random((n, topo[0]), dtype=F32) * 2 - 1,
         "n01": lambda: rng.standard_normal((n, topo[0])).astype(F32)}[inp]()
    fn, _, _ = O.find_sgemm()
    _, want = ref.time_forward_batch(X, 1, fn, 8)
    assert S.lib().spingalett_set_net_activations(net, S.NET_ACTIVATIONS_SPLIT) == 0
    got = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, want) <= 1e-4
    raw, decided = argmax_agreement(got, want)
    assert decided == 1.0
    assert raw >= 0.999, raw


@pytest.mark.parametrize("fmt", ["f16", "bf16", "i8", "i4", "i2"])
@pytest.mark.parametrize("topo,acts,n", [
    ([96, 200, 72, 10], ["tanh", "relu", "softmax"], 5),          # thin kernels with few samples, classifier head
    ([96, 200, 72, 10], ["tanh", "relu", "softmax"], 40),
    ([256, 384, 520, 33], ["sigmoid", "softmax", "none"], 300),   # hidden softmax, streaming kernels, odd widths
    ([77, 130, 65], ["leaky_relu", "foo52"], 129),                # rows that are not whole 16-byte units
    ([512, 1024, 512, 1000], ["relu", "leaky_relu", "softmax"], 2048),   # tiled GEMM with and without K splits
    ([784, 512, 1000, 10], ["relu", "relu", "softmax"], 256),            # small layers in one launch, FP32 input split in it
    ([1000, 136, 2048, 72], ["tanh", "sigmoid", "none"], 70),            # the same with K tails and ragged tiles
])
def test_split_activations_on_every_kernel_family(S, O, fmt, topo, acts, n):
    """The split-activation forward through every matrix-core kernel family (streaming with the weights or the
    activations as the tall operand, K split inside the workgroup, tiled GEMM of both kinds), against the oracle's
    float64 forward on the decoded weights: FP32-grade agreement, which no single 16-bit activation type gives."""
    src = make_oracle_net(O, topo, acts, seed=n + len(topo), bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    X = np.random.default_rng(n).standard_normal((n, topo[0])).astype(F32)
    want = ref.forward_batch_f64(X)
    assert S.lib().spingalett_set_net_activations(net, S.NET_ACTIVATIONS_SPLIT) == 0
    got = S.forward_batch(net, X)
    assert S.lib().spingalett_set_net_activations(net, S.NET_ACTIVATIONS_DEFAULT) == 0
    plain = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, want) <= 2e-5, (fmt, topo, n)
    assert rel_max_abs(plain, want) <= TOL_MFMA


# The split mode of an FP32 net: beyond 64 samples every layer of 128 outputs and more and at least 3 GFLOP runs as
# three FP16 products into one FP32 accumulator (weights and activations as two FP16 parts each) instead of on the
# FP32 matrix instructions; the other layers keep the FP32 kernel.
_F32_SPLIT_CASES = [
    # topology, activations, samples, inputs, input scale, which layers run on the 16-bit matrix cores
    ([784, 512, 1000, 10], ["relu", "relu", "softmax"], 256, "u01", 1.0, (0, 0, 0)),    # configuration 1: too small
    ([784, 512, 1000, 10], ["relu", "relu", "softmax"], 4096, "u01", 1.0, (1, 1, 0)),
    ([1001, 515, 130], ["leaky_relu", "foo52"], 4100, "n01", 1.0, (1, 0)),     # rows that are not whole 16-byte units
    ([2048, 384, 520, 33], ["sigmoid", "softmax", "none"], 3000, "n01", 1.0, (1, 0, 0)),   # hidden softmax behind it
    ([1024, 2048, 1024, 1000], ["tanh", "leaky_relu", "softmax"], 2048, "n01", 1.0, (1, 1, 1)),   # K of 3 x 2048, softmax head
    ([512, 768, 256], ["relu", "none"], 4096, "n01", 3e3, (1, 0)),           # large activations (up to about 1e5 x 0.03)
    ([512, 768, 768], ["relu", "none"], 4096, "n01", 1e-4, (1, 1)),          # small ones: the low parts are FP16 subnormals
]


@pytest.mark.parametrize("topo,acts,n,inp,scale,on16", _F32_SPLIT_CASES)
def test_split_mode_of_an_fp32_net_runs_on_the_16_bit_matrix_cores(S, O, topo, acts, n, inp, scale, on16):
    """FP32 weights, split mode, more than 64 samples: the outputs stay within the FP32 bar (1e-4 of the float64
    forward; measured about 1e-6, as close as the FP32 matrix-core path) while the large layers run in a 16-bit kernel
    over three times the padded row length."""
    src = make_oracle_net(O, topo, acts, seed=n + len(topo), bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, "f32")
    rng = np.random.default_rng(n)
    X = (rng.random((n, topo[0]), dtype=F32) if inp == "u01" else rng.standard_normal((n, topo[0])).astype(F32)) * F32(scale)
    want = ref.forward_batch_f64(X)
    plain = S.forward_batch(net, X)
    assert S.lib().spingalett_set_net_activations(net, S.NET_ACTIVATIONS_SPLIT) == 0
    got = S.forward_batch(net, X)
    m = n * 7 // 8                                                 # a smaller batch through the same buffers
    again = S.forward_batch(net, X[:m])
    h = S.lib().spingalett_hip_handle(net)
    names = [S.lib().sphip_layer_kernel_name(h, l, n, S.SPHIP_SPLIT_ACTIVATIONS).decode() for l in range(1, len(topo))]
    few = S.forward_batch(net, X[:64])                             # too little work for the 16-bit route in every case here
    S.free_network(net)
    assert rel_max_abs(plain, want) <= TOL_VEC
    assert rel_max_abs(got, want) <= 2e-5, (topo, n, rel_max_abs(got, want), rel_max_abs(plain, want))
    assert rel_max_abs(again, want[:m]) <= 2e-5
    assert rel_max_abs(few, want[:64]) <= TOL_VEC
    assert [k.startswith(("sp_gemm16", "sp_skinny16")) for k in names] == [bool(x) for x in on16], names
    assert all(k.startswith("sp_gemm32") for k, x in zip(names, on16) if not x), names
    if not any(on16):
        assert np.array_equal(got, plain)


def test_split_mode_of_an_fp32_net_follows_new_weights(S, O):
    """The FP16 parts of the weights are made on demand and made again after the arrays change on the device: by an
    upload, and by a training step."""
    topo, acts, n = [640, 768, 8], ["tanh", "none"], 3200               # first layer 3.1 GFLOP: on the 16-bit matrix cores
    a = make_oracle_net(O, topo, acts, seed=1)
    b = make_oracle_net(O, topo, acts, seed=2)
    X = np.random.default_rng(0).standard_normal((n, topo[0])).astype(F32)
    d = S.DeviceNet(topo, [S.ACT_TANH, S.ACT_NONE], S.PRECISION_FLOAT32)
    for src in (a, b):
        for l in range(2):
            d.upload(l, 0, np.ascontiguousarray(src.W(l)).ravel())
            d.upload(l, 1, np.ascontiguousarray(src.b(l)).ravel())
        got = d.forward(X, S.SPHIP_SPLIT_ACTIVATIONS)
        assert rel_max_abs(got, src.forward_batch_f64(X)) <= 2e-5
    d.train_begin()
    args = S.SphipTrainArgs(S.OPTIMIZER_SGD, S.LOSS_MSE, 0.05, 0.0, 0.9, 0.9, 0.999, 1e-8, 0.0, 0.9, 0.999)
    T = np.random.default_rng(1).standard_normal((n, topo[-1])).astype(F32)
    d.train_step(X, T, args)
    trained = O.Net.new(topo, [O.ACT[x] for x in acts], 0)
    for l in range(2):
        trained.W(l)[:] = d.train_get(S.SPHIP_TRAIN_W, l).reshape(trained.W(l).shape)
        trained.b(l)[:] = d.train_get(S.SPHIP_TRAIN_B, l)
    got = d.forward(X, S.SPHIP_SPLIT_ACTIVATIONS)
    assert rel_max_abs(got, trained.forward_batch_f64(X)) <= 2e-5
    assert rel_max_abs(got, b.forward_batch_f64(X)) > 1e-3              # the step moved the outputs
    d.destroy()


@pytest.mark.parametrize("fmt", ["f16", "bf16", "i8", "i4", "i2"])
@pytest.mark.parametrize("n", [5, 64, 300])
def test_rows_that_are_not_whole_16_byte_units_split_k_at_few_samples(S, O, fmt, n):
    """Widths like 777 or 1030 keep every 16-bit and integer layer on the single-stage kernel with element-wise loads;
    with few samples that is a handful of workgroups, so K is split over the grid (whole K tiles, partial sums added
    in split order by a second launch).  Same tolerance as every matrix-core path, identical from call to call, with
    plain and with split activations."""
    topo, acts = [777, 1030, 515, 33], ["relu", "tanh", "none"]
    src = make_oracle_net(O, topo, acts, seed=77, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    X = np.random.default_rng(n).standard_normal((n, topo[0])).astype(F32)
    want = ref.forward_batch_f64(X)
    got = S.forward_batch(net, X)
    again = S.forward_batch(net, X)
    h = S.lib().spingalett_hip_handle(net)
    assert S.lib().sphip_layer_kernel_name(h, 1, n, 0).decode() == "sp_gemm16"
    assert S.lib().spingalett_set_net_activations(net, S.NET_ACTIVATIONS_SPLIT) == 0
    fine = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, want) <= TOL_MFMA
    assert np.array_equal(got, again)
    assert rel_max_abs(fine, want) <= 2e-5


@pytest.mark.parametrize("act", ["sigmoid", "relu", "tanh", "leaky_relu", "foo52", "none"])
@pytest.mark.parametrize("n,K,N", [(515, 132, 16390), (512, 128, 16384), (700, 68, 16300)])
def test_large_fp32_layers_take_the_128_by_128_tile(S, O, n, K, N, act):
    """FP32 weights beyond the L2s at 512 samples and more, too few multiply-adds for the BF16 parts: the two-stage
    128 x 128 kernel (ragged M, N and a K that is not a whole number of tiles) with every epilogue, the layer behind it
    and 500 samples the 64 x 64 one; FP32 bar against the float64 forward."""
    src = make_oracle_net(O, [K, N, 40], [act, "none"], seed=12, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, "f32")
    h = S.lib().spingalett_hip_handle(net)
    assert [S.lib().sphip_layer_kernel_name(h, l, n, 0).decode() for l in (1, 2)] == ["sp_gemm32_f32_big", "sp_gemm32_f32"]
    assert S.lib().sphip_layer_kernel_name(h, 1, 500, 0).decode() == "sp_gemm32_f32"
    X = np.random.default_rng(8).standard_normal((n, K)).astype(F32)
    got = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, ref.forward_batch_f64(X)) <= TOL_VEC


@pytest.mark.parametrize("fmt,K,N,act,head,kernel", [
    ("i8", 144, 4112, "tanh", True, "sp_gemm16"),            # an uneven round of large tiles and a short sum
    ("i8", 144, 4112, "relu", True, "sp_gemm16"),
    ("i4", 1056, 4128, "sigmoid", True, "sp_gemm16_big"),    # ... a sum too long for that
    ("f16", 512, 4112, "sigmoid", True, "sp_gemm16"),
    ("f16", 520, 4120, "sigmoid", True, "sp_gemm16_big"),      # 16-bit outputs through the FP32 staging of large tiles
    ("f16", 144, 4112, "leaky_relu", True, "sp_gemm16_big"),
    ("bf16", 640, 4116, "tanh", False, "sp_gemm16_big"),       # FP32 outputs, the last tiles of both kinds in part
])
def test_short_layers_of_uneven_rounds_of_large_tiles(S, O, fmt, K, N, act, head, kernel):
    """306 large tiles on 256 compute units: which kernel takes the layer, and the epilogues with tanh and sigmoid of both."""
    n = 4605
    topo, acts = ([K, N, 24], [act, "none"]) if head else ([K, N], [act])
    src = make_oracle_net(O, topo, acts, seed=K + N, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    h = S.lib().spingalett_hip_handle(net)
    assert S.lib().sphip_layer_kernel_name(h, 1, n, 0).decode() == kernel
    X = np.random.default_rng(N).standard_normal((n, K)).astype(F32)
    got = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, ref.forward_batch_f64(X)) <= TOL_MFMA


@pytest.mark.parametrize("fmt", ["f16", "bf16", "i8", "i4", "i2"])
@pytest.mark.parametrize("n,K,N", [
    (4096, 128, 4096), (4095, 144, 4088), (3841, 192, 4096),    # two and three K tiles, whole and in part: prologue and drain only
    (4090, 320, 4086),                                           # rows of FP32 outputs that are not whole 16-byte units
    (100, 4224, 1023), (100, 3200, 1536),                        # 128-row tiles, K splits of which the last is short
])
def test_large_tiles_at_the_edges_of_their_pipeline(S, O, fmt, n, K, N):
    """sp_gemm16_big where its loop is hardly entered, behind partial K tiles and on both tile heights, FP32 outputs, against
    the float64 forward.  (FP16 inputs: 2^-11 of each, at random over K terms.)"""
    src = make_oracle_net(O, [K, N], ["none"], seed=n + K + N, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    h = S.lib().spingalett_hip_handle(net)
    name = S.lib().sphip_layer_kernel_name(h, 1, n, 0).decode()
    # (rows of 144 packed codes are not whole units; integer layers of few samples are streamed)
    want = "sp_skinny16" if n == 100 and fmt in ("i8", "i4", "i2") else "sp_gemm16" if (fmt, K) in (("i4", 144), ("i2", 144)) else "sp_gemm16_big"
    assert name == want
    X = np.random.default_rng(K).standard_normal((n, K)).astype(F32)
    got = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, ref.forward_batch_f64(X)) <= 2e-3


@pytest.mark.parametrize("fmt", ["f16", "bf16", "i8", "i4", "i2"])
@pytest.mark.parametrize("n,K,N", [
    (9, 2112, 1031), (17, 4160, 130), (33, 2176, 2050), (48, 2560, 126), (64, 2112, 4099),   # one to four sixteens of samples, K
    (65, 8256, 1000), (129, 2496, 1155), (256, 2048, 2047), (200, 2112, 16300),              # splits whose last chunk is partial,
])                                                                                            # rows that end inside a tile
def test_streamed_weights_at_the_edges_of_their_tiles(S, O, fmt, n, K, N):
    """sp_skinny16 (and what takes these layers where it does not) against the float64 forward.  (FP16 inputs: 2^-12 of each, at
    random over K terms.)"""
    src = make_oracle_net(O, [K, N], ["none"], seed=n + K + N, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    h = S.lib().spingalett_hip_handle(net)
    name = S.lib().sphip_layer_kernel_name(h, 1, n, 0).decode()
    packed, wide = fmt in ("i4", "i2"), fmt in ("f16", "bf16")
    want = {65: "sp_gemm16_big" if wide else "sp_skinny16", 200: "sp_skinny16_regs" if packed else "sp_gemm16"}.get(n, "sp_skinny16")
    assert name == want
    X = np.random.default_rng(K).standard_normal((n, K)).astype(F32)
    got = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, ref.forward_batch_f64(X)) <= 2e-3


@pytest.mark.parametrize("fmt,mode", [("f16", "plain"), ("bf16", "plain"), ("bf16", "bf16"), ("i8", "split"), ("i4", "plain"), ("i2", "split")])
@pytest.mark.parametrize("n,K,N,act", [
    (5, 8, 1, "none"), (16, 40, 16, "softmax"), (17, 1000, 17, "softmax"), (33, 2048, 32, "tanh"), (300, 1536, 33, "leaky_relu"),
    (129, 2048, 64, "softmax"), (1001, 3072, 50, "sigmoid"), (40, 8200, 10, "softmax"), (70, 16384, 16, "none"),   # K in parts
    (8192, 264, 31, "softmax"), (8200, 72, 64, "relu"),                                          # two sixteens of samples
])
def test_few_outputs_at_the_edges_of_their_tiles(S, O, fmt, mode, n, K, N, act):
    """sp_skinny16_kw_head against the float64 forward.  (FP16 inputs: 2^-12 of each, at random over K terms; BF16 ones 2^-9; split
    ones 2^-22 beside the sums' 2^-24 per term.)"""
    src = make_oracle_net(O, [K, N], [act], seed=n + K + N, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    if mode != "plain":
        which = S.NET_ACTIVATIONS_SPLIT if mode == "split" else S.NET_ACTIVATIONS_BF16
        assert S.lib().spingalett_set_net_activations(net, which) == 0
    flags = {"plain": 0, "split": S.SPHIP_SPLIT_ACTIVATIONS, "bf16": S.SPHIP_BF16_ACTIVATIONS}[mode]
    assert S.lib().sphip_layer_kernel_name(S.lib().spingalett_hip_handle(net), 1, n, flags).decode() == "sp_skinny16_kw_head"
    X = np.random.default_rng(K).standard_normal((n, K)).astype(F32)
    got = S.forward_batch(net, X)
    part = S.forward_batch(net, X[:n // 2 + 5])                    # other tiles' edges, through the same buffers
    S.free_network(net)
    want, tol = ref.forward_batch_f64(X), {"plain": 2e-3, "bf16": 1.6e-2, "split": 2e-5}[mode]
    assert rel_max_abs(got, want) <= tol
    assert rel_max_abs(part, want[:n // 2 + 5]) <= tol


@pytest.mark.parametrize("fmt,mode", [("f32", "plain"), ("f32", "split"), ("bf16", "bf16"), ("f16", "plain"), ("i8", "split"), ("i2", "plain")])
@pytest.mark.parametrize("n,topo,acts", [
    (19, [4096, 65], ["softmax"]), (37, [6000, 256], ["softmax"]), (50, [4100, 257], ["softmax"]), (9, [8192, 1000], ["softmax"]),
    (300, [8192, 1024], ["softmax"]), (21, [3000, 1025], ["softmax"]), (70, [128, 1027], ["softmax"]), (17, [4096, 4095], ["softmax"]),
    (33, [64, 4097], ["softmax"]), (6, [2048, 16384], ["softmax"]), (5, [64, 16385], ["softmax"]), (1, [96, 2500], ["softmax"]),
    (40, [4096, 1500, 20], ["softmax", "tanh"]), (11, [256, 300, 9], ["softmax", "none"]),       # hidden ones, in each 16-bit form
])
def test_softmax_of_split_sums_and_of_wide_rows(S, O, fmt, mode, n, topo, acts):
    """sp_sum_softmax at the edges of what a thread, a wave and a workgroup hold, against the float64 forward.  (As for few outputs; a
    softmax turns the error of a logit into a relative one, and FP32 logits have 2^-24 per term.)"""
    src = make_oracle_net(O, topo, acts, seed=n + topo[1], bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    if mode != "plain":
        which = S.NET_ACTIVATIONS_SPLIT if mode == "split" else S.NET_ACTIVATIONS_BF16
        assert S.lib().spingalett_set_net_activations(net, which) == 0
    X = np.random.default_rng(n).standard_normal((n, topo[0])).astype(F32)
    got, want = S.forward_batch(net, X), ref.forward_batch_f64(X)
    one = S.forward(net, X[0]).copy()
    S.free_network(net)
    tol = {"plain": 2e-5 if fmt == "f32" else 4e-3, "bf16": 3e-2, "split": 4e-5}[mode]
    assert rel_max_abs(got, want) <= tol
    assert rel_max_abs(one, want[0]) <= 2e-5
    if len(topo) == 2:
        assert np.abs(got.astype(np.float64).sum(axis=1) - 1).max() <= 1e-5


@pytest.mark.parametrize("fmt,mode,n,topo,acts", [
    ("f16", "split", 2048, [64, 512], ["softmax"]), ("i2", "split", 2049, [72, 258], ["softmax"]),           # a wave to a row of
    ("i4", "split", 4096, [64, 513], ["softmax"]), ("bf16", "split", 4099, [64, 768], ["softmax"]),          # up to 768, and
    ("i8", "split", 4097, [64, 769], ["softmax"]), ("f32", "plain", 2100, [300, 401], ["softmax"]),          # just not
    ("i2", "split", 512, [1024, 1025], ["softmax"]), ("f16", "split", 511, [1024, 2051], ["softmax"]),       # with the parts, and not
    ("i8", "split", 600, [256, 8192], ["softmax"]), ("f16", "plain", 513, [64, 8191], ["softmax"]), ("bf16", "plain", 70, [64, 8193], ["softmax"]),
    ("i4", "split", 520, [256, 5001, 9], ["softmax", "none"]),
])
def test_softmax_rows_at_the_lines_between_their_kernels(S, O, fmt, mode, n, topo, acts):
    """sp_sum_softmax's instances at both sides of the lines between them, as above."""
    test_softmax_of_split_sums_and_of_wide_rows(S, O, fmt, mode, n, topo, acts)


def test_rows_of_logits_take_no_longer_past_a_border(S):
    """8192 rows of 4097 logits against 4096 (every thread went through 64 places for 17 values: 2.4 times as long; now 1.2)."""
    n, us = 8192, {}
    for N in (4096, 4097):
        net = S.DeviceNet([64, N], [S.ACT_SOFTMAX], S.PRECISION_FP16)
        net.upload(0, 0, np.zeros(64 * N, np.uint16))
        net.upload(0, 1, np.zeros(N, np.uint16))
        d_x, d_y = S.DeviceBuffer.from_numpy(np.zeros((n, 64), F32)), S.DeviceBuffer(n * N * 4)
        us[N] = np.inf
        for _ in range(6):
            start = time.perf_counter()
            for _ in range(20):
                net.forward_device(d_x, n, d_y)
            S.synchronize()
            us[N] = min(us[N], time.perf_counter() - start)
        net.destroy()
    assert us[4097] <= 1.6 * us[4096]


@pytest.mark.parametrize("fmt", ["f16", "bf16", "i8", "i4", "i2"])
@pytest.mark.parametrize("K,N", [(1279, 70), (1283, 70), (4095, 65), (4097, 65), (4999, 129), (5002, 300), (5003, 64), (9002, 1100), (7297, 901)])
def test_few_samples_of_rows_that_are_no_whole_words(S, O, fmt, K, N):
    """The vector kernels on such rows as they are and padded (raw_rows), one to four samples, against the float64 forward; forward()
    hands out the padded layer's outputs and its input unchanged.  (FP32 sums of K terms: 2^-24 each, at random.)"""
    src = make_oracle_net(O, [K, N, 7], ["tanh", "none"], seed=K + N, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    X = np.random.default_rng(K).standard_normal((4, K)).astype(F32)
    want = ref.forward_batch_f64(X)
    for n in (1, 2, 3, 4):
        assert rel_max_abs(S.forward_batch(net, X[:n]), want[:n]) <= 1e-5
    assert rel_max_abs(S.forward(net, X[1]), want[1]) <= 1e-5
    c = net.contents
    neurons = np.ctypeslib.as_array(c.neurons, shape=(int(c.total_neurons),))
    assert np.array_equal(neurons[:K], X[1])
    hidden = np.tanh(X[1].astype(np.float64) @ ref.W(0).astype(np.float64).T + ref.b(0))
    assert rel_max_abs(neurons[K:K + N], hidden) <= 1e-5
    S.free_network(net)


@pytest.mark.parametrize("fmt,K,N", [("i8", 5003, 1000), ("i8", 7297, 901), ("i4", 5002, 1300), ("i4", 9001, 4100), ("i2", 9002, 1100), ("i2", 4104, 2600)])
def test_few_large_inputs_cost_the_others_no_bits_in_ragged_rows(S, O, fmt, K, N):
    """One to four samples, inputs of a million in front of weights of zero among ones of one: the activations of rows that are whole
    units by padding only stay FP32 values of their own.  (FP32 sums: 2^-24 per term; 22 bits of a chunk's largest would be 0.5.)"""
    src = make_oracle_net(O, [K, N], ["none"], seed=K + N, bias_std=0.1)
    large = [0, 1, K // 3, 2048, K - 1]
    src.W(0)[:, large] = 0.0
    _, ref, net = quantized_pair(O, S, src, fmt)
    X = np.random.default_rng(K).standard_normal((4, K)).astype(F32)
    X[:, large] = np.array([1e6, -3e5, 2e5, -1e6, 7e5], F32)
    want = ref.forward_batch_f64(X)
    for n in (1, 2, 3, 4):
        assert rel_max_abs(S.forward_batch(net, X[:n]), want[:n]) <= 1e-5, n
    assert rel_max_abs(S.forward(net, X[1]), want[1]) <= 1e-5
    S.free_network(net)


@pytest.mark.parametrize("fmt,mode", [("i8", "plain"), ("i4", "plain"), ("i2", "plain"), ("i2", "split")])
@pytest.mark.parametrize("K,N", [(2056, 300), (2072, 260), (4008, 131), (6024, 1030)])
def test_wide_inputs_of_integer_nets_run_padded(S, O, fmt, mode, K, N):
    """Inputs of more than 2048 values whose rows of codes are no whole 16-byte units (padded_width), from a sample to several tiles,
    against the float64 forward.  (FP16 inputs 2^-12, split ones 2^-22.)"""
    src = make_oracle_net(O, [K, N, 12], ["relu", "softmax"], seed=K + N, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    if mode == "split":
        assert S.lib().spingalett_set_net_activations(net, S.NET_ACTIVATIONS_SPLIT) == 0
    X = np.random.default_rng(K).standard_normal((700, K)).astype(F32)
    want = ref.forward_batch_f64(X)
    for n in (1, 4, 5, 17, 64, 300, 700):
        tol = 2e-5 if n <= 4 else 4e-5 if mode == "split" else 5e-3
        assert rel_max_abs(S.forward_batch(net, X[:n]), want[:n]) <= tol, n
    S.free_network(net)


_PLAIN_AND_SPLIT = [("f16", "plain"), ("bf16", "plain"), ("i8", "plain"), ("i4", "plain"), ("i2", "plain"), ("f16", "split"), ("i4", "split")]


@pytest.mark.parametrize("n,K,N,act,fmt,mode", [(*layer, *how) for layer, hows in [
    ((257, 2064, 65, "tanh"), _PLAIN_AND_SPLIT),               # four parts, the last of two K tiles; rows of words in INT4 and INT2
    ((5000, 1168, 75, "softmax"), _PLAIN_AND_SPLIT),           # two parts, the last K tile partial
    ((300, 3024, 200, "softmax"), _PLAIN_AND_SPLIT),           # padded INT4 and INT2 rows
    ((1100, 3024, 73, "tanh"), _PLAIN_AND_SPLIT),
    ((1100, 3000, 73, "softmax"), [("f16", "plain"), ("i8", "plain"), ("i4", "split")]),           # rows of words in INT8
    ((500, 8192, 255, "tanh"), _PLAIN_AND_SPLIT),
    ((1000, 8200, 250, "softmax"), _PLAIN_AND_SPLIT),
    ((1000, 8200, 250, "tanh"), [("f32", "split")]), ((3000, 2056, 250, "softmax"), [("f32", "split")]),   # sums three times as long
] for how in hows])
def test_long_sums_of_few_tiles_are_split(S, O, fmt, mode, n, K, N, act):
    """K splits of sp_gemm16 (gemm16_single_splits): even and uneven ones, partial K tiles, rows of whole words and of 16-byte units,
    against the float64 forward.  (FP16 inputs 2^-12, BF16 2^-9, split ones 2^-22.)"""
    src = make_oracle_net(O, [K, N], [act], seed=n + K + N, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    if mode == "split":
        assert S.lib().spingalett_set_net_activations(net, S.NET_ACTIVATIONS_SPLIT) == 0
    flags = S.SPHIP_SPLIT_ACTIVATIONS if mode == "split" else 0
    assert S.lib().sphip_layer_kernel_name(S.lib().spingalett_hip_handle(net), 1, n, flags).decode() == "sp_gemm16"
    X = np.random.default_rng(K).standard_normal((n, K)).astype(F32)
    got = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, ref.forward_batch_f64(X)) <= (4e-5 if mode == "split" else 2e-2 if fmt == "bf16" else 5e-3)


@pytest.mark.parametrize("fmt", ["f16", "bf16", "i8", "i4", "i2"])
@pytest.mark.parametrize("n,K,N", [(100, 128, 49152), (100, 192, 49160), (128, 320, 49410), (65, 1024, 49153)])
def test_tiles_of_128_rows_in_every_format(S, O, fmt, n, K, N):
    """sp_gemm16_big with 128-row tiles, whole and partial K tiles, against the float64 forward.  (As above.)"""
    src = make_oracle_net(O, [K, N], ["none"], seed=n + K + N, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    h = S.lib().spingalett_hip_handle(net)
    assert S.lib().sphip_layer_kernel_name(h, 1, n, 0).decode() == "sp_gemm16_big"
    X = np.random.default_rng(K).standard_normal((n, K)).astype(F32)
    got = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, ref.forward_batch_f64(X)) <= 2e-3


@pytest.mark.parametrize("fmt,n,K,N,act,name", [
    # one round, as many rounds as tiles fill, three rounds of which a quarter is idle, two of which a third is
    ("f16", 4096, 512, 4096, "sigmoid", "sp_gemm16"), ("f16", 4096, 520, 4096, "tanh", "sp_gemm16_big"),
    ("i8", 4096, 528, 4096, "sigmoid", "sp_gemm16_big"), ("i2", 4096, 512, 4096, "tanh", "sp_gemm16"),
    ("bf16", 8192, 768, 8192, "tanh", "sp_gemm16"), ("bf16", 8192, 776, 8192, "tanh", "sp_gemm16_big"),
    ("i4", 8192, 1024, 8192, "sigmoid", "sp_gemm16"), ("i4", 8192, 1056, 8192, "sigmoid", "sp_gemm16_big"),
    ("f16", 4567, 1536, 8192, "tanh", "sp_gemm16"), ("f16", 4567, 1544, 8192, "sigmoid", "sp_gemm16_big"),
    ("i8", 4567, 2048, 4736, "tanh", "sp_gemm16"), ("i8", 4567, 2064, 4736, "tanh", "sp_gemm16_big"),
    ("i8", 4567, 512, 4736, "relu", "sp_gemm16"), ("i8", 4567, 528, 4736, "relu", "sp_gemm16_big"),
])
def test_which_kernel_takes_short_sums(S, fmt, n, K, N, act, name):
    """Both sides of each line of gemm16_shared_limit (nothing is launched)."""
    bits = {"f16": 16, "bf16": 16, "i8": 8, "i4": 4, "i2": 2}[fmt]
    prec = {"f16": S.PRECISION_FP16, "bf16": S.PRECISION_BFLOAT16, "i8": S.PRECISION_INT8, "i4": S.PRECISION_INT4, "i2": S.PRECISION_INT2}[fmt]
    d = S.DeviceNet([K, N], [{"sigmoid": S.ACT_SIGMOID, "tanh": S.ACT_TANH, "relu": S.ACT_RELU}[act]], prec)
    for which, count in ((0, K * N), (1, N)):
        d.upload(0, which, np.zeros(count * bits // 8, np.uint8), 1.0 if bits < 16 else 0.0)
    got = S.lib().sphip_layer_kernel_name(d.h, 1, n, 0).decode()
    d.destroy()
    assert got == name


@pytest.mark.parametrize("fmt,n,K,N,act", [
    ("f16", 4095, 576, 4088, "tanh"), ("i8", 4090, 576, 4086, "sigmoid"),      # whole units, and rows that are not
    ("i2", 4090, 640, 4086, "tanh"), ("bf16", 3900, 528, 4083, "sigmoid"),
    ("bf16", 1000, 128, 8190, "tanh"), ("f16", 1000, 320, 8184, "sigmoid"),    # 128-row tiles
    ("i4", 100, 192, 49160, "tanh"),
])
def test_large_tiles_with_sigmoid_and_tanh(S, O, fmt, n, K, N, act):
    """The late activations of sp_gemm16_big, once with the layer as the last one (FP32 outputs) and once in front of a small
    one (16-bit outputs, padded widths), against the float64 forward.  A sigmoid or tanh passes at most its argument's error on;
    the 16-bit output adds 2^-9 of at most 1 (BF16), at random over the head's N terms."""
    for topo, acts in (([K, N], [act]), ([K, N, 24], [act, "none"])):
        src = make_oracle_net(O, topo, acts, seed=n + K + N, bias_std=0.1)
        _, ref, net = quantized_pair(O, S, src, fmt)
        h = S.lib().spingalett_hip_handle(net)
        assert S.lib().sphip_layer_kernel_name(h, 1, n, 0).decode() == "sp_gemm16_big"
        X = np.random.default_rng(K).standard_normal((n, K)).astype(F32)
        got = S.forward_batch(net, X)
        S.free_network(net)
        assert rel_max_abs(got, ref.forward_batch_f64(X)) <= (8e-3 if fmt == "bf16" else 2e-3)


def test_large_tiles_apply_the_library_s_tanh(S):
    """tanh of sp_gemm16_big, written without tanhf's branch, bit by bit that of the single-stage kernel: both sides of 0.625,
    zeros of either sign, subnormal and huge sums, infinities and NaN.  (One term per sum, so that no order of sums matters.)"""
    N, n = 4096, 4096
    edge = np.array([0.0, -0.0, 0.625, -0.625, 0.62451171875, 0.62548828125, 6e-8, -6e-8, 1e-4, 9.0, 9.1, -20.0, 65504.0,
                     np.inf, -np.inf, np.nan], np.float16)
    w = np.concatenate([edge, np.linspace(-10, 10, N - edge.size).astype(np.float16)])
    X = np.zeros((n, 576), F32)
    X[:, 0] = np.linspace(0.5, 1.5, n).astype(np.float16)
    out = []
    for K, name in ((576, "sp_gemm16_big"), (512, "sp_gemm16")):
        W = np.zeros((N, K), np.float16)
        W[:, 0] = w
        d = S.DeviceNet([K, N], [S.ACT_TANH], S.PRECISION_FP16)
        d.upload(0, 0, W.ravel().view(np.uint8))
        d.upload(0, 1, np.zeros(N, np.float16).view(np.uint8))
        assert S.lib().sphip_layer_kernel_name(d.h, 1, n, 0).decode() == name
        out.append(d.forward(np.ascontiguousarray(X[:, :K])))
        d.destroy()
    a, b = (o.view(np.uint32) for o in out)
    assert np.array_equal(a[:, :13], b[:, :13]) and np.array_equal(a[:, 16:], b[:, 16:])
    assert np.array_equal(out[0][:, 13:], out[1][:, 13:], equal_nan=True) and np.all(np.isnan(out[0][:, 15]))
    assert np.all(out[0][:, 13] == 1.0) and np.all(out[0][:, 14] == -1.0)


def test_large_tiles_saturate_and_keep_infinities_block_by_block(S):
    """FP16 outputs of sp_gemm16_big: finite sums beyond +-65504 saturate, infinities and NaNs stay and only their own
    samples have them, in row tiles that hold ordinary samples too."""
    n, K, N = 4605, 144, 4112
    rng = np.random.default_rng(5)
    W = (rng.standard_normal((N, K)) * 0.1).astype(np.float16)
    W[:, 3] = 1.0
    V = np.zeros((8, N), np.float16)
    V[np.arange(8), np.arange(8) * 513] = 1.0                    # each output of the net is one neuron of the large layer
    X = rng.standard_normal((n, K)).astype(F32)
    X[17, 3], X[4600, 3] = 65504.0, -65504.0
    X[17, 4:] *= 3000.0                                          # sums on both sides of 65504
    X[33, 3], X[1000, 3], X[4604, 7] = np.inf, -np.inf, np.nan
    d = S.DeviceNet([K, N, 8], [S.ACT_NONE, S.ACT_NONE], S.PRECISION_FP16)
    for l, a in ((0, W), (1, V)):
        d.upload(l, 0, a.ravel().view(np.uint8))
        d.upload(l, 1, np.zeros(a.shape[0], np.float16).view(np.uint8))
    assert S.lib().sphip_layer_kernel_name(d.h, 1, n, 0).decode() == "sp_gemm16_big"
    got = d.forward(X)
    d.destroy()
    odd = [33, 1000, 4604]
    assert not np.isfinite(got[odd]).any()                       # (0 x inf in the second layer)
    keep = np.setdiff1d(np.arange(n), odd)
    sums = X[keep].astype(np.float16).astype(np.float64) @ W[::513][:8].astype(np.float64).T
    want = np.clip(sums, -65504.0, 65504.0)
    # one rounding to FP16, and FP32 sums of 144 terms of up to 65504 before it
    assert np.all(np.abs(got[keep] - want) <= 2.0 ** -11 * np.abs(want) + 1e-5 * np.abs(X[keep]).max(axis=1, keepdims=True))
    assert 0 < np.sum(got[17] == 65504.0) < 8


@pytest.mark.parametrize("n,K,N", [
    (4095, 520, 1000),     # 256 tiles of 128 x 128: rows of 64, a last tile of each kind in part, K 8 beyond its tiles
    (8321, 268, 897),      # rows of 128, no split
    (8321, 269, 897),      # ... rows that are not 16-byte aligned
    (8200, 68, 3600),      # short sums
    (250, 2720, 3000),     # split over K, the last share shorter
    (250, 2721, 3000),
    (128, 4096, 4096),
])
def test_large_fp32_products_on_bf16_parts(S, O, n, K, N):
    """The kernel of products of 2 G multiply-adds and more, against float64 and the FP32 kernels' own accuracy: at most
    6 K / 16 roundings of 2^-24 of a partial sum no larger than about its result's deviation (K = 4096 at random: 2e-6;
    at worst one after the other 1e-4)."""
    src = make_oracle_net(O, [K, N], ["none"], seed=n + K, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, "f32")
    h = S.lib().spingalett_hip_handle(net)
    assert S.lib().sphip_layer_kernel_name(h, 1, n, 0).decode() == "sp_gemm32_bf16_parts"
    X = np.random.default_rng(K).standard_normal((n, K)).astype(F32)
    got = S.forward_batch(net, X)
    S.free_network(net)
    assert rel_max_abs(got, ref.forward_batch_f64(X)) <= 1e-5


@pytest.mark.parametrize("x_exp,w_exp", [(-118, 40), (-122, 0), (-130, 60), (20, -125), (-60, -30), (101, -60), (110, -80), (60, 25)])
def test_large_fp32_products_of_tiny_and_huge_operands_keep_their_bits(S, x_exp, w_exp):
    """Operands down to subnormal ones have BF16 parts that hold all their bits, operands from 2^104 and sums from 2^80 on
    are formed as FP32 chains.  Against 64 bits; the accumulator is rounded six times per 16 k, so the 2-norm of the error
    is about 2^-24 sqrt(6 K / 16) of the result's, a fraction of it since the sums grow; four times that at most, where
    parts that end at 2^-133 give 9e-6 of a result with operands of 2^-118.  (An FP32 chain is rounded K times.)"""
    n, K, N = 700, 1000, 3000
    rng = np.random.default_rng(x_exp + 200)
    X = np.ldexp(rng.standard_normal((n, K)), x_exp).astype(F32)
    W = np.ldexp(rng.standard_normal((N, K)), w_exp).astype(F32)
    d = S.DeviceNet([K, N], [S.ACT_NONE], S.PRECISION_FLOAT32)
    d.upload(0, 0, W.ravel())
    d.upload(0, 1, np.zeros(N, F32))
    assert S.lib().sphip_layer_kernel_name(d.h, 1, n, 0).decode() == "sp_gemm32_bf16_parts"
    got = d.forward(X).astype(np.float64)
    want = X.astype(np.float64) @ W.astype(np.float64).T
    rounds = K if x_exp >= 104 or x_exp + w_exp >= 80 else 6 * K / 16
    assert np.linalg.norm(got - want) <= 4 * 2.0 ** -24 * np.sqrt(rounds) * np.linalg.norm(want), np.linalg.norm(got - want) / np.linalg.norm(want)
    d.destroy()


def test_large_fp32_products_keep_infinities_and_nans(S):
    """Operands without BF16 parts (infinite, beyond the largest BF16, NaN), next to weights whose lower parts are zero."""
    n, K, N = 4096, 784, 640
    rng = np.random.default_rng(3)
    W = (rng.standard_normal((N, K)) * 0.05).astype(F32)
    W[:, 5], W[:, 6], W[::2, 7], W[:, 11] = 1.0, -0.5, 0.0, 0.25
    W[9, 20] = -np.inf
    b = rng.standard_normal(N).astype(F32)
    X = rng.standard_normal((n, K)).astype(F32)
    X[3, 5] = np.inf
    X[70, 5], X[70, 6] = np.inf, np.inf
    X[100, 7] = -np.inf
    X[200, 100] = np.nan
    X[300, 11] = np.finfo(F32).max
    X[4000, 20] = 0.0
    net = S.new_spingalett(S.LOSS_MSE)
    S.layer(net, K)
    S.layer(net, N, S.ACT_NONE, S.WEIGHT_INITIALIZATION_NONE)
    S.weights_view(net, 0)[:] = W
    S.biases_view(net, 0)[:] = b
    got = S.forward_batch(net, X)
    h = S.lib().spingalett_hip_handle(net)
    assert S.lib().sphip_layer_kernel_name(h, 1, n, 0).decode() == "sp_gemm32_bf16_parts"
    S.free_network(net)
    with np.errstate(invalid="ignore"):
        want = X.astype(np.float64) @ W.astype(np.float64).T + b
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want)) and np.array_equal(got[np.isinf(got)], want[np.isinf(want)].astype(F32))
    fine = np.isfinite(want)
    fine[300] = False
    assert fine.sum() > n * N - 5 * n - 5 * N
    assert rel_max_abs(got[fine], want[fine]) <= 1e-5
    row = np.isfinite(want[300])
    assert rel_max_abs(got[300][row], want[300][row]) <= 1e-6


def test_fp32_nets_leave_the_vector_kernel_beyond_four_samples(S, O):
    """From five samples on the FP32 matrix-core kernel is the faster one for FP32 weights, as the 16-bit one is for
    the other formats (configuration 1 at 64 samples: 31 us against 245 us in eight passes of the vector kernel), and
    its K splits need their workspace at those batch sizes too."""
    topo, acts = [784, 512, 1000, 10], ["relu", "relu", "softmax"]
    src = make_oracle_net(O, topo, acts, seed=5, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, "f32")
    h = S.lib().spingalett_hip_handle(net)
    # (512 x 784 at these batch sizes: the one-launch kernel for small layers; at 4096 samples the tiled one)
    assert [S.lib().sphip_layer_kernel_name(h, 1, n, 0).decode() for n in (1, 4, 5, 64, 65, 4096)] == \
        ["sp_gemv", "sp_gemv", "sp_gemm32_small16", "sp_gemm32_small16", "sp_gemm32_small16", "sp_gemm32_f32"]
    # the 1000 -> 10 head: a workgroup per row, up to eight samples (layers of at most 64 outputs)
    assert [S.lib().sphip_layer_kernel_name(h, 3, n, 0).decode() for n in (1, 4, 5, 8, 9)] == \
        ["sp_gemv_words"] * 4 + ["sp_gemm32_small16"]
    X = np.random.default_rng(3).random((4096, topo[0]), dtype=F32)
    want = ref.forward_batch_f64(X)
    for n in (4, 5, 8, 9, 33, 64, 300, 4096):
        assert rel_max_abs(S.forward_batch(net, X[:n]), want[:n]) <= TOL_VEC, n
    S.free_network(net)


def test_net_activation_mode_arguments(S, O):
    src = make_oracle_net(O, [8, 4], ["none"], seed=1)
    _, ref, net = quantized_pair(O, S, src, "i8")
    assert S.lib().spingalett_set_net_activations(net, 3) == 1
    assert S.last_error()[0] == S.SPINGALETT_ERR_INVALID
    S.clear_error()
    assert S.lib().spingalett_set_net_activations(None, 0) == 1
    S.clear_error()
    S.free_network(net)


def _decoded_layer(S, fmt, N, K, seed):
    """One bias-carrying layer with random codes; returns (device net, FP64 weights, FP64 biases)."""
    prec = {"f16": S.PRECISION_FP16, "bf16": S.PRECISION_BFLOAT16, "i8": S.PRECISION_INT8,
            "i4": S.PRECISION_INT4, "i2": S.PRECISION_INT2}[fmt]
    bits = {"f16": 16, "bf16": 16, "i8": 8, "i4": 4, "i2": 2}[fmt]
    rng = np.random.default_rng(seed)
    net = S.DeviceNet([K, N], [S.ACT_LEAKY_RELU], prec)
    if bits == 16:
        w = (rng.standard_normal(N * K) * 0.05).astype(F32)
        b = (rng.standard_normal(N) * 0.1).astype(F32)
        enc = (lambda a: (a.view(np.uint32) >> 16).astype(np.uint16)) if fmt == "bf16" else \
              (lambda a: a.astype(np.float16).view(np.uint16))
        net.upload(0, 0, enc(w))
        net.upload(0, 1, enc(b))
    else:
        net.upload(0, 0, rng.integers(0, 256, size=(N * K * bits + 7) // 8, dtype=np.uint8), 0.37)
        net.upload(0, 1, rng.integers(0, 256, size=(N * bits + 7) // 8, dtype=np.uint8), 0.11)
    W = net.decode(0, 0).astype(np.float64).reshape(N, K)            # decoders are pinned bit-exact elsewhere
    b = net.decode(0, 1).astype(np.float64)
    return net, W, b


@pytest.mark.parametrize("fmt,N,K,n", [
    # few samples, weights streamed: one and two 32-sample tiles, several sample blocks, K splits and K tails
    ("i4", 512, 1024, 5), ("i4", 300, 4096, 33), ("i4", 4096, 2048, 64), ("i4", 2048, 288, 100), ("i4", 1100, 8192, 256),
    ("i8", 512, 144, 7), ("i8", 2100, 2064, 48), ("i8", 8192, 1024, 200),
    ("i2", 640, 4096, 9), ("i2", 4096, 8192, 64), ("i2", 1000, 320, 130),
    ("bf16", 512, 200, 6), ("bf16", 4096, 2048, 40), ("f16", 1500, 1000, 77), ("f16", 96, 4096, 255),
    # at most 8 samples (or outputs): K split among the waves of a workgroup (idle waves, K tails, ragged rows), and
    # the neighbouring sizes that stay on the split-K kernel
    ("i4", 16384, 2048, 8), ("i4", 300, 4352, 7), ("i8", 12288, 1152, 8), ("i2", 12288, 4096, 6), ("i2", 515, 256, 8),
    ("bf16", 12300, 584, 8), ("f16", 640, 8200, 5), ("bf16", 96, 64, 5), ("i8", 8, 4096, 1000), ("i2", 3, 2048, 4096),
    ("i4", 300, 4352, 13), ("i8", 12288, 1152, 16), ("f16", 640, 8200, 12),
    ("i8", 1, 64, 100), ("f16", 2, 8, 9), ("i2", 4, 16, 5),             # one to four outputs, K below one chunk
    # eight-wave workgroups of the streaming kernel: from 16384 outputs, or from 8192 with more than 64 samples;
    # ragged last row block, output counts that are and are not multiples of four (vector / scalar split-K reduction)
    ("i4", 16384, 2048, 40), ("i2", 8192, 1024, 200), ("i4", 16500, 1056, 64), ("i8", 16390, 640, 33),
    ("f16", 16384, 512, 9), ("i2", 20000, 768, 130),
    # few outputs, activations streamed
    ("i8", 10, 1000, 256), ("i8", 10, 1000, 4096), ("i4", 64, 512, 1000), ("i2", 33, 2048, 513),
    ("bf16", 10, 1000, 300), ("f16", 7, 72, 65), ("i4", 10, 4096, 5),
    # a few hundred samples: 256 x 256 tiles with K split over the grid (K of 4096 and more), else the single-stage kernel
    ("i8", 1024, 4096, 700), ("bf16", 2048, 4168, 300),
    ("bf16", 768, 1024, 130), ("f16", 512, 2048, 200), ("bf16", 1024, 1024, 255),
    ("bf16", 4096, 2048, 65), ("f16", 3000, 4096, 100), ("bf16", 4096, 8192, 128), ("i8", 8192, 2048, 129),
    ("i4", 1024, 2048, 300), ("bf16", 768, 1024, 513), ("i2", 2048, 4096, 1000), ("f16", 512, 1024, 257), ("i8", 1280, 1536, 600),
])
def test_thin_and_split_k_shapes(S, fmt, N, K, n):
    """Layers with one thin side (5..256 samples, or at most 64 outputs) run a weight- or
    activation-streaming MFMA kernel with split K, mid-size batches the tiled GEMM with split K;
    checked against FP64 on the decoded arrays."""
    net, W, b = _decoded_layer(S, fmt, N, K, seed=N + K + n)
    X = np.random.default_rng(n).standard_normal((n, K)).astype(F32)
    pre = X.astype(np.float64) @ W.T + b
    want = np.where(pre > 0, pre, 0.01 * pre)
    got = net.forward(X)
    assert rel_max_abs(got, want) <= (4e-3 if fmt == "bf16" else 1e-3)   # 16-bit rounding of the inputs only
    net.destroy()


@pytest.mark.parametrize("fmt,N,K,n", [
    # Too few 256 x 256 tiles and too few K tiles to split K over the grid: the single-stage tiled GEMM; by tile
    # count it runs 64 x 64, 64 x 128 or 128 x 128 tiles (ragged edges in both directions), rows that are not whole
    # 16-byte units take the element-wise loads and always 64 x 64
    # (more than 512 tiles of 32 x 32, or more than 512 K of tiles x K: fewer go to the one-launch kernel below)
    ("bf16", 512, 784, 1200), ("i8", 1000, 528, 4096),
    ("i2", 2048, 1056, 2048),
    ("i8", 300, 1000, 1800), ("i4", 257, 100, 513), ("i2", 1030, 1000, 520), ("i8", 200, 1000, 2400),
    # integer rows that are whole 32-bit words but not whole 16-byte units (784 INT4 codes = 392 bytes): word loads
    ("i4", 512, 784, 2048), ("i2", 300, 784, 2000), ("i8", 1000, 776, 600), ("i4", 520, 1000, 1100), ("i2", 2048, 1008, 2048),
    ("i4", 70, 24, 6000), ("i8", 4096, 72, 4096),
    # K of 1024 and more: K tiles of 128 (layers of up to 2 M weights and K below 4096 stay here instead of splitting K
    # for the 256 x 256 tiles); K tails of 120, 64 and 16 elements, word loads
    ("f16", 1024, 1024, 2048), ("i8", 512, 2048, 4096), ("i4", 520, 1040, 1100), ("bf16", 768, 2040, 3000), ("i2", 1000, 1088, 1800),
    ("f16", 2000, 1000, 2100), ("i4", 2080, 1056, 300), ("i8", 1100, 2000, 700), ("f16", 2001, 1032, 2100),
    ("bf16", 8192, 1000, 100), ("f16", 5000, 1160, 77),
])
def test_single_stage_gemm_tile_shapes(S, fmt, N, K, n):
    net, W, b = _decoded_layer(S, fmt, N, K, seed=N + 3 * K + n)
    X = np.random.default_rng(n + 1).standard_normal((n, K)).astype(F32)
    pre = X.astype(np.float64) @ W.T + b
    want = np.where(pre > 0, pre, 0.01 * pre)
    got = net.forward(X)
    assert _kernel_of(S, net, n) == "sp_gemm16"
    assert rel_max_abs(got, want) <= (4e-3 if fmt == "bf16" else 1e-3)
    net.destroy()


@pytest.mark.parametrize("fmt,N,K,n", [
    # up to 512 tiles of 32 x 32 and K up to 2048: ragged edges in both directions, K tails of 8, 16 and 24 elements
    # (K = 1000, 784, 24, 72), a K shorter than the eight waves' shares, every weight format, 5 samples and up
    ("bf16", 512, 784, 600), ("i8", 300, 1000, 700), ("i8", 200, 1000, 512), ("i4", 512, 784, 1024), ("i2", 300, 784, 300),
    ("i4", 520, 1000, 64), ("i4", 70, 24, 9), ("f16", 1500, 1000, 77), ("i2", 1000, 320, 130), ("bf16", 4096, 2048, 40),
    ("i8", 512, 784, 256), ("i8", 1000, 512, 256), ("f16", 65, 8, 9), ("i2", 97, 2048, 33), ("bf16", 16384, 32, 32),
    ("i8", 256, 256, 2048), ("f16", 1024, 1024, 512), ("i4", 2048, 2048, 128), ("i2", 130, 72, 1000),
    ("i8", 1000, 512, 5), ("f16", 512, 784, 8), ("i2", 8192, 256, 6), ("bf16", 100, 2048, 7),
])
def test_small_layers_run_in_one_launch(S, fmt, N, K, n):
    """Layers of a few hundred 32 x 32 output tiles run in one launch whose workgroups split K among their waves and
    round the FP32 input themselves (no K split over the grid, no second launch, no separate conversion); checked
    against FP64 on the decoded arrays."""
    net, W, b = _decoded_layer(S, fmt, N, K, seed=N + 5 * K + n)
    X = np.random.default_rng(n + 2).standard_normal((n, K)).astype(F32)
    pre = X.astype(np.float64) @ W.T + b
    want = np.where(pre > 0, pre, 0.01 * pre)
    got = net.forward(X)
    assert _kernel_of(S, net, n) == "sp_gemm16_small"
    assert rel_max_abs(got, want) <= (4e-3 if fmt == "bf16" else 1e-3)
    if fmt == "bf16":                                # BF16 activations against the BF16 weights themselves
        assert rel_max_abs(net.forward(X, S.SPHIP_BF16_ACTIVATIONS), want) <= 1e-2
    net.destroy()


@pytest.mark.parametrize("fmt,N,K,n", [
    # K not a multiple of 64 with 16-byte rows: the 256 x 256 tile kernel takes the partial K tile first.
    # Enough tiles for the chip (tails of 40, 8, 48 and 32 elements) ...
    ("bf16", 4096, 1000, 4096), ("f16", 4096, 1096, 3000), ("i8", 4096, 1008, 4096), ("i4", 4096, 1056, 4096),
    # ... K split over the grid, the partial tile in the last split ...
    ("f16", 2200, 4200, 2100), ("bf16", 2048, 1000, 4096), ("i4", 2080, 4128, 300), ("i8", 1100, 4112, 700),
    # ... a single row of 128 x 256 tiles (K split from K = 3072), ragged in M and N, and a K of two tiles and a bit
    ("bf16", 8192, 3080, 100), ("f16", 5000, 4136, 77), ("bf16", 8200, 136, 8200),
    # output rows that are not whole 16-byte units: one element per lane and store, with and without a K split
    ("bf16", 4099, 1024, 4096), ("f16", 2101, 4104, 2100), ("i8", 4102, 1040, 3000),
])
def test_big_tile_gemm_takes_a_partial_k_tile(S, fmt, N, K, n):
    net, W, b = _decoded_layer(S, fmt, N, K, seed=N + 3 * K + n)
    X = np.random.default_rng(n + 1).standard_normal((n, K)).astype(F32)
    pre = X.astype(np.float64) @ W.T + b
    want = np.where(pre > 0, pre, 0.01 * pre)
    got = net.forward(X)
    assert _kernel_of(S, net, n) == "sp_gemm16_big"
    assert rel_max_abs(got, want) <= (4e-3 if fmt == "bf16" else 1e-3)
    net.destroy()


@pytest.mark.parametrize("N,K,n", [
    (512, 1024, 5), (4096, 2048, 64), (1100, 8192, 200),       # weight-streaming kernel, with and without a K split
    (16384, 512, 9), (8192, 1024, 8),                          # eight-wave workgroups; K split inside the workgroup
    (10, 1000, 300), (7, 72, 65),                              # few outputs: activations streamed
    (768, 1024, 130), (4096, 1000, 4096), (2048, 1000, 2100),  # tiles: K split over the grid, partial K tile
    (512, 784, 600), (300, 100, 513),                          # single-stage tiles
])
def test_bf16_weights_with_fp16_activations(S, N, K, n):
    """BF16 weights are multiplied on the FP16 matrix cores against an FP16 copy scaled by a power of two, made at
    upload; SPHIP_BF16_ACTIVATIONS selects the BF16 matrix cores.  Same kernels as FP16 weights (asserted by name
    against an FP16 net of the same shape), outputs compared with FP64 on the decoded BF16 arrays at the FP16 bound of
    the other tests; weights spread over 40 binary orders of magnitude in one array, a re-upload, a clone, and the
    vector path (which has no such copy to use) ride along."""
    net, W, b = _decoded_layer(S, "bf16", N, K, seed=N + 7 * K + n)
    ref16, _, _ = _decoded_layer(S, "f16", N, K, seed=1)
    X = np.random.default_rng(n).standard_normal((n, K)).astype(F32)
    pre = X.astype(np.float64) @ W.T + b
    want = np.where(pre > 0, pre, 0.01 * pre)
    got = net.forward(X)
    assert _kernel_of(S, net, n) == _kernel_of(S, ref16, n)
    assert rel_max_abs(got, want) <= 1e-3
    plain = net.forward(X, S.SPHIP_BF16_ACTIVATIONS)           # BF16 activations: the looser bound, and not the same bits
    assert rel_max_abs(plain, want) <= 4e-3
    assert not np.array_equal(plain, got)
    twin = net.clone()
    assert np.array_equal(twin.forward(X), got)
    twin.destroy()
    # a second array: magnitudes from 2^-30 to 2^10 of the largest; what leaves FP16's range is 2^-29 of it and smaller
    rng = np.random.default_rng(K)
    w = (rng.standard_normal(N * K) * np.exp2(rng.integers(-30, 11, size=N * K))).astype(F32)
    codes = (w.view(np.uint32) >> 16).astype(np.uint16)
    net.upload(0, 0, codes)
    W2 = (codes.astype(np.uint32) << 16).view(F32).astype(np.float64).reshape(N, K)
    pre = X.astype(np.float64) @ W2.T + b
    want2 = np.where(pre > 0, pre, 0.01 * pre)
    assert rel_max_abs(net.forward(X), want2) <= 1e-3
    small = net.forward(X[:3])                                 # vector path: FP32 arithmetic on the BF16 array itself
    assert rel_max_abs(small, want2[:3]) <= 1e-4
    net.destroy(); ref16.destroy()


def _kernel_of(S, net, n, flags=0):
    return S.lib().sphip_layer_kernel_name(net.h, 1, n, flags).decode()


@pytest.mark.parametrize("fmt,N,K", [
    ("i2", 8192, 8192),          # the hidden layers of configuration 5
    ("i4", 16384, 4096),         # the last layer of configuration 3, transposed roles
    ("i8", 2048, 4096),
    ("i8", 2061, 2064), ("i4", 4099, 2080), ("i2", 1035, 4160),      # N not a multiple of 16, K not a whole scale chunk
    ("i8", 60000, 80), ("i4", 30000, 160), ("i2", 9000, 320),        # K just above one 64-byte row segment
    ("i8", 1500, 6144), ("i4", 3000, 10240), ("i2", 2000, 20480),    # several LDS stages of digit planes
])
@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_integer_matrix_core_gemv_one_to_four_samples(S, fmt, N, K, n):
    """Integer weights at one to four samples on layers large enough for the self-quantising INT8 matrix-core
    GEMV (Network.c:229-245 is what it replaces): the kernel that runs is asserted by name, the outputs are
    compared with FP64 on the decoded arrays at the vector path's 1e-4."""
    net, W, b = _decoded_layer(S, fmt, N, K, seed=N + 5 * K)
    assert _kernel_of(S, net, n) == "sp_gemv_i8mfma"
    X = (np.random.default_rng(n + K).standard_normal((n, K)) * 1.7).astype(F32)
    X[0, ::7] *= 1e-3                                   # a wide spread of magnitudes inside one scale chunk
    X[-1, K // 2:] *= 300.0                             # and chunks of very different scale
    pre = X.astype(np.float64) @ W.T + b
    want = np.where(pre > 0, pre, 0.01 * pre)
    got = net.forward(X)
    assert rel_max_abs(got, want) <= TOL_VEC
    for i in range(n):                                   # every sample on its own scale
        assert rel_max_abs(got[i], want[i]) <= TOL_VEC, i
    net.destroy()


@pytest.mark.parametrize("fmt,N,K", [("i8", 4096, 2048), ("i2", 8192, 2048), ("i8", 1030, 1040), ("i2", 2500, 832)])
@pytest.mark.parametrize("n", [5, 8, 9, 13, 17, 24, 25, 33, 48, 49, 64])
def test_integer_matrix_core_gemv_forced_up_to_64_samples(S, fmt, N, K, n):
    """SPHIP_FORCE_GEMV keeps the two-launch form (quantise kernel + planes from memory) reachable up to 64 samples:
    its 2 .. 16 tile instantiations for INT8 and INT2 (INT4: test_vector_path_batch_sizes), 1e-4 against FP64."""
    net, W, b = _decoded_layer(S, fmt, N, K, seed=N + K)
    # INT2 planes of more than 51 samples exceed the LDS of one fetch group: the vector kernel takes those
    fits = fmt != "i2" or n <= 51
    vector = "sp_gemv_words" if K * {"i8": 8, "i2": 2}[fmt] <= 2048 else "sp_gemv"      # rows of at most 16 chunks: a word per lane
    assert _kernel_of(S, net, n, S.SPHIP_FORCE_GEMV) == ("sp_gemv_i8mfma" if fits else vector)
    X = np.random.default_rng(n).standard_normal((n, K)).astype(F32)
    pre = X.astype(np.float64) @ W.T + b
    want = np.where(pre > 0, pre, 0.01 * pre)
    got = net.forward(X, S.SPHIP_FORCE_GEMV)
    assert rel_max_abs(got, want) <= TOL_VEC
    net.destroy()


@pytest.mark.parametrize("fmt,N,K,n,kernel", [
    # either side of where small layers keep the vector kernel: 4 M code-sample products (INT2: 2 M)
    ("i8", 2048, 2048, 1, "sp_gemv"), ("i8", 2064, 2048, 1, "sp_gemv_i8mfma"),
    ("i4", 1024, 1024, 4, "sp_gemv"), ("i4", 1040, 1024, 4, "sp_gemv_i8mfma"),
    ("i2", 1024, 2048, 1, "sp_gemv"), ("i2", 1040, 2048, 1, "sp_gemv_i8mfma"),
    ("i2", 1024, 1024, 2, "sp_gemv_words"), ("i2", 1024, 1024, 3, "sp_gemv_i8mfma"),
    ("i2", 301, 250, 2, "sp_gemv_generic"),            # rows that are not whole 32-bit words
    # rows of whole words: a word per lane when they are not whole 16-byte units, or at most 16 of them
    ("i4", 4096, 2056, 2, "sp_gemv_words"), ("i2", 256, 256, 1, "sp_gemv_words"),
    ("i4", 300, 264, 3, "sp_gemv_words"), ("i8", 100, 36, 4, "sp_gemv_words"), ("i2", 70, 16, 2, "sp_gemv_words"),
    ("i4", 512, 784, 1, "sp_gemv_words"), ("i8", 33, 256, 4, "sp_gemv_words"),
    # at most 64 outputs: a workgroup per row once a row has 256 words, whatever the layer's size
    ("i4", 10, 8192, 4, "sp_gemv_words"), ("i4", 64, 16384, 3, "sp_gemv_words"), ("i2", 10, 8192, 2, "sp_gemv_words"),
    ("i8", 7, 4100, 4, "sp_gemv_words"), ("i8", 64, 1024, 1, "sp_gemv_words"), ("i2", 65, 16384, 4, "sp_gemv_i8mfma"),
    # ... 16-bit weights too (two values per word)
    ("f16", 10, 8192, 4, "sp_gemv_words"), ("bf16", 64, 1000, 2, "sp_gemv_words"), ("bf16", 3, 514, 1, "sp_gemv_words"),
    ("f16", 65, 8192, 4, "sp_gemv"), ("bf16", 10, 500, 3, "sp_gemv_generic"),
])
def test_small_integer_layers_keep_the_vector_kernel(S, fmt, N, K, n, kernel):
    net, W, b = _decoded_layer(S, fmt, N, K, seed=3 * N + K + n)
    assert _kernel_of(S, net, n) == kernel
    X = np.random.default_rng(n + 2).standard_normal((n, K)).astype(F32)
    pre = X.astype(np.float64) @ W.T + b
    want = np.where(pre > 0, pre, 0.01 * pre)
    assert rel_max_abs(net.forward(X), want) <= TOL_VEC
    net.destroy()


def test_config5_int2_full_size_one_to_four_samples(S, O):
    """Configuration 5 at its real layer sizes (2048 -> 4 x 8192 -> 1000 softmax, INT2 through the serializer,
    inputs U[-1,1]) at one to four samples, and one sample through the public forward(), against the oracle."""
    topo = [2048, 8192, 8192, 8192, 8192, 1000]
    acts = ["sigmoid", "relu", "relu", "tanh", "softmax"]
    src = make_oracle_net(O, topo, acts, seed=55)
    _, ref, net = quantized_pair(O, S, src, "i2")
    h = S.lib().spingalett_hip_handle(net)
    X = (np.random.default_rng(56).random((4, 2048), dtype=F32) * 2 - 1)
    want = ref.forward_batch_f64(X)
    for n in (1, 2, 3, 4):
        got = S.forward_batch(net, X[:n])
        names = [S.lib().sphip_layer_kernel_name(h, l, n, 0).decode() for l in range(1, 6)]
        assert names[:4] == ["sp_gemv_i8mfma"] * 4, names
        assert rel_max_abs(got, want[:n]) <= TOL_VEC, n
        assert np.allclose(got.sum(axis=1), 1.0, atol=1e-5)
    y = S.forward(net, X[2])
    assert rel_max_abs(y, want[2]) <= TOL_VEC
    S.free_network(net)


def _same_nonfinite(got, want):
    """NaNs in the same places, infinities in the same places with the same sign."""
    return (np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
            and np.array_equal(np.isneginf(got), np.isneginf(want)))


@pytest.mark.parametrize("fmt,N,K,n,flags,kernel", [
    ("i8", 2064, 2048, 1, 0, "sp_gemv_i8mfma"), ("i4", 4099, 2080, 3, 0, "sp_gemv_i8mfma"),
    ("i2", 8192, 8192, 4, 0, "sp_gemv_i8mfma"), ("i8", 1030, 1040, 17, 16, "sp_gemv_i8mfma"),
    ("i4", 512, 1024, 2, 0, "sp_gemv"), ("bf16", 600, 512, 4, 0, "sp_gemv"), ("i2", 301, 250, 3, 0, "sp_gemv_generic"),
    ("i4", 16384, 2048, 8, 0, "sp_skinny16_kw"), ("i8", 2100, 2064, 48, 0, "sp_skinny16"),
    ("f16", 1500, 4096, 60, 0, "sp_skinny16"), ("bf16", 10, 1000, 300, 0, "sp_skinny16_kw_head"),
    ("f16", 1500, 1000, 77, 0, "sp_gemm16_small"), ("i2", 600, 1000, 200, 0, "sp_gemm16_small"),
    ("bf16", 2048, 4096, 600, 0, "sp_gemm16_big"), ("i2", 2048, 4096, 1000, 0, "sp_gemm16_big"),
    ("bf16", 2048, 2048, 600, 0, "sp_gemm16"),
    ("i8", 1000, 528, 700, 0, "sp_gemm16"), ("i4", 257, 100, 513, 0, "sp_gemm16"),
])
def test_infinities_and_nans_travel_like_in_fp32(S, fmt, N, K, n, flags, kernel):
    """The reference's FP32 products propagate non-finite inputs (cblas_sgemv / the FP32 dot product,
    Network.c:229-245; cblas_sgemm, Training.c:327-333): an infinite input gives +-inf where its weight is
    positive or negative and NaN where it is zero or where infinities of both signs meet, a NaN input gives
    NaN everywhere in its sample, and other samples are untouched.  Every kernel family, one layer, against
    FP64 on the decoded arrays (finite outputs at the path's tolerance)."""
    net, W, b = _decoded_layer(S, fmt, N, K, seed=N + K + n)
    assert _kernel_of(S, net, n, flags) == kernel
    rng = np.random.default_rng(n + N)
    X = rng.standard_normal((n, K)).astype(F32)
    X[0, K // 3] = np.inf                                  # one infinity
    if n > 1:
        X[1, 5] = np.nan                                   # one NaN
    if n > 2:
        X[2, 1], X[2, K - 1] = np.inf, -np.inf             # both signs in one sample: NaN unless a weight is zero ...
    if n > 3:
        X[3, K // 2] = -np.inf
        X[3, K // 2 + 1] = -np.inf                         # ... two of one sign
    with np.errstate(invalid="ignore", over="ignore"):
        pre = np.zeros((n, N))
        for i in range(n):                                 # row by row: products with zero weights must give NaN
            pre[i] = (W * X[i].astype(np.float64)).sum(axis=1) + b
        want = np.where(pre > 0, pre, 0.01 * pre)
    got = net.forward(X, flags)
    assert _same_nonfinite(got, want)
    fin = np.isfinite(want)
    assert fin[4:].all() and (n < 2 or not fin[1].any())
    tol = TOL_VEC if kernel.startswith("sp_gemv") else (4e-3 if fmt == "bf16" else 1e-3)
    if fin.any():
        assert np.max(np.abs(got[fin] - want[fin])) <= tol * np.max(np.abs(want[fin]))
    net.destroy()


@pytest.mark.parametrize("fmt,n", [("i8", 1), ("i8", 64), ("i8", 600), ("bf16", 600), ("f32", 100)])
def test_nonfinite_inputs_through_a_softmax_net(S, O, fmt, n):
    """Whole nets against the oracle: the sample that carries a NaN or an infinity shows the oracle's pattern after
    ReLU (NaN -> 0, Activation.c:26) and softmax (Activation.c:5-21: no normalisation when the sum is NaN), the others
    are unaffected."""
    src = make_oracle_net(O, [2048, 2064, 10], ["leaky_relu", "softmax"], seed=91)
    _, ref, net = quantized_pair(O, S, src, fmt)
    X = np.random.default_rng(92).standard_normal((n, 2048)).astype(F32)
    X[0, 7] = np.inf
    if n > 1:
        X[n - 1, 100] = np.nan
    with np.errstate(invalid="ignore", over="ignore"):
        want = ref.forward_batch(X)
    got = S.forward_batch(net, X)
    assert _same_nonfinite(got, want)
    fin = np.isfinite(want).all(axis=1)
    if fin.any():
        assert rel_max_abs(got[fin], want[fin]) <= tol_for(fmt, n)
    S.free_network(net)


def test_fp16_activation_range_saturates(S, O):
    """Matrix-core paths carry FP16 activations between layers: a finite hidden activation beyond +-65504 becomes
    +-65504 (documented deviation: the reference keeps FP32 activations, Training.c:327-343), so the outputs equal
    the oracle's on activations clamped to that range; BF16 weights with BF16 activations selected (FP32's range) and
    the vector path at up to four samples do not saturate."""
    src = make_oracle_net(O, [64, 96, 8], ["none", "none"], seed=93, bias_std=0.0)
    src.W(0)[:] *= 4000.0
    X = np.random.default_rng(94).standard_normal((40, 64)).astype(F32) * 30
    for fmt in ("i8", "bf16"):
        _, ref, net = quantized_pair(O, S, src, fmt)
        hidden = X.astype(np.float64) @ ref.W(0).astype(np.float64).T + ref.b(0)
        assert np.abs(hidden).max() > 3 * 65504
        full = hidden @ ref.W(1).astype(np.float64).T + ref.b(1)
        clamped = np.clip(hidden, -65504, 65504) @ ref.W(1).astype(np.float64).T + ref.b(1)
        got = S.forward_batch(net, X)
        assert np.isfinite(got).all()
        assert rel_max_abs(got, clamped) <= TOL_MFMA
        if fmt == "bf16":
            S.lib().spingalett_set_bf16_activations(1)
            try:
                wide_range = S.forward_batch(net, X)
            finally:
                S.lib().spingalett_set_bf16_activations(0)
            assert rel_max_abs(wide_range, full) <= TOL_MFMA
        assert rel_max_abs(S.forward_batch(net, X[:4]), full[:4]) <= TOL_VEC
        S.free_network(net)


def _random_shapes(count, seed):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        fmt = ["i8", "i4", "i2", "bf16", "f16"][int(rng.integers(0, 5))]
        N = int(rng.choice([1, 3, 8, 10, 31, 64, 65, 100, 257, 640, 1500]))
        K = int(rng.choice([8, 24, 64, 136, 256, 520, 1024, 2056, 4096]))
        n = int(rng.choice([5, 6, 8, 9, 16, 31, 33, 64, 65, 100, 128, 129, 200, 256, 257, 400]))
        out.append((fmt, N, K, n))
    return out


@pytest.mark.parametrize("fmt,N,K,n", _random_shapes(48, seed=2024))
def test_seeded_random_layer_shapes(S, fmt, N, K, n):
    """Shapes drawn around every boundary of the planner (8 / 64 / 128 / 256 samples, 8 / 64 outputs, K below and
    across chunk sizes, rows that are and are not whole 16-byte units), one layer each, against FP64."""
    net, W, b = _decoded_layer(S, fmt, N, K, seed=N * 7 + K + n)
    X = np.random.default_rng(n + K).standard_normal((n, K)).astype(F32)
    pre = X.astype(np.float64) @ W.T + b
    want = np.where(pre > 0, pre, 0.01 * pre)
    got = net.forward(X)
    assert rel_max_abs(got, want) <= (8e-3 if fmt == "bf16" else 2e-3)
    net.destroy()


def test_large_host_input_goes_up_in_chunks(S):
    """Host inputs of 10 MB and more are uploaded through a ring of pinned chunks, of 0.5 to 4.5 MB up to the eighth megabyte and of 8
    from there, filled by several threads, and from 16 MB on the layers of the rows that have landed run beside the rest; sizes
    that are no multiple of a chunk, twice in a row (the ring is reused), against FP64 on every row."""
    net, W, b = _decoded_layer(S, "bf16", 16, 1030, seed=77)
    for n in (5000, 4200):                                  # 20.6 MB and 17.3 MB
        X = np.random.default_rng(n).standard_normal((n, 1030)).astype(F32)
        pre = X.astype(np.float64) @ W.T + b
        want = np.where(pre > 0, pre, 0.01 * pre)
        got = net.forward(X)
        assert rel_max_abs(got, want) <= 4e-3
        bad = np.abs(got - want).max(axis=1) > 4e-3 * np.abs(want).max()
        assert not bad.any(), np.nonzero(bad)[0][:10]
    net.destroy()


def test_batch_permutation_and_row_independence(S, O):
    """Samples are independent: permuting the batch permutes the outputs bit for bit."""
    src = make_oracle_net(O, [256, 384, 64], ["foo52", "softmax"], seed=31)
    _, ref, net = quantized_pair(O, S, src, "i8")
    rng = np.random.default_rng(32)
    X = rng.standard_normal((333, 256)).astype(F32)
    perm = rng.permutation(333)
    a = S.forward_batch(net, X)
    b = S.forward_batch(net, X[perm])
    assert np.array_equal(a[perm], b)
    S.free_network(net)


@pytest.mark.parametrize("fmt,topo,acts,n", [
    # 16-bit activation buffers of more than 128 MiB: the batch runs as equal blocks of rows, all layers per block
    ("i2", [64, 8192, 1000], ["relu", "softmax"], 9000),          # 3 blocks of 3072 rows (the last one smaller: 2856)
    ("bf16", [32, 16384, 24], ["tanh", "none"], 4500),            # 3 blocks of 1536 rows, ragged remainder 1428
])
def test_large_batches_run_in_blocks_of_rows(S, fmt, topo, acts, n):
    """A batch cut into blocks of rows gives the whole batch's outputs (rows are independent; Training.c:313-345 has
    one sgemm over all rows): against SPHIP_WHOLE_BATCH within FP32 rounding (the K splits of a block may differ from
    those of the whole batch), and bit for bit against the blocks run as separate calls."""
    act = {"relu": S.ACT_RELU, "softmax": S.ACT_SOFTMAX, "tanh": S.ACT_TANH, "none": S.ACT_NONE}
    prec = {"i2": S.PRECISION_INT2, "bf16": S.PRECISION_BFLOAT16}[fmt]
    rng = np.random.default_rng(n)
    net = S.DeviceNet(topo, [act[a] for a in acts], prec)
    for l in range(len(topo) - 1):
        K, N = topo[l], topo[l + 1]
        if fmt == "bf16":
            w = (rng.standard_normal(N * K) * np.sqrt(1.0 / K)).astype(F32)
            net.upload(l, 0, (w.view(np.uint32) >> 16).astype(np.uint16))
            net.upload(l, 1, ((rng.standard_normal(N) * 0.1).astype(F32).view(np.uint32) >> 16).astype(np.uint16))
        else:
            net.upload(l, 0, rng.integers(0, 256, size=(N * K * 2 + 7) // 8, dtype=np.uint8), 0.5 / np.sqrt(K))
            net.upload(l, 1, rng.integers(0, 256, size=(N * 2 + 7) // 8, dtype=np.uint8), 0.1)
    X = rng.standard_normal((n, topo[0])).astype(F32)
    whole = net.forward(X, S.SPHIP_WHOLE_BATCH)
    blocks = net.forward(X)
    assert np.isfinite(whole).all()
    assert rel_max_abs(blocks, whole) <= 1e-5
    per_row = 2 * max(topo)
    rows = (64 << 20) // per_row // 256 * 256
    nb = -(-n // rows)
    rows = -(-(-(-n // nb)) // 256) * 256
    assert rows < n
    parts = np.concatenate([net.forward(X[r0:r0 + rows], S.SPHIP_WHOLE_BATCH) for r0 in range(0, n, rows)])
    assert np.array_equal(blocks.view(np.uint32), parts.view(np.uint32))
    net.destroy()


def test_integer_gemv_with_a_very_long_row_falls_back_to_the_vector_kernel(S):
    """A K so long that the self-quantising integer GEMV's two digit-plane buffers plus its scale records exceed the
    LDS of a compute unit (2 M columns at four samples: 64 KB of scale records next to two 48 KB plane buffers): the layer must route to the vector kernel, not fail at
    launch; and it must still compute the product."""
    K, N, n = 1 << 21, 80, 4                            # (more than 64 outputs: thinner layers never take that kernel)
    rng = np.random.default_rng(5)
    net = S.DeviceNet([K, N], [S.ACT_NONE], S.PRECISION_INT8)
    codes = rng.integers(-127, 128, size=N * K, dtype=np.int8)
    net.upload(0, 0, codes.view(np.uint8), 0.25)
    net.upload(0, 1, np.zeros(N, np.uint8), 0.0)
    assert _kernel_of(S, net, n) == "sp_gemv"
    assert _kernel_of(S, net, 1) in ("sp_gemv", "sp_gemv_i8mfma")
    X = rng.standard_normal((n, K)).astype(F32)
    want = X.astype(np.float64) @ (codes.reshape(N, K).astype(np.float64) * (0.25 / 127.0)).T
    assert rel_max_abs(net.forward(X), want) <= TOL_VEC
    net.destroy()


def test_device_resident_entry_and_argument_checks(S, O):
    src = make_oracle_net(O, [128, 64, 8], ["relu", "none"], seed=41)
    _, ref, net = quantized_pair(O, S, src, "bf16")
    X = np.random.default_rng(42).standard_normal((100, 128)).astype(F32)
    d_x = S.DeviceBuffer.from_numpy(X)
    d_y = S.DeviceBuffer(100 * 8 * 4)
    assert S.lib().spingalett_forward_batch_device(net, d_x.ptr, 100, d_y.ptr) == 0
    assert S.lib().spingalett_hip_synchronize() == 0
    got = d_y.to_numpy(F32, (100, 8))
    assert np.array_equal(got, S.forward_batch(net, X))
    assert S.lib().spingalett_forward_batch_device(net, None, 100, d_y.ptr) == 1
    assert S.last_error()[0] == S.SPINGALETT_ERR_INVALID
    S.clear_error()
    assert S.lib().spingalett_forward_batch_device(None, d_x.ptr, 100, d_y.ptr) == 1
    S.clear_error()
    assert S.lib().spingalett_forward_batch(net, None, 3, got.ctypes.data) is None
    assert S.last_error()[0] == 0                                   # silent, like forward()
    S.free_network(net)


def test_zero_scale_arrays_forward_to_bias_only(S, O):
    """An all-zero weight matrix is written with scale 0 and decodes to zeros
    (Serialize.c:231-236): the layer outputs act(bias)."""
    src = make_oracle_net(O, [32, 16], ["none"], seed=51)
    src.W(0)[:] = 0
    _, ref, net = quantized_pair(O, S, src, "i4")
    X = np.random.default_rng(52).standard_normal((3, 32)).astype(F32)
    got = S.forward_batch(net, X)
    assert np.allclose(got, np.broadcast_to(ref.b(0), (3, 16)), rtol=1e-6, atol=0)
    S.free_network(net)


def test_full_size_layer_unit_vector_probe(S):
    """16384 x 16384 INT4 (the largest layer of config 3, 128 MiB of codes):
    x = e_k reads column k of W exactly, and f(2x) = 2 f(x) for a bias-free
    linear layer — properties that hold at any size."""
    K = N = 16384
    rng = np.random.default_rng(61)
    codes = rng.integers(0, 256, size=N * K // 2, dtype=np.uint8)
    mx = 7.0                                                         # scale max/7 = 1: outputs are the integer codes
    net = S.DeviceNet([K, N], [S.ACT_NONE], S.PRECISION_INT4)
    net.upload(0, 0, codes, mx)
    net.upload(0, 1, np.zeros(N // 2, np.uint8), 0.0)
    ks = [0, 1, 7, 4095, 8192, 16383]
    X = np.zeros((len(ks), K), F32)
    for i, k in enumerate(ks):
        X[i, k] = 1.0
    got = net.forward(X)
    rows = codes.reshape(N, K // 2)
    for i, k in enumerate(ks):
        nib = (rows[:, k // 2] >> ((k & 1) * 4)) & 15
        q = nib.astype(np.int32) - np.where(nib & 8, 16, 0)
        assert np.array_equal(got[i], q.astype(F32)), k
    x = rng.standard_normal((1, K)).astype(F32)
    y1, y2 = net.forward(x), net.forward(2 * x)
    assert np.array_equal(2 * y1, y2)
    # and the matrix-core path reads the same codes: one-hot rows are exact in bf16
    Xg = np.zeros((65, K), F32)
    Xg[np.arange(65), np.arange(65) * 251] = 1.0
    gg = net.forward(Xg)
    for i in (0, 17, 64):
        k = i * 251
        nib = (rows[:, k // 2] >> ((k & 1) * 4)) & 15
        q = nib.astype(np.int32) - np.where(nib & 8, 16, 0)
        assert np.array_equal(gg[i], q.astype(F32)), k
    net.destroy()


@pytest.mark.parametrize("fmt,acts,loss,n", [
    ("i8", ["relu", "relu", "softmax"], 1, 300),         # classifier: cross-entropy on softmax outputs
    ("bf16", ["tanh", "sigmoid"], 1, 77),                # sigmoid output layer: binary cross-entropy
    ("i4", ["leaky_relu", "none"], 0, 3),                # squared error, vector path
    ("f32", ["relu", "softmax"], 1, 1000),
])
def test_evaluate_batch_matches_oracle(S, O, fmt, acts, loss, n):
    """spingalett_evaluate_batch = forward + compute_sample_loss (SIMD.c:522-552) summed over the
    batch (Training.c:421-435) + per-sample argmax, all on the device.  The loss is compared with the
    oracle's loss of the library's own outputs (so that only the evaluation step is under test), the
    predictions with the argmax of those outputs."""
    topo = [64, 128, 96, 10][:len(acts) + 1] if len(acts) == 3 else [48, 80, 12]
    src = make_oracle_net(O, topo, acts, seed=71, loss=loss)
    _, ref, net = quantized_pair(O, S, src, fmt)
    assert net.contents.loss_func == loss
    rng = np.random.default_rng(72)
    X = rng.standard_normal((n, topo[0])).astype(F32)
    labels = rng.integers(0, topo[-1], n)
    T = np.eye(topo[-1], dtype=F32)[labels]
    if loss == 0:
        T = rng.standard_normal((n, topo[-1])).astype(F32)
    Y = S.forward_batch(net, X)
    total, pred, correct = S.evaluate_batch(net, X, T)
    want = O.batch_loss(Y, T, loss, O.ACT[acts[-1]])
    assert abs(total - want) <= 2e-5 * abs(want)
    assert np.array_equal(pred, O.argmax_rows(Y))
    assert correct == int((O.argmax_rows(Y) == O.argmax_rows(T)).sum())
    # and end to end against the oracle's own forward, at the forward's tolerance
    want_ref = O.batch_loss(ref.forward_batch(X), T, loss, O.ACT[acts[-1]])
    assert abs(total - want_ref) <= (1e-3 if fmt == "f32" or n <= 4 else 3e-2) * abs(want_ref)
    S.free_network(net)


def test_evaluate_batch_argument_checks(S, O):
    src = make_oracle_net(O, [16, 8], ["softmax"], seed=73, loss=1)
    _, _, net = quantized_pair(O, S, src, "i8")
    X = np.zeros((2, 16), F32)
    T = np.zeros((2, 8), F32)
    loss = C.c_float(0)
    assert S.lib().spingalett_evaluate_batch(net, None, T.ctypes.data, 2, C.byref(loss), None, None) == 1
    assert S.last_error()[0] == S.SPINGALETT_ERR_INVALID
    S.clear_error()
    assert S.lib().spingalett_evaluate_batch(net, X.ctypes.data, T.ctypes.data, 0, C.byref(loss), None, None) == 1
    S.clear_error()
    assert S.lib().spingalett_evaluate_batch(net, X.ctypes.data, T.ctypes.data, 2, C.byref(loss), None, None) == 0
    assert loss.value == pytest.approx(0.0)                      # all-zero targets: nothing to add
    S.free_network(net)


@pytest.mark.parametrize("activations", ["f16", "bf16"])
def test_full_size_gemm_layer_properties(S, activations):
    """8192 x 8192 BF16 at batch 8192 (one layer of config 4, the tiled GEMM at its benchmark shape), with the
    default FP16 activations and with BF16 activations selected: one-hot rows read columns of W exactly, duplicated
    rows give identical outputs wherever they sit in the batch, and random rows agree with FP64 dot products of the
    weights and the inputs rounded to the activation type."""
    flags = S.SPHIP_BF16_ACTIVATIONS if activations == "bf16" else 0
    K = N = n = 8192
    rng = np.random.default_rng(81)
    w = (rng.standard_normal(N * K, dtype=F32) * F32(0.02))
    codes = (w.view(np.uint32) >> 16).astype(np.uint16)
    net = S.DeviceNet([K, N], [S.ACT_NONE], S.PRECISION_BFLOAT16)
    net.upload(0, 0, codes)
    net.upload(0, 1, np.zeros(N, np.uint16))
    Wd = (codes.astype(np.uint32) << 16).view(F32).reshape(N, K)
    X = rng.standard_normal((n, K), dtype=F32)
    hot = [0, 1, 255, 256, 4097, 8191]
    for i, r in enumerate(hot):
        X[r] = 0
        X[r, (r * 37 + 5) % K] = 1.0
    X[7000] = X[3]                                                   # duplicates in different tiles
    X[8190] = X[3]
    Y = net.forward(X, flags)
    for r in hot:
        assert np.array_equal(Y[r], Wd[:, (r * 37 + 5) % K]), r
    assert np.array_equal(Y[7000], Y[3]) and np.array_equal(Y[8190], Y[3])
    for r in (3, 1234, 8189):
        if activations == "bf16":
            xb = ((X[r].view(np.uint32) + 0x7FFF + ((X[r].view(np.uint32) >> 16) & 1)) & 0xFFFF0000).view(F32)   # BF16 RNE
        else:
            xb = X[r].astype(np.float16).astype(F32)
        want = Wd.astype(np.float64) @ xb.astype(np.float64)
        assert rel_max_abs(Y[r], want) <= 1e-4, r                    # products exact, FP32 accumulation over 8192 terms
    net.destroy()


def test_full_batch_int2_first_layer_properties(S):
    """2048 -> 8192 INT2 at batch 65536 (first layer of config 5 at the top of its sweep): every row of the
    batch is one of 97 distinct inputs; equal inputs must give bit-identical outputs in all 65536 positions,
    and the distinct ones agree with FP64 on the decoded codes."""
    K, N, n = 2048, 8192, 65536
    rng = np.random.default_rng(82)
    net = S.DeviceNet([K, N], [S.ACT_TANH], S.PRECISION_INT2)
    net.upload(0, 0, rng.integers(0, 256, size=N * K // 4, dtype=np.uint8), 0.03)
    net.upload(0, 1, rng.integers(0, 256, size=N // 4, dtype=np.uint8), 0.2)
    W = net.decode(0, 0).astype(np.float64).reshape(N, K)
    b = net.decode(0, 1).astype(np.float64)
    base = (rng.random((97, K), dtype=F32) * 2 - 1)
    idx = rng.integers(0, 97, n)
    Y = net.forward(base[idx])
    first = {int(v): int(np.nonzero(idx == v)[0][0]) for v in range(97)}
    ref_rows = np.stack([Y[first[int(v)]] for v in idx[::997]])
    assert np.array_equal(Y[::997], ref_rows)
    assert np.array_equal(Y[np.nonzero(idx == 5)[0]], np.broadcast_to(Y[first[5]], (int((idx == 5).sum()), N)))
    want = np.tanh(base[:8].astype(np.float16).astype(np.float64) @ W.T + b)
    got = np.stack([Y[first[v]] for v in range(8)])
    assert rel_max_abs(got, want) <= 2e-3
    net.destroy()


@pytest.mark.parametrize("fmt", ["f16", "bf16", "i8", "i4", "i2"])
@pytest.mark.parametrize("topo,acts", [
    ([777, 1030, 515, 33], ["sigmoid", "tanh", "softmax"]),       # every layer padded (activation(0) of the padding is 0.5)
    ([33, 7, 1, 70, 5], ["foo52", "sigmoid", "relu", "none"]),    # widths below one unit
    ([130, 1101, 90, 9], ["softmax", "relu", "none"]),            # a hidden softmax keeps its width: the layer behind it is ragged
    ([512, 1000, 640, 11], ["relu", "sigmoid", "softmax"]),       # whole words, padded for its half a million weights
])
def test_padded_widths_leave_the_outputs_alone(S, O, fmt, topo, acts):
    """Hidden widths and inputs whose weight rows are not whole 16-byte units run padded with zero weights: outputs
    against the float64 forward at one to four samples (vector kernels, FP32-grade) and on both sides of the small,
    streaming and tiled kernels' ranges, plain and split; every activation of a single forward; a clone."""
    src = make_oracle_net(O, topo, acts, seed=sum(topo), bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, fmt)
    X = np.random.default_rng(1).standard_normal((1500, topo[0])).astype(F32)
    want = ref.forward_batch_f64(X)
    for n in (1, 3, 4, 5, 33, 260, 1500):
        assert rel_max_abs(S.forward_batch(net, X[:n]), want[:n]) <= (TOL_VEC if n <= 4 else TOL_MFMA), n
    assert S.lib().spingalett_set_net_activations(net, S.NET_ACTIVATIONS_SPLIT) == 0
    for n in (5, 260):
        assert rel_max_abs(S.forward_batch(net, X[:n]), want[:n]) <= 2e-5, n
    assert rel_max_abs(S.forward(net, X[2]), want[2]) <= TOL_VEC
    h = S.lib().spingalett_hip_handle(net)
    d = S.DeviceNet(topo, [O.ACT[a] for a in acts], O.PREC[fmt], handle=h)
    d.owned = False
    twin = d.clone()
    assert np.array_equal(twin.forward(X[:300]), d.forward(X[:300]))
    twin.destroy()
    S.free_network(net)


@pytest.mark.parametrize("fmt", ["f16", "bf16", "i8", "i4", "i2"])
@pytest.mark.parametrize("act", ["tanh", "sigmoid", "leaky_relu", "foo52"])
@pytest.mark.parametrize("topo,sizes", [
    ([777, 1030, 33], (1, 3, 5, 33, 260, 1500)),                   # vector, small, streaming and single-stage kernels
    ([200, 37, 90, 9], (2, 64, 700)),                              # widths below one unit, thin layers
    ([640, 4500, 2300, 10], (4, 8, 130, 2100)),                    # large tiles, K splits, a padded last column of tiles
])
def test_padded_widths_keep_infinities_and_nans_where_they_are(S, fmt, act, topo, sizes):
    """A padded neuron sees the infinite input too: 0 x inf must not reach the outputs.  Single infinities of either sign,
    and NaNs, in samples of their own, against FP64 on the decoded arrays.  (A zero code of a real neuron makes a NaN of an
    infinity, as in the reference's FP32 sums: integer weights are drawn without zeros.)"""
    rng = np.random.default_rng(len(topo) + topo[1])
    levels = {"i8": 127, "i4": 7, "i2": 1}.get(fmt)
    W, b = [], []
    for l in range(len(topo) - 1):
        w = rng.standard_normal((topo[l + 1], topo[l])) / np.sqrt(topo[l])
        if levels:
            top = np.abs(w).max()
            q = np.rint(w / top * levels)
            w = np.where(q == 0, np.where(w < 0, -1, 1), q) * (top / levels)
            w.ravel()[0] = top                                     # the scale that the writer finds again
        W.append(w.astype(F32)); b.append((rng.standard_normal(topo[l + 1]) * 0.1).astype(F32))
    acts = [act] * (len(topo) - 2) + ["none"]
    src = S.new_spingalett()
    S.layer(src, topo[0])
    for l, a in enumerate(acts):
        S.layer(src, topo[l + 1], {"tanh": S.ACT_TANH, "sigmoid": S.ACT_SIGMOID, "leaky_relu": S.ACT_LEAKY_RELU,
                                   "foo52": S.ACT_FOO52, "none": S.ACT_NONE}[a], S.WEIGHT_INITIALIZATION_NONE)
        S.weights_view(src, l)[:] = W[l]
        S.biases_view(src, l)[:] = b[l]
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "net.nn")
        prec = {"f16": S.PRECISION_FP16, "bf16": S.PRECISION_BFLOAT16, "i8": S.PRECISION_INT8, "i4": S.PRECISION_INT4,
                "i2": S.PRECISION_INT2}[fmt]
        S.save_spingalett(src, path, prec, do_not_save_optimizer=True)
        net = S.load_spingalett(path)
    S.free_network(src)
    D = [(S.weights_view(net, l).astype(np.float64), S.biases_view(net, l).astype(np.float64)) for l in range(len(acts))]
    f = {"tanh": np.tanh, "sigmoid": lambda z: 1 / (1 + np.exp(-z)), "leaky_relu": lambda z: np.where(z > 0, z, 0.01 * z),
         "foo52": lambda z: np.where(z > 1, 1 + 0.01 * (z - 1), np.where(z < 0, 0.01 * z, z)), "none": lambda z: z}
    X = rng.standard_normal((max(sizes), topo[0])).astype(F32)
    X[0, 5] = np.inf
    X[1::7, topo[0] - 1] = -np.inf
    X[2::7, 3] = np.nan
    with np.errstate(invalid="ignore", over="ignore"):
        a = X.astype(np.float64)
        for (w, c), name in zip(D, acts):
            a = f[name](a @ w.T + c)
    for n in sizes:
        for split in ([False, True] if n > 4 else [False]):
            assert S.lib().spingalett_set_net_activations(net, S.NET_ACTIVATIONS_SPLIT if split else S.NET_ACTIVATIONS_DEFAULT) == 0
            got = S.forward_batch(net, X[:n])
            assert _same_nonfinite(got, a[:n]), (n, split)
            fin = np.isfinite(a[:n])
            assert not fin.any() or rel_max_abs(got[fin], a[:n][fin]) <= (TOL_VEC if n <= 4 else TOL_MFMA), (n, split)
    S.free_network(net)


@pytest.mark.parametrize("N,K,n,tile", [
    (16, 16, 5, 16), (17, 33, 16, 16), (1, 3, 9, 16), (512, 784, 64, 16), (300, 2000, 33, 16),   # 16 x 16 tiles: whole and partial steps, few rows
    (233, 1038, 64, 16), (65, 1, 40, 16), (90, 1023, 100, 16), (31, 1026, 17, 16),               # ... rows that start anywhere
    (1000, 512, 128, 16), (1024, 1024, 128, 16), (65, 1024, 1365, 32),                           # ... at their bound, and 32 x 32 tiles beyond it
    (500, 1000, 512, 32), (512, 1020, 1024, 32),
])
@pytest.mark.parametrize("act", ["tanh", "softmax"])
def test_small_fp32_layers_run_in_one_launch(S, O, N, K, n, tile, act):
    """Small FP32 layers whose workgroups split K among their waves; a softmax of at most a tile's width in the same
    launch, wider ones by the row kernel.  1e-4 against the float64 forward, like every FP32 path."""
    src = make_oracle_net(O, [K, N], [act], seed=N + K, bias_std=0.1)
    _, ref, net = quantized_pair(O, S, src, "f32")
    X = np.random.default_rng(n).standard_normal((n, K)).astype(F32)
    got = S.forward_batch(net, X)
    name = S.lib().sphip_layer_kernel_name(S.lib().spingalett_hip_handle(net), 1, n, 0).decode()
    S.free_network(net)
    assert rel_max_abs(got, ref.forward_batch_f64(X)) <= TOL_VEC
    if N > 64 or n > 8:
        assert name == ("sp_gemm32_small16" if tile == 16 else "sp_gemm32_small")


@pytest.mark.parametrize("nbytes", [(16 << 20) - 1, 16 << 20, (16 << 20) + 1, (17 << 20) + 17, (35 << 20) + 4])
def test_large_uploads_arrive_whole(S, nbytes):
    """Uploads through the ring of chunks, at and off its multiples and the helpers' pages, several in a row."""
    rng = np.random.default_rng(nbytes)
    dst = S.DeviceBuffer(nbytes + 4)
    for shift in (0, 4, 0):
        a = rng.integers(0, 256, nbytes, dtype=np.uint8)
        assert S.lib().sphip_memcpy_h2d(dst.ptr.value + shift, a.ctypes.data, nbytes) == 0
        assert np.array_equal(dst.to_numpy(np.uint8, nbytes + 4)[shift:shift + nbytes], a)


@pytest.mark.parametrize("nbytes", [(4 << 20) - 4, 4 << 20, (4 << 20) + 4, (11 << 19) + 4, (15 << 19) - 4, (35 << 20) + 4])
def test_large_downloads_arrive_whole(S, nbytes):
    """Downloads at, below and past the line of the ring of chunks and its borders: a net that hands out what it was given."""
    net = S.new_spingalett(S.LOSS_MSE)
    S.layer(net, 1)
    S.layer(net, 1, S.ACT_NONE, S.WEIGHT_INITIALIZATION_NONE)
    S.weights_view(net, 0)[:] = 1.0
    S.biases_view(net, 0)[:] = 0.0
    for seed in (nbytes, 1):
        X = np.random.default_rng(seed).standard_normal((nbytes // 4, 1)).astype(F32)
        assert np.array_equal(S.forward_batch(net, X), X)
    S.free_network(net)


class _Busy:
    """enqueue(): about 0.15 s of kernels."""

    def __init__(self, S):
        self.n = 16384
        self.net = S.DeviceNet([4096] * 4, [S.ACT_RELU] * 3, S.PRECISION_FP16)
        for l in range(3):
            self.net.upload(l, 0, np.zeros(4096 * 4096, np.uint16))
            self.net.upload(l, 1, np.zeros(4096, np.uint16))
        self.x, self.y = S.DeviceBuffer.from_numpy(np.zeros((self.n, 4096), F32)), S.DeviceBuffer(self.n * 4096 * 4)
        self.net.forward_device(self.x, self.n, self.y)
        S.synchronize()

    def enqueue(self):
        for _ in range(120):
            self.net.forward_device(self.x, self.n, self.y)


def test_nobody_spins_behind_a_busy_stream(S):
    """A large upload behind kernels: the threads that copy sleep until a chunk is free (the caller and three helpers looked for one
    all the time, four processors for as long as the kernels ran), and what arrives is whole."""
    busy = _Busy(S)
    a = np.random.default_rng(3).random(16 << 20, dtype=F32)
    dst = S.DeviceBuffer.from_numpy(a[::-1].copy())
    busy.enqueue()
    wall, cpu = time.perf_counter(), time.process_time()
    assert S.lib().sphip_memcpy_h2d(dst.ptr, a.ctypes.data, a.nbytes) == 0
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert wall >= 0.05                                             # (it did wait)
    assert cpu <= 2.0 * wall, (cpu, wall)
    assert np.array_equal(dst.to_numpy(F32, a.size), a)
    busy.net.destroy()


class _LargeBatch:
    """A net, a batch of 22.5 MB and what a step on it makes of the first layer's gradients."""

    def __init__(self, S):
        self.topo, n, rng = [256, 16, 10], 23000, np.random.default_rng(5)
        self.net = S.DeviceNet(self.topo, [S.ACT_TANH, S.ACT_SOFTMAX], S.PRECISION_FLOAT32)
        for l in range(2):
            self.net.upload(l, 0, (rng.standard_normal(self.topo[l] * self.topo[l + 1]) * 0.1).astype(F32))
            self.net.upload(l, 1, np.zeros(self.topo[l + 1], F32))
        self.net.train_begin()
        self.x, self.t = rng.standard_normal((n, 256)).astype(F32), np.zeros((n, 10), F32)
        self.t[np.arange(n), rng.integers(0, 10, n)] = 1.0
        self.args = S.SphipTrainArgs(S.OPTIMIZER_SGD, S.LOSS_CROSS_ENTROPY, 0.0, 0.0, 0.9, 0.9, 0.999, 1e-8, 0.0, 0.9, 0.999)
        self.step()
        self.want = self.gradients(S)

    def step(self, x=None):
        self.net.train_step(self.x if x is None else x, self.t, self.args)

    def gradients(self, S):
        return self.net.train_get(S.SPHIP_TRAIN_GW, 0).copy()


def test_large_batch_is_staged_behind_a_busy_stream(S):
    """A step's batch of 22.5 MB: the slots hold all of it, the call returns long before the kernels in front of it are done, and has
    read the caller's array by then."""
    busy, batch = _Busy(S), _LargeBatch(S)
    for _ in range(2):
        x = batch.x.copy()
        S.synchronize()
        busy.enqueue()
        start = time.perf_counter()
        batch.step(x)
        back = time.perf_counter() - start
        x[:] = 0.0
        S.synchronize()
        done = time.perf_counter() - start
        assert done >= 0.05 and back <= 0.5 * done, (back, done)
        assert np.array_equal(batch.gradients(S), batch.want)
    busy.net.destroy()


def test_upload_does_not_wait_for_another_threads_download(S):
    """Thread A waits for 8 MB of outputs behind a busy stream; a large batch of this thread's is staged meanwhile (the two shared a
    lock)."""
    busy, batch = _Busy(S), _LargeBatch(S)
    net, W, b = _fp32_layer(S, 2000, 64, seed=9)
    X = np.random.default_rng(9).standard_normal((1000, 64)).astype(F32)
    net.forward(X)                                                  # (its buffers and the slots are there)
    S.synchronize()
    busy.enqueue()
    got = []
    other = threading.Thread(target=lambda: got.append(net.forward(X)))
    other.start()
    time.sleep(0.02)                                                # (it waits by then)
    start = time.perf_counter()
    batch.step()
    back = time.perf_counter() - start
    other.join()
    done = time.perf_counter() - start
    S.synchronize()
    assert done >= 0.05 and back <= 0.5 * done, (back, done)
    pre = X.astype(np.float64) @ W.T + b
    assert rel_max_abs(got[0], np.where(pre > 0, pre, 0.01 * pre)) <= 1e-5
    assert np.array_equal(batch.gradients(S), batch.want)
    net.destroy()
    busy.net.destroy()


@pytest.mark.parametrize("fmt", ["i4", "i2"])
def test_streamed_rows_a_little_below_8192_take_no_longer(S, fmt):
    """sp_skinny16_regs at 256 samples: workgroups of 256 rows, and planned as such where the rows are fewer than 8192 too
    (planned as 128 rows each, every other workgroup had none and the others twice the K: 1.4 times as long; now even)."""
    n, K = 256, 8192
    us = {}
    for N in (8100, 8192):
        net, W, b = _decoded_layer(S, fmt, N, K, seed=N)
        assert S.lib().sphip_layer_kernel_name(net.h, 1, n, 0).decode() == "sp_skinny16_regs"
        X = np.random.default_rng(N).standard_normal((n, K)).astype(F32)
        pre = X.astype(np.float64) @ W.T + b
        assert rel_max_abs(net.forward(X), np.where(pre > 0, pre, 0.01 * pre)) <= 1e-3
        us[N] = min(S.time_layer([net], 1, n, 100) for _ in range(5))
        net.destroy()
    assert us[8100] <= 1.2 * us[8192]


@pytest.mark.parametrize("fmt", ["f16", "i8"])
def test_sums_too_short_for_a_split_take_no_longer(S, fmt):
    """gemm16_single_splits: a million outputs of 1024 terms in 256 tiles, against a tenth more in 288 tiles, which are never split
    (in two parts 1.3 times as long; now 0.95)."""
    N, K, us = 1000, 1024, {}
    net, W, b = _decoded_layer(S, fmt, N, K, seed=N)
    for n in (1000, 1100):
        assert S.lib().sphip_layer_kernel_name(net.h, 1, n, 0).decode() == "sp_gemm16"
        X = np.random.default_rng(n).standard_normal((n, K)).astype(F32)
        pre = X.astype(np.float64) @ W.T + b
        assert rel_max_abs(net.forward(X), np.where(pre > 0, pre, 0.01 * pre)) <= 1e-3
        us[n] = min(S.time_layer([net], 1, n, 100) for _ in range(5))
    net.destroy()
    assert us[1000] <= 1.12 * us[1100]


def test_shorter_sums_of_few_outputs_take_no_longer(S):
    """sp_skinny16_kw_head with split activations: 4096 terms a sum against 6144 (in one part against three 1.15 times as long; in
    four now 0.9)."""
    us = {}
    for K in (4096, 6144):
        net, _, _ = _decoded_layer(S, "f16", 16, K, seed=K)
        us[K] = min(S.time_layer([net], 1, 16, 200, S.SPHIP_SPLIT_ACTIVATIONS) for _ in range(7))
        net.destroy()
    assert us[4096] <= 1.05 * us[6144]


def test_padded_integer_inputs_take_no_longer_than_unpadded_ones(S):
    """700 to 4000 samples of 4104 INT4 codes into 1030 outputs, which run padded, against 4088 codes of the kernel of one stage (on
    large tiles split over K 1.2 to 1.3 times as long; now even)."""
    us = {}
    for K in (4088, 4104):
        net, _, _ = _decoded_layer(S, "i4", 1030, K, seed=K)
        for n in (700, 1500, 4000):
            assert S.lib().sphip_layer_kernel_name(net.h, 1, n, 0).decode() == "sp_gemm16"
            us[K, n] = min(S.time_layer([net], 1, n, 50) for _ in range(5))
        net.destroy()
    for n in (700, 1500, 4000):
        assert us[4104, n] <= 1.12 * us[4088, n], n


def _fp32_layer(S, N, K, seed):
    rng = np.random.default_rng(seed)
    W, b = (rng.standard_normal((N, K)) * 0.05).astype(F32), (rng.standard_normal(N) * 0.1).astype(F32)
    net = S.DeviceNet([K, N], [S.ACT_LEAKY_RELU], S.PRECISION_FLOAT32)
    net.upload(0, 0, W)
    net.upload(0, 1, b)
    return net, W.astype(np.float64), b.astype(np.float64)


@pytest.mark.parametrize("n,K,N,kernel", [
    (17000, 128, 10, "head"), (6000, 129, 10, "tiles"), (17000, 512, 16, "head"), (10001, 319, 3, "head"), (9999, 319, 3, "tiles"),
    (10001, 321, 3, "tiles"), (8192, 511, 10, "tiles"), (32769, 511, 2, "head"), (8192, 516, 10, "tiles"),
])
def test_few_fp32_outputs_on_both_sides_of_their_kernels(S, n, K, N, kernel):
    """gemm32_head_takes: rows of whole 16-byte units up to K = 512, others where the kernel of tiles is the slower one, against
    float64.  (FP32 sums: 2^-24 per term.)"""
    net, W, b = _fp32_layer(S, N, K, seed=n + K)
    name = S.lib().sphip_layer_kernel_name(net.h, 1, n, 0).decode()
    assert (name == "sp_gemm32_head") == (kernel == "head"), name
    X = np.random.default_rng(n).standard_normal((n, K)).astype(F32)
    pre = X.astype(np.float64) @ W.T + b
    got = net.forward(X)
    net.destroy()
    assert rel_max_abs(got, np.where(pre > 0, pre, 0.01 * pre)) <= 1e-5


def test_ragged_rows_into_few_fp32_outputs_take_no_longer(S):
    """8192 samples of 511 values into 10 outputs against 513, which the kernel of tiles takes (sp_gemm32_head 1.4 times as long)."""
    us = {}
    for K in (511, 513):
        net, _, _ = _fp32_layer(S, 10, K, seed=K)
        us[K] = min(S.time_layer([net], 1, 8192, 100) for _ in range(5))
        net.destroy()
    assert us[511] <= 1.15 * us[513]


def test_streamed_rows_of_8_kib_take_no_longer_than_others(S):
    """sp_skinny16 on rows that are a power of two of bytes long: read in step, they lay in a few of the memory's channels
    (16384 x 16384 INT4 1.35 times as long as 16384 x 15872; now even).  Weights larger than the memory-side cache."""
    n, N, us = 16, 16384, {}
    for K in (15872, 16384):
        rng = np.random.default_rng(K)
        nets = [S.DeviceNet([K, N], [S.ACT_RELU], S.PRECISION_INT4) for _ in range(4)]
        for net in nets:
            net.upload(0, 0, rng.integers(0, 256, N * K // 2, dtype=np.uint8), 0.01)
            net.upload(0, 1, rng.integers(0, 256, N // 2, dtype=np.uint8), 0.1)
        assert S.lib().sphip_layer_kernel_name(nets[0].h, 1, n, 0).decode() == "sp_skinny16"
        us[K] = min(S.time_layer(nets, 1, n, 100) for _ in range(5))
        for net in nets:
            net.destroy()
    assert us[16384] <= 1.15 * us[15872]


@pytest.mark.parametrize("fmt", ["f32", "f16", "i8"])
@pytest.mark.parametrize("topo,n", [([784, 96, 33], 5350), ([784, 96, 33], 8193), ([2100, 40, 10], 2049), ([2100, 40, 10], 6145)])
def test_layers_over_the_rows_that_have_landed(S, O, fmt, topo, n):
    """Batches whose upload is followed block by block: the first size of a block and of an upload in chunks, a last block of
    one row more than a whole one, sizes that leave whole blocks.  A row's result does not depend on the block it is in, up to
    the order of a K split's sums: two orders of K products differ by at most K 2^-24 of the sum of their magnitudes (784
    of them: 5e-5), and 16-bit activations may round the other way once per layer."""
    src = make_oracle_net(O, topo, ["relu", "softmax"], seed=74, loss=1)
    _, _, net = quantized_pair(O, S, src, fmt)
    X = np.random.default_rng(75).random((n, topo[0])).astype(F32)
    got = S.forward_batch(net, X)
    want = sphip_forward(S, net, X, S.SPHIP_WHOLE_BATCH)
    assert rel_max_abs(got, want) <= (TOL_VEC if fmt == "f32" else 2.0 ** -9)
    T = np.eye(topo[-1], dtype=F32)[np.arange(n) % topo[-1]]
    total, pred, correct = S.evaluate_batch(net, X, T)
    loss = O.batch_loss(got, T, 1, O.ACT["softmax"])
    assert abs(total - loss) <= 2e-5 * abs(loss)
    assert np.array_equal(pred, O.argmax_rows(got))
    assert correct == int((O.argmax_rows(got) == O.argmax_rows(T)).sum())
    S.free_network(net)


def test_landed_blocks_keep_the_arithmetic_of_the_whole_batch(S, O):
    """10,000 samples make this layer one for the BF16 parts, and for the FP16 parts in split mode, whose inputs saturate at
    65504; the rows of a block that has landed are too few for either."""
    topo, n = [784, 512], 10000
    src = make_oracle_net(O, topo, ["none"], seed=81)
    _, ref, net = quantized_pair(O, S, src, "f32")
    X = np.random.default_rng(82).standard_normal((n, topo[0])).astype(F32)
    true = ref.forward_batch_f64(X)
    got, whole = (np.linalg.norm(sphip_forward(S, net, X, f).astype(np.float64) - true) for f in (0, S.SPHIP_WHOLE_BATCH))
    assert got <= 1.2 * whole
    X[5000, 7] = 1e6
    got, whole = (sphip_forward(S, net, X, S.SPHIP_SPLIT_ACTIVATIONS | f) for f in (0, S.SPHIP_WHOLE_BATCH))
    assert rel_max_abs(got, whole) <= TOL_VEC
    S.free_network(net)


def test_pinned_batches_run_whole(S, O):
    """Memory that the copy engine reads as it is arrives in one piece: bit for bit the whole batch's outputs (whose 784 sums
    the blocks of a pageable batch cut differently)."""
    topo, n = [784, 512], 10000
    src = make_oracle_net(O, topo, ["none"], seed=83)
    _, _, net = quantized_pair(O, S, src, "f32")
    X = np.random.default_rng(84).random((n, topo[0]), dtype=F32)
    whole = sphip_forward(S, net, X, S.SPHIP_WHOLE_BATCH)
    with open("/proc/self/maps") as f:
        hip = C.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))      # (the one the library runs on)
    at = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(at), C.c_size_t(X.nbytes), 0) == 0
    pinned = np.frombuffer((C.c_float * X.size).from_address(at.value), dtype=F32).reshape(X.shape)
    pinned[:] = X
    got = sphip_forward(S, net, pinned, 0)
    assert hip.hipHostFree(at) == 0
    assert np.array_equal(got, whole)
    assert not np.array_equal(sphip_forward(S, net, X, 0), whole)
    S.free_network(net)


def test_uploads_in_a_row_do_not_share_a_chunk(S, O):
    """Targets of four chunks, then samples of two: the samples' first chunk goes where the targets' last one lay."""
    topo, n = [512, 24, 1000], 8192
    src = make_oracle_net(O, topo, ["relu", "none"], seed=76)
    _, _, net = quantized_pair(O, S, src, "f32")
    rng = np.random.default_rng(77)
    X = rng.random((n, topo[0]), dtype=F32)
    T = rng.random((n, topo[-1]), dtype=F32) + F32(8)
    want = float(((S.forward_batch(net, X).astype(np.float64) - T) ** 2).sum())
    for _ in range(3):
        total, _, _ = S.evaluate_batch(net, X, T)
        assert abs(total - want) <= 2e-5 * abs(want)
    S.free_network(net)


@pytest.mark.parametrize("topo", [[1200, 1630, 1010], [1200, 1631, 1010], [1200, 2640], [1200, 2641], [65] * 16, [65] * 17])
@pytest.mark.parametrize("last", ["softmax", "none"])
def test_single_sample_ends_on_both_sides_of_one_launch(S, O, topo, last):
    """3840 values and 16 layers are gathered by one workgroup, more by the launches before it; the call is repeated."""
    src = make_oracle_net(O, topo, ["tanh"] * (len(topo) - 2) + [last], seed=79, init="xavier")
    _, ref, net = quantized_pair(O, S, src, "f16")
    rng = np.random.default_rng(80)
    for _ in range(3):
        x = rng.standard_normal(topo[0]).astype(F32)
        y = S.forward(net, x)
        assert rel_max_abs(y, ref.forward_batch(x[None])[0]) <= TOL_VEC
        v = S.neurons_view(net)
        assert np.array_equal(v[:topo[0]], x) and np.array_equal(v[-topo[-1]:], y)
        hidden = np.tanh(ref.W(0).astype(np.float64) @ x + ref.b(0)) if len(topo) > 2 else y
        assert rel_max_abs(v[topo[0]:topo[0] + topo[1]], hidden) <= TOL_VEC
    S.free_network(net)
