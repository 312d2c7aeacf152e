"""The training steps in LDS: over rounds of 64 samples (trainRoundKernel), for half networks outside the fused kernels'
shapes and networks of float that fit a compute unit's LDS, and with every wave by itself (trainWaveKernel), for the smaller
of the float networks.

Two bars.  Networks of small whole numbers, in which every product, sum and rounding is exact (weights of -1, 0, 1 with three
entries to a row, so that values stay below 2048, a half's range of exact whole numbers): gradients and loss equal the
reference bit for bit, ties of max() included.  Random networks: the bars of the other training tests, 1e-3 of a layer's
gradient norm for half (hidden values that round the other way), 2e-5 for float."""
import numpy as np
import pytest
import torch

import oracle_binding as ob
from gpu_util import DEV, as_bytes, to_dev
from slang_amd import coopvec as cv
from slang_amd.coopvec import Activation, CoopVecComponentType as CT, CoopVecMatrixLayout as ML, FeedForwardLayer
from test_gpu_train import read_grads, rel_err

pytestmark = pytest.mark.gpu


def reference(specs, x, t, scale):
    """The step in float64 with Slang's rule for max(): (dW, db, every sample's loss).  ReLU of NaN is 0 and passes nothing."""
    hs, zs = [x.astype(np.float64)], []
    for s in specs:
        z = hs[-1] @ s["W"].astype(np.float64).T + (s["b"].astype(np.float64) if s["b"] is not None else 0.0)
        zs.append(z)
        hs.append(np.where(z > 0, z, 0.0) if s["act"] == 1 else np.maximum(z, z * s["slope"]) if s["act"] == 2 else z)
    diff = hs[-1] - t.astype(np.float64)
    g, dW, dB = 2.0 * diff * scale, [], []
    for l in range(len(specs) - 1, -1, -1):
        z, sl = zs[l], specs[l]["slope"]
        if specs[l]["act"] == 1: g = g * np.where(z > 0, 1.0, np.where(z == 0, 0.5, 0.0))
        if specs[l]["act"] == 2: g = g * np.where(z > 0, 1.0, np.where(z == 0, 0.5 + 0.5 * sl, sl))
        dW.append(g.T @ hs[l]); dB.append(g.sum(axis=0))
        g = g @ specs[l]["W"].astype(np.float64)
    return dW[::-1], dB[::-1], (diff ** 2).sum(axis=1)


def build(specs, ct, layout=ML.RowMajor, grad_layout=ML.TrainingOptimal, preset=0.0):
    layers = []
    for s in specs:
        out, fan_in = s["W"].shape
        esz = s["W"].itemsize
        w, stride = as_bytes(to_dev(np.ascontiguousarray(s["W"]))), fan_in * esz
        if layout == ML.ColumnMajor:
            w, stride = as_bytes(to_dev(np.ascontiguousarray(s["W"].T))), out * esz
        elif layout != ML.RowMajor:
            size = cv.getCooperativeVectorMatrixSize(out, fan_in, ct, layout)
            D, dst = cv.CooperativeVectorMatrixDesc, torch.zeros(size, dtype=torch.uint8, device=DEV)
            cv.convertCooperativeVectorMatrix(dst, [D(out, fan_in, ct, layout, size, 0, 0)], w, [D(out, fan_in, ct, ML.RowMajor, out * stride, 0, stride)])
            w, stride = dst, 0
        wg = torch.full((cv.getCooperativeVectorMatrixSize(out, fan_in, CT.Float32, grad_layout) // 4,), preset, device=DEV)
        bg = torch.full((out,), preset, device=DEV)
        layers.append(FeedForwardLayer(fan_in, out, w, as_bytes(to_dev(s["b"])) if s["b"] is not None else None, layout, stride, s["act"], s["slope"],
                                       wg.view(torch.uint8), bg.view(torch.uint8), grad_layout, 0))
    return layers


def kernel_of(elem, dims):
    """float networks whose dW fits a wave's registers (36 tiles of 16 x 16 at 1, 2 or 4 tiles per layer) run on
    trainWaveKernel, the others on trainRoundKernel"""
    up = lambda v: next((t for t in (1, 2, 4) if v <= 16 * t), 99)
    ht, it, hidden = max(up(d) for d in dims[1:-1]), up(dims[0]), len(dims) - 2
    wave = elem == "f32" and ht * it + ht * ht * (hidden - 1) + ht <= 36
    return "train%sKernel<%s" % ("Wave" if wave else "Round", elem)


def whole_number_network(rng, dims, dtype, act, slope, last_act):
    specs = []
    for i, (fi, fo) in enumerate(zip(dims, dims[1:])):
        W = np.zeros((fo, fi))
        for row in W:
            row[rng.choice(fi, min(3, fi), replace=False)] = rng.integers(-1, 2, min(3, fi))
        b = rng.integers(-1, 2, fo).astype(np.float64)
        if i + 2 < len(dims):
            W[::5] = 0; b[::5] = 0          # pre-activations that are always exactly 0
        specs.append(dict(W=W.astype(dtype), b=b.astype(dtype), act=int(last_act if i == len(dims) - 2 else act), slope=slope))
    return specs


# (sizes at the edges of tiles, of the rows a wave takes and of the LDS; batches around a round of 64 samples)
CASES = [
    ("f32", [32, 64, 64, 8], 64), ("f32", [5, 17, 3], 1), ("f32", [16, 16, 16], 63), ("f32", [33, 64, 48, 33, 1], 65), ("f32", [64, 64, 16], 1000),
    ("f32", [31, 32, 32, 32, 31, 16], 129), ("f32", [1, 1, 1], 200), ("f32", [100, 128, 4], 130), ("f32", [65, 65, 20, 3], 77), ("f32", [16, 64, 64, 64, 64, 2], 300),
    ("f32", [64, 64, 64, 9], 4097), ("f32", [40, 32, 20, 32, 32, 16], 128), ("f32", [16, 10, 16, 16, 16, 1], 17), ("f32", [12, 50, 2], 2049), ("f32", [30, 40, 33, 64, 7], 190),
    ("f16", [16, 128, 128, 128, 8], 64), ("f16", [16, 128, 128, 128, 8], 40001), ("f16", [33, 16, 2], 1), ("f16", [64, 64, 64, 16], 65), ("f16", [40, 20, 49, 5], 127),
    ("f16", [8, 128, 128, 128, 128, 4], 1), ("f16", [32, 128, 128, 128, 128, 16], 33), ("f16", [21, 128, 128, 128, 128, 5], 20011), ("f16", [7, 128, 113, 128, 97, 1], 1000),
    ("f16", [128, 128, 128, 128, 9], 95),
    # (rows of weights that begin at any half: every remainder of a piece, matrices of few bytes)
    ("f16", [33, 65, 1, 66, 2], 70), ("f16", [1, 67, 3, 68, 1], 70), ("f16", [34, 69, 5, 70, 16], 70), ("f16", [39, 71, 79, 2], 70), ("f16", [36, 73, 2, 6], 70),
    ("f16", [127, 33, 12], 300), ("f16", [48, 96, 80, 3], 200), ("f16", [10, 65, 33, 97, 16], 63), ("f16", [20, 129 - 1, 17, 64, 30, 7], 500), ("f16", [50, 30, 30, 30, 30, 1], 70),
]


@pytest.mark.parametrize("elem,dims,B", CASES)
@pytest.mark.parametrize("act,slope,last", [(Activation.ReLU, 0.0, Activation.NoActivation), (Activation.LeakyReLU, 0.5, Activation.LeakyReLU)])
def test_whole_number_networks_are_exact(elem, dims, B, act, slope, last):
    rng = np.random.default_rng(sum(dims) * 7 + B)
    dtype, ct = (np.float32, CT.Float32) if elem == "f32" else (np.float16, CT.Float16)
    if act == Activation.LeakyReLU and len(dims) > (5 if elem == "f32" else 4):
        # Every leaky layer halves the unit the values are multiples of, forward and backward: with three hidden layers and the
        # loss scale the gradients are multiples of 2^-7, and sums of a column's entries reach 80, more than 2048 of them (a
        # half's 11 bits); float's 24 bits last one layer longer in the products of dW.  Slope 0 keeps the units.
        slope = 0.0
    specs = whole_number_network(rng, dims, dtype, act, slope, last)
    x = rng.integers(-1, 2, (B, dims[0])).astype(dtype)
    t = rng.integers(-2, 3, (B, dims[-1])).astype(dtype)
    scale = 1.0 / 16
    dW, dB, loss = reference(specs, x, t, scale)
    layers = build(specs, ct, preset=1.0)
    lmax = torch.zeros(1, device=DEV)
    ws, got = cv.mlpTrainStep(layers, to_dev(x), to_dev(t), lossScale=scale, weightType=ct, lossMax=lmax)
    assert cv.lastKernelName().startswith(kernel_of(elem, dims)), cv.lastKernelName()
    gW, gB = read_grads(layers, specs, CT.Float32, ML.TrainingOptimal)
    for l in range(len(specs)):
        assert np.array_equal(gW[l] - 1.0, dW[l]), (l, np.abs(gW[l] - 1.0 - dW[l]).max())
        assert np.array_equal(gB[l] - 1.0, dB[l]), l
    assert got.item() == loss.sum() and lmax.item() == loss.max()
    # the same weights in other layouts, vectors that are no aligned 16-byte pieces: the same bits
    layouts = [ML.ColumnMajor, ML.InferencingOptimal, ML.TrainingOptimal]
    other = build(specs, ct, layouts[B % 3], ML.RowMajor, preset=1.0)
    xs = torch.zeros(B, dims[0] + 3, dtype=torch.float32 if elem == "f32" else torch.float16, device=DEV)
    xs[:, 1:1 + dims[0]] = to_dev(x)
    _, got2 = cv.mlpTrainStep(other, xs[:, 1:1 + dims[0]], to_dev(t), lossScale=scale, weightType=ct, workspace=ws)
    oW, oB = read_grads(other, specs, CT.Float32, ML.RowMajor)
    for l in range(len(specs)):
        assert np.array_equal(oW[l], gW[l]) and np.array_equal(oB[l], gB[l]), l
    assert got2.item() == got.item()


@pytest.mark.parametrize("elem,dims,B", [("f32", [32, 64, 64, 8], 5000), ("f32", [9, 30, 12, 3], 777), ("f16", [16, 128, 128, 128, 8], 3000), ("f16", [60, 48, 20, 4], 1500)])
@pytest.mark.parametrize("act,slope", [(Activation.ReLU, 0.0), (Activation.LeakyReLU, 0.125)])
@pytest.mark.parametrize("targets", [True, False])
def test_random_networks(elem, dims, B, act, slope, targets):
    rng = np.random.default_rng(sum(dims) + B)
    dtype, ct = (np.float32, CT.Float32) if elem == "f32" else (np.float16, CT.Float16)
    specs = []
    for i, (fi, fo) in enumerate(zip(dims, dims[1:])):
        specs.append(dict(W=(rng.standard_normal((fo, fi)) * np.sqrt(2.0 / fi)).astype(dtype), b=rng.uniform(-0.1, 0.1, fo).astype(dtype) if i != 1 else None,
                          act=int(Activation.NoActivation if i == len(dims) - 2 else act), slope=slope))
    x = rng.uniform(-1, 1, (B, dims[0])).astype(dtype)
    t = rng.uniform(-1, 1, (B, dims[-1])).astype(dtype) if targets else None
    want_t = t if targets else np.repeat(np.sin(x.astype(np.float64).sum(axis=1, keepdims=True)), dims[-1], axis=1)
    if elem == "f16":
        rW, rB, rloss = ob.ref_mlp_train(specs, x, t, 1.0, tie_rule=True)
        bar = 1e-3
    else:
        rW, rB, rloss = reference(specs, x, want_t, 1.0)
        rloss = rloss.sum()
        bar = 2e-5
    layers, again = build(specs, ct), build(specs, ct)
    _, loss = cv.mlpTrainStep(layers, to_dev(x), to_dev(t) if targets else None, weightType=ct)
    assert cv.lastKernelName().startswith(kernel_of(elem, dims)), cv.lastKernelName()
    _, loss2 = cv.mlpTrainStep(again, to_dev(x), to_dev(t) if targets else None, weightType=ct)
    dW, dB = read_grads(layers, specs, CT.Float32, ML.TrainingOptimal)
    for l in range(len(specs)):
        assert rel_err(dW[l], rW[l]) <= bar and rel_err(dB[l], rB[l]) <= bar, (l, rel_err(dW[l], rW[l]), rel_err(dB[l], rB[l]))
        assert torch.equal(layers[l].weightsGrad, again[l].weightsGrad) and torch.equal(layers[l].biasesGrad, again[l].biasesGrad)
    assert abs(loss.item() - rloss) <= bar * rloss and loss.item() == loss2.item()


KERNELS = [("f32", [32, 64, 64, 8], "trainWaveKernel"), ("f32", [100, 128, 4], "trainRoundKernel"), ("f16", [64, 64, 64, 16], "trainRoundKernel"),
           ("f16", [16, 128, 128, 128, 8], "trainRoundKernel"), ("f32", [9, 30, 12, 3], "trainWaveKernel"), ("f16", [60, 48, 20, 4], "trainRoundKernel")]


@pytest.mark.filterwarnings("ignore:invalid value encountered in matmul")
@pytest.mark.parametrize("flags", [0, cv.FLAG_LAYERWISE_TRAINING])
@pytest.mark.parametrize("elem,dims,kernel", KERNELS)
def test_nan_at_a_relu_is_no_tie(elem, dims, kernel, flags):
    # Samples with a NaN of either sign: every hidden unit of the first layer is NaN, which ReLU turns into 0 and whose gradient
    # is 0 (not the half of a tie), so the loss is finite and these samples add to the layers above alone.  In dW of the first
    # layer their 0 x NaN shows in the NaN's column, nowhere else (over memory half vectors spread it to neighbouring columns).
    # A third sample has infinities of both signs, which make the NaN, and two units are NaN for every sample, by their biases.
    # Whole numbers: exact.  The step over memory has the same rule.
    rng = np.random.default_rng(sum(dims))
    dtype, ct = (np.float32, CT.Float32) if elem == "f32" else (np.float16, CT.Float16)
    B = 150
    specs = whole_number_network(rng, dims, dtype, Activation.ReLU, 0.0, Activation.NoActivation)
    x = rng.integers(-1, 2, (B, dims[0])).astype(dtype)
    t = rng.integers(-2, 3, (B, dims[-1])).astype(dtype)
    x[77, 1], x[78, 1], x[140, 1], x[140, 2] = np.nan, -np.nan, np.inf, -np.inf
    specs[0]["W"][:, 1:3] = 1
    specs[0]["b"][3], specs[0]["b"][4] = np.nan, -np.nan
    dW, dB, loss = reference(specs, x, t, 1.0 / 16)
    assert np.isfinite(loss).all()
    layers = build(specs, ct)
    _, got = cv.mlpTrainStep(layers, to_dev(x), to_dev(t), lossScale=1.0 / 16, weightType=ct, flags=flags)
    assert (kernel in cv.lastKernelName()) == (flags == 0), cv.lastKernelName()
    gW, gB = read_grads(layers, specs, CT.Float32, ML.TrainingOptimal)
    assert got.item() == loss.sum()
    for l in range(len(specs)):
        assert np.array_equal(gB[l], dB[l]), (l, np.abs(gB[l] - dB[l]).max())
        keep = np.ones(dims[l], bool)
        if l == 0: keep[slice(1, 3) if elem == "f32" or flags == 0 else slice(None)] = False
        assert np.array_equal(gW[l][:, keep], dW[l][:, keep]), l
    assert np.isnan(gW[0][:, 1:3]).all()


@pytest.mark.parametrize("value", ["nan", "inf", "infinite loss"])
@pytest.mark.parametrize("elem,dims,kernel", KERNELS + [("f16", [8, 64, 64, 64, 64, 1], "mlpTrainPairKernel"), ("f16", [4, 16, 4], "mlpTrainKernel")])
def test_a_loss_that_is_not_finite_voids_the_step(elem, dims, kernel, value):
    # lossSum, lossMax and every gradient element are NaN, whatever is in the gradients before; so they are where a sample's
    # loss is infinite and its gradients are not (float: the square of a difference of 2^66)
    rng = np.random.default_rng(sum(dims) + 1)
    dtype, ct = (np.float32, CT.Float32) if elem == "f32" else (np.float16, CT.Float16)
    B = 16 if dims == [4, 16, 4] else 300
    specs = []
    for i, (fi, fo) in enumerate(zip(dims, dims[1:])):
        specs.append(dict(W=(rng.standard_normal((fo, fi)) / np.sqrt(fi)).astype(dtype), b=np.zeros(fo, dtype),
                          act=int(Activation.NoActivation if i == len(dims) - 2 else Activation.LeakyReLU), slope=0.125))
    x = rng.uniform(-1, 1, (B, dims[0])).astype(dtype)
    t = rng.uniform(-1, 1, (B, dims[-1])).astype(dtype)
    at = B - 3
    if value != "infinite loss":
        x[at, 1] = float(value)
    elif elem == "f32":
        t[at, 0] = 2.0 ** 66
    else:
        specs[-1]["b"][0], t[:, 0], t[at, 0] = 60000, 60000, -60000       # (the difference is infinite in half)
    layers = build(specs, ct, preset=1.0)
    lmax = torch.zeros(1, device=DEV)
    _, loss = cv.mlpTrainStep(layers, to_dev(x), to_dev(t), weightType=ct, lossMax=lmax)
    assert kernel in cv.lastKernelName(), cv.lastKernelName()
    assert np.isnan(loss.item()) and np.isnan(lmax.item()), (loss.item(), lmax.item())
    gW, gB = read_grads(layers, specs, CT.Float32, ML.TrainingOptimal)
    for l in range(len(specs)):
        assert np.isnan(gW[l]).all() and np.isnan(gB[l]).all(), l


@pytest.mark.parametrize("elem,dims,kernel", KERNELS)
def test_workspace_grows_with_the_batch_and_is_enough(elem, dims, kernel):
    # One set of gradients for every 64 samples until the chip is full.  The step stays inside what the query says (what lies
    # behind it keeps its bytes), and gives the same bits whatever the workspace held before.
    rng = np.random.default_rng(sum(dims) + 5)
    dtype, ct = (np.float32, CT.Float32) if elem == "f32" else (np.float16, CT.Float16)
    specs = whole_number_network(rng, dims, dtype, Activation.ReLU, 0.0, Activation.NoActivation)
    size = lambda B: cv.mlpTrainStepWorkspaceSize(build(specs, ct), B, weightType=ct)
    one, full = size(1), size(1 << 30)
    assert one == size(64) and size(65) == 2 * one and full % one == 0 and full >= 256 * one and size(0xffffffff) == full
    for B in (1, 64, 65, 1000, 64 * 255 + 1, 64 * 600):
        x = to_dev(rng.integers(-1, 2, (B, dims[0])).astype(dtype))
        t = to_dev(rng.integers(-2, 3, (B, dims[-1])).astype(dtype))
        need, got = size(B), []
        assert need == min(-(-B // 64) * one, full)
        for fill in (0xff, 0x3c):
            layers = build(specs, ct)
            room = torch.full((need + 4096,), fill, dtype=torch.uint8, device=DEV)
            _, loss = cv.mlpTrainStep(layers, x, t, lossScale=1.0 / 16, weightType=ct, workspace=room[:need])
            assert kernel in cv.lastKernelName(), cv.lastKernelName()
            assert (room[need:] == fill).all()
            got.append((loss.item(), [v.clone() for y in layers for v in (y.weightsGrad, y.biasesGrad)]))
        assert got[0][0] == got[1][0] and all(torch.equal(a, b) for a, b in zip(got[0][1], got[1][1]))
        assert np.isfinite(got[0][0])


def test_the_largest_batch():
    # 2^32 - 1 samples: rounds and tiles are counted without leaving 32 bits.  All samples are 0 but the first and the last.
    B = 0xffffffff
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 34 GB of memory")
    x, t = torch.zeros(B, 1, device=DEV), torch.zeros(B, 1, device=DEV)
    x[0], x[-1] = 1, 1
    for dims, kernel in (([1, 1, 1], "trainWaveKernel"), ([1, 65, 1], "trainRoundKernel")):
        specs = [dict(W=np.zeros((fo, fi), np.float32), b=np.zeros(fo, np.float32), act=int(a), slope=0.0)
                 for fi, fo, a in ((1, dims[1], Activation.ReLU), (dims[1], 1, Activation.NoActivation))]
        for s in specs:
            s["W"][0, 0] = 1
        layers = build(specs, CT.Float32, grad_layout=ML.RowMajor)
        _, loss = cv.mlpTrainStep(layers, x, t, weightType=CT.Float32)
        assert kernel in cv.lastKernelName(), cv.lastKernelName()
        gW, gB = read_grads(layers, specs, CT.Float32, ML.RowMajor)
        assert loss.item() == 2 and gW[1][0, 0] == 4 and gB[1][0] == 4 and gW[0][0, 0] == 4 and gB[0][0] == 4
        assert not gW[0][1:].any() and not gB[0][1:].any() and not gW[1][0, 1:].any()
