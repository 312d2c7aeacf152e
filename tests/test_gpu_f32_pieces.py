"""fp32 matrix products as sums of bfloat16 pieces (F32Mma, slang_amd/csrc/cv_device.h), and where the fp32 instruction stays: accuracy against 64 bits, infinities,
NaN, the largest and the smallest values, and the kernel for equal hidden layers against the chain of single-layer operators.

Bound of a sum of K terms: an operand (times 2^24) is three pieces exactly; of the nine products the three dropped ones are below 2^-26 of the
term each, the others are exact; of the sums, one rounding to 24 bits per matrix instruction (K/32 of them on the h*h products;
the five small ones count below 2^-7 of it) and two at the end, where the bias and the small products join."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, as_bytes, to_dev
from slang_amd import coopvec as cv
from slang_amd.coopvec import Activation, CoopVecComponentType as CT, CoopVecMatrixLayout as ML, FeedForwardLayer

pytestmark = pytest.mark.gpu


def matmul(x, W, b, act=Activation.NoActivation):
    M, K = W.shape
    return cv.coopVecMatMulAdd(to_dev(x), CT.Float32, as_bytes(to_dev(W)), 0, CT.Float32, as_bytes(to_dev(b)), 0, CT.Float32,
                               ML.RowMajor, False, 4 * K, M=M, resultType=CT.Float32, activation=act).cpu().numpy()


def bound(x, W, b):
    K = W.shape[1]
    mag = np.abs(x.astype(np.float64)) @ np.abs(W.astype(np.float64)).T + np.abs(b.astype(np.float64))
    return (K / 32 + 4) * 2.0 ** -24 * mag


# remainders of tiles; 16 x 32 and 64 x 64 in the streaming form; from 20 x 1664 on the fp32 instruction, whose roundings, one for every term,
# mostly cancel
@pytest.mark.parametrize("M,K,B", [(1, 1, 1), (16, 32, 64), (17, 33, 100), (64, 64, 1027), (65, 64, 500), (128, 192, 400), (130, 200, 300),
                                   (20, 1664, 60), (20, 1680, 60), (33, 2048, 50)])
def test_products_against_64_bits(M, K, B):
    rng = np.random.default_rng(M * 3000 + K)
    x = (rng.standard_normal((B, K)) * np.exp2(rng.integers(-12, 13, (B, K)))).astype(np.float32)
    W = (rng.standard_normal((M, K)) * np.exp2(rng.integers(-6, 7, (M, K)))).astype(np.float32)
    b = rng.standard_normal(M).astype(np.float32)
    ref = x.astype(np.float64) @ W.astype(np.float64).T + b
    assert (np.abs(matmul(x, W, b) - ref) <= bound(x, W, b)).all()


# the rule between the pieces and the fp32 instruction (one rounding for every term and for the bias), at its edges; up to 256 terms of vectors that
# are no aligned groups of four the packed kernel, else matmulLargeKernel
@pytest.mark.parametrize("M,K,whole", [(16, 192, False), (16, 193, True), (17, 193, False), (16, 200, True), (17, 200, False), (32, 320, False), (32, 321, True),
                                       (33, 321, False), (130, 384, False), (33, 385, True), (100, 1025, True), (3, 2048, True)])
def test_large_products_take_the_faster_instruction(M, K, whole):
    rng = np.random.default_rng(M * 5000 + K)
    for B in (1, 37, 4000):
        x, W, b = (rng.standard_normal(s).astype(np.float32) for s in ((B, K), (M, K), (M,)))
        got = matmul(x, W, b)
        kernel = "matmulPackedKernel<%s,KT=7," if K == 193 else "matmulLargeKernel<%s,"
        assert cv.lastKernelName().startswith(kernel % ("f32-whole" if whole else "f32")), cv.lastKernelName()
        ref = x.astype(np.float64) @ W.astype(np.float64).T + b
        mag = np.abs(x.astype(np.float64)) @ np.abs(W.astype(np.float64)).T + np.abs(b)
        assert (np.abs(got - ref) <= ((K + 1) * 2.0 ** -24 * mag if whole else bound(x, W, b))).all()


# (the packed kernel; the streaming form of 64 x 64 takes NaN through a maximum; then matmulLargeKernel on pieces and on the fp32 instruction)
@pytest.mark.parametrize("M,K", [(24, 40), (63, 64), (100, 96), (40, 300), (8, 1700)])
def test_values_at_the_ends_of_the_range(M, K):
    rng = np.random.default_rng(M + K)
    B = 200
    x, W, b = (rng.standard_normal(s).astype(np.float32) for s in ((B, K), (M, K), (M,)))
    plain = matmul(x, W, b)
    big = np.float32(3.4e38)                             # its nearest bfloat16 is infinite
    y = x.copy()
    y[3, 5], y[20, 0], y[40, K - 1], y[60, 7] = np.inf, -np.inf, np.nan, big
    y[80] = np.where(np.arange(K) % 3 == 0, np.inf, y[80])
    y[100] = x[100] * np.float32(1e-38)                  # down into the subnormal numbers
    V = W.copy()
    V[2, 5], V[5, 7], V[6, 9] = 0.0, 1e-3, np.inf
    def want(xs, ws):
        with np.errstate(all="ignore"):
            return (xs.astype(np.float64) @ ws.astype(np.float64).T + b).astype(np.float32)
    got = matmul(y, W, b)
    special = [3, 20, 40, 60, 80]
    others = np.setdiff1d(np.arange(B), special + [100])
    assert np.array_equal(got[others].view(np.uint32), plain[others].view(np.uint32))
    for rows in ([3], [20], [40], [80]):
        ref = want(y[rows], W)
        assert np.array_equal(np.isnan(got[rows]), np.isnan(ref)) and np.array_equal(got[rows][~np.isnan(ref)], ref[~np.isnan(ref)])
    ref = y[[60, 100]].astype(np.float64) @ W.astype(np.float64).T + b
    fits = np.abs(ref) < 1e38
    assert (np.abs(got[[60, 100]] - ref)[fits] <= bound(y[[60, 100]], W, b)[fits]).all() and fits[1].all()
    ref = y[[100]].astype(np.float64) @ W.astype(np.float64).T      # ... of which the bias hides everything
    assert (np.abs(matmul(y[[100]], W, 0 * b) - ref) <= bound(y[[100]], W, 0 * b) + 2.0 ** -149).all()
    # an infinite element of the matrix: its row alone
    got = matmul(x, V, b)
    ref = want(x, V)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(got[:, 6][~np.isnan(ref[:, 6])], ref[:, 6][~np.isnan(ref[:, 6])])
    same = np.setdiff1d(np.arange(M), [2, 5, 6])
    assert np.array_equal(got[:, same].view(np.uint32), plain[:, same].view(np.uint32))
    got = matmul(y, V, b)                                # ... and infinite vectors before it: 0 x inf is NaN
    ref = want(y[special], V)
    ok = np.isfinite(ref) & (np.abs(ref) < 1e38)
    assert np.array_equal(np.isnan(got[special]), np.isnan(ref)) and np.array_equal(np.isinf(got[special]) & ~ok, np.isinf(ref) & ~ok)


def large(rng, *shape):
    return (10.0 ** rng.uniform(22, 30, shape) * rng.choice([-1.0, 1.0], shape)).astype(np.float32)


# (64 x 64: the streaming kernel, 37 samples beyond its whole tiles on the packed one, as the next two; then matmulLargeKernel on pieces and on the fp32
# instruction)
@pytest.mark.parametrize("M,K", [(64, 64), (24, 40), (100, 96), (40, 300), (8, 1700)])
def test_products_of_finite_operands_that_overflow(M, K):
    rng = np.random.default_rng(M * 7 + K)
    B = 293
    x, W, b = rng.standard_normal((B, K)).astype(np.float32), rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal(M).astype(np.float32)
    rows, samples = rng.permutation(M)[: M // 2], rng.permutation(B)[:40]
    V = W.copy()
    V[rows, 3] = large(rng, len(rows))
    plain = matmul(x, V, b)
    y = x.copy()
    y[samples, 3] = large(rng, 40)
    ref = y.astype(np.float64) @ V.astype(np.float64).T + b
    over = np.abs(ref) > 3.5e38
    assert over[np.ix_(samples, rows)].all()
    got = matmul(y, V, b)
    assert np.array_equal(got[over], np.where(ref[over] > 0, np.inf, -np.inf).astype(np.float32))
    assert (np.abs(got - ref)[~over] <= bound(y, V, b)[~over]).all()
    others = np.setdiff1d(np.arange(B), samples)
    assert np.array_equal(got[others].view(np.uint32), plain[others].view(np.uint32))
    # what other samples hold, infinities too, changes nothing
    z = y.copy()
    z[others[::5], 1] = np.inf
    keep = np.setdiff1d(np.arange(B), others[::5])
    assert np.array_equal(matmul(z, V, b)[keep].view(np.uint32), got[keep].view(np.uint32))
    # every element of a vector and of a row
    y[samples], V[rows] = np.abs(large(rng, 40, K)), np.abs(large(rng, len(rows), K))
    got = matmul(y, V, b, Activation.ReLU)
    assert (got[np.ix_(samples, rows)] == np.inf).all()
    assert np.array_equal(matmul(y, -V, b, Activation.ReLU)[np.ix_(samples, rows)], np.zeros((40, len(rows)), np.float32))


def same_as(got, ref):
    # bit for bit; a subnormal result, which is the sum of two values rounded to multiples of 2^-149, within one of these
    return (np.abs(got - ref) <= np.where(np.abs(ref) < 2.0 ** -126, 2.0 ** -149, 0.0)).all()


@pytest.mark.parametrize("M,K", [(64, 64), (24, 40), (100, 96), (8, 1700)])
def test_small_operands(M, K):
    # one element of every row: the products are exact
    rng = np.random.default_rng(M * 11 + K)
    B = 160
    zero = np.zeros(M, np.float32)
    pick = rng.integers(0, K, M)
    for e in (-60, -100, -110, -118, -124, -126, -135, -147):
        x = np.ldexp(rng.uniform(1, 2, (B, K)), e).astype(np.float32)
        for s in (0, 31, -20, 100):
            W = np.zeros((M, K), np.float32)
            W[np.arange(M), pick] = 2.0 ** s
            assert same_as(matmul(x, W, zero).astype(np.float64), x[:, pick].astype(np.float64) * 2.0 ** s), (e, s)
            y = np.zeros((B, K), np.float32)                          # ... the small ones in the matrix
            y[np.arange(B), np.arange(B) % K] = 2.0 ** s
            assert same_as(matmul(y, x[:M], zero).astype(np.float64), x[:M, np.arange(B) % K].T.astype(np.float64) * 2.0 ** s), (e, s)
    # full rows, of every size within 2^24: the bound of the products alone
    for s in (0, 20, 100):
        x = (rng.standard_normal((B, K)) * np.exp2(rng.integers(-136, -111, (B, K)))).astype(np.float32)
        W = (rng.standard_normal((M, K)) * np.exp2(rng.integers(-6, 7, (M, K)) + s)).astype(np.float32)
        ref = x.astype(np.float64) @ W.astype(np.float64).T
        # (from 2^32 on, the fp32 instruction: a rounding for every term)
        b = bound(x, W, zero) if s < 32 else K * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(W.astype(np.float64)).T)
        assert (np.abs(matmul(x, W, zero) - ref) <= b + 2.0 ** -149).all(), s


# hidden values of 2^-127 to 2^-107, brought back by the last layer
@pytest.mark.parametrize("dims,last", [([32, 64, 64, 8], Activation.NoActivation), ([20, 48, 24, 5], Activation.NoActivation), ([20, 48, 24, 5], Activation.Sigmoid)])
def test_networks_with_small_hidden_values(dims, last):
    rng = np.random.default_rng(sum(dims))
    layers, params = network(rng, dims, [Activation.ReLU, Activation.NoActivation, last])
    for fi, fo, wd, bd, act in params:
        bd.zero_()
    params[0][2].view(torch.float32).mul_(2.0 ** -60)
    params[1][2].view(torch.float32).mul_(2.0 ** -57)
    params[2][2].view(torch.float32).mul_(2.0 ** 117)
    x = to_dev(rng.uniform(-1, 1, (3000, dims[0])).astype(np.float32))
    y = cv.mlpForward(layers, x, weightType=CT.Float32)
    assert torch.equal(y.view(torch.int32), chain(params, x).view(torch.int32))
    h, mag = x.double(), x.double().abs()
    for l, (fi, fo, wd, bd, act) in enumerate(params):
        w = wd.view(torch.float32).view(fo, fi).double()
        h, mag = h @ w.T, mag @ w.abs().T
        h = torch.relu(h) if l == 0 else h
    h = torch.sigmoid(h) if last == Activation.Sigmoid else h
    assert ((y - h).abs() <= 2.0 ** -18 * mag).all()


# the kernels for equal hidden layers, for any, and with a smooth activation
@pytest.mark.parametrize("dims,last", [([32, 64, 64, 8], Activation.ReLU), ([8, 128, 128, 3], Activation.NoActivation), ([20, 48, 24, 5], Activation.ReLU),
                                       ([64, 112, 96, 12], Activation.NoActivation), ([16, 112, 112, 112, 8], Activation.ReLU), ([20, 48, 24, 5], Activation.Sigmoid)])
def test_networks_whose_hidden_layers_overflow(dims, last):
    rng = np.random.default_rng(sum(dims))
    acts = [Activation.ReLU] * (len(dims) - 2) + [last]
    layers, params = network(rng, dims, acts)
    for fi, fo, wd, bd, act in params:
        wd.view(torch.float32).abs_()
    B = 20000
    x = rng.uniform(0.1, 1, (B, dims[0])).astype(np.float32)
    x[::33] *= np.float32(1e30)
    x[5::66] *= np.float32(1e20)
    params[1][2].view(torch.float32)[:dims[1]] *= 1e25                 # the first unit of the second layer
    x = to_dev(x)
    y = cv.mlpForward(layers, x, weightType=CT.Float32)
    ref = chain(params, x)
    assert torch.equal(y.view(torch.int32), ref.view(torch.int32)), cv.lastKernelName()
    want = x.double()
    for fi, fo, wd, bd, act in params[:-1]:
        want = torch.relu(want @ wd.view(torch.float32).view(fo, fi).double().T + bd.view(torch.float32).double()).float().double()
    fi, fo, wd, bd, act = params[-1]
    want = (want @ wd.view(torch.float32).view(fo, fi).double().T + bd.view(torch.float32).double()).float()
    want = torch.sigmoid(want) if last == Activation.Sigmoid else torch.relu(want) if last == Activation.ReLU else want
    assert not torch.isnan(y).any()
    if last != Activation.Sigmoid:
        assert torch.equal(torch.isinf(y), torch.isinf(want)) and torch.isinf(y).any(dim=1).sum() >= B // 33
    assert torch.allclose(y.nan_to_num(posinf=0.0), want.nan_to_num(posinf=0.0), rtol=1e-5, atol=1e-5)


def network(rng, dims, acts):
    layers, params = [], []
    for fi, fo, act in zip(dims, dims[1:], acts):
        W = (rng.standard_normal((fo, fi)) * np.sqrt(2.0 / fi)).astype(np.float32)
        b = (rng.standard_normal(fo) * 0.1).astype(np.float32)
        wd, bd = as_bytes(to_dev(W)), as_bytes(to_dev(b))
        layers.append(FeedForwardLayer(fi, fo, wd, bd, ML.RowMajor, fi * 4, act, 0.125))
        params.append((fi, fo, wd, bd, act))
    return layers, params


def chain(params, x):
    for fi, fo, wd, bd, act in params:
        x = cv.coopVecMatMulAdd(x, CT.Float32, wd, 0, CT.Float32, bd, 0, CT.Float32, ML.RowMajor, False, fi * 4, M=fo, resultType=CT.Float32,
                                activation=act, leakySlope=0.125)
    return x


@pytest.mark.parametrize("dims", [[4, 16, 1], [3, 16, 16, 16], [32, 32, 5], [20, 20, 24, 31, 8], [8, 64, 64, 64, 3], [33, 50, 64, 16], [64, 60, 60, 9],
                                  [7, 128, 4], [64, 120, 113, 16], [40, 16, 16, 16, 16, 16, 2], [36, 30, 7]])
def test_equal_hidden_layers_equal_the_chain_of_single_layer_operators(dims):
    rng = np.random.default_rng(sum(dims))
    acts = [[Activation.ReLU, Activation.NoActivation, Activation.LeakyReLU][l % 3] for l in range(len(dims) - 1)]
    layers, params = network(rng, dims, acts)
    for B, pad in ((1, 0), (15, 0), (65, 3), (20000, 0), (5001, 4)):      # `pad`: rows at a pitch, of which 3 leaves them unaligned
        wide = torch.zeros((B, dims[0] + pad), dtype=torch.float32, device=DEV)
        wide[:, :dims[0]] = to_dev(rng.uniform(-1, 1, (B, dims[0])).astype(np.float32))
        if B > 100:
            wide[7, 0], wide[B - 1, dims[0] - 1], wide[50, 1] = float("inf"), float("-inf"), 3.4e38
        x = wide[:, :dims[0]]
        y = cv.mlpForward(layers, x, weightType=CT.Float32)
        assert cv.lastKernelName().startswith("mlpChainKernelEqualF32"), cv.lastKernelName()
        ref = chain(params, x)
        assert torch.equal(torch.isnan(y), torch.isnan(ref))
        assert torch.equal(y[~torch.isnan(y)].view(torch.int32), ref[~torch.isnan(ref)].view(torch.int32)), (B, pad)


# the last and the first network whose pieces fit the LDS and do not, on either kernel; workgroups of eight waves, the last partly filled
@pytest.mark.parametrize("dims,last,split", [([128, 128, 80], Activation.NoActivation, False), ([128, 128, 96], Activation.NoActivation, True),
                                             ([101, 128, 67], Activation.NoActivation, False), ([101, 113, 85], Activation.NoActivation, True),
                                             ([128, 128, 48], Activation.Tanh, False), ([128, 128, 64], Activation.Tanh, True)])
def test_networks_that_fill_the_lds_equal_the_chain_of_single_layer_operators(dims, last, split):
    rng = np.random.default_rng(sum(dims))
    layers, params = network(rng, dims, [Activation.LeakyReLU, last])
    for B in (1, 113, 70001):
        x = to_dev(rng.uniform(-1, 1, (B, dims[0])).astype(np.float32))
        if B > 100:
            x[7, 0], x[B - 1, dims[0] - 1], x[50, 1], x[9, 2] = float("inf"), float("-inf"), 3.4e38, float("nan")
        y = cv.mlpForward(layers, x, weightType=CT.Float32)
        name = cv.lastKernelName()
        assert name.startswith("mlpChainKernel<" if last == Activation.NoActivation else "mlpFloatKernel<") and ("split at use" in name) == split, name
        ref = chain(params, x)
        assert torch.equal(torch.isnan(y), torch.isnan(ref))
        assert torch.equal(y[~torch.isnan(y)].view(torch.int32), ref[~torch.isnan(ref)].view(torch.int32)), B


# A training step over memory stays on the fp32 instruction, whose roundings, to nearest, cancel over samples; what the bfloat16 instruction
# drops it drops in one direction (means off by 1.3e-8 of the products there, by 6e-10 here).  Targets are the results in 64 bits,
# so that the bias gradient is the sum of the errors alone: each at most K roundings of 2^-24 of the sum so far, with signs as they
# come, hence over B samples a mean within 6 * sqrt(K / 12) * 2^-23 / sqrt(B) of the products' magnitudes, and a rounding of the targets.
# (The first layer is the identity.)
@pytest.mark.parametrize("dims", [[64, 24], [40, 130], [100, 48]])
def test_training_over_memory_keeps_the_means_of_rows(dims):
    rng = np.random.default_rng(sum(dims))
    B, (K, M) = 1 << 17, dims
    x = (rng.uniform(0, 1, (B, K)) * np.exp2(-rng.integers(0, 12, (B, K)))).astype(np.float32)
    W = (rng.uniform(0, 1, (M, K)) * np.exp2(-rng.integers(0, 6, (M, K)))).astype(np.float32)
    ref = x.astype(np.float64) @ W.astype(np.float64).T
    layers = [FeedForwardLayer(K, w.shape[0], as_bytes(to_dev(w)), None, ML.RowMajor, K * 4, Activation.NoActivation, 0.0,
                               as_bytes(torch.zeros(w.shape, device=DEV)), as_bytes(torch.zeros(w.shape[0], device=DEV)), ML.RowMajor, K * 4)
              for w in (np.eye(K, dtype=np.float32), W)]
    t = ref.astype(np.float32)
    cv.mlpTrainStep(layers, to_dev(x), to_dev(t), lossScale=0.5, weightType=CT.Float32)
    assert "layer-by-layer" in cv.lastKernelName(), cv.lastKernelName()
    mean = (layers[1].biasesGrad.view(torch.float32).cpu().numpy() + (t - ref).sum(axis=0)) / ref.sum(axis=0)
    print("mean errors of rows:", np.abs(mean).max(), np.abs(mean).mean())
    assert (np.abs(mean) <= 6 * np.sqrt(K / 12) * 2.0 ** -23 / np.sqrt(B)).all(), np.abs(mean).max()
