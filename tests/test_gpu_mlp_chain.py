"""mlpChainKernel (networks of any layer sizes, one straight-line arm per number of row tiles) against the chain of
single-layer operators, bit for bit, where it can go wrong: every number of row tiles, odd numbers of them, inputs of
whole groups of four elements and others, batches that end inside a tile and inside a pair of tiles, both rules of tiles
per wave, inputs and results inside larger buffers.  What lies around the input is NaN, so a read of a neighbour shows."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, to_dev
from slang_amd import coopvec as cv
from slang_amd.coopvec import Activation, CoopVecComponentType as CT, CoopVecMatrixLayout as ML
from test_gpu_mlp import chain_of_single_layers, gpu_layers, make_net
from test_gpu_mlp_float import TORCH, build, chain, to_T

pytestmark = pytest.mark.gpu

BATCHES = [1, 15, 16, 17, 33, 4097, 32769, 70001]      # 32768: above it (256 compute units) two tiles per wave
DIMS = [[20, 48, 24, 5], [3, 33, 80, 4], [64, 112, 96, 128, 12], [17, 16, 49, 1], [128, 65, 8], [4, 128, 7, 100]]


def surrounded(x, pad):
    """x inside a larger buffer of NaN bytes, rows `pad` elements further apart"""
    B, k = x.shape
    big = torch.full(((B * (k + pad) + 32) * x.element_size(),), 0xff, dtype=torch.uint8, device=DEV)
    rows = big.view(x.dtype)[16:16 + B * (k + pad)].view(B, k + pad)[:, :k]
    rows.copy_(x)
    return rows


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("ct", [CT.Float16, CT.FloatE4M3, CT.Float32, CT.BFloat16])
def test_chain_kernel_equals_single_layers(dims, ct):
    rng = np.random.default_rng(sum(dims) + int(ct))
    hidden = Activation.ReLU if len(dims) % 2 or ct == CT.FloatE4M3 else Activation.LeakyReLU
    floats = ct in TORCH
    L = len(dims) - 1
    if floats:
        acts = [hidden] * (L - 1) + [Activation.NoActivation]
        acts[min(1, L - 1)] = Activation.NoActivation              # (that layer has no bias)
        layers, params = build(rng, dims, ct, acts, ML.RowMajor)
    else:
        specs = make_net(rng, dims, ct, act=hidden, slope=0.125, bias="rand", init="he" if ct == CT.Float16 else "half")
        layers = gpu_layers(specs, ct, ML.InferencingOptimal)
    for B in BATCHES:
        for pad in (0, 1, 4):
            x64 = rng.uniform(-1, 1, (B, dims[0]))
            x = to_T(x64, ct) if floats else to_dev(x64.astype(np.float16))
            if ct == CT.FloatE4M3:
                x = x.to(torch.float8_e4m3fn)
            want = chain(params, x, ct, acts) if floats else chain_of_single_layers(specs, x, ct)
            out = torch.full((B + 2, dims[-1] + pad), -7.0, dtype=want.dtype, device=DEV)
            cv.mlpForward(layers, surrounded(x, pad), weightType=ct, out=out[1:B + 1, :dims[-1]])
            name = cv.lastKernelName()
            assert name.startswith("mlpChainKernel"), name
            bits = torch.int32 if want.element_size() == 4 else torch.int16
            assert torch.equal(out[1:B + 1, :dims[-1]].contiguous().view(bits), want.contiguous().view(bits)), (dims, ct, B, pad, name)
            assert (out[0] == -7).all() and (out[B + 1] == -7).all() and (out[:, dims[-1]:] == -7).all()


@pytest.mark.parametrize("ct", [CT.Float16, CT.Float32, CT.BFloat16])
def test_chain_kernel_keeps_non_finite_values_to_their_sample(ct):
    rng = np.random.default_rng(int(ct))
    dims, B = [20, 48, 24, 5], 40000
    acts = [Activation.ReLU, Activation.NoActivation, Activation.NoActivation]
    if ct in TORCH:
        layers, params = build(rng, dims, ct, acts, ML.RowMajor)
    else:
        specs = make_net(rng, dims, ct, act=Activation.ReLU, bias="rand", init="he")
        layers = gpu_layers(specs, ct, ML.RowMajor)
    x64 = rng.uniform(-1, 1, (B, dims[0]))
    x = to_T(x64, ct) if ct in TORCH else to_dev(x64.astype(np.float16))
    clean = cv.mlpForward(layers, x, weightType=ct).clone()
    x[37, 19], x[38, 0], x[B - 1, 3] = float("nan"), float("inf"), -float("inf")
    got = cv.mlpForward(layers, x, weightType=ct)
    want = chain(params, x, ct, acts) if ct in TORCH else chain_of_single_layers(specs, x, ct)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
    keep = torch.ones(B, dtype=torch.bool, device=DEV)
    keep[[37, 38, B - 1]] = False
    assert torch.equal(got[keep], clean[keep])


@pytest.mark.parametrize("ct,other", [(CT.Float16, "mlpGenericKernel"), (CT.FloatE4M3, "mlpGenericKernel"), (CT.Float32, "mlpFloatKernel"), (CT.BFloat16, "mlpFloatKernel")])
def test_rows_far_apart(ct, other):
    # sixteen vectors up to 2^26 bytes apart lie within the reach of a tile's descriptor; beyond that the kernel with run-time
    # sizes takes the network, with the same bits
    rng = np.random.default_rng(int(ct))
    dims, B = [20, 48, 24, 5], 33
    floats = ct in TORCH
    if floats:
        acts = [Activation.ReLU, Activation.NoActivation, Activation.NoActivation]
        layers, _ = build(rng, dims, ct, acts, ML.RowMajor)
    else:
        layers = gpu_layers(make_net(rng, dims, ct, act=Activation.ReLU, bias="rand", init="he" if ct == CT.Float16 else "half"), ct, ML.RowMajor)
    x64 = rng.uniform(-1, 1, (B, dims[0]))
    x = to_T(x64, ct) if floats else to_dev(x64.astype(np.float16))
    if ct == CT.FloatE4M3:
        x = x.to(torch.float8_e4m3fn)
    want = cv.mlpForward(layers, x, weightType=ct).clone()
    big = torch.zeros((B * ((1 << 26) + 16),), dtype=torch.uint8, device=DEV).view(x.dtype)
    for pitch, name in (((1 << 26), "mlpChainKernel"), ((1 << 26) + 16, other)):
        rows = big.as_strided((B, dims[0]), (pitch // x.element_size(), 1))
        rows.copy_(x)
        got = cv.mlpForward(layers, rows, weightType=ct)
        assert cv.lastKernelName().startswith(name), cv.lastKernelName()
        bits = torch.int32 if want.element_size() == 4 else torch.int16
        assert torch.equal(got.view(bits), want.view(bits))


# Vectors that begin at any element: every number of k-slots beyond a whole fragment and half of one (inputs 1 to 40), results of one to
# four rows beyond whole groups, matrices in rows that begin at any element; the last vector ends its buffer.  (What is read
# behind it does not show in the results: test_vector_reads.py checks that nothing is.)
@pytest.mark.parametrize("ct", [CT.Float16, CT.FloatE4M3, CT.Float32, CT.BFloat16])
def test_chain_kernel_takes_vectors_at_any_element(ct):
    floats = ct in TORCH
    bits = torch.int32 if ct == CT.Float32 else torch.int16
    for k in [1, 2, 5, 6, 7, 9, 15, 18, 31, 33, 34, 37, 39, 63, 97]:
        rng = np.random.default_rng(1000 * int(ct) + k)
        dims = [k, 19 if k < 64 else 70, 39, 24 + k % 4]      # (two sizes of hidden layer: not the kernel for equal ones)
        acts = [Activation.LeakyReLU, Activation.NoActivation, Activation.NoActivation]
        if floats:
            layers, params = build(rng, dims, ct, acts, ML.RowMajor)
        else:
            specs = make_net(rng, dims, ct, act=Activation.LeakyReLU, slope=0.125, bias="rand", init="he" if ct == CT.Float16 else "half")
            layers = gpu_layers(specs, ct, ML.RowMajor)
        for B, pad in [(1, 0), (23, 0), (23, 3), (32785, 1)]:
            x64 = rng.uniform(-1, 1, (B, k))
            x = to_T(x64, ct) if floats else to_dev(x64.astype(np.float16))
            if ct == CT.FloatE4M3:
                x = x.to(torch.float8_e4m3fn)
            want = chain(params, x, ct, acts) if floats else chain_of_single_layers(specs, x, ct)
            # the last vector ends where its buffer does; NaN before the first and between them
            size, each = x.element_size(), (k + pad) * x.element_size()
            big = torch.full(((B - 1) * each + k * size + size,), 0xff, dtype=torch.uint8, device=DEV)
            rows = big.view(x.dtype).as_strided((B, k), (k + pad, 1), 1)
            rows.copy_(x)
            out = torch.full((B * (dims[-1] + pad) + 1,), -7.0, dtype=want.dtype, device=DEV)
            res = out[1:].view(B, dims[-1] + pad)
            cv.mlpForward(layers, rows, weightType=ct, out=res[:, :dims[-1]])
            name = cv.lastKernelName()
            assert name.startswith("mlpChainKernel"), name
            assert torch.equal(res[:, :dims[-1]].contiguous().view(bits), want.contiguous().view(bits)), (k, ct, B, pad, name)
            assert out[0] == -7 and (res[:, dims[-1]:] == -7).all()


@pytest.mark.parametrize("slope", [2.0 ** -24, 0.001, 1.0, 1.5, 0.0, -0.5])
@pytest.mark.parametrize("ct", [CT.Float16, CT.FloatE4M3])
def test_leaky_slopes(ct, slope):
    # a positive slope takes the packed product, any other the choice element by element
    rng = np.random.default_rng(5)
    dims, B = [20, 48, 24, 5], 600
    specs = make_net(rng, dims, ct, act=Activation.LeakyReLU, slope=slope, bias="rand", init="he" if ct == CT.Float16 else "half")
    x = to_dev(rng.uniform(-1, 1, (B, dims[0])).astype(np.float16))
    x[3] = 0.0
    if ct == CT.FloatE4M3:
        x = x.to(torch.float8_e4m3fn)
    layers = gpu_layers(specs, ct, ML.InferencingOptimal)
    got = cv.mlpForward(layers, x, weightType=ct)
    assert cv.lastKernelName().startswith("mlpChainKernel")
    want = chain_of_single_layers(specs, x, ct)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
