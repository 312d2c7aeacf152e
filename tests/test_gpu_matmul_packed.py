"""matMul on vectors of any length, stride and alignment, through the C-ABI, against sums in 64 bits.

Every size runs on packed vectors, on vectors inside wider rows that begin at an odd element (with NaN, or bytes of the largest
magnitude, around them) and in the accumulate form; results inside wider rows must leave what lies beside them alone."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, as_bytes, matrix_in_layout, to_dev
from slang_amd import coopvec as cv
from slang_amd.coopvec import Activation, CoopVecComponentType as CT, CoopVecMatrixLayout as ML

pytestmark = pytest.mark.gpu

TYPES = {"f16": (torch.float16, CT.Float16, torch.float16, CT.Float16), "bf16": (torch.bfloat16, CT.BFloat16, torch.bfloat16, CT.BFloat16),
         "f32": (torch.float32, CT.Float32, torch.float32, CT.Float32), "i8": (torch.int8, CT.SignedInt8, torch.int32, CT.SignedInt32),
         "u8": (torch.uint8, CT.UnsignedInt8, torch.int32, CT.SignedInt32), "f16to32": (torch.float16, CT.Float16, torch.float32, CT.Float32)}
HALF_UNIT = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 0.0, "f16to32": 0.0}      # one rounding of the result (bfloat16: half of 2^-7)

# one row and one slot; remainders of 16 rows, of a fragment and of a tile; k-tiles 1 to 8; rows split between workgroups (few samples)
# and over the LDS (fp32 250 x 224); enough samples for two tiles a wave; a streaming size with samples left over
SIZES = [(1, 1, 1), (3, 5, 1), (15, 17, 16), (17, 33, 31), (16, 8, 33), (118, 13, 1000), (43, 101, 517), (156, 211, 70), (20, 160, 300),
         (33, 192, 200), (250, 224, 400), (256, 64, 333), (64, 64, 37), (9, 250, 129), (29, 30, 70003)]


def values(kind, rng, *shape):
    if kind in ("i8", "u8"):
        t = torch.from_numpy(rng.integers(-128 if kind == "i8" else 0, 128 if kind == "i8" else 256, shape).astype(np.int64))
        return t.to(TYPES[kind][0]).to(DEV)
    return torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).to(DEV).to(TYPES[kind][0])


def beside(kind, t, before, behind):
    """t as the middle columns of a wider tensor, and that tensor."""
    fill = {"i8": -128, "u8": 255}.get(kind, float("nan"))
    wide = torch.full((t.shape[0], before + t.shape[1] + behind), fill, dtype=t.dtype, device=DEV)
    wide[:, before:before + t.shape[1]] = t
    return wide[:, before:before + t.shape[1]]


@pytest.mark.parametrize("kind", list(TYPES))
@pytest.mark.parametrize("M,K,B", SIZES)
def test_any_length_stride_and_alignment(kind, M, K, B):
    rng = np.random.default_rng(M * 1000 + K)
    dt, ct, odt, oct = TYPES[kind]
    x, W = values(kind, rng, B, K), values(kind, rng, M, K)
    whole = kind in ("i8", "u8")
    b = torch.from_numpy(rng.integers(-65536, 65537, M).astype(np.int32)).to(DEV) if whole else values(kind, rng, M)
    x64, W64, b64 = x.cpu().double(), W.cpu().double(), b.cpu().double()
    ref = x64 @ W64.T + b64
    mag = x64.abs() @ W64.abs().T + b64.abs()

    def check(y, want, act=lambda v: v, magnitude=mag):
        want = act(want)
        if whole:
            assert torch.equal(y.cpu().double(), want), cv.lastKernelName()
            return
        bound = (K + 2) * 2.0 ** -23 * magnitude + HALF_UNIT[kind] * 1.01 * want.abs() + 2.0 ** -24
        assert ((y.cpu().double() - want).abs() <= bound).all(), cv.lastKernelName()

    def run(xs, layout=ML.RowMajor, out=None, act=Activation.NoActivation, bias=b, accumulate=False):
        if layout == ML.RowMajor:
            data, stride = as_bytes(W), K * W.element_size()
        elif layout == ML.ColumnMajor:
            data, stride = as_bytes(W.t()), M * W.element_size()
        else:
            raw = W.cpu().view(torch.int16).numpy() if kind == "bf16" else W.cpu().numpy()
            data, stride = to_dev(matrix_in_layout(raw, CT.Float16 if kind == "bf16" else ct, layout)), 0
        if accumulate:
            return cv.coopVecMatMul(xs, ct, data, 0, ct, layout, False, stride, M=M, resultType=oct, out=out, accumulate=True)
        return cv.coopVecMatMulAdd(xs, ct, data, 0, ct, as_bytes(bias), 0, oct if whole else ct, layout, False, stride, M=M, resultType=oct,
                                   out=out, activation=act)

    for layout in (ML.RowMajor, ML.ColumnMajor, ML.InferencingOptimal):
        check(run(x, layout), ref)
    plain = run(x)
    check(run(x, act=Activation.ReLU), ref, lambda v: v.clamp(min=0))
    odd = beside(kind, x, 3, 2)
    wide = torch.full((B, M + 4), 77, dtype=odt, device=DEV)
    y = run(odd, out=wide[:, 1:M + 1])
    assert torch.equal(y, plain)                         # the same bits, whatever lies beside the vectors
    assert (wide[:, 0] == 77).all() and (wide[:, M + 1:] == 77).all()
    start = values("f32", rng, B, M).to(odt)
    acc = beside("f32", start, 1, 1) if odt == torch.float32 else start.clone()
    run(odd, out=acc, accumulate=True)
    s64 = start.cpu().double()
    if kind in ("f16", "bf16"):                          # two roundings: of the product, of the sum
        bound = (K + 2) * 2.0 ** -23 * mag + HALF_UNIT[kind] * 1.01 * ((ref - b64).abs() + (ref - b64 + s64).abs()) + 2.0 ** -23
        assert ((acc.cpu().double() - (ref - b64 + s64)).abs() <= bound).all()
    else:
        check(acc, ref - b64 + s64, magnitude=mag + s64.abs())


@pytest.mark.parametrize("act", [Activation.LeakyReLU, Activation.Sigmoid, Activation.Tanh, Activation.Exp, Activation.Sine, Activation.SiLU,
                                 Activation.QuickGELU])
def test_activations_are_those_of_aligned_vectors(act):
    """Vectors of 40 elements in rows of 40 and in rows of 47: the same activation of the same sums (in half: of the rounded sum)."""
    rng = np.random.default_rng(int(act))
    for kind in ("f16", "f32"):
        dt, ct, _, _ = TYPES[kind]
        x, W, b = values(kind, rng, 97, 40), values(kind, rng, 37, 40) / 6, values(kind, rng, 37)
        y = cv.coopVecMatMulAdd(beside(kind, x, 3, 4), ct, as_bytes(W), 0, ct, as_bytes(b), 0, ct, ML.RowMajor, False, 40 * W.element_size(), M=37,
                                resultType=ct, activation=act, leakySlope=0.25)
        z = cv.coopVecMatMulAdd(x, ct, as_bytes(W), 0, ct, as_bytes(b), 0, ct, ML.RowMajor, False, 40 * W.element_size(), M=37, resultType=ct).double()
        s = 1.702 * z
        want = {Activation.LeakyReLU: torch.maximum(z, z * 0.25), Activation.Sigmoid: torch.sigmoid(z), Activation.Tanh: torch.tanh(z),
                Activation.Exp: torch.exp(z), Activation.Sine: torch.sin(z), Activation.SiLU: z * torch.sigmoid(z),
                Activation.QuickGELU: z * torch.sigmoid(s)}[act]
        # fp32 functions to a few of their own units, then one rounding to half
        tolerance = (2.0 ** -20 if kind == "f32" else 2.0 ** -11 * 1.01) * want.abs() + 2.0 ** -21
        assert ((y.double() - want).abs() <= tolerance).all(), (kind, cv.lastKernelName())


# Results on top of the vectors.  Small batches, whose rows would otherwise be split between workgroups; more samples than a round of tiles; whole
# aligned rows (streaming, and what it leaves), odd ones, results longer and shorter than the vectors.
@pytest.mark.parametrize("kind", list(TYPES))
@pytest.mark.parametrize("M,K,B", [(72, 72, 1000), (120, 120, 300), (128, 128, 2000), (64, 64, 1003), (33, 128, 517), (128, 17, 70), (1, 1, 40), (57, 59, 70003)])
def test_results_on_their_vectors(kind, M, K, B):
    if kind == "f32":
        M, K = min(M, 64), min(K, 64)
    rng = np.random.default_rng(M * 1000 + K)
    dt, ct, odt, oct = TYPES[kind]
    x, W = values(kind, rng, B, K), values(kind, rng, M, K)
    b = torch.from_numpy(rng.integers(-65536, 65537, M).astype(np.int32)).to(DEV) if oct == CT.SignedInt32 else values(kind, rng, M)

    def run(xs, out, accumulate=False):
        if accumulate:
            return cv.coopVecMatMul(xs, ct, as_bytes(W), 0, ct, ML.RowMajor, False, K * W.element_size(), M=M, resultType=oct, out=out, accumulate=True)
        return cv.coopVecMatMulAdd(xs, ct, as_bytes(W), 0, ct, as_bytes(b), 0, oct if oct == CT.SignedInt32 else ct, ML.RowMajor, False, K * W.element_size(),
                                   M=M, resultType=oct, out=out)

    isz, osz = x.element_size(), torch.empty(0, dtype=odt).element_size()
    pitch = -(-max(K * isz, M * osz) // osz) * osz
    for values_ in (x, x * 2 ** 16 if kind == "f32" else x):      # (fp32 from 2^32 on: the sums are formed again from the vectors)
        if kind == "f32" and values_ is not x:
            values_ = values_.clone()
            values_[::3, K // 2] = 2.0 ** 33
        for accumulate in (False, True):
            raw = torch.zeros(B * pitch, dtype=torch.uint8, device=DEV)
            vectors = raw.view(dt).as_strided((B, K), (pitch // isz, 1))
            vectors.copy_(values_)
            results = raw.view(odt).as_strided((B, M), (pitch // osz, 1))
            before = results.clone()
            want = run(values_, before if accumulate else torch.empty(B, M, dtype=odt, device=DEV), accumulate)
            run(vectors, results, accumulate)
            bits = torch.int16 if osz == 2 else torch.int32
            assert torch.equal(results.contiguous().view(bits), want.view(bits)), (accumulate, cv.lastKernelName())


# The same of the flavours that matmulKernel's general instantiation serves: half vectors taken as e4m3, e5m2 vectors, e4m3 ones on the e4m3 pipeline.
@pytest.mark.parametrize("vector,interpretation,flags", [(torch.float16, CT.FloatE4M3, 0), (torch.uint8, CT.FloatE5M2, 0), (torch.uint8, CT.FloatE4M3, 0),
                                                         (torch.uint8, CT.FloatE4M3, cv.FLAG_FP8_MATRIX_PIPELINE)])
@pytest.mark.parametrize("M,K,B", [(100, 100, 1000), (128, 128, 517), (17, 128, 40)])
def test_eight_bit_float_results_on_their_vectors(vector, interpretation, flags, M, K, B):
    rng = np.random.default_rng(M + K + int(interpretation))
    W = torch.from_numpy(rng.integers(0, 0x41, (M, K)).astype(np.uint8)).to(DEV)      # moderate values of either type
    x = torch.from_numpy(rng.standard_normal((B, K)).astype(np.float16)).to(DEV) if vector == torch.float16 else torch.from_numpy(rng.integers(0, 0x41, (B, K)).astype(np.uint8)).to(DEV)

    def run(xs, out):
        return cv.coopVecMatMul(xs, interpretation, W.flatten(), 0, interpretation, ML.RowMajor, False, K, M=M, resultType=CT.Float16, out=out, flags=flags)

    pitch = max(K * x.element_size(), 2 * M)
    raw = torch.zeros(B * pitch, dtype=torch.uint8, device=DEV)
    vectors, results = raw.view(vector).as_strided((B, K), (pitch // x.element_size(), 1)), raw.view(torch.float16).as_strided((B, M), (pitch // 2, 1))
    vectors.copy_(x)
    want = run(x, torch.empty(B, M, dtype=torch.float16, device=DEV))
    run(vectors, results)
    assert torch.equal(results.contiguous().view(torch.int16), want.view(torch.int16)), cv.lastKernelName()
