"""GPU parity of the input encodings in front of the MLP, through the C-ABI.

The example's encoding (network.slang:35-38) and loss (network.slang:58-75) are evaluated in half; the
test restates them with numpy float16 arithmetic (IEEE half, one rounding per operation) and feeds the
encoded vectors / targets to the un-encoded entry points, which the other tests hold to the oracle:
encoded and un-encoded launches must agree bit for bit."""
import numpy as np
import pytest
import torch

import oracle_binding as ob
from gpu_util import DEV, as_bytes, to_dev
from slang_amd import coopvec as cv
from slang_amd.coopvec import Activation, CoopVecComponentType as CT, CoopVecMatrixLayout as ML, FeedForwardLayer, InputEncoding
from test_gpu_train import build, make_specs, read_grads

pytestmark = pytest.mark.gpu


def encode_xy_squares(xy32: np.ndarray) -> np.ndarray:
    h = xy32.astype(np.float16)                                # (half2)inputs[tid], kernels.slang:19
    return np.concatenate([h, h * h], axis=1)                  # CoopVec<half,4>(x, y, x*x, y*y), network.slang:37


def groundtruth(xy32: np.ndarray) -> np.ndarray:
    h = xy32.astype(np.float16)
    x, y = h[:, 0], h[:, 1]
    one, two, hlf, c12 = np.float16(1), np.float16(2), np.float16(0.5), np.float16(1.2)
    return np.stack([(x + y) / (one + y * y), two * x + y, hlf * x * x + c12 * y, x + hlf * y * y], axis=1)   # network.slang:67-75


@pytest.mark.parametrize("dims,B", [([4, 16, 4], 1000), ([4, 64, 64, 4], 4099), ([4, 24, 9], 333)])
def test_forward_with_example_encoding(dims, B):
    rng = np.random.default_rng(sum(dims))
    specs = make_specs(rng, dims, act=Activation.LeakyReLU, slope=float(np.float16(0.001)))
    xy = rng.uniform(0, 1, (B, 2)).astype(np.float32)
    layers = build(specs)
    y_enc = cv.mlpForward(layers, to_dev(xy), inputEncoding=InputEncoding.XYSquares)
    y_ref = cv.mlpForward(layers, to_dev(encode_xy_squares(xy)))
    assert torch.equal(y_enc.view(torch.int16), y_ref.view(torch.int16))
    # strided float2 samples (two of every four floats)
    wide = to_dev(np.concatenate([xy, -xy], axis=1))
    y_str = cv.mlpForward(layers, wide[:, :2], inputEncoding=InputEncoding.XYSquares)
    assert torch.equal(y_str.view(torch.int16), y_ref.view(torch.int16))


@pytest.mark.parametrize("dims,B", [([4, 16, 4], 16), ([4, 16, 4], 2000), ([4, 64, 64, 4], 1500)])
def test_training_step_with_example_encoding_and_loss(dims, B):
    # learnGradient of the example: float2 samples in, encoding, loss against groundtruth(x, y) -- all in the kernel
    rng = np.random.default_rng(B)
    specs = make_specs(rng, dims, act=Activation.LeakyReLU, slope=float(np.float16(0.001)))
    specs[-1]["act"] = int(Activation.LeakyReLU)            # the example activates the last layer too (fflayer.slang:60-66)
    specs[-1]["slope"] = float(np.float16(0.001))
    xy = rng.uniform(0, 1, (B, 2)).astype(np.float32)
    la = build(specs, CT.Float32, ML.TrainingOptimal)
    _, loss_a = cv.mlpTrainStep(la, to_dev(xy), None, inputEncoding=InputEncoding.XYSquares)
    lb = build(specs, CT.Float32, ML.TrainingOptimal)
    _, loss_b = cv.mlpTrainStep(lb, to_dev(encode_xy_squares(xy)), to_dev(groundtruth(xy)))
    for a, b in zip(la, lb):
        assert torch.equal(a.weightsGrad, b.weightsGrad) and torch.equal(a.biasesGrad, b.biasesGrad)
    assert loss_a.item() == loss_b.item()
    # and the un-encoded launch is the one the oracle checks
    dW, dB = read_grads(lb, specs, CT.Float32, ML.TrainingOptimal)
    rW, rB, rloss = ob.ref_mlp_train(specs, encode_xy_squares(xy), groundtruth(xy), 1.0, tie_rule=True)
    for l in range(len(specs)):
        assert np.linalg.norm(dW[l] - rW[l]) <= 1e-3 * np.linalg.norm(rW[l])
    assert abs(loss_a.item() - rloss) <= 1e-3 * rloss


def test_encoding_argument_validation():
    rng = np.random.default_rng(0)
    layers = build(make_specs(rng, [8, 16, 4]))
    xy = torch.zeros(10, 2, dtype=torch.float32, device=DEV)
    with pytest.raises(cv.CoopVecError) as e:
        cv.mlpForward(layers, xy, inputEncoding=InputEncoding.XYSquares)     # first layer must take 4 inputs
    assert e.value.result == cv.SLANG_E_NOT_AVAILABLE
    layers = build(make_specs(rng, [4, 16, 3]))
    with pytest.raises(cv.CoopVecError) as e:
        cv.mlpTrainStep(layers, xy, None, inputEncoding=InputEncoding.XYSquares)    # the example's loss has 4 outputs
    assert e.value.result == cv.SLANG_E_INVALID_ARG


# ---- grid hashes and the permutohedral encoder ---------------------------------------------------
import json
import os

NG = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "neural_goldens.json")))


def test_grid_hash_goldens_and_random_positions():
    # integer work: bit-exact against tests/neural/hash-function-test.slang and the oracle
    pos = NG["hash"]["positions"]
    got = []
    for t in (cv.HashType.Prime, cv.HashType.CoherentPrime, cv.HashType.ReversedPrime, cv.HashType.BaseConvert, cv.HashType.Rng):
        for d in "1234":
            p = torch.tensor([pos[d]], dtype=torch.int32, device=DEV)
            got.append(int(cv.gridHash(t, p).cpu().numpy().view(np.uint32)[0]))
    p3 = torch.tensor([pos["3"]], dtype=torch.int32, device=DEV)
    got.append(int(cv.gridHash(cv.HashType.Prime, p3).cpu().numpy().view(np.uint32)[0]))
    got.append(int(cv.gridHash(cv.HashType.BaseConvert, p3).cpu().numpy().view(np.uint32)[0]))
    assert got == NG["hash"]["expected"]
    rng = np.random.default_rng(1)
    for dims in (1, 2, 3, 5, 7):
        grid = rng.integers(0, 2 ** 32, (3000, dims), dtype=np.uint64).astype(np.uint32)
        gd = to_dev(grid.view(np.int32))
        for t in range(5):
            want = np.array([ob.grid_hash(t, row) for row in grid[:300]], np.uint32)
            assert np.array_equal(cv.gridHash(t, gd).cpu().numpy().view(np.uint32)[:300], want), (t, dims)


def _reference_setup():
    from test_oracle_encoders import reference_setup
    return reference_setup()


def test_permuto_encoder_reference_data():
    # tests/neural/permuto-encoder-test.slang and -backward: the reference's expected values, to its epsilon
    P = NG["permuto"]; cfg = P["config"]
    pos, table, levels, max_level = _reference_setup()
    enc = cv.PermutoEncoder(2, 2, 8, 4, baseScale=cfg["baseScale"], log2PerLevelScale=cfg["log2PerLevelScale"],
                            maxLevelRatio=cfg["maxLevelRatio"], seed=cfg["seed"])
    out = enc.encode(to_dev(pos), to_dev(table)).cpu().numpy()
    want = np.array(P["expectedForward"]).reshape(16, 8)
    assert np.abs(out[P["verifyPositions"]] - want).max() <= cfg["epsilon"]
    assert np.array_equal(out, ob.permuto_encode(levels, 2, max_level, pos, table))      # same fp32 operations, same order
    d_pos, d_table = enc.backward(to_dev(pos), to_dev(table), torch.ones(256, 8, device=DEV))
    want_pos = np.array(P["expectedDLdPos"]).reshape(16, 2)
    got_pos = d_pos.cpu().numpy()[P["verifyPositions"]]
    assert (np.abs(got_pos - want_pos) <= cfg["epsilon"] + 1e-5 * np.abs(want_pos)).all()
    assert np.abs(d_table.cpu().numpy()[P["verifyParamIndices"]] - np.array(P["expectedDLdParams"])).max() <= cfg["epsilon"]


@pytest.mark.parametrize("D,F,levels_n", [(1, 1, 3), (3, 4, 6), (4, 2, 8), (6, 8, 2), (8, 2, 4)])
def test_permuto_encoder_against_oracle(D, F, levels_n):
    rng = np.random.default_rng(D * 100 + F)
    log2 = 10
    enc = cv.PermutoEncoder(D, F, log2, levels_n, baseScale=2.0, log2PerLevelScale=0.8, maxLevelRatio=0.8, seed=7)
    levels = ob.permuto_levels(D, log2, levels_n, 2.0, 0.8, 7)
    max_level = float(np.float32(0.8) * np.float32(levels_n))
    B = 5000
    pos = rng.uniform(0, 1, (B, D)).astype(np.float32)
    table = rng.standard_normal(enc.featureTableElements).astype(np.float32)
    out = enc.encode(to_dev(pos), to_dev(table)).cpu().numpy()
    assert np.array_equal(out, ob.permuto_encode(levels, F, max_level, pos, table))
    g = rng.standard_normal((B, levels_n * F)).astype(np.float32)
    d_pos, d_table = enc.backward(to_dev(pos), to_dev(table), to_dev(g))
    r_pos, r_table = ob.permuto_encode_backward(levels, F, max_level, pos, table, g)
    assert np.linalg.norm(d_pos.cpu().numpy() - r_pos) <= 1e-4 * np.linalg.norm(r_pos)
    assert np.linalg.norm(d_table.cpu().numpy() - r_table) <= 1e-4 * np.linalg.norm(r_table)
    # fp16 data: every product and sum rounded to half, as the generic T of the reference does
    enc16 = cv.PermutoEncoder(D, F, log2, levels_n, baseScale=2.0, log2PerLevelScale=0.8, maxLevelRatio=0.8, seed=7, dtype=torch.float16)
    p16, t16 = pos.astype(np.float16), table.astype(np.float16)
    o16 = enc16.encode(to_dev(p16), to_dev(t16)).cpu().numpy()
    assert np.array_equal(o16, ob.permuto_encode(levels, F, max_level, p16, t16))


@pytest.mark.parametrize("D,F,levels_n,log2", [(2, 2, 5, 8), (3, 8, 3, 6), (4, 1, 7, 12), (2, 4, 16, 4), (3, 2, 8, 14), (5, 4, 2, 9)])
def test_permuto_encoder_kernel_choices(D, F, levels_n, log2):
    # one thread per (position, level) with the table in LDS or in memory, level counts that are no power of two,
    # positions outside the unit cube, output rows at a pitch, and the one-thread-per-position kernel for what the
    # other does not take (more than four dimensions, entries over 16 bytes, unaligned buffers): all bit for bit the oracle
    rng = np.random.default_rng(D * 1000 + F * 10 + levels_n)
    levels = ob.permuto_levels(D, log2, levels_n, 1.5, 0.7, 99)
    max_level = float(np.float32(1.1) * np.float32(levels_n))
    B = 3001
    pos = rng.uniform(-4, 4, (B, D)).astype(np.float32)
    for dt, npdt in ((torch.float32, np.float32), (torch.float16, np.float16)):
        enc = cv.PermutoEncoder(D, F, log2, levels_n, baseScale=1.5, log2PerLevelScale=0.7, maxLevelRatio=1.1, seed=99, dtype=dt)
        p, t = pos.astype(npdt), rng.standard_normal(enc.featureTableElements).astype(npdt)
        want = ob.permuto_encode(levels, F, max_level, p, t)
        out = enc.encode(to_dev(p), to_dev(t))
        name = cv.lastKernelName()
        pairs = D <= 4 and F * np.dtype(npdt).itemsize <= 16
        assert name.startswith("permutoEncodePairsKernel" if pairs else "permutoEncodeKernel"), name
        assert np.array_equal(out.cpu().numpy(), want)
        # rows at a pitch of one extra entry; then a table that starts one element into its allocation
        wide = torch.zeros(B, levels_n * F + F, dtype=dt, device=DEV)
        enc.encode(to_dev(p), to_dev(t), out=wide[:, :levels_n * F])
        assert np.array_equal(wide[:, :levels_n * F].cpu().numpy(), want) and not wide[:, levels_n * F:].any()
        shifted = torch.zeros(t.size + 1, dtype=dt, device=DEV)
        shifted[1:] = to_dev(t)
        out2 = enc.encode(to_dev(p), shifted[1:])
        assert np.array_equal(out2.cpu().numpy(), want)
        if F > 1:
            assert cv.lastKernelName().startswith("permutoEncodeKernel"), cv.lastKernelName()


@pytest.mark.parametrize("D,F,levels_n,log2,B,kernel", [
    (2, 2, 4, 8, 2047, "permutoTableGradKernel<D=2,positions>"),           # the whole table in one workgroup's LDS
    (2, 2, 4, 8, 5000, "permutoTableGradKernel<D=2,4 parts,positions beside>"),   # the same table, a level to a part
    (3, 1, 2, 6, 1, "permutoTableGradKernel<D=3,positions>"),
    (2, 4, 3, 10, 1025, "permutoTableGradKernel<D=2,2 parts,positions beside>"),   # two levels, then one
    (3, 2, 8, 12, 4099, "permutoTableGradKernel<D=3,8 parts,positions beside>"),   # a level to a part
    (3, 4, 2, 12, 1023, "permutoTableGradKernel<D=3,2 parts,positions beside>"),   # beyond half a unit's LDS
    (2, 5, 2, 12, 300, "permutoTableGradKernel<D=2,2 parts,positions beside>"),    # the LDS full to the byte
    (2, 3, 2, 13, 2000, "permutoTableGradKernel<D=2,4 parts> + permutoBackwardKernel<D=2,positions>"),   # two slices to a level
    (3, 2, 2, 17, 3000, "permutoTableGradKernel<D=3,26 parts> + permutoBackwardKernel<D=3,positions>"),  # thirteen slices
    (2, 2, 1, 18, 2000, "permutoBackwardKernel<D=2,positions,table>"),     # too many slices: added in memory
])
def test_permuto_backward_table_parts(D, F, levels_n, log2, B, kernel):
    # Bound: the weights of an addend are differences of single-precision values below 2, off by at most 2^-22 against the
    # oracle's double ones, their mean is 1/(D+1), so a sum of addends is off by less than 2^-20 of its norm for D <= 3; the
    # sums (in double, or one by one in memory: at most 2^12 addends on an entry, each rounding 2^-25) stay within 2^-16.
    rng = np.random.default_rng(D * 1000 + F * 100 + levels_n * 10 + log2)
    enc = cv.PermutoEncoder(D, F, log2, levels_n, baseScale=3.0, log2PerLevelScale=1.0, maxLevelRatio=1.0, seed=11)
    levels = ob.permuto_levels(D, log2, levels_n, 3.0, 1.0, 11)
    pos = rng.uniform(-1, 1, (B, D)).astype(np.float32)
    table = rng.standard_normal(enc.featureTableElements).astype(np.float32)
    g = rng.standard_normal((B, levels_n * F)).astype(np.float32)
    r_pos, r_table = ob.permuto_encode_backward(levels, F, float(levels_n), pos, table, g)
    start = rng.standard_normal(table.size).astype(np.float32)              # gradients are added to what is there
    d_table = to_dev(start)
    d_pos, _ = enc.backward(to_dev(pos), to_dev(table), to_dev(g), dFeatureTable=d_table)
    assert cv.lastKernelName() == kernel
    got = d_table.cpu().numpy().astype(np.float64) - start
    rounding = 2.0 ** -23 * np.linalg.norm(start)                           # of the last sum, and of taking `start` out again
    assert np.linalg.norm(got - r_table) <= 2.0 ** -16 * np.linalg.norm(r_table) + rounding
    untouched = r_table == 0
    assert np.array_equal(d_table.cpu().numpy()[untouched], start[untouched])
    assert np.linalg.norm(d_pos.cpu().numpy() - r_pos) <= 1e-4 * np.linalg.norm(r_pos)
    # the table gradient alone: the same sums
    alone = torch.zeros_like(d_table)
    none, _ = enc.backward(to_dev(pos), to_dev(table), to_dev(g), dFeatureTable=alone, wantPositionGrad=False)
    assert none is None
    assert np.linalg.norm(alone.cpu().numpy() - r_table) <= 2.0 ** -16 * np.linalg.norm(r_table)


@pytest.mark.parametrize("F,tables,B,kernel", [
    # a third of the entries would be 1366 x 15 (683 x 30, 6827 x 3) doubles, ten (ten, one) more than the LDS holds
    (15, [(0, 4096), (4096, 4096)], 700, "permutoTableGradKernel<D=2,8 parts> + permutoBackwardKernel<D=2,positions>"),
    (30, [(0, 2048)], 500, "permutoTableGradKernel<D=2,4 parts> + permutoBackwardKernel<D=2,positions>"),
    (3, [(0, 20480)], 900, "permutoTableGradKernel<D=2,4 parts> + permutoBackwardKernel<D=2,positions>"),
    # small tables with gaps, in reverse order, on shared entries: up to 2047 positions all of them a single part, beyond a level to a part, but for
    # levels on the same entries
    (2, [(3, 256), (267, 256), (531, 100), (700, 256)], 2000, "permutoTableGradKernel<D=2,positions>"),
    (4, [(384, 128), (256, 128), (128, 128), (0, 128)], 2047, "permutoTableGradKernel<D=2,positions>"),
    (2, [(0, 256), (0, 256), (128, 256)], 1500, "permutoTableGradKernel<D=2,positions>"),
    (2, [(3, 256), (267, 256), (531, 100), (700, 256)], 5000, "permutoTableGradKernel<D=2,4 parts,positions beside>"),
    (4, [(384, 128), (256, 128), (128, 128), (0, 128)], 4097, "permutoTableGradKernel<D=2,4 parts,positions beside>"),
    (2, [(0, 256), (0, 256), (128, 256)], 4500, "permutoTableGradKernel<D=2,positions>"),
    # larger ones, a part to a level or in slices
    (2, [(20000, 4096), (3000, 8192), (3000, 8192)], 3000, "permutoTableGradKernel<D=2,3 parts,positions beside>"),
    (1, [(50, 40000), (0, 60), (45, 9000)], 2500, "permutoTableGradKernel<D=2,3 parts> + permutoBackwardKernel<D=2,positions>"),
])
def test_permuto_backward_of_other_tables(F, tables, B, kernel):
    # tables: (offset, size) in entries of every level.  The bound is that of test_permuto_backward_table_parts.
    rng = np.random.default_rng(F * 100 + B)
    n = len(tables)
    enc = cv.PermutoEncoder(2, F, 12, n, baseScale=3.0, log2PerLevelScale=1.0, maxLevelRatio=1.0, seed=11)
    levels = ob.permuto_levels(2, 12, n, 3.0, 1.0, 11)
    for l, (offset, size) in enumerate(tables):
        for record in (enc.desc.levelInfo[l], levels[l]):
            record.offsetOfFeatureTable, record.featureTableSize = offset, size
    pos = rng.uniform(-1, 1, (B, 2)).astype(np.float32)
    table = rng.standard_normal(max(o + s for o, s in tables) * F).astype(np.float32)
    g = rng.standard_normal((B, n * F)).astype(np.float32)
    r_pos, r_table = ob.permuto_encode_backward(levels, F, float(n), pos, table, g)
    d_table = torch.zeros(table.size, dtype=torch.float32, device=DEV)
    d_pos, _ = enc.backward(to_dev(pos), to_dev(table), to_dev(g), dFeatureTable=d_table)
    assert cv.lastKernelName() == kernel
    assert np.linalg.norm(d_table.cpu().numpy() - r_table) <= 2.0 ** -16 * np.linalg.norm(r_table)
    assert not d_table.cpu().numpy()[r_table == 0].any()
    assert np.linalg.norm(d_pos.cpu().numpy() - r_pos) <= 1e-4 * np.linalg.norm(r_pos)


@pytest.mark.parametrize("D,F,tables,B,parts", [
    (3, 2, [(4096 * l, 4096) for l in range(8)], 31745, 8),      # the fewest positions whose table workgroups fill 256 compute units
    (3, 2, [(4096 * l, 4096) for l in range(8)], 70001, 8),      # a last unit of 49 positions
    (2, 1, [(4096 * l, 4096) for l in range(5)], 131073, 3),     # two levels to a part, then one
    (4, 4, [(4096 * l, 4096) for l in range(2)], 131013, 2),     # the LDS of a compute unit to a part
    (2, 3, [(0, 8192), (8192, 8192)], 66000, 4),                 # slices
    (3, 2, [(0, 5000), (5000, 4096), (9096, 777)], 140000, 2),   # tables that are not 2^n entries
    (5, 2, [(4096 * l, 4096) for l in range(4)], 65536, 4),
    (2, 5, [(2048 * l, 2048) for l in range(4)], 65000, 4),
])
def test_permuto_backward_positions_beside_the_table(D, F, tables, B, parts):
    # One launch for both gradients: the position gradients are those of a launch of their own, bit for bit, which they have where they
    # are written on top of the positions; the table's the sum of parts of the batch by itself (in another order: bound as in
    # test_permuto_backward_table_parts).
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the batches are those of 256 compute units")
    rng = np.random.default_rng(D * 100 + F * 10 + len(tables))
    n = len(tables)
    enc = cv.PermutoEncoder(D, F, 12, n, baseScale=4.0, log2PerLevelScale=0.5, maxLevelRatio=1.0, seed=11)
    for l, (offset, size) in enumerate(tables):
        enc.desc.levelInfo[l].offsetOfFeatureTable, enc.desc.levelInfo[l].featureTableSize = offset, size
    pos = rng.uniform(-1, 1, (B, D)).astype(np.float32)
    pos[rng.integers(0, B, 20)] *= 3e6                            # beyond LatticeSimplex's reach
    pos, g = to_dev(pos), to_dev(rng.standard_normal((B, n * F)).astype(np.float32))
    table = to_dev(rng.standard_normal(max(o + s for o, s in tables) * F).astype(np.float32))
    d_table = torch.zeros_like(table)
    d_pos, _ = enc.backward(pos, table, g, dFeatureTable=d_table)
    assert cv.lastKernelName() == "permutoTableGradKernel<D=%d,%d parts,positions beside>" % (D, parts)
    into, both = pos.clone(), torch.zeros_like(table)
    rc = cv._lib.load().cvPermutoEncodeBackward(torch.cuda.current_stream().cuda_stream, cv.ctypes.byref(enc.desc), into.data_ptr(), 4 * D, table.data_ptr(),
                                                g.data_ptr(), 4 * n * F, into.data_ptr(), 4 * D, both.data_ptr(), B)
    assert rc == 0 and cv.lastKernelName().endswith(" + permutoBackwardKernel<D=%d,positions>" % D), cv.lastKernelName()
    assert torch.equal(d_pos, into)
    want_table = torch.zeros(table.numel(), dtype=torch.float64, device=DEV)
    for i in range(0, B, 16384):
        part = torch.zeros_like(table)
        enc.backward(pos[i:i + 16384], table, g[i:i + 16384], dFeatureTable=part, wantPositionGrad=False)
        want_table += part
    assert torch.linalg.norm(both - want_table) <= 2.0 ** -16 * torch.linalg.norm(want_table)
    assert torch.linalg.norm(d_table - want_table) <= 2.0 ** -16 * torch.linalg.norm(want_table)


@pytest.mark.parametrize("D,F,size", [(4, 4, 256), (4, 4, 255), (3, 4, 256), (4, 1, 1024)])
def test_permuto_backward_in_one_pass_of_one_and_two_workgroups(D, F, size):
    # one part of half the LDS or less, table and positions in a pass: up to 256 x 1024 positions one workgroup on a compute unit,
    # beyond that two, whose waves have half the registers.  Position gradients are the same, bit for bit.
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the batches are those of 256 compute units")
    L, B, part = 4, 256 * 1024 + 77, 256 * 1024
    enc = cv.PermutoEncoder(D, F, 4, L, baseScale=4.0, log2PerLevelScale=0.5, seed=3)
    for l in range(L):
        enc.desc.levelInfo[l].featureTableSize, enc.desc.levelInfo[l].offsetOfFeatureTable = size, size * l
    rng = np.random.default_rng(D * F + size)
    pos, table, g = (to_dev(rng.standard_normal(s).astype(np.float32)) for s in ((B, D), size * L * F, (B, L * F)))
    pos[torch.randint(0, B, (20,), device=DEV)] *= 3e6                # beyond LatticeSimplex's reach
    d_pos, d_table = enc.backward(pos, table, g)
    assert cv.lastKernelName() == "permutoTableGradKernel<D=%d,positions>" % D
    a_pos, want = enc.backward(pos[:part], table, g[:part])
    b_pos, _ = enc.backward(pos[part:], table, g[part:], dFeatureTable=want)
    assert torch.equal(d_pos, torch.cat((a_pos, b_pos)))
    assert torch.linalg.norm((d_table - want).double()) <= 2.0 ** -16 * torch.linalg.norm(want.double())


def test_permuto_backward_of_many_parts():
    # 144 parts, one workgroup each: the positions beside them up to 2^16, by a kernel of their own beyond
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the batches are those of 256 compute units")
    D, F, n, L, B = 2, 2, 16 * 10240, 9, (1 << 16) + 1
    enc = cv.PermutoEncoder(D, F, 4, L, baseScale=4.0, log2PerLevelScale=0.5, seed=3)
    for l in range(L):
        enc.desc.levelInfo[l].featureTableSize, enc.desc.levelInfo[l].offsetOfFeatureTable = n, n * l
    rng = np.random.default_rng(9)
    pos, table, g = (to_dev(rng.standard_normal(s).astype(np.float32)) for s in ((B, D), n * L * F, (B, L * F)))
    d_pos, d_table = enc.backward(pos, table, g)
    assert cv.lastKernelName() == "permutoTableGradKernel<D=2,144 parts> + permutoBackwardKernel<D=2,positions>", cv.lastKernelName()
    d_pos2, d_table2 = enc.backward(pos[:-1], table, g[:-1])
    assert cv.lastKernelName() == "permutoTableGradKernel<D=2,144 parts,positions beside>", cv.lastKernelName()
    enc.backward(pos[-1:], table, g[-1:], dFeatureTable=d_table2)
    assert torch.equal(d_pos[:-1], d_pos2)
    assert torch.linalg.norm((d_table - d_table2).double()) <= 2.0 ** -16 * torch.linalg.norm(d_table.double())


@pytest.mark.parametrize("D,F,tables,B,parts,kernel", [(3, 2, [1 << 12] * 8, 1 << 16, 8, "permutoTableGradKernel<D=3,8 parts> + permutoBackwardKernel<D=3,positions>"),
                                                        (2, 4, [1 << 8] * 4, 4099, 4, "permutoTableGradKernel<D=2,positions>"),
                                                        (3, 1, [1 << 15] * 3, 70001, 6, "permutoTableGradKernel<D=3,6 parts> + permutoBackwardKernel<D=3,positions>")])
@pytest.mark.parametrize("where", ["positions", "dOut"])
def test_permuto_backward_positions_on_top_of_inputs(D, F, tables, B, parts, kernel, where):
    # dPositions row on row of positions, or of the gradients that come in: as into a buffer of its own (beside the table's `parts` there)
    rng = np.random.default_rng(B)
    enc = cv.PermutoEncoder(D, F, 4, len(tables), baseScale=2.0, log2PerLevelScale=0.5, seed=5)
    for l, n in enumerate(tables):
        enc.desc.levelInfo[l].featureTableSize, enc.desc.levelInfo[l].offsetOfFeatureTable = n, sum(tables[:l])
    pos = to_dev(rng.uniform(-1, 1, (B, D)).astype(np.float32))
    table = to_dev(rng.standard_normal(sum(tables) * F).astype(np.float32))
    g = to_dev(rng.integers(-4, 5, (B, len(tables) * F)).astype(np.float32))
    want_pos, want_table = enc.backward(pos, table, g)
    assert cv.lastKernelName() == "permutoTableGradKernel<D=%d,%d parts,positions beside>" % (D, parts), cv.lastKernelName()
    d_table, into = torch.zeros_like(table), pos if where == "positions" else g
    lib = cv._lib.load()
    rc = lib.cvPermutoEncodeBackward(torch.cuda.current_stream().cuda_stream, cv.ctypes.byref(enc.desc), pos.data_ptr(), 4 * D, table.data_ptr(), g.data_ptr(),
                                     4 * g.shape[1], into.data_ptr(), 4 * into.shape[1], d_table.data_ptr(), B)
    assert rc == 0 and cv.lastKernelName() == kernel, cv.lastKernelName()
    assert torch.equal(into[:, :D], want_pos)
    assert torch.allclose(d_table, want_table, rtol=1e-6, atol=1e-4)


@pytest.mark.parametrize("D,F,levels_n,log2,B,in_memory", [
    (2, 4, 3, 10, 1, True), (2, 4, 3, 10, 40, True), (2, 4, 3, 10, 41, False),       # 36 additions to a position
    (3, 2, 8, 12, 22, True), (3, 2, 8, 12, 23, False), (1, 1, 4, 15, 64, True), (1, 1, 4, 15, 65, False),
    (2, 2, 9, 12, 3, False), (2, 3, 3, 12, 3, False),                                # 18 features; three to an entry
])
def test_permuto_backward_of_a_handful_of_positions(D, F, levels_n, log2, B, in_memory):
    # both sides of the rule that sends a few positions to the kernel that adds in memory; the bound is that of
    # test_permuto_backward_table_parts
    rng = np.random.default_rng(D * 1000 + F * 100 + levels_n * 10 + B)
    enc = cv.PermutoEncoder(D, F, log2, levels_n, baseScale=3.0, log2PerLevelScale=0.5, maxLevelRatio=1.0, seed=3)
    levels = ob.permuto_levels(D, log2, levels_n, 3.0, 0.5, 3)
    pos = rng.uniform(-1, 1, (B, D)).astype(np.float32)
    table = rng.standard_normal(enc.featureTableElements).astype(np.float32)
    g = rng.standard_normal((B, levels_n * F)).astype(np.float32)
    r_pos, r_table = ob.permuto_encode_backward(levels, F, float(levels_n), pos, table, g)
    for want_pos in (True, False):
        d_table = torch.zeros(table.size, dtype=torch.float32, device=DEV)
        d_pos, _ = enc.backward(to_dev(pos), to_dev(table), to_dev(g), dFeatureTable=d_table, wantPositionGrad=want_pos)
        assert cv.lastKernelName().startswith("permutoBackwardKernel" if want_pos and in_memory else "permutoTableGradKernel"), cv.lastKernelName()
        assert np.linalg.norm(d_table.cpu().numpy() - r_table) <= 2.0 ** -16 * np.linalg.norm(r_table)
        if want_pos:
            assert np.linalg.norm(d_pos.cpu().numpy() - r_pos) <= 1e-4 * np.linalg.norm(r_pos)


def test_permuto_backward_of_the_largest_batch():
    # 2^32 - 1 positions: workgroups are counted without leaving 32 bits.  Only the first and the last have a gradient, each
    # position's weights sum to 1.
    B = 0xffffffff
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 52 GB of memory")
    enc = cv.PermutoEncoder(1, 1, 6, 1, baseScale=3.0, log2PerLevelScale=1.0, maxLevelRatio=1.0, seed=11)
    pos, g = torch.zeros(B, 1, device=DEV), torch.zeros(B, 1, device=DEV)
    pos[-1], g[0], g[-1] = 0.75, 1, 2
    table = torch.randn(enc.featureTableElements, device=DEV)
    d_table = torch.zeros_like(table)
    d_pos, _ = enc.backward(pos, table, g, dFeatureTable=d_table)
    assert cv.lastKernelName().startswith("permutoTableGradKernel")
    want_pos, want_table = enc.backward(pos[[0, -1]].contiguous(), table, g[[0, -1]].contiguous())
    assert torch.equal(d_pos[[0, -1]], want_pos) and not d_pos[1:-1].any()
    assert torch.allclose(d_table, want_table, rtol=0, atol=2.0 ** -20) and abs(d_table.sum().item() - 3) <= 2.0 ** -20


def test_encoder_feeds_the_mlp():
    # encode positions, run the decoder MLP on the fp16 features: the neural-texture shape
    rng = np.random.default_rng(8)
    enc = cv.PermutoEncoder(3, 2, 12, 8, baseScale=4.0, log2PerLevelScale=1.0, dtype=torch.float16)
    B = 4096
    pos = to_dev(rng.uniform(0, 1, (B, 3)).astype(np.float16))
    table = to_dev((rng.standard_normal(enc.featureTableElements) * 0.5).astype(np.float16))
    feats = enc.encode(pos, table)
    specs = make_specs(rng, [16, 64, 64, 3])
    layers = build(specs)
    y = cv.mlpForward(layers, feats)
    ref = ob.ref_mlp_forward(specs, feats.cpu().numpy(), ob.F16)
    assert (np.abs(y.cpu().numpy().astype(np.float32) - ref.astype(np.float32)) <= 2e-2 * np.abs(ref.astype(np.float32)) + 2e-2).mean() > 0.999


@pytest.mark.parametrize("D,F,levels_n,log2,dims,B,kernel", [
    (3, 2, 8, 12, [16, 64, 64, 3], 4099, "permutoWide16Kernel"),     # the neural-texture shape; table (128 KB) and network in LDS
    (2, 2, 16, 8, [32, 32, 4], 777, "permutoWide16Kernel"),
    (4, 2, 8, 10, [16, 64, 8], 64, "permutoWide16Kernel"),
    (3, 2, 16, 11, [32, 64, 64, 1], 3000, "permutoWide16Kernel"),
    (2, 4, 4, 8, [16, 32, 5], 17, "permutoMlpKernel"),               # four features per entry
    (4, 1, 12, 10, [12, 128, 128, 7], 1000, "permutoMlpKernel"),     # 128-wide layers; a first layer narrower than its 16-column tile
    (3, 2, 8, 15, [16, 64, 64, 3], 2500, "permutoMlpKernel"),        # a 1 MB table stays in memory
    (1, 2, 16, 6, [32, 48, 16, 1], 1, "permutoMlpKernel"),
])
def test_encoder_and_network_in_one_kernel(D, F, levels_n, log2, dims, B, kernel):
    # cvPermutoMlpForward == cvPermutoEncode followed by cvMlpForward, bit for bit, on the 32-sample-tile kernel where the
    # decoder allows it and on the run-time-size kernel otherwise (or when asked for)
    rng = np.random.default_rng(D * 100 + F * 10 + len(dims))
    enc = cv.PermutoEncoder(D, F, log2, levels_n, baseScale=2.0, log2PerLevelScale=0.9, maxLevelRatio=0.9, seed=5, dtype=torch.float16)
    pos = to_dev(rng.uniform(-1, 2, (B, D)).astype(np.float16))
    table = to_dev((rng.standard_normal(enc.featureTableElements) * 0.5).astype(np.float16))
    specs = make_specs(rng, dims)
    if kernel == "permutoMlpKernel":
        specs[0]["act"], specs[0]["slope"] = 2, float(np.float16(0.01))      # a leaky layer among the ReLU ones
    layers = build(specs)
    feats = enc.encode(pos, table)
    want = cv.mlpForward(layers, feats)
    got = enc.encodeAndEval(pos, table, layers)
    name = cv.lastKernelName()
    assert name.startswith(kernel + "<D=%d,F=%d" % (D, F)), name
    if kernel == "permutoMlpKernel":
        assert name.endswith("memory>" if log2 == 15 else "LDS>"), name
    assert torch.equal(got, want)
    got16 = enc.encodeAndEval(pos, table, layers, flags=cv.FLAG_FORWARD_TILE16)
    assert cv.lastKernelName().startswith("permutoMlpKernel"), cv.lastKernelName()
    assert torch.equal(got16, want)
    levels = ob.permuto_levels(D, log2, levels_n, 2.0, 0.9, 5)
    max_level = float(np.float32(0.9) * np.float32(levels_n))
    f_ref = ob.permuto_encode(levels, F, max_level, pos.cpu().numpy(), table.cpu().numpy())
    assert np.array_equal(feats.cpu().numpy(), f_ref)
    # rows of the result at a pitch
    wide = torch.full((B, dims[-1] + 3), 7.0, dtype=torch.float16, device=DEV)
    enc.encodeAndEval(pos, table, layers, out=wide[:, :dims[-1]])
    assert torch.equal(wide[:, :dims[-1]], want) and bool((wide[:, dims[-1]:] == 7.0).all())


def test_encoder_and_network_argument_checks():
    rng = np.random.default_rng(3)
    enc = cv.PermutoEncoder(3, 2, 8, 4, baseScale=1.0, log2PerLevelScale=1.0, dtype=torch.float16)
    pos = to_dev(rng.uniform(0, 1, (8, 3)).astype(np.float16))
    table = to_dev(rng.standard_normal(enc.featureTableElements).astype(np.float16))
    with pytest.raises(cv.CoopVecError) as e:          # first layer does not match the encoder's output
        enc.encodeAndEval(pos, table, build(make_specs(rng, [16, 32, 4])))
    assert e.value.result == cv.SLANG_E_INVALID_ARG
    with pytest.raises(cv.CoopVecError) as e:          # a single layer is not a network
        enc.encodeAndEval(pos, table, build(make_specs(rng, [8, 4])))
    assert e.value.result == cv.SLANG_E_NOT_AVAILABLE
    enc5 = cv.PermutoEncoder(5, 2, 8, 4, baseScale=1.0, log2PerLevelScale=1.0, dtype=torch.float16)
    with pytest.raises(cv.CoopVecError) as e:          # five dimensions: the two-call form
        enc5.encodeAndEval(to_dev(rng.uniform(0, 1, (8, 5)).astype(np.float16)),
                           to_dev(rng.standard_normal(enc5.featureTableElements).astype(np.float16)), build(make_specs(rng, [8, 16, 4])))
    assert e.value.result == cv.SLANG_E_NOT_AVAILABLE


@pytest.mark.parametrize("D,F,levels_n,log2,dims,B", [
    (3, 2, 8, 12, [16, 64, 64, 3], 4099),       # permutoWide16Kernel, 16 inputs
    (2, 2, 16, 8, [32, 32, 4], 777),            # 32 inputs
    (4, 2, 8, 10, [16, 64, 8], 65),
    (4, 2, 16, 9, [32, 32, 32, 4], 1000),
    (2, 4, 4, 8, [16, 32, 5], 17),              # permutoMlpKernel
    (3, 2, 8, 15, [16, 64, 64, 3], 2500),       # a table in memory
])
@pytest.mark.parametrize("reach", [2.0, 3000.0])
def test_encoder_with_all_levels_in_use(D, F, levels_n, log2, dims, B, reach):
    # every level active and every table of 2^n entries, the kernels without branches inside a level: against the oracle, and
    # against the general kernels, which an encoder takes as soon as one of its tables has another size.  `reach`: lattice
    # coordinates beyond 24 bits of hash
    rng = np.random.default_rng(D * 100 + F * 10 + len(dims))
    enc = cv.PermutoEncoder(D, F, log2, levels_n, baseScale=2.0, log2PerLevelScale=0.9, seed=5, dtype=torch.float16)
    pos = to_dev(rng.uniform(-reach, reach, (B, D)).astype(np.float16))
    table = to_dev((rng.standard_normal(enc.featureTableElements) * 0.5).astype(np.float16))
    layers = build(make_specs(rng, dims))
    feats = enc.encode(pos, table)
    ref = ob.permuto_encode(ob.permuto_levels(D, log2, levels_n, 2.0, 0.9, 5), F, float(np.float32(1.1) * np.float32(levels_n)),
                            pos.cpu().numpy(), table.cpu().numpy())
    assert np.array_equal(feats.cpu().numpy(), ref)
    want = cv.mlpForward(layers, feats)
    assert torch.equal(enc.encodeAndEval(pos, table, layers), want)
    assert torch.equal(enc.encodeAndEval(pos, table, layers, flags=cv.FLAG_FORWARD_TILE16), want)
    odd = levels_n // 2
    enc.desc.levelInfo[odd].featureTableSize = (1 << log2) - 3
    feats2 = enc.encode(pos, table)
    keep = [i for i in range(levels_n * F) if i // F != odd]
    assert torch.equal(feats2[:, keep], feats[:, keep]) and (B < 32 or not torch.equal(feats2, feats))
    want2 = cv.mlpForward(layers, feats2)
    assert torch.equal(enc.encodeAndEval(pos, table, layers), want2)
    assert torch.equal(enc.encodeAndEval(pos, table, layers, flags=cv.FLAG_FORWARD_TILE16), want2)


@pytest.mark.parametrize("D", [1, 2, 3, 4])
def test_encoder_at_half_way_values(D):
    # The rounding to the nearest lattice point on the GPU (one instruction where D + 1 is a power of two) against the steps as the
    # reference has them, which a wave takes when one of its positions is out of reach: values in the middle between two lattice
    # points, their neighbours among the floats, and any others, up to the reach.
    L, F, log2, B = 1, 4, 12, 1 << 21
    enc = cv.PermutoEncoder(D, F, log2, L, baseScale=1.0, log2PerLevelScale=0.0, seed=1)
    lv = enc.desc.levelInfo[0]
    for d in range(D):
        lv.scalesPerDim[d], lv.shiftsPerDim[d] = 1.0, 0.0
    reach = 4194304.0 / sum(d + 2 for d in range(D))
    rng = np.random.default_rng(D)
    pos = (rng.integers(-1 << 22, 1 << 22, (B, D)) * 0.5 * np.exp2(-rng.integers(0, 21, (B, 1)))).astype(np.float32)
    pos = np.where(rng.random((B, D)) < 0.7, np.rint(2 * pos) / 2, pos).astype(np.float32)          # whole and half numbers
    if D == 1:
        pos[: 1 << 20, 0] = np.arange(1 << 20) * 2.0 + 1 - (1 << 20)                                # every middle to 2^20
    step = np.where(pos == 0, 0, rng.integers(-1, 2, (B, D)))     # (values below 2^-147 count as zero)
    pos = np.where(step == 0, pos, np.nextafter(pos, np.where(step > 0, np.inf, -np.inf).astype(np.float32))).clip(-reach, reach)
    table = to_dev(rng.standard_normal(enc.featureTableElements).astype(np.float32))
    pos = to_dev(pos.astype(np.float32))
    far = pos.clone()
    far[::64] = 1e30
    got, want = enc.encode(pos, table), enc.encode(far, table)
    keep = torch.arange(B, device=DEV) % 64 != 0
    assert torch.equal(got[keep].view(torch.int32), want[keep].view(torch.int32))
    g = to_dev(rng.standard_normal((B, F)).astype(np.float32))
    got, want = enc.backward(pos, table, g)[0], enc.backward(far, table, g)[0]
    assert torch.equal(got[keep], want[keep]), pos[keep][(got != want)[keep].any(dim=1)][:8]


@pytest.mark.parametrize("D,F,tables,B,kernel", [
    # one part; several levels to a part, then one: from 2048 positions on a level to a part
    (3, 4, [(512 * l, 512) for l in range(6)], 2047, "permutoTableGradKernel<D=3,2 parts,positions beside>"),
    (3, 4, [(512 * l, 512) for l in range(6)], 2048, "permutoTableGradKernel<D=3,6 parts,positions beside>"),
    (2, 1, [(64 * l, 64) for l in range(8)], 2049, "permutoTableGradKernel<D=2,8 parts,positions beside>"),
    (4, 2, [(300, 256), (0, 256), (700, 100), (800, 100)], 4097, "permutoTableGradKernel<D=4,4 parts,positions beside>"),      # gaps, another order
    (4, 2, [(300, 256), (0, 256), (700, 100), (700, 100)], 4097, "permutoTableGradKernel<D=4,positions>"),                     # levels on the same entries stay together
    (2, 4, [(1024 * l, 1024) for l in range(3)], 20001, "permutoTableGradKernel<D=2,3 parts,positions beside>"),
    # fewer units of positions than waves, one, and as many of them as waves; entries of three features
    (3, 2, [(4096 * l, 4096) for l in range(8)], 7168, "permutoTableGradKernel<D=3,8 parts,positions beside>"),
    (3, 2, [(4096 * l, 4096) for l in range(8)], 65, "permutoTableGradKernel<D=3,8 parts,positions beside>"),
    (4, 4, [(512 * l, 512) for l in range(8)], 1, "permutoTableGradKernel<D=4,2 parts,positions beside>"),
    (3, 2, [(4096 * l, 4096) for l in range(2)], 2048, "permutoTableGradKernel<D=3,2 parts,positions beside>"),
    (3, 3, [(2048 * l, 2048) for l in range(5)], 4096, "permutoTableGradKernel<D=3,5 parts,positions beside>"),
    (3, 1, [(4096, 4096)], 3000, "permutoTableGradKernel<D=3,positions>"),                                     # one level
])
def test_permuto_backward_spread_over_levels(D, F, tables, B, kernel):
    # the bounds are those of test_permuto_backward_table_parts
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the batches are those of 256 compute units")
    rng = np.random.default_rng(F * 100 + B)
    n = len(tables)
    enc = cv.PermutoEncoder(D, F, 12, n, baseScale=3.0, log2PerLevelScale=0.5, maxLevelRatio=1.0, seed=11)
    levels = ob.permuto_levels(D, 12, n, 3.0, 0.5, 11)
    for l, (offset, size) in enumerate(tables):
        for record in (enc.desc.levelInfo[l], levels[l]):
            record.offsetOfFeatureTable, record.featureTableSize = offset, size
    pos = rng.uniform(-1, 1, (B, D)).astype(np.float32)
    table = rng.standard_normal(max(o + s for o, s in tables) * F).astype(np.float32)
    g = rng.standard_normal((B, n * F)).astype(np.float32)
    r_pos, r_table = ob.permuto_encode_backward(levels, F, float(n), pos, table, g)
    d_table = torch.zeros(table.size, dtype=torch.float32, device=DEV)
    d_pos, _ = enc.backward(to_dev(pos), to_dev(table), to_dev(g), dFeatureTable=d_table)
    assert cv.lastKernelName() == kernel
    assert np.linalg.norm(d_table.cpu().numpy() - r_table) <= 2.0 ** -16 * np.linalg.norm(r_table)
    assert not d_table.cpu().numpy()[r_table == 0].any()
    assert np.linalg.norm(d_pos.cpu().numpy() - r_pos) <= 1e-4 * np.linalg.norm(r_pos)
    alone = torch.zeros_like(d_table)                                 # the table's gradient by itself
    enc.backward(to_dev(pos), to_dev(table), to_dev(g), dFeatureTable=alone, wantPositionGrad=False)
    assert np.linalg.norm(alone.cpu().numpy() - r_table) <= 2.0 ** -16 * np.linalg.norm(r_table)
