"""Performance cases: what a program built on this library has it do, through slang_amd.coopvec.

Each case is one pass over a batch of vectors already in GPU memory, into buffers the program keeps:

  matmul    one coopVecMatMulAdd (+ activation) over a batch
  forward   a whole network (MlpForwardPlan, or the neural module's FFLayer chain over one parameter block)
  train     a training step: forward, backward, gradients of every weight and bias
  iterate   a training step and the parameter update of the example's loop
  texture   permutohedral encoder + decoder network, one call
  encoder   reverse mode of the permutohedral encoder: gradients of feature table and positions

listed() holds the sizes the repository's own configurations and tests name (and ragged neighbours of them); draw()
gives sizes between the smallest and the largest of each kind.
"""
from __future__ import annotations

import math

import torch

from slang_amd import coopvec as cv
from slang_amd.coopvec import Activation, CoopVecComponentType as CT, CoopVecMatrixLayout as ML

DEVICE = "cuda"

DTYPE = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "i8": torch.int8, "e4m3": torch.float8_e4m3fn}
COMPONENT = {"f16": CT.Float16, "bf16": CT.BFloat16, "f32": CT.Float32, "i8": CT.SignedInt8, "e4m3": CT.FloatE4M3}
SIZE = {"f16": 2, "bf16": 2, "f32": 4, "i8": 1, "e4m3": 1}
# element type of biases and results
RESULT = {"f16": "f16", "bf16": "bf16", "f32": "f32", "i8": "i32", "e4m3": "f16"}
RESULT_DTYPE = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "i32": torch.int32}
RESULT_COMPONENT = {"f16": CT.Float16, "bf16": CT.BFloat16, "f32": CT.Float32, "i32": CT.SignedInt32}
RESULT_SIZE = {"f16": 2, "bf16": 2, "f32": 4, "i32": 4}
LAYOUT = {"row": ML.RowMajor, "column": ML.ColumnMajor, "optimal": ML.InferencingOptimal}
ACTIVATION = {"none": Activation.NoActivation, "relu": Activation.ReLU, "leaky": Activation.LeakyReLU}


def listed():
    return [
        # One iteration of the coopvec training example: 16 samples, a 4-16-4 network, step and Adam update; latency.
        dict(name="example_iteration", kind="iterate", elem="f16", widths="4-16-4", act="leaky", encode=True, batch=16),
        # A tiny network over a 256x256 image of coordinates: the smallest forward call that fills the card.
        dict(name="forward_f16_tiny", kind="forward", elem="f16", widths="2-16-16-16-1", act="relu", layout="row", block=False, batch=1 << 16),
        # The operator itself over a full-screen sized batch, fp16, weights converted once.
        dict(name="matmul_f16", kind="matmul", elem="f16", m=64, k=64, layout="optimal", act="none", batch=1 << 22),
        # Quantised inference layer: int8 vectors and matrix, int32 sums, weights as they lie in a file.
        dict(name="matmul_i8", kind="matmul", elem="i8", m=128, k=128, layout="column", act="none", batch=1 << 21),
        # 8-bit float network over 2^24 vectors: the largest forward batch.
        dict(name="forward_e4m3", kind="forward", elem="e4m3", widths="32-64-64-8", act="relu", layout="optimal", block=False, batch=1 << 24),
        # The neural module's FFLayer<float> chain over one parameter block.
        dict(name="forward_f32", kind="forward", elem="f32", widths="32-64-64-8", act="relu", layout="optimal", block=True, batch=1 << 22),
        # A network with layers of no particular size over a ragged batch.
        dict(name="forward_f16_ragged", kind="forward", elem="f16", widths="20-48-24-5", act="relu", layout="row", block=False, batch=2000003),
        # Training a radiance-cache sized half network, one large batch.
        dict(name="train_f16", kind="train", elem="f16", widths="8-64-64-64-64-1", act="relu", batch=1 << 20),
        # Training a wide half network (three 128-wide hidden layers) on an ordinary, ragged batch.
        dict(name="train_f16_wide", kind="train", elem="f16", widths="16-128-128-128-8", act="relu", batch=200003),
        # Training an FFLayer<float> network.
        dict(name="train_f32", kind="train", elem="f32", widths="32-64-64-8", act="relu", batch=1 << 20),
        # Neural texture lookup: encoder and decoder for every pixel of a 2048x2048 target.
        dict(name="texture_eval", kind="texture", elem="f16", dims=3, features=2, log2=12, levels=8, widths="16-64-64-3", batch=1 << 22),
        # Training the feature table of such an encoder: its reverse mode (which takes float vectors) over one training batch.
        dict(name="encoder_backward", kind="encoder", elem="f32", dims=3, features=2, log2=12, levels=8, batch=1 << 18),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_widths(rng, most_layers, widest):
    hidden = rng.randint(1, most_layers)
    if rng.random() < 0.6:      # most networks: equal hidden layers of a round size
        inner = [rng.choice([w for w in (16, 32, 64, 128) if w <= widest])] * hidden
    else:
        inner = [_spread(rng, 8, widest) for _ in range(hidden)]
    return "-".join(str(w) for w in [_spread(rng, 2, 64)] + inner + [_spread(rng, 1, 16)])


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "forward", "forward", "forward", "train", "train", "train", "iterate", "texture", "encoder"])
    if kind == "matmul":
        case = dict(kind=kind, elem=rng.choice(["f16", "bf16", "i8", "f32"]), m=_spread(rng, 8, 256), k=_spread(rng, 8, 256),
                    layout=rng.choice(["row", "column", "optimal"]), act=rng.choice(["none", "relu"]))
        low, high = 1 << 10, 1 << 22
    elif kind == "forward":
        elem = rng.choice(["f16", "f16", "e4m3", "f32", "bf16"])
        case = dict(kind=kind, elem=elem, widths=_draw_widths(rng, 4, 128), act=rng.choice(["relu", "relu", "leaky"]),
                    layout=rng.choice(["row", "optimal"]), block=False)
        low, high = 1 << 10, 1 << 22
    elif kind == "train":
        elem = rng.choice(["f16", "f16", "f32"])
        case = dict(kind=kind, elem=elem, widths=_draw_widths(rng, 4, 128 if elem == "f16" else 64), act=rng.choice(["relu", "relu", "leaky"]))
        low, high = 1 << 8, 1 << 20
    elif kind == "iterate":
        case = dict(kind=kind, elem="f16", widths=_draw_widths(rng, 2, 64), act="leaky", encode=False)
        low, high = 16, 1 << 14
    elif kind == "texture":
        features, levels = rng.choice([(2, 4), (2, 8), (4, 4), (2, 16), (4, 8)])
        hidden = rng.choice(["32", "64", "32-32", "64-64"])
        case = dict(kind=kind, elem="f16", dims=rng.choice([2, 3]), features=features, log2=rng.randint(8, 12), levels=levels,
                    widths="%d-%s-%d" % (features * levels, hidden, rng.randint(1, 8)))
        low, high = 1 << 12, 1 << 21
    else:
        case = dict(kind=kind, elem="f32", dims=rng.choice([2, 3]), features=rng.choice([1, 2, 4]),
                    log2=rng.randint(6, 12), levels=rng.randint(2, 8))
        low, high = 1 << 12, 1 << 18
    # no more work than the listed case of the kind
    case["batch"] = 1
    one = work(case)
    most = dict(matmul=(1.1e9, 1.4e11), forward=(1.1e9, 5.6e10), train=(4e8, 3.7e10), iterate=(4e8, 1e10), texture=(4e8, 5.4e10), encoder=(1e8, 1e12))[kind]
    case["batch"] = max(low, min(_spread(rng, low, high), int(most[0] / one["bytes"]), int(most[1] / max(1.0, one["flops"]))))
    return case


def _widths(case):
    return [int(w) for w in case["widths"].split("-")]


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _uniform(g, *shape):
    return torch.rand(*shape, device=DEVICE, generator=g) * 2 - 1


def _bytes(t):
    return t.contiguous().view(torch.uint8).flatten()


def _converted(t, rows, cols, component, layout):
    """The bytes of the row-major matrix `t` in `layout`, as a program lays its weights out once."""
    if layout == ML.RowMajor:
        return _bytes(t), cols * t.element_size()
    if layout == ML.ColumnMajor:
        return _bytes(t.t()), rows * t.element_size()
    size = cv.getCooperativeVectorMatrixSize(rows, cols, component, layout)
    out = torch.empty(size, dtype=torch.uint8, device=DEVICE)
    src = cv.CooperativeVectorMatrixDesc(rows, cols, component, ML.RowMajor, rows * cols * t.element_size(), 0, cols * t.element_size())
    dst = cv.CooperativeVectorMatrixDesc(rows, cols, component, layout, size, 0, 0)
    cv.convertCooperativeVectorMatrix(out, [dst], _bytes(t), [src])
    return out, 0


def _layers(g, case, layout, grad_dtype=None, last_act="none"):
    """The network's layers with He-initialised weights and small biases; gradients (all in one buffer, which is the second
    value) where grad_dtype is given."""
    widths, elem = _widths(case), case["elem"]
    component, carrier = COMPONENT[elem], RESULT_DTYPE[RESULT[elem]]
    layers, spans, total = [], [], 0
    grad_component = CT.Float32 if grad_dtype == torch.float32 else CT.Float16
    for fan_in, fan_out in zip(widths, widths[1:]):
        last = len(layers) == len(widths) - 2
        w = (torch.randn(fan_out, fan_in, device=DEVICE, generator=g) * (2.0 / fan_in) ** 0.5).to(DTYPE[elem])
        b = (_uniform(g, fan_out) * 0.1).to(carrier)
        data, stride = _converted(w, fan_out, fan_in, component, layout)
        layers.append(cv.FeedForwardLayer(fan_in, fan_out, data, _bytes(b), layout, stride,
                                          ACTIVATION[last_act if last else case["act"]], 0.001))
        if grad_dtype is not None:
            wsize = cv.getCooperativeVectorMatrixSize(fan_out, fan_in, grad_component, ML.TrainingOptimal)
            bsize = -(-fan_out * (4 if grad_dtype == torch.float32 else 2) // 16) * 16
            spans.append((total, wsize, total + wsize, fan_out * (4 if grad_dtype == torch.float32 else 2)))
            total += -(-(wsize + bsize) // 256) * 256
    if grad_dtype is None:
        return layers, None
    grads = torch.zeros(total // (4 if grad_dtype == torch.float32 else 2), dtype=grad_dtype, device=DEVICE)
    raw = grads.view(torch.uint8)
    for layer, (wo, wn, bo, bn) in zip(layers, spans):
        layer.weightsGrad, layer.biasesGrad = raw[wo:wo + wn], raw[bo:bo + bn]
        layer.gradLayout, layer.gradStride = ML.TrainingOptimal, 0
    return layers, grads


def prepare(case, seed):
    g = _generator(seed)
    kind, elem, batch = case["kind"], case["elem"], case["batch"]
    if kind == "matmul":
        m, k = case["m"], case["k"]
        if elem == "i8":
            x = torch.randint(-128, 128, (batch, k), dtype=torch.int8, device=DEVICE, generator=g)
            w = torch.randint(-127, 128, (m, k), dtype=torch.int8, device=DEVICE, generator=g)
            b = torch.randint(-65536, 65537, (m,), dtype=torch.int32, device=DEVICE, generator=g)
        else:
            x = torch.randn(batch, k, device=DEVICE, generator=g, dtype=DTYPE[elem])
            w = (torch.randn(m, k, device=DEVICE, generator=g) / k ** 0.5).to(DTYPE[elem])
            b = (_uniform(g, m) * 0.1).to(DTYPE[elem])
        data, stride = _converted(w, m, k, COMPONENT[elem], LAYOUT[case["layout"]])
        out = torch.empty(batch, m, dtype=RESULT_DTYPE[RESULT[elem]], device=DEVICE)
        return dict(case=case, x=x, w=data, stride=stride, b=_bytes(b), out=out)
    if kind == "forward":
        widths = _widths(case)
        x = (_uniform(g, batch, widths[0])).to(DTYPE[elem])
        out = torch.empty(batch, widths[-1], dtype=RESULT_DTYPE[RESULT[elem]], device=DEVICE)
        if case["block"]:
            conv = cv.NetworkParameterLayoutConverter(DTYPE[elem], (1 << (len(widths) - 1)) - 1, *widths)
            flat = [torch.randn(fo * fi, device=DEVICE, generator=g) * (2.0 / fi) ** 0.5 for fi, fo in zip(widths, widths[1:])]
            flat += [_uniform(g, fo) * 0.1 for fo in widths[1:]]
            params = conv.toOptimalLayout(torch.cat(flat).to(DTYPE[elem]))
            acts = [ACTIVATION[case["act"]]] * (len(widths) - 2) + [ACTIVATION["none"]]
            return dict(case=case, x=x, out=out, conv=conv, params=params, acts=acts)
        layers, _ = _layers(g, case, LAYOUT[case["layout"]])
        return dict(case=case, x=x, out=out, plan=cv.MlpForwardPlan(layers, weightType=COMPONENT[elem]))
    if kind in ("train", "iterate"):
        widths = _widths(case)
        iterate = kind == "iterate"
        encode = 1 if case.get("encode") else 0
        grad_dtype = torch.float16 if iterate else torch.float32
        layers, grads = _layers(g, case, ML.RowMajor, grad_dtype, last_act=case["act"] if iterate else "none")
        grad_type = CT.Float16 if iterate else CT.Float32
        x = torch.rand(batch, 2, device=DEVICE, generator=g) if encode else _uniform(g, batch, widths[0]).to(DTYPE[elem])
        t = None if encode else _uniform(g, batch, widths[-1]).to(DTYPE[elem])
        size = cv.mlpTrainStepWorkspaceSize(layers, batch, gradType=grad_type, inputEncoding=encode, weightType=COMPONENT[elem])
        state = dict(case=case, layers=layers, grads=grads, x=x, t=t, encode=encode, grad_type=grad_type,
                     workspace=torch.empty(size, dtype=torch.uint8, device=DEVICE), loss=torch.zeros(1, device=DEVICE))
        if iterate:
            # the mean over the samples, scaled so that half gradients neither overflow nor vanish; the example itself sums over its 16
            state["scale"] = 1.0 if batch <= 256 else 256.0 / batch
            state["weight_states"] = [torch.zeros(a * b * cv.ADAM_STATE_BYTES, dtype=torch.uint8, device=DEVICE) for a, b in zip(widths, widths[1:])]
            state["bias_states"] = [torch.zeros(b * cv.ADAM_STATE_BYTES, dtype=torch.uint8, device=DEVICE) for b in widths[1:]]
        else:
            state["scale"] = 1.0
        return state
    enc = cv.PermutoEncoder(case["dims"], case["features"], case["log2"], case["levels"], baseScale=4.0, log2PerLevelScale=0.5, dtype=DTYPE[elem])
    x = torch.rand(batch, case["dims"], device=DEVICE, generator=g).to(DTYPE[elem])
    table = (torch.randn(enc.featureTableElements, device=DEVICE, generator=g) * 0.5).to(DTYPE[elem])
    if kind == "texture":
        layers, _ = _layers(g, dict(case, act="relu"), ML.RowMajor)
        out = torch.empty(batch, _widths(case)[-1], dtype=torch.float16, device=DEVICE)
        return dict(case=case, enc=enc, x=x, table=table, layers=layers, out=out)
    grad = (_uniform(g, batch, enc.outputSize) / batch ** 0.5).to(DTYPE[elem])
    return dict(case=case, enc=enc, x=x, table=table, grad=grad)


def run(state):
    case = state["case"]
    kind, elem = case["kind"], case["elem"]
    if kind == "matmul":
        result = RESULT_COMPONENT[RESULT[elem]]
        return cv.coopVecMatMulAdd(state["x"], COMPONENT[elem], state["w"], 0, COMPONENT[elem], state["b"], 0, result, LAYOUT[case["layout"]],
                                   False, state["stride"], M=case["m"], resultType=result, out=state["out"], activation=ACTIVATION[case["act"]])
    if kind == "forward":
        if case["block"]:
            return state["conv"].eval(state["params"], state["x"], optimalLayout=True, activations=state["acts"], out=state["out"])
        return state["plan"](state["x"], state["out"])
    if kind == "train":
        state["grads"].zero_()
        cv.mlpTrainStep(state["layers"], state["x"], state["t"], lossScale=state["scale"], gradType=state["grad_type"],
                        workspace=state["workspace"], lossSum=state["loss"], weightType=COMPONENT[elem])
        return [state["grads"], state["loss"]]
    if kind == "iterate":
        cv.mlpTrainStep(state["layers"], state["x"], state["t"], lossScale=state["scale"], gradType=state["grad_type"],
                        workspace=state["workspace"], lossSum=state["loss"], inputEncoding=state["encode"])
        cv.mlpAdjustParameters(state["layers"], state["weight_states"], state["bias_states"], gradType=state["grad_type"])
        return [v.view(torch.float16) for layer in state["layers"] for v in (layer.weights, layer.biases)] + [state["loss"]]
    if kind == "texture":
        return state["enc"].encodeAndEval(state["x"], state["table"], state["layers"], out=state["out"])
    return state["enc"].backward(state["x"], state["table"], state["grad"])


def work(case):
    """Inputs read once, outputs written once; two flops per multiply-add of the unpadded layers."""
    kind, elem, batch = case["kind"], case["elem"], case["batch"]
    if kind == "matmul":
        m, k, out = case["m"], case["k"], RESULT_SIZE[RESULT[elem]]
        return {"bytes": float(batch * (k * SIZE[elem] + m * out) + m * k * SIZE[elem] + m * out), "flops": 2.0 * batch * m * k}
    if kind in ("texture", "encoder"):
        size = SIZE[elem]
        table = (1 << case["log2"]) * case["levels"] * case["features"] * size
        outputs, lookups = case["features"] * case["levels"], (case["dims"] + 1) * case["levels"] * case["features"]
        if kind == "encoder":      # per output feature and vertex: two multiply-adds into the table, two towards the positions
            return {"bytes": float(batch * (2 * case["dims"] + outputs) * size + 2 * table), "flops": 4.0 * batch * lookups}
        widths = _widths(case)
        macs = sum(a * b for a, b in zip(widths, widths[1:])) + lookups
        params = sum(a * b + b for a, b in zip(widths, widths[1:]))
        return {"bytes": float(batch * (case["dims"] + widths[-1]) * size + table + params * 2), "flops": 2.0 * batch * macs}
    widths = _widths(case)
    macs = sum(a * b for a, b in zip(widths, widths[1:]))
    params = macs + sum(widths[1:])
    if kind == "forward":
        return {"bytes": float(batch * (widths[0] * SIZE[elem] + widths[-1] * RESULT_SIZE[RESULT[elem]]) + params * SIZE[elem]), "flops": 2.0 * batch * macs}
    # forward, weight gradients, and input gradients of all layers but the first
    flops = 2.0 * batch * (3 * macs - widths[0] * widths[1])
    sample = 8 if case.get("encode") else (widths[0] + widths[-1]) * SIZE[elem]
    per_param = SIZE[elem] + 4
    if kind == "iterate":      # parameters, Adam state and gradients read and written
        per_param = 2 * (2 + 8 + 2)
    return {"bytes": float(batch * sample + params * per_param), "flops": flops}


def tolerance(case):
    """About four times what the path was seen to differ by from the same network evaluated with 64-bit sums and the same
    roundings between layers, or from itself with the batch in another order."""
    kind, elem = case["kind"], case["elem"]
    if kind == "matmul":
        if elem == "i8":
            return "exact"
        # one rounding of the sum: 2.1e-4 (half) and 1.7e-3 (bfloat16) of the norm; fp32 2e-7
        return {"f16": {"rel": 8e-4, "max": 4e-3}, "bf16": {"rel": 6e-3, "max": 3e-2}, "f32": {"rel": 1e-6, "max": 8e-6}}[elem]
    if kind in ("forward", "texture"):
        # hidden values whose sums lie at a rounding boundary take the other neighbour: half 6e-5 / 4e-3, bfloat16 1e-5 / 5e-3 (few
        # of them, each a whole unit of bfloat16); an e4m3 neighbour is a sixteenth away; fp32 2.6e-7 / 1.9e-6
        return {"f16": {"rel": 2.5e-4, "max": 1.5e-2}, "bf16": {"rel": 1e-3, "max": 2e-2}, "e4m3": {"rel": 1e-3, "max": 5e-2},
                "f32": {"rel": 1e-6, "max": 8e-6}}[elem]
    if kind == "train":
        # half: 1.4e-5 / 1e-4 in the worst layer; fp32: 3.2e-6 / 3e-5
        return {"f16": {"rel": 6e-5, "max": 1e-3}, "f32": {"rel": 1.5e-5, "max": 2e-4}}[elem]
    if kind == "iterate":
        # updated half parameters: one that rounds the other way is 1e-3 of itself
        return {"rel": 1e-3, "max": 5e-2}
    # fp32 sums in the order in which the positions arrive: 3.7e-6 / 2.2e-4 from run to run
    return {"rel": 1.5e-5, "max": 1e-3}
