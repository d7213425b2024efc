"""The framework's workloads as timed cases: what a user's program has it do, through its public entry points.

Kinds of case (the "kind" of each dict):

* linear     one eager call of an installed group-64 layer (actune_amd.layers.ResidentLinear): quantize + packed GEMM.
* mlp        one eager gated MLP: gate / up as sibling projections, act(gate) * up inside the down projection's
             quantizer, the down projection.
* layer      decoder blocks (q/k/v siblings, o, residual, gated MLP, residual) replayed by GraphReplay, as a decode or
             denoise step runs them.
* tokenwise  one eager call of a per-row layer of actune_amd.kernels.tokenwise (quantize + packed GEMM).
* calibrate  actune_amd.calibration.calibrate_linear of one layer: the channel scale, the clips and the errors.

Weights are N(0, 0.02), activations N(0, 1) with one percent of the channels ten times larger, as transformer layers
show them.
"""
import math

import torch

from actune_amd.calibration import calibrate_linear
from actune_amd.graph import GraphReplay
from actune_amd.kernels import tokenwise
from actune_amd.kernels.grouped import gated_down_forward, grouped_sibling_forward
from actune_amd.layers import ResidentLinear
from actune_amd.precision import CONFIGURATIONS

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
TOKENWISE = {"w4a8": tokenwise.W4A8TritonLinear, "w8a8": tokenwise.W8A8TritonLinear, "w2a8": tokenwise.W2A8TritonLinear,
             "w4a4": tokenwise.W4A4NativeLinear, "w2a4": tokenwise.W2A4NativeLinear,
             "w8a4": tokenwise.W8A4NativeLinear}
PAIRS = ["w%da%d" % (w, a) for w in (2, 4, 8) for a in (2, 4, 8)]
# the modes of a mixed-precision bank's block (an action expert: W8 keys, W2 output, the rest W4, all at A4)
MIXED = {"q": "w4a4", "k": "w8a4", "v": "w4a4", "o": "w2a4", "gate": "w4a4", "up": "w4a4", "down": "w4a4"}
MOST_FLOPS = 2 * 2000 * 11008 * 4096


def listed():
    return [
        # one projection of a 7B model for one token, called eagerly: the smallest call, launch and host latency
        dict(name="linear_m1", kind="linear", m=1, n=4096, k=4096, mode="w4a8", dtype="bf16", bias=False, scale=False),
        # one decoder layer of a 7B model for one token, as a replayed decode step: the packed weights' bandwidth
        dict(name="layer_m1", kind="layer", m=1, hidden=4096, kv=4096, inner=11008, blocks=1, mode="w4a8", act="silu"),
        # the action expert of a VLA policy (width 1024) on its 50-token chunk, mixed weight widths, replayed
        dict(name="expert_m50", kind="layer", m=50, hidden=1024, kv=256, inner=4096, blocks=2, mode="mixed", act="gelu"),
        # a 7B model's MLP for a ragged batch of decoding requests (between the decode and prefill ranges)
        dict(name="mlp_m40", kind="mlp", m=40, hidden=4096, inner=11008, mode="w4a8", dtype="bf16", act="silu"),
        # a VLA backbone's MLP (width 2048) on its 256 image and text tokens, 4-bit activations
        dict(name="mlp_m256_w4a4", kind="mlp", m=256, hidden=2048, inner=16384, mode="w4a4", dtype="bf16", act="gelu"),
        # prefill of a 512-token prompt: an attention projection at 8 bits with a calibrated channel scale and a bias
        dict(name="linear_m512_w8a8", kind="linear", m=512, n=4096, k=4096, mode="w8a8", dtype="bf16", bias=True,
             scale=True),
        # prefill of a 512-token prompt: the MLP of a 7B model
        dict(name="mlp_m512", kind="mlp", m=512, hidden=4096, inner=11008, mode="w4a8", dtype="bf16", act="silu"),
        # prefill of a long, ragged prompt: the largest call
        dict(name="linear_m2000", kind="linear", m=2000, n=11008, k=4096, mode="w4a8", dtype="bf16", bias=False,
             scale=False),
        # the per-row family: one token through a 7B model's down projection (its captured decode plan)
        dict(name="tokenwise_m1", kind="tokenwise", m=1, n=4096, k=11008, mode="w4a8", dtype="bf16"),
        # the per-row family: a 512-token prompt at 4 bits
        dict(name="tokenwise_m512_w4a4", kind="tokenwise", m=512, n=4096, k=4096, mode="w4a4", dtype="bf16"),
        # the per-row family: a long, ragged prompt at 8 bits
        dict(name="tokenwise_m1500_w8a8", kind="tokenwise", m=1500, n=11008, k=4096, mode="w8a8", dtype="bf16"),
        # calibration of one layer on a fitting set
        dict(name="calibrate", kind="calibrate", m=512, n=1024, k=1024, budget="w4a4"),
    ]


def draw(rng):
    def size(lo, hi, step=1):
        return max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step)

    kind = rng.choices(("linear", "mlp", "layer", "tokenwise", "calibrate"), (8, 3, 2, 5, 1))[0]
    dtype = rng.choices(("bf16", "f16", "f32"), (6, 1, 1))[0]
    mode = rng.choice(PAIRS + ["w4a8", "w4a4", "w8a8"] * 2)
    act = rng.choice(("silu", "gelu"))
    m = size(1, 2000)
    if kind == "linear":
        c = dict(kind=kind, m=m, n=size(256, 11008, rng.choice((1, 16))), k=size(256, 11008, 64), mode=mode, dtype=dtype,
                 bias=rng.random() < 0.3, scale=rng.random() < 0.3)
        c["m"] = max(1, min(m, MOST_FLOPS // (2 * c["n"] * c["k"])))
        return c
    if kind == "mlp":
        hidden = size(512, 4096, 64)
        inner = size(1024, 11008, 64)
        return dict(kind=kind, m=max(1, min(m, MOST_FLOPS // (6 * hidden * inner))), hidden=hidden, inner=inner, mode=mode,
                    dtype=dtype, act=act)
    if kind == "layer":
        hidden = size(512, 2560, 128)
        return dict(kind=kind, m=size(1, 300), hidden=hidden, kv=rng.choice((256, hidden)), inner=size(1024, 8192, 128),
                    blocks=rng.choice((1, 2)), mode=rng.choice(["mixed", "w4a8", "w4a4", "w8a8"]), act=act)
    if kind == "tokenwise":
        c = dict(kind=kind, m=m, n=size(256, 11008, rng.choice((1, 16))), k=size(256, 11008, 128),
                 mode=rng.choice(sorted(TOKENWISE)), dtype=dtype)
        c["m"] = max(1, min(m, MOST_FLOPS // (2 * c["n"] * c["k"])))
        return c
    return dict(kind=kind, m=size(64, 512), n=size(256, 1024, 16), k=size(256, 1024, 64),
                budget=rng.choice(("w4a4", "w4a8")))


# ------------------------------------------------------------------ inputs
def _normal(gen, *shape):
    return torch.randn(*shape, device=DEVICE, generator=gen)


def _weight(gen, n, k, dtype):
    return _normal(gen, n, k).mul_(0.02).to(dtype)


def _rows(gen, m, k, dtype):
    x = _normal(gen, m, k)
    x[:, torch.rand(k, device=DEVICE, generator=gen) < 0.01] *= 10
    return x.to(dtype)


def _shapes(case):
    """The case's linear layers: {name: (n, k, mode)} of one block, MLP or call."""
    kind = case["kind"]
    if kind in ("linear", "tokenwise"):
        return {"proj": (case["n"], case["k"], case["mode"])}
    h, i = case["hidden"], case["inner"]
    names = {"gate": (i, h), "up": (i, h), "down": (h, i)}
    if kind == "layer":
        names = {"q": (h, h), "k": (case["kv"], h), "v": (case["kv"], h), "o": (h, h), **names}
    return {name: (*nk, MIXED[name] if case["mode"] == "mixed" else case["mode"]) for name, nk in names.items()}


def _data(case, seed):
    """What the seed gives: the rows, and each block's weights (bias, channel scale) by layer name."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = DTYPES[case.get("dtype", "bf16")]
    k = case["k"] if "k" in case else case["hidden"]
    x = _rows(gen, case["m"], k, dtype)
    blocks = []
    for _ in range(case.get("blocks", 1)):
        block = {}
        for name, (n, kk, _mode) in _shapes(case).items():
            bias = _normal(gen, n).mul_(0.1).to(dtype) if case.get("bias") else None
            scale = (0.5 + 1.5 * torch.rand(kk, device=DEVICE, generator=gen)).to(dtype) if case.get("scale") else None
            block[name] = (_weight(gen, n, kk, dtype), bias, scale)
        blocks.append(block)
    return x, blocks


def _linear(weight, bias=None):
    fc = torch.nn.utils.skip_init(torch.nn.Linear, weight.shape[1], weight.shape[0], bias=bias is not None,
                                  device=weight.device, dtype=weight.dtype)
    with torch.no_grad():
        fc.weight.copy_(weight)
        if bias is not None:
            fc.bias.copy_(bias)
    return fc


def _resident(weight, bias, scale, mode):
    return ResidentLinear(_linear(weight, bias), {q: mode for q in CONFIGURATIONS}, {mode: None}, scale)


class _Block(torch.nn.Module):
    def __init__(self, layers, act):
        super().__init__()
        for name, layer in layers.items():
            setattr(self, name, layer)
        self.act = act

    def forward(self, x):
        q, k, v = grouped_sibling_forward(x, [self.q, self.k, self.v])
        h = x + self.o(q)
        gate, up = grouped_sibling_forward(h, [self.gate, self.up])
        return [k, v, h + gated_down_forward(self.down, gate, up, self.act)]


def _act(case):
    return torch.nn.SiLU() if case["act"] == "silu" else torch.nn.GELU(approximate="tanh")


def prepare(case, seed):
    if case["kind"] == "calibrate":
        gen = torch.Generator(device=DEVICE).manual_seed(seed)
        return {"case": case, "x": _rows(gen, case["m"], case["k"], torch.bfloat16),
                "linear": _linear(_weight(gen, case["n"], case["k"], torch.bfloat16))}
    x, blocks = _data(case, seed)
    state = {"case": case, "x": x}
    if case["kind"] == "tokenwise":
        weight, bias, _scale = blocks[0]["proj"]
        state["layer"] = TOKENWISE[case["mode"]](_linear(weight, bias))
        return state
    layers = [{name: _resident(*block[name], mode) for name, (_n, _k, mode) in _shapes(case).items()} for block in blocks]
    if case["kind"] == "linear":
        state["layer"] = layers[0]["proj"]
    elif case["kind"] == "mlp":
        state.update(layers[0], act=_act(case))
    else:
        modules = [_Block(block, _act(case)) for block in layers]

        def step(x):
            outs = []
            for module in modules:
                outs += module(x)
                x = outs[-1]
            return outs

        named = {"%d.%s" % (i, name): layer for i, block in enumerate(layers) for name, layer in block.items()}
        state["step"] = GraphReplay(step, named, shared_a8=True)
        state["step"].enabled = True
        state["step"](x)  # captures the graph that the program keeps
    return state


def run(state):
    kind = state["case"]["kind"]
    if kind == "calibrate":
        return calibrate_linear(state["linear"], state["x"], budget=state["case"]["budget"])
    with torch.inference_mode():
        if kind == "layer":
            return state["step"](state["x"])
        if kind == "mlp":
            gate, up = grouped_sibling_forward(state["x"], [state["gate"], state["up"]])
            return [gate, up, gated_down_forward(state["down"], gate, up, state["act"])]
        return state["layer"](state["x"])


# ------------------------------------------------------------------ what a pass needs
def _candidates(case):
    """GEMMs of a calibration: the float reference, five channel scales, nine clips of each pair."""
    return 6 + 9 * 3 * (3 if case["budget"] == "w4a4" else 1)


def work(case):
    m = case["m"]
    if case["kind"] == "calibrate":
        n, k = case["n"], case["k"]
        pairs = 9 if case["budget"] == "w4a4" else 3
        return {"bytes": 2 * n * k + 2 * m * k + 2 * k + 4 * n * pairs, "flops": 2 * m * n * k * _candidates(case)}
    size = 4 if case.get("dtype") == "f32" else 2
    shapes = _shapes(case)
    many = case.get("blocks", 1)
    weights = sum(n * k * int(mode[1]) // 8 + 4 * n for n, k, mode in shapes.values()) * many
    flops = sum(2 * m * n * k for n, k, _mode in shapes.values()) * many
    if case["kind"] in ("linear", "tokenwise"):
        n, k = case["n"], case["k"]
        extra = (n if case.get("bias") else 0) + (k if case.get("scale") else 0)
        return {"bytes": weights + size * (m * k + m * n + extra), "flops": flops}
    if case["kind"] == "mlp":
        return {"bytes": weights + size * m * (2 * case["hidden"] + 2 * case["inner"]), "flops": flops}
    return {"bytes": weights + size * m * (case["hidden"] + many * (2 * case["kv"] + case["hidden"])), "flops": flops}


def tolerance(case):
    # Codes and integer sums are exact; another correct order of the fp32 sums changes the last bit of some outputs, and
    # behind a second quantizer the codes that such a bit moves over a rounding boundary, more with each layer of a
    # block. Each line is four times what the path differs by from exact() rounded to the output's type: one layer
    # 7e-5 (bf16) and 1.5e-7 (f32), the largest single difference one last bit; an MLP 5e-4; two mixed blocks 1.9e-2.
    kind, dtype = case["kind"], case.get("dtype", "bf16")
    if kind == "calibrate":
        return {"rel": 2e-3, "max": 0.3}  # sums to 1e-7; a clip moves to its neighbour where two candidates nearly tie
    if kind == "layer":
        return {"rel": 3e-2, "max": 0.95}
    if kind == "mlp":
        return {"rel": 2e-3, "max": 0.1}
    if dtype == "f32":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 3e-4, "max": 4e-2} if dtype == "bf16" else {"rel": 4e-5, "max": 5e-3}


# ------------------------------------------------------------------ in 64 bits
def _codebook(weight, mode):
    """Weight codes (float64) and row scales (float64) of a layer on the GPU (divisions by 7 and 127 are products with
    their fp32 reciprocals there)."""
    w, a = int(mode[1]), int(mode[3])
    v = weight.float()
    amax = v.abs().amax(1).clamp_min(1e-8)

    def codes(scale, lo, hi):
        return (v / scale[:, None]).round().clamp(lo, hi)

    if w == 2:
        return codes(amax, -2, 1).double(), amax.double()
    if w == 8 and a != 4:
        scale = amax * (torch.ones((), device=DEVICE) / 127)
        return codes(scale, -128, 127).double(), scale.double()
    scale = amax * (torch.ones((), device=DEVICE) / 7)
    q4 = codes(scale, -8, 7)
    if w == 4:
        return q4.double(), scale.double()
    r4 = (16 * (v / scale[:, None] - q4)).round().clamp(-8, 7)
    r4 = torch.minimum(torch.maximum(r4, (-128 - 16 * q4).clamp_min(-8)), (127 - 16 * q4).clamp_max(7))
    return (16 * q4 + r4).double(), (scale / 16).double()


def _group64(x, a):
    """The group-64 activation codes times their scales, in float64."""
    p = 2 ** (a - 1) - 1
    g = x.float().reshape(x.shape[0], -1, 64)
    scale = g.abs().amax(2, keepdim=True).clamp_min(1e-8) / torch.full((), float(p), device=DEVICE)
    return ((g / scale).round().clamp(-p - 1, p).double() * scale.double()).reshape(x.shape)


def _exact_linear(x, weight, bias, scale, mode):
    a = int(mode[3])
    if scale is not None:
        weight = (weight * scale[None, :]).to(weight.dtype)
        x = (x / scale).to(x.dtype)
    if x.shape[1] % 128:
        pad = -x.shape[1] % 128
        x, weight = torch.nn.functional.pad(x, (0, pad)), torch.nn.functional.pad(weight, (0, pad))
    codes, ws = _codebook(weight, mode)
    y = (_group64(x, a) @ codes.t()) * ws
    return y if bias is None else y + bias.double()


def _exact_tokenwise(x, weight, mode):
    p = 2 ** (int(mode[3]) - 1) - 1
    v = x.float()
    scale = v.abs().amax(1, keepdim=True).clamp_min(1e-8) * (torch.ones((), device=DEVICE) / p)
    q = (v / scale).round().clamp(-p - 1, p).double()
    codes, ws = _codebook(weight, mode)
    return (q @ codes.t()) * scale.double() * ws


def _exact_mlp(x, block, shapes, act):
    """(gate, up, down) in float64; each layer's input is rounded to the activations' type, as the path does."""
    gate, up = (_exact_linear(x, *block[name], shapes[name][2]) for name in ("gate", "up"))
    product = act(gate.to(x.dtype)).mul_(up.to(x.dtype))
    return gate, up, _exact_linear(product, *block["down"], shapes["down"][2])


def _exact_calibration(case, x, weight):
    gains = torch.ones(case["n"], device=DEVICE, dtype=torch.float64)
    reference = x.double() @ weight.double().t()
    moment = x.float().abs().mean(0).clamp_min(1e-4)

    def clipped(w16, mode, ratio):
        # the clip shrinks the row scale; W8 with A2 or A8 takes none
        w, a = int(mode[1]), int(mode[3])
        v = w16.float()
        amax = v.abs().amax(1).clamp_min(1e-8)
        if w == 8 and a != 4:
            return _codebook(w16, mode)
        amax = amax if ratio is None else amax * ratio
        if w == 2:
            return (v / amax[:, None]).round().clamp(-2, 1).double(), amax.double()
        scale = amax / 7.0
        q4 = (v / scale[:, None]).round().clamp(-8, 7)
        if w == 4:
            return q4.double(), scale.double()
        r4 = (16.0 * (v / scale[:, None] - q4)).round().clamp(-8, 7)
        r4 = torch.minimum(torch.maximum(r4, (-128 - 16 * q4).clamp_min(-8)), (127 - 16 * q4).clamp_max(7))
        return (16 * q4 + r4).double(), (scale / 16.0).double()

    def loss(xs, w16, mode, ratio):
        codes, ws = clipped(w16, mode, ratio)
        return ((_group64(xs, int(mode[3])) @ codes.t()) * ws - reference).square().mean(0)

    base = "w4a4" if case["budget"] == "w4a4" else "w4a8"
    best = None
    for alpha in (0., .25, .5, .75, 1.):
        scale = moment.pow(alpha)
        scale = (scale / (scale.max() * scale.min()).sqrt()).clamp(1 / 16, 16).to(x.dtype)
        score = float((loss((x / scale).to(x.dtype), (weight * scale[None, :]).to(x.dtype), base, None) * gains).sum())
        if best is None or score < best[0]:
            best = score, scale
    scale = best[1]
    xs, w16 = (x / scale).to(x.dtype), (weight * scale[None, :]).to(x.dtype)
    clips, errors = {}, {}
    for w in (2, 4, 8):
        for a in ((8,) if base == "w4a8" else (2, 4, 8)):
            mode = "w%da%d" % (w, a)
            row = torch.full((case["n"],), math.inf, device=DEVICE, dtype=torch.float64)
            kept = torch.ones_like(row)
            for ratio in (1, .975, .95, .925, .9, .875, .85, .8, .75):
                now = loss(xs, w16, mode, ratio)
                better = now < row
                kept[better], row[better] = ratio, now[better]
            clips[mode], errors[mode] = kept, float((row * gains).sum())
    return dict(channel_scale=scale.double(), clips=clips, errors=errors, group_size=64)


def exact(case, seed):
    if case["kind"] == "calibrate":
        gen = torch.Generator(device=DEVICE).manual_seed(seed)
        x = _rows(gen, case["m"], case["k"], torch.bfloat16)
        return _exact_calibration(case, x, _weight(gen, case["n"], case["k"], torch.bfloat16))
    x, blocks = _data(case, seed)
    if case["kind"] == "linear":
        return _exact_linear(x, *blocks[0]["proj"], case["mode"])
    if case["kind"] == "tokenwise":
        return _exact_tokenwise(x, blocks[0]["proj"][0], case["mode"])
    shapes, act = _shapes(case), _act(case)
    if case["kind"] == "mlp":
        return list(_exact_mlp(x, blocks[0], shapes, act))
    outs = []
    for block in blocks:
        q, k, v = (_exact_linear(x, *block[name], shapes[name][2]) for name in ("q", "k", "v"))
        h = x + _exact_linear(q.to(x.dtype), *block["o"], shapes["o"][2]).to(x.dtype)
        out = h + _exact_mlp(h, block, shapes, act)[2].to(x.dtype)
        outs += [k, v, out.double()]
        x = out
    return outs
