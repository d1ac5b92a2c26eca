"""The work this framework's users have it do, as timed cases.

Each case is one pass through public entry points: the export of a layer at
round to nearest or from tuned parameters (``quantize_pack``), a layer's fake
quantization and fused sign step, the candidate-scale search, a step of the
single-layer loop, a decoder block's tuning step (forward, loss, backward), a
block's forward over the calibration stream, and the whole-model scoring pass.
The geometries are those of the repository's configurations (135M: hidden 576;
0.5B: 896; 3B: 2048; 7B: 3584) and, in the drawn cases, generic ones between
them.
"""

from __future__ import annotations

import math

import torch

from mround_amd import kernels as K
from mround_amd.core.quantizer import fake_quantize, quantize_pack
from mround_amd.core.scale_search import SearchGrid, search_scales
from mround_amd.core.signsgd import fused_step
from mround_amd.pipeline.block import LAYERS, QKV, BlockEngine, BlockShape, BlockWeights, aligned_length, placements
from mround_amd.pipeline.causal_lm import CausalLM
from mround_amd.pipeline.checkpoint import DecoderModel
from mround_amd.pipeline.runner import DecoderBlock
from mround_amd.schemes import QuantScheme, ScaleInit, Symmetry

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
# The last rate of a 200-step run at 1/200 (linear decay): repeated passes over
# one state leave its parameters where a tune has them.
LATE_LR = 0.005 / 200
EPS = 1e-8

G135M = dict(hidden=576, heads=9, kv=3, d=64, mlp=1536, bias=False)
G05B = dict(hidden=896, heads=14, kv=2, d=64, mlp=4864, bias=True)
G3B = dict(hidden=2048, heads=16, kv=2, d=128, mlp=11008, bias=True)
G7B = dict(hidden=3584, heads=28, kv=4, d=128, mlp=18944, bias=True)
GEOMETRIES = (G135M, G05B, G3B, G7B)


def listed() -> list[dict]:
    return [
        # Round-to-nearest export of the smallest linear there is (a 135M k
        # projection): latency of one call.
        dict(name="pack-192x576", kind="pack", rows=192, cols=576, bits=4, group=64, mode="asym", dtype="bf16",
             tuned=False),
        # Export of a tuned 7B gate projection at 3 bits, whose codes straddle words.
        dict(name="pack-18944x3584", kind="pack", rows=18944, cols=3584, bits=3, group=64, mode="sym", dtype="bf16",
             tuned=True),
        # One tuning step's fake quantization and sign step of a small linear:
        # seven of these run per step of a 135M block.
        dict(name="step-1536x576", kind="step", rows=1536, cols=576, bits=4, group=64, mode="asym", dtype="bf16"),
        # The same of the largest linear of the headline 2-bit workload.
        dict(name="step-18944x3584", kind="step", rows=18944, cols=3584, bits=2, group=64, mode="asym", dtype="bf16"),
        # One scale per output channel on a float16 checkpoint's weight (0.5B gate projection).
        dict(name="step-channel-f16", kind="step", rows=4864, cols=896, bits=4, group=-1, mode="sym", dtype="f16"),
        # The candidate-scale search that starts every symmetric tune below 4
        # bits, importance-weighted (3B gate projection).
        dict(name="search-11008x2048", kind="search", rows=11008, cols=2048, bits=2, group=64, dtype="bf16",
             importance=True),
        # A step of the single-layer loop on a 0.5B down projection, an uneven sample count.
        dict(name="layer-896x4864", kind="layer", rows=896, cols=4864, samples=1000, bits=3, group=64, mode="asym"),
        # A tuning step of a 135M block on the small calibration set (8 x 512): launches and latency.
        dict(name="block-135m", kind="block", **G135M, seqs=8, length=512, suppress=False),
        # A tuning step of a 0.5B block on sequences that are not whole tiles, with the outlier rule.
        dict(name="block-0.5b", kind="block", **G05B, seqs=4, length=1000, suppress=True),
        # The headline: a tuning step of a 7B block on 8 x 2048 tokens with the outlier rule.
        dict(name="block-7b", kind="block", **G7B, seqs=8, length=2048, suppress=True),
        # The targets pass of an 8-bit 3B block, which runs in split precision.
        dict(name="stream-3b-split", kind="stream", **G3B, seqs=2, length=2048, split=True),
        # A scoring batch of the mixed-precision planner: two 0.5B blocks under the full vocabulary.
        dict(name="score-0.5b", kind="score", **G05B, layers=2, vocab=151936, seqs=4, tokens=512, bits=4, group=64,
             mode="sym"),
    ]


# ------------------------------------------------------------------- drawn --

def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _geometry(rng) -> dict:
    """A repository geometry, or a generic one inside their range."""
    if rng.random() < 0.5:
        return dict(rng.choice(GEOMETRIES))
    d = rng.choice((64, 128))
    kv = rng.choice((1, 2, 4))
    per = rng.choice((1, 2, 3, 4, 7))
    heads = kv * per
    hidden = 64 * _log_int(rng, 4, 56) if rng.random() < 0.3 else d * heads
    return dict(hidden=hidden, heads=heads, kv=kv, d=d, mlp=64 * max(2, int(hidden * rng.uniform(2.5, 5.5)) // 64),
                bias=rng.random() < 0.5)


def _linear(rng) -> tuple[int, int]:
    """The shape of a linear of some geometry, or an uneven one."""
    if rng.random() < 0.75:
        g = _geometry(rng)
        q, kv = g["heads"] * g["d"], g["kv"] * g["d"]
        return rng.choice(((q, g["hidden"]), (kv, g["hidden"]), (g["hidden"], q), (g["mlp"], g["hidden"]),
                           (g["hidden"], g["mlp"])))
    return _log_int(rng, 33, 12000), 128 * _log_int(rng, 1, 32)


def draw(rng) -> dict:
    kind = rng.choice(("pack", "step", "step", "search", "layer", "block", "block", "block", "stream", "score"))
    if kind in ("pack", "step", "search"):
        rows, cols = _linear(rng)
        group = rng.choice([g for g in (32, 64, 64, 128) if cols % g == 0])
        dtype = "bf16" if rng.random() < 0.7 else "f32"
        if kind == "search":
            return dict(kind=kind, rows=rows, cols=cols, bits=rng.choice((2, 3)), group=group, dtype=dtype,
                        importance=rng.random() < 0.6)
        if kind == "pack":
            return dict(kind=kind, rows=rows, cols=cols, bits=rng.choice((2, 3, 4, 5, 6, 8)), group=group,
                        mode=rng.choice(("asym", "sym", "searched")), dtype=dtype, tuned=rng.random() < 0.5)
        u = rng.random()
        if u < 0.15:
            group, dtype = -1, rng.choice(("bf16", "f32", "f16"))
        elif u < 0.3:
            dtype = "f16"
        mode = rng.choice(("asym", "sym") if group == -1 else ("asym", "sym", "searched"))
        return dict(kind=kind, rows=rows, cols=cols, bits=rng.choice((2, 3, 4, 4, 8)), group=group, mode=mode,
                    dtype=dtype)
    if kind == "layer":
        return dict(kind=kind, rows=_log_int(rng, 16, 2048), cols=64 * _log_int(rng, 1, 48),
                    samples=_log_int(rng, 100, 6000), bits=rng.choice((2, 3, 4)), group=64,
                    mode=rng.choice(("asym", "sym")))
    g = _geometry(rng)
    length = rng.choice((128, 256, 512, 1024, 2048)) if rng.random() < 0.5 else _log_int(rng, 100, 2048)
    if kind == "score":
        return dict(kind=kind, **g, layers=rng.choice((1, 2)), vocab=_log_int(rng, 4000, 152064), seqs=rng.choice((1, 2, 4)),
                    tokens=min(length, 1024), bits=rng.choice((2, 3, 4)), group=64, mode=rng.choice(("asym", "sym")))
    seqs = rng.choice((1, 2, 3, 4, 8))
    if kind == "stream":
        split = rng.random() < 0.5
        return dict(kind=kind, **g, seqs=min(seqs, 4) if split else seqs, length=length, split=split)
    return dict(kind=kind, **g, seqs=seqs, length=length, suppress=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs --

class _Source:
    """Random inputs made on the device from one seed."""

    def __init__(self, seed: int) -> None:
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device=DEV) * std

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def weight(self, rows, cols, dtype):
        """N(0, 0.02) with 0.1 % of the entries ten times larger, as trained linears have."""
        w = self.normal(rows, cols, std=0.02)
        big = torch.rand(rows, cols, generator=self.g, device=DEV) < 1e-3
        return torch.where(big, w * 10, w).to(dtype)

    def stream(self, rows, cols):
        """A residual stream: unit variance, a few channels much larger than the rest."""
        return self.normal(rows, cols) * torch.exp(self.normal(cols, std=0.5))

    def params(self, rows, ng, gs):
        return {"v": self.uniform(rows, ng, gs, lo=-0.5, hi=0.5), "alpha": self.uniform(rows, ng, 1, lo=0.8, hi=1.0),
                "beta": self.uniform(rows, ng, 1, lo=0.8, hi=1.0)}


def _scheme(c) -> QuantScheme:
    mode = c.get("mode", "sym")
    return QuantScheme(bits=c["bits"], group_size=c["group"],
                       symmetry=Symmetry.ASYMMETRIC if mode == "asym" else Symmetry.SYMMETRIC,
                       scale_init=ScaleInit.SEARCHED if mode == "searched" else ScaleInit.OBSERVED_RANGE)


def _absmax_scale(w, gs, bits):
    """A starting scale per group near what the search finds: the clipped signed extreme."""
    x = w.float().reshape(w.shape[0], -1, gs)
    top = x.gather(2, x.abs().argmax(2, keepdim=True))
    return -0.9 * top / 2 ** (bits - 1)


def _layer_inputs(c, seed):
    src = _Source(seed)
    w = src.weight(c["rows"], c["cols"], DTYPES[c["dtype"]])
    gs = c["cols"] if c["group"] == -1 else c["group"]
    s = {"w": w, "scheme": _scheme(c), "params": None, "init": None}
    if c["kind"] == "step" or c["tuned"]:
        s["params"] = src.params(c["rows"], c["cols"] // gs, gs)
    if c["mode"] == "searched":
        s["init"] = _absmax_scale(w, gs, c["bits"])
        if s["params"] is not None:
            s["params"]["alpha"].fill_(1.0)
    if c["kind"] == "step":
        s["grad"] = src.normal(c["rows"], c["cols"], std=1e-4)
        s["out"] = torch.empty(c["rows"], c["cols"], dtype=torch.bfloat16, device=DEV)
    return s


def _shape(c) -> BlockShape:
    return BlockShape(hidden=c["hidden"], n_heads=c["heads"], n_kv_heads=c["kv"], head_dim=c["d"],
                      intermediate=c["mlp"], norm_eps=1e-6, rope_theta=1e6, attn_bias=c["bias"])


def _rtn(w, bits, gs):
    """Asymmetric round to nearest of a weight whose rows are whole groups, float32."""
    x = w.float().reshape(w.shape[0], -1, gs)
    hi, lo = x.amax(2, keepdim=True).clamp_min(0), x.amin(2, keepdim=True).clamp_max(0)
    s = ((hi - lo) / (2**bits - 1)).clamp_min(EPS)
    z = torch.round(-lo / s)
    return (s * ((torch.round(x / s) + z).clamp(0, 2**bits - 1) - z)).reshape(w.shape)


def _block_weights(src, shape) -> BlockWeights:
    lin = {n: src.weight(*shape.linear_shape(n), torch.bfloat16) for n in LAYERS}
    biases = {n: src.normal(shape.linear_shape(n)[0], std=0.1) for n in QKV} if shape.attn_bias else {}
    return BlockWeights(lin, biases, src.uniform(shape.hidden, lo=0.5, hi=1.5), src.uniform(shape.hidden, lo=0.5, hi=1.5))


def _block_inputs(c, seed):
    """Weights, W', input and target of a block case. The target differs from
    the input by heavy-tailed noise, so that the residual, a block's
    contribution less that noise, has the tails that the outlier rule cuts."""
    src, shape = _Source(seed), _shape(c)
    rows = aligned_length(c["length"])
    w = _block_weights(src, shape)
    bits = 8 if c["kind"] == "stream" else 3
    wq = {n: _rtn(t, bits, 64) for n, t in w.linears.items()}
    if not c.get("split"):
        wq = {n: t.to(torch.bfloat16) for n, t in wq.items()}
    T = c["seqs"] * rows
    x = src.stream(T, shape.hidden)
    target = x + src.normal(T, shape.hidden, std=0.3) * torch.exp(src.normal(T, 1, std=0.5)) if c["kind"] == "block" else None
    return shape, w, wq, x, target


def _model(c, seed):
    src, shape = _Source(seed), _shape(c)
    blocks = [DecoderBlock(i, f"model.layers.{i}", shape, _block_weights(src, shape)) for i in range(c["layers"])]
    embed = src.normal(c["vocab"], shape.hidden, std=0.02).to(torch.bfloat16)
    norm = src.uniform(shape.hidden, lo=0.5, hi=1.5)
    tokens = torch.randint(0, c["vocab"], (c["seqs"], c["tokens"]), generator=src.g, device=DEV)
    return DecoderModel({}, torch.bfloat16, embed, blocks, norm, None), tokens


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("pack", "step"):
        return dict(_layer_inputs(c, seed), kind=kind)
    if kind == "search":
        src = _Source(seed)
        return dict(kind=kind, w=src.weight(c["rows"], c["cols"], DTYPES[c["dtype"]]), scheme=_search_scheme(c),
                    imp=torch.exp(src.normal(c["cols"])) if c["importance"] else None)
    if kind == "layer":
        src, rows, cols, n = _Source(seed), c["rows"], c["cols"], c["samples"]
        w = src.weight(rows, cols, torch.bfloat16)
        e = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=DEV)
        zero = torch.zeros(n, rows, dtype=torch.float32, device=DEV)
        return dict(kind=kind, w=w, w32=w.float(), x=src.stream(n, cols), scheme=_scheme(c),
                    params=src.params(rows, cols // 64, 64), qdq=e(rows, cols), res=e(n, rows), zero=zero,
                    dres=e(n, rows), dw=e(rows, cols), loss=e(1), thr=e(1), ws=K.loss_workspace(zero.device, n * rows))
    if kind in ("block", "stream"):
        shape, w, wq, x, target = _block_inputs(c, seed)
        eng = BlockEngine(shape, batch=c["seqs"], seq_len=aligned_length(c["length"]), real_len=c["length"], device=DEV,
                          split=bool(c.get("split")))
        eng.set_block(w)
        eng.load_dense(wq)
        return dict(kind=kind, eng=eng, x=x, target=target, out=torch.empty_like(x), suppress=c.get("suppress"))
    model, tokens = _model(c, seed)
    lm = CausalLM(model, batch=c["seqs"], seq_len=c["tokens"], device=DEV, keep_activations=True)
    scheme = _scheme(c)
    lm.set_weights({f"{b.name}.{n}": scheme for b in model.blocks for n in LAYERS})
    return dict(kind=kind, lm=lm, model=model, tokens=tokens, scheme=scheme, place=placements(lm.shape),
                mode="asym" if c["mode"] == "asym" else "sym")


def _search_scheme(c):
    return QuantScheme(bits=c["bits"], group_size=c["group"], symmetry=Symmetry.SYMMETRIC, scale_init=ScaleInit.SEARCHED)


# --------------------------------------------------------------------- run --

def run(state):
    return {"pack": _run_pack, "step": _run_step, "search": _run_search, "layer": _run_layer, "block": _run_block,
            "stream": _run_stream, "score": _run_score}[state["kind"]](state)


def _run_pack(s):
    packed, scales, biases = quantize_pack(s["w"], s["params"], s["scheme"], init_scale=s["init"])
    return {"packed": packed.view(torch.int32), "scales": scales, "biases": biases}


def _run_step(s):
    fake_quantize(s["w"], s["params"], s["scheme"], init_scale=s["init"], out=s["out"])
    fused_step(s["w"], s["params"], s["grad"], s["scheme"], LATE_LR, init_scale=s["init"])
    return {"wq": s["out"], **s["params"]}


def _run_search(s):
    return search_scales(s["w"], s["scheme"], importance=s["imp"])


def _run_layer(s):
    """A step of ``core.tuning.tune_layer``'s loop, by the calls that make it:
    its results (the parameters after many sign steps) amplify every rounding
    error, a step's do not."""
    (rows, cols), n = s["w"].shape, s["x"].shape[0]
    fake_quantize(s["w"], s["params"], s["scheme"], out=s["qdq"])
    K.gemm_f32("nt", s["x"], s["qdq"], s["res"], M=n, N=rows, K=cols, b_minus=s["w32"])
    if s["scheme"].bits < 4:
        K.loss_outlier(s["res"], s["zero"], k=max(1, int(n * rows * 0.001)), denom=n * rows, loss_out=s["loss"],
                       threshold_out=s["thr"], grad_out=s["dres"], workspace=s["ws"])
    else:
        K.loss_mse(s["res"], s["zero"], denom=n * rows, loss_out=s["loss"], grad_out=s["dres"], workspace=s["ws"])
    K.gemm_f32("tn", s["dres"], s["x"], s["dw"], M=rows, N=cols, K=n)
    fused_step(s["w"], s["params"], s["dw"], s["scheme"], LATE_LR)
    return {"loss": s["loss"], "qdq": s["qdq"], "res": s["res"], "dw": s["dw"], "params": s["params"]}


def _run_block(s):
    eng = s["eng"]
    eng.forward(s["x"], s["out"], save=True)
    loss = eng.loss(s["out"], s["target"], suppress=s["suppress"], with_grad=True)
    eng.backward()
    out = s["out"].view(eng.batch, eng.seq_len, -1)[:, :eng.real_len]
    return {"loss": loss, "out": out, "dw": dict(eng.dw)}


def _run_stream(s):
    eng = s["eng"]
    eng.forward(s["x"], s["out"], save=False)
    return s["out"].view(eng.batch, eng.seq_len, -1)[:, :eng.real_len]


def _run_score(s):
    lm, model, place = s["lm"], s["model"], s["place"]
    scores = torch.zeros(len(model.blocks), len(LAYERS), 1, dtype=torch.float64, device=DEV)

    def on_block(b, dw):
        for i, name in enumerate(LAYERS):
            p = place[name]
            K.delta_loss_mapped(model.blocks[b].weights.linears[name], dw[p.operand], group_size=s["scheme"].group_size,
                                bits_list=[s["scheme"].bits], mode=s["mode"], eps=EPS, scores_out=scores[b, i],
                                row_block=p.row_block, row_stride=p.row_stride, row_offset=p.row_offset)

    loss = lm.run(s["tokens"], on_block)
    dlogits = lm.logits.view(lm.batch, -1, lm.logits.shape[1])[:, :lm.n_in, :lm.vocab]
    return {"loss": loss, "dlogits": dlogits, "scores": scores, "dw0": dict(lm.eng.dw)}


# -------------------------------------------------------------------- work --

def _block_params(c):
    h, q, kv = c["hidden"], c["heads"] * c["d"], c["kv"] * c["d"]
    return h * (q + 2 * kv) + h * q + 3 * h * c["mlp"]


def _block_flops(c, tokens, length, backward):
    """Products of a block, attention at its causal half; the backward is twice
    the linears (without the input gradient of q/k/v) and 2.5 times the attention."""
    lin = 2.0 * tokens * _block_params(c)
    attn = 2.0 * tokens * length * c["heads"] * c["d"]
    if not backward:
        return lin + attn
    qkv = 2.0 * tokens * c["hidden"] * (c["heads"] + 2 * c["kv"]) * c["d"]
    return 3 * lin - qkv + 3.5 * attn


def work(case):
    c, kind = case, case["kind"]
    wb = {"bf16": 2, "f16": 2, "f32": 4}
    if kind in ("pack", "step", "search"):
        n = c["rows"] * c["cols"]
        g = n // (c["cols"] if c["group"] == -1 else c["group"])
        size = wb[c["dtype"]]
        if kind == "pack":
            return {"bytes": n * (size + c["bits"] / 8 + 4 * c["tuned"]) + g * (4 + 8 * c["tuned"] + 4 * (c["mode"] == "searched")),
                    "flops": 0}
        if kind == "step":
            # forward: W, v in, W' out; step: W, v, gradient in, v out
            return {"bytes": n * (size + 4 + 2 + size + 4 + 4 + 4) + g * 24, "flops": 0}
        step, half = SearchGrid().steps(c["bits"])
        return {"bytes": n * size + g * 4, "flops": 8.0 * n * (2 * half + 1)}
    if kind == "layer":
        n = c["rows"] * c["cols"]
        return {"bytes": n * 22 + 4 * c["samples"] * (c["cols"] + c["rows"]), "flops": 4.0 * n * c["samples"]}
    P = _block_params(c)
    if kind == "block":
        T = c["seqs"] * c["length"]
        return {"bytes": P * (2 + 4) + T * c["hidden"] * 12, "flops": _block_flops(c, T, c["length"], True)}
    if kind == "stream":
        T, k = c["seqs"] * c["length"], 3 if c["split"] else 1
        return {"bytes": P * (4 if c["split"] else 2) + T * c["hidden"] * 8, "flops": k * _block_flops(c, T, c["length"], False)}
    L, T = c["tokens"] - 1, c["seqs"] * (c["tokens"] - 1)
    head = c["vocab"] * c["hidden"]
    return {"bytes": c["layers"] * P * 8 + head * 4 + T * c["vocab"] * 4,
            "flops": c["layers"] * _block_flops(c, T, L, True) + 4.0 * T * head}


# --------------------------------------------------------------- tolerance --

def tolerance(case):
    kind = case["kind"]
    if kind == "pack" or kind == "search":
        return "exact"
    if kind == "step":
        # v and W' are the same arithmetic everywhere; alpha and beta move by
        # the sign of a float32 sum, which its order can turn for a few groups.
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "layer":
        # Float32 products of a few thousand terms; the sign steps as above.
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "stream" and case["split"]:
        return {"rel": 1e-4}
    return {"rel": 0.025}


# ------------------------------------------------------------------- exact --

def _round_half_even(x):
    return torch.round(x)


def _quantize64(w, params, bits, gs, mode, init, dtype=torch.float64):
    """Fake quantization in float64 (or ``dtype``): W', the terms its gradient needs."""
    x = w.to(dtype).reshape(w.shape[0], -1, gs)
    if params is None:
        v, a, b = 0.0, 1.0, 1.0
    else:
        v, a, b = (params[k].to(dtype) for k in ("v", "alpha", "beta"))
    hi, lo = x.amax(2, keepdim=True).clamp_min(0), x.amin(2, keepdim=True).clamp_max(0)
    z, pos = 0.0, None
    if mode == "asym":
        maxq, qmin, qmax = 2**bits - 1, 0, 2**bits - 1
        s = ((hi * a - lo * b) / maxq).clamp_min(EPS)
        z = _round_half_even(-(lo * b) / s)
    else:
        maxq, qmin, qmax = 2 ** (bits - 1), -(2 ** (bits - 1)), 2 ** (bits - 1) - 1
        if mode == "searched":
            signed = init.to(dtype).reshape(x.shape[0], -1, 1) * b
        else:
            pos = hi * a >= -(lo * b)
            signed = torch.where(pos, -(hi * a), -(lo * b)) / maxq
        s = torch.where(signed < 0, -1.0, 1.0) * signed.abs().clamp_min(EPS)
    raw = _round_half_even(x / s + v) + z
    code = raw.clamp(qmin, qmax)
    inside = (raw >= qmin) & (raw <= qmax)
    q = (s * (code - z)).reshape(w.shape)
    return q, dict(x=x, s=s, z=z, code=code, inside=inside, hi=hi, lo=lo, pos=pos, maxq=maxq, b=b, init=init)


def _grad64(t, grad, mode):
    """Straight-through gradients of (v, alpha, beta) from ``_quantize64``'s terms."""
    g = grad.double().reshape(t["x"].shape)
    gv = g * t["s"] * t["inside"]
    if mode == "asym":
        off = t["lo"] * t["b"] / t["s"]
        ds = (g * (t["code"] - t["z"] - torch.where(t["inside"], t["x"] / t["s"], off))).sum(2, keepdim=True)
        direct = (g * ~t["inside"] * t["lo"]).sum(2, keepdim=True)
        return gv, ds * t["hi"] / t["maxq"], -ds * t["lo"] / t["maxq"] + direct
    ds = (g * (t["code"] - t["inside"] * t["x"] / t["s"])).sum(2, keepdim=True)
    if mode == "searched":
        return gv, torch.zeros_like(ds), ds * t["init"].double().reshape(ds.shape)
    zero = torch.zeros_like(ds)
    return gv, torch.where(t["pos"], -ds * t["hi"] / t["maxq"], zero), torch.where(t["pos"], zero, -ds * t["lo"] / t["maxq"])


def _stepped64(params, grads, lr, mode):
    lo, hi = (0.5, 1.5) if mode == "searched" else (0.1, 1.0)
    gv, ga, gb = grads
    return {"v": (params["v"].double() - lr * gv.sign()).clamp(-0.5, 0.5),
            "alpha": (params["alpha"].double() - lr * ga.sign()).clamp(lo, hi),
            "beta": (params["beta"].double() - lr * gb.sign()).clamp(lo, hi)}


def _rope64(x, theta):
    S, d = x.shape[-2], x.shape[-1]
    inv = theta ** (-torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)
    ang = torch.arange(S, dtype=torch.float64, device=x.device)[:, None] * inv
    a, b = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _block64(c, wq, w, x):
    """A block over ``[B, S, h]`` in float64 (autograd follows it to ``wq`` and ``x``)."""
    B, S, _ = x.shape
    d, hq, kv = c["d"], c["heads"], c["kv"]
    norm = lambda t, g: t * torch.rsqrt((t * t).mean(-1, keepdim=True) + 1e-6) * g.double()
    x1 = norm(x, w.input_norm)
    proj = lambda n: x1 @ wq[n].t() + (w.biases[n].double() if n in w.biases else 0.0)
    q = _rope64(proj("self_attn.q_proj").view(B, S, hq, d).transpose(1, 2), 1e6)
    k = _rope64(proj("self_attn.k_proj").view(B, S, kv, d).transpose(1, 2), 1e6)
    v = proj("self_attn.v_proj").view(B, S, kv, d).transpose(1, 2)
    hidden = torch.ones(S, S, dtype=torch.bool, device=x.device).triu(1)
    heads = []
    for h in range(hq):
        kk, vv = k[:, h * kv // hq], v[:, h * kv // hq]
        s = (q[:, h] @ kk.transpose(1, 2).contiguous() * d**-0.5).masked_fill(hidden, float("-inf"))
        heads.append(torch.softmax(s, -1) @ vv)
    h = x + torch.cat(heads, -1) @ wq["self_attn.o_proj"].t()
    x2 = norm(h, w.post_norm)
    act = torch.nn.functional.silu(x2 @ wq["mlp.gate_proj"].t()) * (x2 @ wq["mlp.up_proj"].t())
    return h + act @ wq["mlp.down_proj"].t()


def _fused(dw):
    """Per-layer gradients in the engine's operand layouts: q/k/v stacked, gate and up rows interleaved by 32."""
    g, u = dw["mlp.gate_proj"], dw["mlp.up_proj"]
    gu = torch.stack([g.view(-1, 32, g.shape[1]), u.view(-1, 32, u.shape[1])], 1).reshape(-1, g.shape[1])
    return {"qkv": torch.cat([dw[n] for n in QKV]), "o": dw["self_attn.o_proj"], "gu": gu, "down": dw["mlp.down_proj"]}


def _exact_block(c, seed):
    shape, w, wq, x, target = _block_inputs(c, seed)
    S, r = aligned_length(c["length"]), c["length"]
    leaf = {n: t.double().requires_grad_(c["kind"] == "block") for n, t in wq.items()}
    rows = lambda t: t.view(c["seqs"], S, -1)[:, :r]
    if c["kind"] == "stream":
        return torch.cat([_block64(c, leaf, w, rows(x)[i:i + 1].double()) for i in range(c["seqs"])])
    n = c["seqs"] * r * c["hidden"]
    out = torch.cat([_block64(c, {k: t.detach() for k, t in leaf.items()}, w, rows(x)[i:i + 1].double())
                     for i in range(c["seqs"])])
    res = out - rows(target).double()
    keep = torch.ones_like(res, dtype=torch.bool)
    if c["suppress"]:
        k = max(1, int(n * 0.001))
        thr = res.abs().reshape(-1).kthvalue(n - k + 1).values if n < 1 << 24 else _kth_largest(res.abs().reshape(-1), k)
        keep = res.abs() < thr
    for i in range(c["seqs"]):
        _block64(c, leaf, w, rows(x)[i:i + 1].double()).backward((2 * res * keep / n)[i:i + 1])
    return {"loss": None, "out": out, "dw": _fused({k: t.grad for k, t in leaf.items()})}


def _kth_largest(a, k):
    """The k-th largest of a long vector: candidates first, then a sort of those."""
    cut = a[torch.randperm(a.numel(), device=a.device)[:1 << 20]].kthvalue((1 << 20) - 4 * ((k << 20) // a.numel()) - 64).values
    top = a[a >= cut]
    return top.sort(descending=True).values[k - 1]


def _exact_score(c, seed):
    model, tokens = _model(c, seed)
    mode = "asym" if c["mode"] == "asym" else "sym"
    leaf = []
    for blk in model.blocks:
        leaf.append({n: _quantize64(t, None, c["bits"], 64, mode, None)[0].to(torch.bfloat16).double().requires_grad_()
                     for n, t in blk.weights.linears.items()})
    x = model.embed[tokens[:, :-1]].double()
    for blk, wq in zip(model.blocks, leaf):
        x = _block64(c, wq, blk.weights, x)
    xn = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * model.norm.double()
    logits = xn @ model.embed.double().t()
    logits.retain_grad()
    loss = torch.nn.functional.cross_entropy(logits.view(-1, c["vocab"]), tokens[:, 1:].reshape(-1))
    loss.backward()
    scores = [[(wq[n].grad * (_quantize64(blk.weights.linears[n], None, c["bits"], 64, mode, None)[0]
                              - blk.weights.linears[n].double())).abs().sum() for n in LAYERS]
              for blk, wq in zip(model.blocks, leaf)]
    return {"loss": None, "dlogits": logits.grad,
            "scores": torch.stack([torch.stack(r) for r in scores])[..., None],
            "dw0": _fused({n: leaf[0][n].grad for n in LAYERS})}


def _exact_layer(c, seed):
    s = prepare(c, seed)
    w, x = s["w"].double(), s["x"].double()
    n, k = c["samples"] * c["rows"], max(1, int(c["samples"] * c["rows"] * 0.001))
    # The codes are those of float32 arithmetic: one that rounds the other way
    # would show in a whole row of the residual.
    q, t = _quantize64(s["w"], s["params"], c["bits"], 64, c["mode"], None, torch.float32)
    t = {k: y.double() if isinstance(y, torch.Tensor) and y.is_floating_point() else y for k, y in t.items()}
    r = x @ (q.double() - w).t()
    keep = r.abs() < r.abs().reshape(-1).topk(k).values[-1] if c["bits"] < 4 else torch.ones_like(r, dtype=torch.bool)
    dw = (2 * r * keep / n).t() @ x
    return {"loss": None, "qdq": q.double(), "res": r, "dw": dw,
            "params": _stepped64(s["params"], _grad64(t, dw, c["mode"]), LATE_LR, c["mode"])}


def exact(case, seed):
    """What ``run`` returns, from plain torch in float64; None for whole numbers,
    for the search, whose choice among candidates is defined in float32, and
    for the loss, one number in which errors of either sign cancel by chance."""
    c, kind = case, case["kind"]
    if kind == "search":
        return None
    if kind in ("pack", "step"):
        s = _layer_inputs(c, seed)
        gs = c["cols"] if c["group"] == -1 else c["group"]
        q, t = _quantize64(s["w"], s["params"], c["bits"], gs, c["mode"], s["init"])
        if kind == "pack":
            z = t["z"] if c["mode"] == "asym" else 2.0 ** (c["bits"] - 1)
            return {"packed": None, "scales": t["s"][..., 0], "biases": (-t["s"] * z)[..., 0]}
        return {"wq": q, **_stepped64(s["params"], _grad64(t, s["grad"], c["mode"]), LATE_LR, c["mode"])}
    if kind == "layer":
        return _exact_layer(c, seed)
    if kind == "score":
        return _exact_score(c, seed)
    return _exact_block(c, seed)
