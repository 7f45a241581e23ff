"""Timing cases of HeatViT-T's integer inference path on one MI355X.

Each case is one call that a program makes through the framework's entry
points: whole forwards (heatvit_amd.model.Engine and Pipeline), one
transformer block, one token selector, and the row kernels (attention core,
LayerNorm, softmax) of the C ABI (include/heatvit_hip.h).  The weights are the
seeded synthetic HeatViT-T of heatvit_amd.synth, with its scale exponents and
its calibrated selectors (197 -> 88 -> 45 -> 32 tokens); images, tokens and
scores are drawn from the seed.

Every output is a whole number that the golden model defines bit for bit, so
every tolerance is "exact" and there is no rounding for a 64-bit reference to
measure.
"""

import functools
import math
import random

import numpy as np
import torch

from heatvit_amd import _lib, synth
from heatvit_amd.device import DeviceBlock, DeviceSelector
from heatvit_amd.model import Engine, Pipeline

TOKENS = 197          # patch rows plus the class row
DIM, HIDDEN, HEADS, CLASSES = 192, 768, 3, 1000
IMAGE_BYTES = 224 * 224 * 3
STAGE_TOKENS = (197, 88, 45, 32)   # the calibrated budget before and after each selector
MAX_BATCH = 256
PIPELINE_DEPTH = 3


def listed():
    return [
        # one transformer block over one image: the golden model's transformer_block
        {"name": "block_b1", "kind": "block", "batch": 1, "low": 197, "high": 197, "block": 1},
        # the same over a ragged batch, as between selectors
        {"name": "block_ragged_b100", "kind": "block", "batch": 100, "low": 20, "high": 197,
         "block": 6},
        # one image through the whole unpruned model: interactive latency
        {"name": "model_unpruned_b1", "kind": "model", "batch": 1, "pruned": False,
         "images": "int8"},
        # a small server batch, with the selectors
        {"name": "model_pruned_b32", "kind": "model", "batch": 32, "pruned": True,
         "images": "int8"},
        # the benchmark batch, one at a time, with and without the selectors
        {"name": "model_pruned_b256", "kind": "model", "batch": 256, "pruned": True,
         "images": "int8"},
        {"name": "model_unpruned_b256", "kind": "model", "batch": 256, "pruned": False,
         "images": "int8"},
        # preprocessed float images, quantised on the device
        {"name": "model_float_b256", "kind": "model", "batch": 256, "pruned": True,
         "images": "float32"},
        # throughput serving: batches in flight on their own streams
        {"name": "pipeline_b256", "kind": "pipeline", "batch": 256, "pruned": True},
        # the token selector alone over 64 token sets
        {"name": "selector_b64", "kind": "selector", "batch": 64, "tokens": 197,
         "package": False},
        # the attention core over a ragged batch of images
        {"name": "attention_b96", "kind": "attention", "batch": 96, "low": 60, "high": 197,
         "block": 3},
        # LayerNorm over the rows of 256 images
        {"name": "layernorm_50432", "kind": "layernorm", "rows": 50432, "block": 2},
        # the attention softmax over every score row of 256 images
        {"name": "softmax_b256", "kind": "softmax", "batch": 256, "low": 197, "high": 197,
         "outputs": "attention"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("model", "model", "model", "model", "block", "block", "selector",
                       "attention", "layernorm", "softmax", "pipeline"))
    if kind == "model":
        return {"kind": kind, "batch": _log_int(rng, 1, MAX_BATCH), "pruned": rng.random() < 0.6,
                "images": rng.choice(("int8", "int8", "float32"))}
    if kind == "pipeline":
        return {"kind": kind, "batch": _log_int(rng, 16, MAX_BATCH), "pruned": True}
    if kind == "selector":
        return {"kind": kind, "batch": _log_int(rng, 1, 512), "tokens": rng.randint(8, 197),
                "package": rng.random() < 0.5}
    if kind == "layernorm":
        return {"kind": kind, "rows": _log_int(rng, 197, 50432), "block": rng.randint(1, 12)}
    low = rng.randint(8, 197)
    case = {"kind": kind, "batch": _log_int(rng, 1, MAX_BATCH), "low": low,
            "high": rng.randint(low, 197)}
    if kind == "softmax":
        case["outputs"] = rng.choice(("attention", "selector", "both"))
    else:
        case["block"] = rng.randint(1, 12)
    return case


# ------------------------------------------------------------------ the model

@functools.lru_cache(maxsize=None)
def _params(pruned):
    params = synth.pruned_params()
    return params if pruned else synth.unpruned_control(params)


@functools.lru_cache(maxsize=None)
def _selector_params():
    return synth.selector_workload()[1]


def _lengths(case):
    """Token counts of the case's images, spread over [low, high]."""
    rng = random.Random("%d %d %d" % (case["batch"], case["low"], case["high"]))
    return [rng.randint(case["low"], case["high"]) for _ in range(case["batch"])]


def _offsets(lengths):
    return np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform_i8(g, shape):
    return torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=g)


def _normal_i8(g, shape, sigma=40.0):
    x = torch.randn(shape, device="cuda", generator=g) * sigma
    return x.round_().clamp_(-128, 127).to(torch.int8)


def _images(g, batch):
    return _uniform_i8(g, (batch, IMAGE_BYTES))


def _stream():
    return torch.cuda.current_stream().cuda_stream


# ---------------------------------------------------------------- preparation

def prepare(case, seed):
    return _PREPARE[case["kind"]](case, _generator(seed))


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_model(case, g):
    params = _params(case["pruned"])
    engine = Engine(params, case["batch"])
    images = _images(g, case["batch"])
    if case["images"] == "float32":
        scale = 2.0 ** params.patch.image_scale_exp
        x = images.view(-1, 224, 224, 3).permute(0, 3, 1, 2).to(torch.float32)
        # off the quantiser's grid, as preprocessed photographs are
        x += torch.rand(x.shape, device="cuda", generator=g) - 0.5
        images = (x * scale).contiguous()
    return {"kind": "model", "engine": engine, "images": images}


def _run_model(s):
    return s["engine"].forward(s["images"])


def _prepare_pipeline(case, g):
    pipe = Pipeline(_params(case["pruned"]), case["batch"], depth=PIPELINE_DEPTH)
    return {"kind": "pipeline", "pipe": pipe,
            "images": [_images(g, case["batch"]) for _ in range(PIPELINE_DEPTH)]}


def _run_pipeline(s):
    tickets = [s["pipe"].submit(images) for images in s["images"]]
    return [t.wait() for t in tickets]


def _prepare_block(case, g):
    lengths = _lengths(case)
    rows, batch = sum(lengths), case["batch"]
    lib = _lib.lib()
    return {"kind": "block", "batch": batch, "rows": rows,
            "block": DeviceBlock(_params(True).blocks[case["block"] - 1]),
            "x": _normal_i8(g, (rows, DIM)),
            "offsets": torch.from_numpy(_offsets(lengths)).cuda(),
            "z": torch.empty((rows, DIM), dtype=torch.int8, device="cuda"),
            "status": torch.empty(batch, dtype=torch.int32, device="cuda"),
            "warnings": torch.empty(batch, dtype=torch.int32, device="cuda"),
            "workspace": torch.empty(lib.hv_block_workspace_bytes(batch, rows),
                                     dtype=torch.uint8, device="cuda")}


def _run_block(s):
    _lib.check(_lib.lib().hv_block_forward(
        s["block"].struct, s["x"].data_ptr(), s["offsets"].data_ptr(), s["batch"], s["rows"],
        s["z"].data_ptr(), None, s["status"].data_ptr(), s["warnings"].data_ptr(),
        s["workspace"].data_ptr(), s["workspace"].numel(), _stream()), "block")
    return s["z"], s["status"], s["warnings"]


def _prepare_selector(case, g):
    batch, n = case["batch"], case["tokens"]

    def zeros(shape, dtype):
        return torch.zeros(shape, dtype=dtype, device="cuda")

    return {"kind": "selector", "batch": batch, "selector": DeviceSelector(_selector_params()),
            "tokens": _uniform_i8(g, (batch * n, DIM)),
            "offsets": torch.arange(batch + 1, dtype=torch.int32, device="cuda") * n,
            "package": torch.full((batch,), int(case["package"]), dtype=torch.uint8,
                                  device="cuda"),
            "out": zeros((batch * (n + 1), DIM), torch.int8),
            "out_offsets": zeros(batch + 1, torch.int32),
            "out_package": zeros(batch, torch.uint8), "fused": zeros((batch, 196), torch.int32),
            "kept": zeros((batch, 196), torch.int32), "state": zeros((batch, 5), torch.int32),
            "workspace": torch.empty(_lib.lib().hv_selector_workspace_bytes(batch),
                                     dtype=torch.uint8, device="cuda")}


def _run_selector(s):
    _lib.check(_lib.lib().hv_selector_forward(
        s["selector"].struct, s["tokens"].data_ptr(), s["offsets"].data_ptr(),
        s["package"].data_ptr(), s["batch"], s["out"].data_ptr(), s["out_offsets"].data_ptr(),
        s["out_package"].data_ptr(), s["fused"].data_ptr(), s["kept"].data_ptr(),
        s["state"].data_ptr(), None, s["workspace"].data_ptr(), s["workspace"].numel(),
        _stream()), "selector")
    return (s["out"], s["out_offsets"], s["out_package"], s["fused"], s["kept"], s["state"])


def _prepare_attention(case, g):
    lengths = _lengths(case)
    m = _params(True).blocks[case["block"] - 1].mhsa
    rows = sum(lengths)
    return {"kind": "attention", "batch": case["batch"], "rows": rows,
            "exps": (m.qkv_out_scale_exp, m.score_scale_exp, m.prob_scale_exp,
                     m.context_out_scale_exp),
            "qkv": _normal_i8(g, (rows, 3 * DIM)),
            "offsets": torch.from_numpy(_offsets(lengths)).cuda(),
            "ctx": torch.empty((rows, DIM), dtype=torch.int8, device="cuda"),
            "status": torch.empty(case["batch"], dtype=torch.int32, device="cuda")}


def _run_attention(s):
    _lib.check(_lib.lib().hv_attention_i8(
        s["qkv"].data_ptr(), s["offsets"].data_ptr(), s["batch"], s["rows"],
        s["ctx"].data_ptr(), None, None, *s["exps"], s["status"].data_ptr(), _stream()),
        "attention")
    return s["ctx"], s["status"]


def _prepare_layernorm(case, g):
    m = _params(True).blocks[case["block"] - 1].mhsa
    rows = case["rows"]
    return {"kind": "layernorm", "rows": rows,
            "gamma": torch.from_numpy(np.array(m.ln_gamma, np.int8)).cuda(),
            "beta": torch.from_numpy(np.array(m.ln_beta, np.int8)).cuda(),
            "exps": (m.x_scale_exp, m.gamma1_scale_exp, m.beta1_scale_exp, m.ln1_out_scale_exp),
            "x": _normal_i8(g, (rows, DIM)),
            "y": torch.empty((rows, DIM), dtype=torch.int8, device="cuda"),
            "negative": torch.empty(rows, dtype=torch.uint8, device="cuda")}


def _run_layernorm(s):
    _lib.check(_lib.lib().hv_layernorm_i8(
        s["x"].data_ptr(), s["gamma"].data_ptr(), s["beta"].data_ptr(), s["y"].data_ptr(),
        s["rows"], None, *s["exps"], s["negative"].data_ptr(), _stream()), "layernorm")
    return s["y"], s["negative"]


def _prepare_softmax(case, g):
    lengths = np.repeat(_lengths(case), [HEADS * n for n in _lengths(case)])
    offsets = _offsets(lengths)
    total = int(offsets[-1])

    def out(wanted, dtype):
        return (torch.empty(total, dtype=dtype, device="cuda")
                if case["outputs"] in (wanted, "both") else None)

    return {"kind": "softmax", "rows": len(lengths),
            "x": torch.randint(-(1 << 18), 1 << 18, (total,), dtype=torch.int32, device="cuda",
                               generator=g),
            "offsets": torch.from_numpy(offsets).cuda(),
            "attention": out("attention", torch.uint8), "selector": out("selector", torch.int32)}


def _run_softmax(s):
    outputs = [t for t in (s["attention"], s["selector"]) if t is not None]
    _lib.check(_lib.lib().hv_softmax_rows(
        s["x"].data_ptr(), s["offsets"].data_ptr(), s["rows"],
        None if s["attention"] is None else s["attention"].data_ptr(),
        None if s["selector"] is None else s["selector"].data_ptr(), _stream()), "softmax")
    return outputs


_PREPARE = {"model": _prepare_model, "pipeline": _prepare_pipeline, "block": _prepare_block,
            "selector": _prepare_selector, "attention": _prepare_attention,
            "layernorm": _prepare_layernorm, "softmax": _prepare_softmax}
_RUN = {"model": _run_model, "pipeline": _run_pipeline, "block": _run_block,
        "selector": _run_selector, "attention": _run_attention, "layernorm": _run_layernorm,
        "softmax": _run_softmax}


# --------------------------------------------------- what a pass cannot do without

_BLOCK_WEIGHTS = DIM * (3 * DIM + DIM + 2 * HIDDEN)
_ROW_OPS = 2 * _BLOCK_WEIGHTS                   # QKV, projection and the two FFN layers
_SELECTOR_OPS = 2 * HEADS * (64 * 32 + 64 * 32 + 32 * 16 + 16 * 2)   # per candidate


def _block_ops(lengths):
    return sum(_ROW_OPS * n + 2 * 2 * DIM * n * n for n in lengths)


def _model_work(case):
    batch = case["batch"]
    ops = batch * (2 * HIDDEN * DIM * (TOKENS - 1) + 2 * DIM * CLASSES)
    for block in range(12):
        n = STAGE_TOKENS[block // 3] if case["pruned"] else TOKENS
        ops += batch * _block_ops([n])
    if case["pruned"]:
        ops += batch * _SELECTOR_OPS * sum(n - 1 for n in STAGE_TOKENS[:3])
    image = IMAGE_BYTES * (4 if case.get("images") == "float32" else 1)
    weights = 12 * _BLOCK_WEIGHTS + HIDDEN * DIM + DIM * CLASSES + TOKENS * DIM
    return batch * (image + 4 * CLASSES) + weights, ops


def work(case):
    kind = case["kind"]
    if kind == "model":
        nbytes, ops = _model_work(case)
    elif kind == "pipeline":
        nbytes, ops = (PIPELINE_DEPTH * v for v in _model_work(case))
    elif kind == "block":
        lengths = _lengths(case)
        nbytes, ops = 2 * DIM * sum(lengths) + _BLOCK_WEIGHTS, _block_ops(lengths)
    elif kind == "selector":
        rows = case["batch"] * case["tokens"]
        nbytes, ops = DIM * (rows + 0.45 * rows), _SELECTOR_OPS * (rows - case["batch"])
    elif kind == "attention":
        lengths = _lengths(case)
        nbytes, ops = 4 * DIM * sum(lengths), sum(2 * 2 * DIM * n * n for n in lengths)
    elif kind == "layernorm":
        nbytes, ops = (2 * DIM + 1) * case["rows"], 8 * DIM * case["rows"]
    else:
        scores = sum(HEADS * n * n for n in _lengths(case))
        per = 4 + {"attention": 1, "selector": 4, "both": 5}[case["outputs"]]
        nbytes, ops = per * scores, 8 * scores
    return {"bytes": nbytes, "flops": ops}


def tolerance(case):
    return "exact"
