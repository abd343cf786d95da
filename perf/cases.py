"""The work that a training program has this package do, as timed cases.

A case is one call that the program makes again and again: an optimizer step over its parameters (by far the most
frequent), a step tensor by tensor as gradients arrive, saving and restoring the optimizer, exporting and importing the
fp32 master weights.  ``listed`` names the cases that are always timed, ``draw`` gives more of the same ranges.

Every case starts in the middle of a training run: weights ~N(0, 0.02) (norm weights 1), gradients ~N(0, 1e-3) times a
factor per tensor log-uniform in [0.1, 10] (Student-t with 3 degrees of freedom for the ragged lists), moments as such
gradients leave them behind, correction bits uniform.  The optimizer has stepped before, so that its states and launch
tables exist.

Parameters, gradients and optimizer states of a step are carved from one flat buffer per kind at offsets of 512
elements, which is how a caching allocator lays out tensors that are allocated one after the other; the flat
buffers are what a step returns, so that lists of thousands of tensors come back whole.
"""

from __future__ import annotations

import math
import warnings

import torch

import flashoptim_amd as fo
from flashoptim_amd.state import _MaybeQuantizedTensor

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_WIDTH = {"bf16": 2, "fp16": 2, "fp32": 4}
_GROUP = 32
_ALIGN = 512          # elements between the starts of carved tensors
_STEP = 100.0         # how long the run has been going
_DRAW_CHUNK = 1 << 26  # random values drawn at a time


# ------------------------------------------------------------------------------------------------- the cases


def _case(name, task, optimizer, dtype, master, layout, quantize=True, compress=False, **sizes):
    return dict(name=name, task=task, optimizer=optimizer, dtype=dtype, master=master, quantize=quantize,
                compress=compress, layout=layout, **sizes)


def listed():
    layer = dict(hidden=4096, ffn=14336, kv=1024)
    return [
        # the smallest program: a two-layer perceptron, 4 tensors, 35.6 thousand weights; latency and launches
        _case("mlp-adamw-24", "step", "adamw", "bf16", 24, "mlp", d_in=128, hidden=256, d_out=10),
        # what is trained when most of a model is frozen: hundreds of short tensors (norms, biases, adapters)
        _case("short-adamw-24", "step", "adamw", "bf16", 24, "ragged", tensors=512, longest=1 << 14, lengths_seed=1),
        # two layers of the 8B-parameter transformer that the package's benchmark steps, default masters
        _case("block-adamw-24", "step", "adamw", "bf16", 24, "block", layers=2, **layer),
        # one flat tensor of 2^30 weights (a sharded model's local shard): bandwidth alone
        _case("flat-adamw-24", "step", "adamw", "bf16", 24, "flat", n=1 << 30),
        # one layer with 32-bit masters, the other width of the correction term
        _case("block-adamw-32", "step", "adamw", "bf16", 32, "block", layers=1, **layer),
        # a ragged list, odd lengths among them, under the sign-based optimizer
        _case("ragged-lion-24", "step", "lion", "bf16", 24, "ragged", tensors=1024, longest=1 << 22, lengths_seed=2),
        # a smaller model in fp16, widths that are no powers of two
        _case("block-sgdw-24-fp16", "step", "sgdw", "fp16", 24, "block", layers=4, hidden=1000, ffn=2730, kv=250),
        # fp32 weights stepped tensor by tensor in reverse order, as the hooks of gradient release do
        _case("release-adamw-fp32", "release", "adamw", "fp32", 0, "block", layers=4, hidden=2048, ffn=5632, kv=512),
        # a checkpoint in the default format (bf16 moments), written and read back
        _case("save-adamw-24", "save", "adamw", "bf16", 24, "block", layers=1, **layer),
        _case("load-adamw-24", "load", "adamw", "bf16", 24, "block", layers=1, **layer),
        # the fp32 master weights out of (evaluation, export) and into (fine-tuning start) the optimizer
        _case("export-fp32-24", "export", "adamw", "bf16", 24, "block", layers=1, **layer),
        _case("import-fp32-24", "import", "adamw", "bf16", 24, "block", layers=1, **layer),
    ]


def draw(rng):
    task = rng.choice(["step"] * 6 + ["release", "save", "load", "export", "import"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    optimizer = rng.choice(["adamw", "adamw", "adam", "lion", "sgdw", "sgd"])
    master = 0 if dtype == "fp32" else rng.choice([24, 24, 32])
    quantize = rng.random() < 0.9
    compress = quantize and master != 32 and dtype != "fp32" and rng.random() < 0.3
    layout = rng.choice(["mlp", "block", "flat", "ragged"] if task == "step" else ["mlp", "block"])
    if task in ("save", "load") and not master:
        compress = False
    if task in ("export", "import") and not master:
        dtype, master = "bf16", 24
    if layout == "flat":
        sizes = dict(n=int(2 ** rng.uniform(10, 29)) | rng.randint(0, 1))
    elif layout == "mlp":
        sizes = dict(d_in=int(2 ** rng.uniform(3, 12)), hidden=int(2 ** rng.uniform(4, 13)), d_out=int(2 ** rng.uniform(1, 10)))
    elif layout == "block":
        hidden = int(2 ** rng.uniform(5, 12))
        sizes = dict(layers=rng.randint(1, 6) if task in ("step", "release") and hidden < 2048 else 1, hidden=hidden,
                     ffn=int(hidden * rng.uniform(2, 4)), kv=max(1, hidden // rng.choice([1, 4, 8])))
    else:
        sizes = dict(tensors=int(2 ** rng.uniform(4, 11)), longest=int(2 ** rng.uniform(8, 21)), lengths_seed=rng.randint(3, 1 << 20))
    case = _case("", task, optimizer, dtype, master, layout, quantize, compress, **sizes)
    del case["name"]
    return case


# ------------------------------------------------------------------------------------------------- shapes


def _shapes(case):
    if case["layout"] == "flat":
        return [(case["n"],)]
    if case["layout"] == "mlp":
        return [(case["hidden"], case["d_in"]), (case["hidden"],), (case["d_out"], case["hidden"]), (case["d_out"],)]
    if case["layout"] == "block":
        h, f, kv = case["hidden"], case["ffn"], case["kv"]
        return [(h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f), (h,), (h,)] * case["layers"]
    # lengths log-uniform in [1, longest], the shortest and the group's edges among them
    g = torch.Generator().manual_seed(case["lengths_seed"])
    lens = torch.exp2(math.log2(case["longest"]) * torch.rand(case["tensors"], generator=g, dtype=torch.float64))
    lens[:3] = torch.tensor([1.0, 31.0, 33.0])
    return [(int(n),) for n in lens.floor().clamp(1, case["longest"]).tolist()]


def _moments(case):
    """State names of the case's optimizer: (key, signed, sqrt, softsign)."""
    if case["optimizer"] in ("adam", "adamw"):
        return [("exp_avg", True, False, True), ("exp_avg_sq", False, True, False)]
    return [("exp_avg" if case["optimizer"] == "lion" else "momentum_buffer", True, False, True)]


def _ecc_bytes(case):
    return max(0, case["master"] // 8 - _WIDTH[case["dtype"]])


# ------------------------------------------------------------------------------------------------- inputs


class _Flat:
    """Tensors of `shapes` carved from one flat buffer; `per` elements of the shapes share one of the buffer."""

    def __init__(self, shapes, dtype, device, per=1):
        counts = [-(-math.prod(s) // per) for s in shapes]
        step = _ALIGN // per
        self.starts = []
        total = 0
        for c in counts:
            self.starts.append(total)
            total += -(-c // step) * step
        self.buffer = torch.zeros(total, dtype=dtype, device=device)
        self.views = [self.buffer[o:o + c] if per > 1 else self.buffer[o:o + c].view(s)
                      for o, c, s in zip(self.starts, counts, shapes)]


def _fill(buffer, values):
    """Fills a flat buffer piecewise from values(count)."""
    for o in range(0, buffer.numel(), _DRAW_CHUNK):
        m = min(_DRAW_CHUNK, buffer.numel() - o)
        buffer[o:o + m] = values(m)


class _Holder(torch.nn.Module):
    """A module that owns the case's parameters."""

    def __init__(self, params):
        super().__init__()
        for i, p in enumerate(params):
            self.register_parameter(f"w{i}", p)


def _make_optimizer(case, params):
    kw = dict(quantize=case["quantize"], compress_state_dict=case["compress"], master_weight_bits=case["master"] or None)
    if case["optimizer"] == "adamw":
        return fo.FlashAdamW(params, lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01, **kw)
    if case["optimizer"] == "adam":
        return fo.FlashAdam(params, lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01, **kw)
    if case["optimizer"] == "lion":
        return fo.FlashLion(params, lr=1e-4, betas=(0.9, 0.99), weight_decay=0.1, **kw)
    if case["optimizer"] == "sgdw":
        return fo.FlashSGDW(params, momentum=0.9, lr=1e-2, weight_decay=1e-4, **kw)
    return fo.FlashSGD(params, momentum=0.9, nesterov=True, lr=1e-2, weight_decay=1e-4, **kw)


def prepare(case, seed):
    device, dtype = torch.device("cuda"), _DTYPES[case["dtype"]]
    shapes = _shapes(case)
    heavy = case["layout"] == "ragged"
    g = torch.Generator(device=device).manual_seed(seed)

    def normal(m):
        return torch.randn(m, generator=g, device=device)

    def student(m):
        chi = normal(m).square_() + normal(m).square_() + normal(m).square_()
        return normal(m) / (chi / 3.0).sqrt_()

    # weights and gradients; every tensor's gradient scale is its own
    param, grad = _Flat(shapes, dtype, device), _Flat(shapes, dtype, device)
    scales = (10.0 ** (torch.rand(len(shapes), generator=torch.Generator().manual_seed(seed)) * 2 - 1)).tolist()
    _fill(param.buffer, lambda m: normal(m) * 0.02)
    _fill(grad.buffer, lambda m: (student(m) if heavy else normal(m)) * 1e-3)
    for s, p, x, shape in zip(scales, param.views, grad.views, shapes):
        x.mul_(s)
        if len(shape) == 1 and case["layout"] == "block":
            p.fill_(1.0)
    params = [torch.nn.Parameter(v) for v in param.views]
    for p, x in zip(params, grad.views):
        p.grad = x
    flats = {"param": param.buffer}
    per_param = [{} for _ in params]

    # correction bits of the masters
    ecc_bytes = _ecc_bytes(case)
    if ecc_bytes:
        ecc = _Flat(shapes, torch.int8 if ecc_bytes == 1 else torch.int16, device)
        top = 127 if ecc_bytes == 1 else 32767
        _fill(ecc.buffer, lambda m: torch.randint(-top, top + 1, (m,), generator=g, device=device, dtype=ecc.buffer.dtype))
        flats["error_bits"] = ecc.buffer
        for st, e in zip(per_param, ecc.views):
            st["error_bits"] = e

    # moments after _STEP steps: first moments are averages of gradients of mean zero, second moments their mean square
    spread = {"adam": 0.23, "adamw": 0.23, "lion": 0.07, "sgd": 2.3, "sgdw": 2.3}[case["optimizer"]] * 1e-3
    for key, signed, sqrt, softsign in _moments(case):
        spec = dict(signed=signed, sqrt=sqrt, softsign=softsign)
        plain = _Flat(shapes, dtype if not case["quantize"] else torch.float32, device)
        if signed:
            _fill(plain.buffer, lambda m: normal(m) * spread)
        else:
            _fill(plain.buffer, lambda m: (0.3 * normal(m)).exp_() * (0.095 * 1e-6))
        for s, x in zip(scales, plain.views):
            x.mul_(s if signed else s * s)
        holders = [_MaybeQuantizedTensor(None, try_quantize=case["quantize"], storage_dtype=dtype, **spec) for _ in params]
        if case["quantize"]:
            codes = _Flat(shapes, torch.int8 if signed else torch.uint8, device)
            scale = _Flat(shapes, torch.float16, device, per=_GROUP)
            whole = _MaybeQuantizedTensor(plain.buffer, **spec)
            codes.buffer.copy_(whole.quantized)
            scale.buffer.copy_(whole.scales)
            flats[key], flats[key + "_scales"] = codes.buffer, scale.buffer
            for h, c, s in zip(holders, codes.views, scale.views):
                h.load_state_dict({"x::quantized": c, "x::scales": s}, "x")
        else:
            flats[key] = plain.buffer
            for h, x in zip(holders, plain.views):
                h.load_state_dict({"x": x}, "x")
        for st, h in zip(per_param, holders):
            st[key] = h
        del plain

    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        opt = _make_optimizer(case, params)
    for p, st in zip(params, per_param):
        if case["optimizer"] in ("adam", "adamw"):
            st["step"] = torch.tensor(_STEP)
        opt.state[p].update(st)

    state = dict(case=case, params=params, opt=opt, flats=flats)
    task = case["task"]
    if task == "step":
        opt.step()
    elif task == "release":
        for p in reversed(params):
            opt.step_param(p, opt.param_groups[0])
    elif task == "load":
        # the checkpoint of this run, read into the optimizer of a restarted one
        state["checkpoint"] = opt.state_dict()
        state["opt"] = _make_optimizer(case, params)
    elif task == "import":
        masters = {}
        for i, s in enumerate(shapes):
            w = torch.empty(math.prod(s), device=device)
            _fill(w, lambda m: normal(m) * 0.02)
            masters[f"w{i}"] = w.view(s)
        state["masters"] = masters
    if task in ("export", "import"):
        state["model"] = _Holder(params)
    return state


# ------------------------------------------------------------------------------------------------- one pass


def run(state):
    task, opt = state["case"]["task"], state["opt"]
    if task == "step":
        opt.step()
        return state["flats"]
    if task == "release":
        group = opt.param_groups[0]
        for p in reversed(state["params"]):
            opt.step_param(p, group)
        return state["flats"]
    if task == "save":
        return opt.state_dict()["state"]
    if task == "load":
        opt.load_state_dict(state["checkpoint"])
        return [_state_tensors(opt.state[p]) for p in state["params"]]
    if task == "export":
        return opt.get_fp32_model_state_dict(state["model"])
    opt.set_fp32_model_state_dict(state["model"], state["masters"])
    return [(p, opt.state[p]["error_bits"]) for p in state["params"]]


def _state_tensors(st):
    out = {}
    for key, value in st.items():
        if not isinstance(value, _MaybeQuantizedTensor):
            out[key] = value
        elif value.is_quantized():
            out[key], out[key + "_scales"] = value.quantized, value.scales
        else:
            out[key] = value.data
    return out


# ------------------------------------------------------------------------------------------------- its cost and its exactness


def work(case):
    n = sum(math.prod(s) for s in _shapes(case))
    width, ecc, moments = _WIDTH[case["dtype"]], _ecc_bytes(case), len(_moments(case))
    held = 1.0 + 2.0 / _GROUP if case["quantize"] else float(width)   # bytes of one moment of one weight
    task = case["task"]
    if task in ("step", "release"):
        per, ops = 3 * width + 2 * ecc + 2 * moments * held, 12 + 20 * moments
    elif task in ("save", "load"):
        # moments between their stored form and bf16 (a compressed checkpoint holds them as they are), 1-byte
        # correction bits between int8 and the parameter's dtype
        per, ops = (0 if case["compress"] else moments * (held + 2)) + (3 if ecc == 1 else 0), 8 * moments
    else:
        per, ops = 4 + width + ecc, 8
    return {"bytes": n * per, "flops": n * ops}


def tolerance(case):
    # Adam on bf16 with 24-bit masters lets a master weight differ by one unit of its precision from an evaluation
    # operation by operation.  Three steps from the same state in either form, gradients included: codes and scales
    # the same, correction bits differ in 0.31 % of the weights, bf16 weights by 1.9e-5 (2-norm) and by at most one of
    # their own units, 2^-7.  Everything else is exact.
    if case["task"] in ("step", "release") and case["optimizer"] in ("adam", "adamw") and case["dtype"] == "bf16" and case["master"] == 24:
        return {"rel": 8e-5, "max": 0.032, "differ": 0.01}
    return "exact"
