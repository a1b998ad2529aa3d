"""The work this backend is measured on: what a user of the mi355x backend has it do, through its public entry points.

Four families, each a dict of plain values:

    block    a nanoGPT-style int8 block stack (models.BlockSpec) compiled and planned once, its quantized input resident
             in HBM: run() is one forward (CompiledModel.launch) and its results are the device values that `keep` returns
    run      CompiledModel.run as a caller of the reference's driver uses it: a host float input (or token ids) in, the
             device quantization, the forward, and the integers and dequantized outputs back on the host
    linear   one int8 linear layer with its requant (and optionally a GELU table): x (M, K) @ w (K, N)
    frozen   the reference's frozen 2-layer models (contract v1, int8; v2, int16 residual stream) over a batch

`replay` is the launch mode: the plan's kernels replayed as one captured HIP graph, or launched from the host.

Every result is an integer defined by the graph, so outputs are compared exactly. exact() evaluates the same graph in
torch in 64 bits: the graph's constants are data, the arithmetic is its own.
"""
import gzip
import json
import math
import sys
from functools import lru_cache
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT / "anvil-compiler_amd"))

import anvil_mi355x as anvil  # noqa: E402
from anvil_mi355x import ir, models, quantize  # noqa: E402
from anvil_mi355x import runtime as rt  # noqa: E402

CALIB_TAG = 11           # calibration seed of the blocks that the tracked calibrations do not cover
TORCH_DTYPE = {"i8": torch.int8, "i16": torch.int16, "i32": torch.int32}
TYPESTR = {"i8": "|i1", "i16": "<i2", "i32": "<i4"}


# ------------------------------------------------------------------------------------------------------ cases

def _block(family, C, H, T, B, layers=1, vocab=0, causal=True, gelu="fused", keep="outputs", replay=True):
    return {"family": family, "n_embd": C, "n_head": H, "seq": T, "batch": B, "layers": layers, "vocab": vocab,
            "causal": causal, "gelu": gelu, "keep": keep, "replay": replay}


def _linear(M, K, N, lut=False, replay=False):
    return {"family": "linear", "M": M, "K": K, "N": N, "lut": lut, "replay": replay}


def listed():
    named = [
        # the smallest whole call: one short sequence, host floats in, integers and floats out
        ("run-block64", _block("run", 64, 4, 32, 1)),
        # a token model served in small batches: ids in, logits out
        ("run-model128", _block("run", 128, 4, 128, 8, layers=2, vocab=512)),
        # the 2-layer token model with its logits head, a full batch resident on the device
        ("model128", _block("block", 128, 4, 128, 128, layers=2, vocab=512)),
        # a mid-size block with every intermediate returned (a parity run, or a debugger's view of the graph)
        ("block256-all", _block("block", 256, 8, 256, 16, keep="all")),
        # the GPT-2-small-shaped block at the benchmark's batch: throughput
        ("block768", _block("block", 768, 12, 1024, 32, replay=False)),
        # the same block on one sequence: latency
        ("block768-one", _block("block", 768, 12, 1024, 1)),
        # a prompt that is no multiple of any tile, a batch of them
        ("block384-ragged", _block("block", 384, 6, 250, 16)),
        # an encoder block (no mask) with its GELU as an op of its own
        ("block512-full", _block("block", 512, 8, 384, 12, causal=False, gelu="lut")),
        # a few rows against a wide weight, as in decoding
        ("linear-rows16", _linear(16, 768, 3072, lut=True)),
        ("linear-rows256", _linear(256, 3072, 3072)),
        # a long prefill through one wide layer
        ("linear-rows16384", _linear(16384, 3072, 3072)),
        # the reference's frozen model with its int16 residual stream, a large batch of its short sequences
        ("frozen-v2", {"family": "frozen", "model": "v2", "batch": 16384, "replay": True}),
    ]
    return [dict(c, name=n) for n, c in named]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_block(rng, family, most):
    """A block of up to `most` activations (batch x seq x n_embd): any sequence length, odd ones among them, heads of
    the usual sizes, one or two layers."""
    while True:
        d = rng.choice([16, 32, 32, 64, 64, 64, 128])
        H = rng.randint(1, 12)
        C = d * H
        T = _log(rng, 16, 1024)
        if rng.random() < 0.4:
            T = max(32, T // 32 * 32)
        if 64 <= C <= 768 and C * T <= most:
            break
    B = _log(rng, 1, max(1, most // (C * T)))
    layers = rng.choice([1, 1, 2])
    vocab = rng.choice([0, 0, 512]) if family == "block" else 0
    keep = "all" if family == "block" and rng.random() < 0.2 and B * H * T * T <= 1 << 26 else "outputs"
    return _block(family, C, H, T, B, layers, vocab, rng.random() < 0.75, rng.choice(["fused", "fused", "lut"]), keep,
                  rng.random() < 0.7)


def draw(rng):
    family = rng.choice(["block"] * 5 + ["linear"] * 3 + ["run", "frozen"])
    if family == "linear":
        M, K, N = _log(rng, 1, 16384), _log(rng, 64, 3072), _log(rng, 64, 3072)
        if rng.random() < 0.6:                       # layer widths are mostly multiples of 64; the rest are odd ones
            K, N = max(64, K // 64 * 64), max(64, N // 64 * 64)
        return _linear(M, K, N, rng.random() < 0.3, rng.random() < 0.3)
    if family == "frozen":
        return {"family": "frozen", "model": rng.choice(["v1", "v2"]), "batch": _log(rng, 1, 16384),
                "replay": rng.random() < 0.7}
    return _draw_block(rng, family, 1 << 22 if family == "block" else 1 << 18)


# --------------------------------------------------------------------------------------------- graphs and inputs

def _spec(case):
    for spec, tag, _ in models.CONFIGS.values():     # a tracked calibration serves its configuration at any batch
        if all(case[k] == getattr(spec, k) for k in ("n_embd", "n_head", "seq", "layers", "vocab", "causal", "gelu")):
            return spec, tag
    return models.BlockSpec(case["n_embd"], case["n_head"], case["seq"], layers=case["layers"], vocab=case["vocab"],
                            causal=case["causal"], gelu=case["gelu"], calib_batches=2), CALIB_TAG


@lru_cache(maxsize=4)
def _built(spec, tag):
    return models.build(spec, tag)


@lru_cache(maxsize=4)
def _linear_graph(M, K, N, lut):
    """Weights uniform in [-127, 127] and the requant that maps the accumulator's largest magnitude, about 5.5 of its
    standard deviations, to 127 / 1.5 (the quantizer's headroom)."""
    rng = np.random.default_rng([K, N])
    w = rng.integers(-127, 128, (K, N))
    acc = 5.5 * math.sqrt(K) * 127 * 128 / 3
    (mult,), shift = quantize.choose_shift([127 / (quantize.HEADROOM * acc)], [128 * int(np.abs(w).sum(axis=0).max())])
    b = ir.GraphBuilder("linear")
    consts = {"w": w}
    table = None
    if lut:
        consts["gelu"] = quantize.activation_table(models.gelu, 0.03, 0.03)
        table = b.const("gelu", [256], "i8", 0.03)
    b.output(b.qlinear("y", b.input("x", [M, K], "i8", 1.0), b.const("w", [K, N], "i8", 1.0), mult, shift, 1.0,
                       lut=table))
    return b.module(), consts


@lru_cache(maxsize=2)
def _frozen_graph(model):
    with gzip.open(ROOT / "tests" / "golden" / f"model_graph_{model}.json.gz", "rt") as f:
        body = json.load(f)
    return anvil.parse_ir(body["ir"]), {k: np.asarray(v, dtype=np.int64).reshape(body["shapes"][k])
                                        for k, v in body["consts"].items()}


def _graph(case):
    """(module, consts, what compile() takes) of a case."""
    if case["family"] == "linear":
        m, c = _linear_graph(case["M"], case["K"], case["N"], case["lut"])
        return m, c, (m, c)
    if case["family"] == "frozen":
        m, c = _frozen_graph(case["model"])
        return m, c, (m, c)
    b = _built(*_spec(case))
    return b.module, b.consts, b


def _inputs(case, seed):
    """The case's input of a seed, as the caller holds it: float32 N(0, 1) activations or token ids (blocks), integers
    of the input's whole range (linear and frozen)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["family"] == "linear":
        return torch.randint(-127, 128, (1, case["M"], case["K"]), generator=gen, device="cuda", dtype=torch.int8)
    if case["family"] == "frozen":
        dims = (case["batch"], 16, 32)
        lo, dt = (-128, torch.int8) if case["model"] == "v1" else (-(1 << 15), torch.int16)
        return torch.randint(lo, -lo, dims, generator=gen, device="cuda", dtype=dt)
    lead = (case["batch"], case["seq"])
    if case["vocab"]:
        return torch.randint(0, case["vocab"], lead, generator=gen, device="cuda")
    return torch.randn((*lead, case["n_embd"]), generator=gen, device="cuda")


class _Span:
    """A planned device buffer as torch sees it (and what keeps it alive)."""

    def __init__(self, view):
        self.mem = view.buf.mem
        self.__cuda_array_interface__ = {"shape": (view.buf.nbytes // view.itemsize,), "typestr": TYPESTR[view.dtype],
                                         "data": (self.mem.ptr, False), "strides": None, "version": 3}


def _tensor(view):
    """A graph value's device buffer as a torch view in its logical order; a last dim of whole 64-element blocks is
    shown split into them, whether or not the value is stored K-blocked."""
    base = torch.as_tensor(_Span(view), device="cuda")
    dims, st = list(view.dims), list(view.strides)
    if dims[-1] % 64 == 0:
        dims, st = [*dims[:-1], dims[-1] // 64, 64], [*st[:-1], view.kb or 64 * st[-1], st[-1]]
    return base.as_strided(dims, st, view.offset)


class Resident:
    """A compiled model with its plan, and its input on the device."""

    def __init__(self, case, seed):
        module, consts, model = _graph(case)
        self.cm = anvil.compile(model)
        self.replay = case["replay"]
        keep = case.get("keep", "outputs")
        self.plan = self.cm.plan(case.get("batch", 1), keep)
        x, sym = _inputs(case, seed), self.cm.inputs[0]
        dev, view = self.cm.dev, self.plan.views[self.cm.input_ops[0].result]
        if x.dtype == torch.int64:
            self.cm.upload_tokens(self.plan, x.cpu().numpy())
        elif x.dtype == torch.float32:
            torch.cuda.synchronize()
            dev.quantize(x.data_ptr(), False, self.cm.scale(sym), x.numel(), view.ptr, view.dtype)
        else:
            torch.cuda.synchronize()
            dev.copy_strided(x.data_ptr(), view.ptr, x.element_size(), [x.numel()], [1])
        dev.sync()
        by_sym = {op.sym_str: op.result for op in self.cm.ops if op.sym_str is not None}
        syms = self.cm.outputs if keep == "outputs" else self.cm.readable("all")
        self.outputs = {s: _tensor(self.plan.views[by_sym[s]]) for s in syms}
        if self.replay:                              # a serving program captures its plan before the first request
            self.cm.launch(self.plan, graph=True)
            dev.sync()


class HostCall:
    """A compiled model and a host input, for whole run() calls. The first calls (which choose the launch mode) are
    the program's warm-up."""

    def __init__(self, case, seed):
        module, consts, model = _graph(case)
        self.cm = anvil.compile(model)
        self.x = _inputs(case, seed).cpu().numpy()
        self.tokens = bool(case["vocab"])
        self.replay = case["replay"]
        self.call()

    def call(self):
        return self.cm.run(self.x, "mi355x", batch=True, tokens=self.tokens, graph=self.replay)


def prepare(case, seed):
    return HostCall(case, seed) if case["family"] == "run" else Resident(case, seed)


def run(state):
    if isinstance(state, HostCall):
        res = state.call()
        return {"output": res.output, "ints": res.ints}
    state.cm.launch(state.plan, graph=state.replay)
    return state.outputs


# ------------------------------------------------------------------------------------------------ what it must do

def work(case):
    """Each input and constant read once, each returned value written once, two operations a multiply-add; of a causal
    chain's square products the kept half."""
    module, consts, _ = _graph(case)
    nb = case.get("batch", 1)
    flops = nbytes = 0
    ops = ir.func_of(module).ops
    outs = next(op for op in ops if isinstance(op, ir.OutputOp)).values
    fixed = set()
    for op in ops:
        if isinstance(op, ir.OutputOp):
            continue
        t = ir.qt(op.result)
        size = math.prod(t.dims) * rt.ITEMSIZE[t.dtype]
        if isinstance(op, ir.ConstOp) or (op.operands and all(v in fixed for v in op.operands)):
            fixed.add(op.result)
            nbytes += size if isinstance(op, ir.ConstOp) else 0
            continue
        if isinstance(op, (ir.QMatmulOp, ir.QLinearOp)):
            K = ir.qt(op.a).dims[-1]
            n = 2 * nb * math.prod(t.dims) * K
            square = op.b not in fixed and case.get("causal", True) and case.get("keep") != "all"
            flops += n // 2 if square else n
        if isinstance(op, ir.InputOp):
            nbytes += nb * (math.prod(t.dims) * 4 if case["family"] == "run" else size)
        elif case.get("keep") == "all" and not isinstance(op, (ir.TransposeOp, ir.ReshapeOp)):
            nbytes += nb * size
        elif op.result in outs:
            nbytes += nb * math.prod(t.dims) * 16 if case["family"] == "run" else nb * size
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    return "exact"


# --------------------------------------------------------------------------------------------- the same in 64 bits

LIMITS = {"i8": (-128, 127), "i16": (-(1 << 15), (1 << 15) - 1), "i32": (-(1 << 31), (1 << 31) - 1)}


def _round_shift(v, s, dtype):
    """clamp((v + 2^(s-1)) >> s); s a number or a tensor of shifts."""
    s = torch.as_tensor(s, device=v.device, dtype=torch.int64)
    half = torch.where(s > 0, torch.ones_like(s) << (s - 1).clamp(min=0), torch.zeros_like(s))
    return ((v + half) >> s).clamp(*LIMITS[dtype])


def _matmul(a, b):
    return (a.double() @ b.double().contiguous()).round().long()       # every sum below 2^53: exact


def _rmsnorm(x, w, table, op):
    c, n = op.ss_shift_int, table.numel()
    sq = x * x
    ss = ((sq + (1 << (c - 1))) >> c if c else sq).sum(-1, keepdim=True) + op.ss_init_int
    k = torch.zeros_like(ss)
    for _ in range(16):
        big = ss >= n
        ss, k = torch.where(big, ss >> 2, ss), k + big
    return _round_shift(x * w * table[ss] * int(op.M), int(op.s) + k, "i8")


def _softmax(x, table, one, causal):
    keep = torch.ones(x.shape[-2:], dtype=torch.bool, device=x.device)
    keep = keep.tril() if causal else keep
    top = torch.where(keep, x, -128).amax(-1, keepdim=True)
    e = torch.where(keep, table[(x - top + 255).clamp(max=255)], 0)
    total = e.sum(-1, keepdim=True)
    return (e * one + total // 2) // total


def _evaluate(module, consts, x):
    """Every value of the graph for a batch of integer inputs x, by sym, as int64 tensors."""
    env, fixed, named = {}, set(), {}
    for op in ir.func_of(module).ops:
        if isinstance(op, ir.OutputOp):
            return named
        r, t = op.result, ir.qt(op.result)
        v = lambda n: env[op._operands[n]]                              # noqa: E731
        if isinstance(op, ir.InputOp):
            y = x
        elif isinstance(op, ir.ConstOp):
            y = torch.as_tensor(np.asarray(op.value if op.value is not None else consts[op.sym_str], dtype=np.int64))
            y = y.reshape(t.dims).to(x.device)
            fixed.add(r)
        elif isinstance(op, (ir.QMatmulOp, ir.QLinearOp)):
            y = _round_shift(_matmul(v("a"), v("b")) * int(op.M), int(op.s), t.dtype)
            y = y if op.lut is None else v("lut")[y + 128]
        elif isinstance(op, ir.LutOp):
            y = v("table")[v("x") + 128]
        elif isinstance(op, ir.LutMulOp):
            y = _round_shift(v("table")[v("x") + 128] * v("y") * int(op.M), int(op.s), "i8")
        elif isinstance(op, ir.AddRequantOp):
            y = _round_shift(v("a") * int(op.Ma) + v("b") * int(op.Mb), int(op.s), t.dtype)
        elif isinstance(op, ir.RmsNormIntOp):
            y = _rmsnorm(v("x"), v("w"), v("lut"), op)
        elif isinstance(op, ir.SoftmaxLutOp):
            y = _softmax(v("x"), v("lut"), int(op.one), bool(op.causal))
        elif isinstance(op, ir.TransposeOp):
            k = 0 if op.x in fixed else 1
            y = v("x").permute(list(range(k)) + [p + k for p in op.perm_list])
        else:                                                           # reshape
            y = v("x").reshape(([] if op.x in fixed else [len(x)]) + list(t.dims))
        if isinstance(op, (ir.TransposeOp, ir.ReshapeOp)) and op.x in fixed:
            fixed.add(r)
        env[r] = y
        if op.sym_str is not None and r not in fixed:
            named[op.sym_str] = y
    raise ValueError("a graph without an output op")


def exact(case, seed):
    module, consts, model = _graph(case)
    func = ir.func_of(module)
    inp = next(op for op in func.ops if isinstance(op, ir.InputOp))
    t = ir.qt(inp.result)
    x = _inputs(case, seed)
    if x.dtype == torch.int64:
        wte, wpe = (torch.as_tensor(model.params[n]).double().to(x.device) for n in ("wte", "wpe"))
        x = wte[x] + wpe[None, : x.shape[1]]
    if x.is_floating_point():
        x = (x.double() / t.scale).round().clamp(*LIMITS[t.dtype])
    x = x.long()
    outs = [v.owner.sym_str for v in next(op for op in func.ops if isinstance(op, ir.OutputOp)).values]
    parts = {}
    step = max(1, (1 << 24) // (math.prod(t.dims) * max(1, case.get("seq", 16) // 64)))
    for lo in range(0, len(x), step):                                   # sequences are independent
        for s, v in _evaluate(module, consts, x[lo:lo + step]).items():
            if case.get("keep") == "all" or s in outs or s == inp.sym_str:
                parts.setdefault(s, []).append(v)
    val = {s: torch.cat(v) for s, v in parts.items()}
    if case["family"] == "run":
        scale = ir.qt(next(op for op in func.ops if op.sym_str == outs[0]).result).scale
        return {"output": (val[outs[0]].double() * scale).cpu().numpy(), "ints": {s: v.cpu().numpy()
                                                                                  for s, v in val.items()}}
    keep = val if case.get("keep") == "all" else {s: val[s] for s in outs}
    return {s: v.unflatten(-1, (-1, 64)) if v.shape[-1] % 64 == 0 else v for s, v in keep.items()}
