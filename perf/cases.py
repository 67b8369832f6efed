"""The work a user of the decode worker has it do, as cases that can be timed and compared.

Three kinds of case, each through a public entry point:

* ``request``: one request on a sequence context (tiles_amd.runtime): reset, prefill a prompt,
  generate ``new`` tokens greedily (0: the prompt alone, as a scoring program calls it), wait,
  collect the last step's logits.  Returns the tokens and the logits.
* ``step``: a host of the launch boundary that owns every buffer (``ti_enqueue_worker``) and a
  cache filled up to ``position``: one launch decodes ``steps`` given tokens.  Returns the last
  step's logits and the K/V rows that the launch wrote.
* ``head``: the isolated LM-head step, ``rounds`` times on a hidden vector from the host.

Widths are Llama-3.2-1B's (hidden 2048, FFN 8192, 32 query and 8 K/V heads of 64 dims).  The
whole model has 16 layers and 128,256 tokens; the cases of single layers run a stack of 2 (1
layer's outputs alone are not visible in a prefill: its cache rows do not depend on its attention)
with 4,096 tokens.  Weights are N(0, 0.02) and norm weights 1, as the benchmark's, with two
differences: embedding rows are N(0, 1) and tied, so that the greedy choice is decisive, as a
trained model's mostly is, and a rounding does not change which tokens follow; and the matrices
that write to the residual stream (Wo, Wdown) are scaled by 1 / sqrt(2 layers), as usual inits do,
so that a rounding in one layer is not blown up by those after it.

Packages are planned as the benchmark plans them: 384 positions with the planner's own chunking
(one fused chunk), 4,160 positions in 130-step chunks, 32,832 in 1,026-step chunks.  A program
keeps its model and its contexts, so models are loaded once per process and a state holds a context.
"""

from __future__ import annotations

import atexit
import ctypes as C
import hashlib
import math
import os
import random
import shutil
import tempfile
from pathlib import Path

import torch

from tiles_amd import runtime as R
from tiles_amd.tileplan import package as K
from tiles_amd.tileplan import plan as P
from tiles_amd.tileplan import probe

# Largest context -> attention chunk steps of its package (None: the planner's default).
TIERS = {384: None, 4160: 130, 32832: 1026}
LAYER_TIER = 4160  # the 2-layer stacks' package: every range of the single-layer cases fits it
LAYER_VOCAB = 4096
HIDDEN, FFN, HEADS, KV_HEADS, DIM = 2048, 8192, 32, 8, 64
KV_WIDTH = KV_HEADS * DIM


def listed() -> list[dict]:
    def request(name, prompt, new, layers=16, dtype="bfloat16"):
        return {"name": name, "kind": "request", "dtype": dtype, "layers": layers, "prompt": prompt, "new": new}

    def step(name, position, steps, layers, dtype="bfloat16"):
        return {"name": name, "kind": "step", "dtype": dtype, "layers": layers, "position": position, "steps": steps}

    return [
        # One token through two layers at a short context: the smallest call, all launch and latency.
        step("step_layers_ctx40", 40, 1, 2),
        # The same in fp32, well into a split context: the option for exact comparisons.
        step("step_layers_f32_ctx1500", 1500, 1, 2, "float32"),
        # One decode step of the whole model for a program that samples on its own.
        step("step_model_ctx600", 600, 1, 16),
        # The benchmark's isolated LM-head step, 20 rounds.
        {"name": "lm_head", "kind": "head", "dtype": "bfloat16", "rounds": 20},
        # The layers of a prefill alone: a ragged prompt through two of them.
        request("prefill_layers_1000", 1001, 0, layers=2),
        # A short question: the time to its first token's logits.
        request("prompt_37", 37, 0),
        # An ordinary chat turn, prompt and answer.
        request("chat_211_48", 211, 48),
        # A page of text scored.
        request("prompt_1500", 1531, 0),
        # The benchmark's generations: from one token, and after 4,096.
        request("generate_1_256", 1, 256),
        request("prompt_4096_64", 4096, 64),
        # A document of about the longest context with an odd length, and a short answer.
        request("prompt_30011_32", 30011, 32),
        # An fp32 request (the worker prefills and decodes; layers alone).
        request("request_f32_29_8", 29, 8, layers=2, dtype="float32"),
    ]


def draw(rng: random.Random) -> dict:
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    if rng.random() < 0.3:
        layers = rng.choice((2, 2, 16))
        dtype = "float32" if layers == 2 and rng.random() < 0.35 else "bfloat16"
        steps = 1 if rng.random() < 0.6 else log(2, 64)
        return {"kind": "step", "dtype": dtype, "layers": layers, "position": log(1, 4000), "steps": steps}
    if rng.random() < 0.15:
        return {"kind": "request", "dtype": "float32", "layers": 2, "prompt": log(1, 300), "new": rng.choice((0, log(1, 64)))}
    layers = rng.choice((2, 16, 16, 16))
    prompt = log(2, 4000 if layers == 2 else 28000)
    new = 0 if rng.random() < 0.5 else log(1, 24 if prompt > 8000 else 200)
    return {"kind": "request", "dtype": "bfloat16", "layers": layers, "prompt": prompt, "new": min(new, 4100 - prompt) if layers == 2 else new}


# ---------------------------------------------------------------- models

_weights: dict = {}
_models: dict = {}
_scratch: Path | None = None


def _vocab(layers: int) -> int:
    return 128256 if layers == 16 else LAYER_VOCAB


def _spec(layers: int, max_context: int) -> P.StackSpec:
    spec = P.llama32_1b(max_context)
    return spec if layers == 16 else P.StackSpec(spec.block, layers, LAYER_VOCAB, True)


def _stack_weights(layers: int, dtype: str) -> dict:
    """The stack's weights on the GPU, from a fixed seed, in the package's type (Wdown [d, f])."""
    if (layers, dtype) not in _weights:
        generator = torch.Generator(device="cuda").manual_seed(1234)
        kind = torch.bfloat16 if dtype == "bfloat16" else torch.float32
        spec, out = _spec(layers, 384), {}
        for name in K.weight_names(spec):
            shape = K.weight_shape(spec, name)
            if name.endswith("norm"):
                out[name] = torch.ones(shape, dtype=kind, device="cuda")
            else:
                std = 1.0 if name == "embedding" else 0.02
                if name.endswith((".Wo", ".Wdown")):
                    std /= math.sqrt(2 * layers)
                out[name] = (torch.randn(shape, generator=generator, device="cuda") * std).to(kind)
        _weights[layers, dtype] = out
    return _weights[layers, dtype]


def _package(layers: int, dtype: str, tier: int) -> Path:
    """The package's directory.  The tiers of one stack hold the same weights: the first is built
    whole, the others are planned against a link to its weights.bin."""
    global _scratch
    if _scratch is None:
        _scratch = Path(tempfile.mkdtemp(prefix="perf_cases_"))
        atexit.register(shutil.rmtree, _scratch, ignore_errors=True)
    out = _scratch / f"{layers}_{dtype}_{tier}"
    target, spec = probe.probe_library(), _spec(layers, tier)
    built = sorted(_scratch.glob(f"{layers}_{dtype}_*"))
    if not built:
        weights = {name: value.cpu() for name, value in _stack_weights(layers, dtype).items()}
        K.build_stack_package(spec, weights, target, out, dtype, chunk_steps=TIERS[tier])
    else:
        digest = K.read_plan(built[0])["integrity"]["weights_sha256"]
        out.mkdir()
        os.link(built[0] / "weights.bin", out / "weights.bin")
        plan = P.json_bytes(P.stack_plan(spec, P.plan_target(target), dtype, digest, TIERS[tier]))
        (out / "plan.json").write_bytes(plan)
    return out


def _model(layers: int, dtype: str, length: int):
    """The loaded model of the smallest package that holds `length` positions, and its plan."""
    tier = LAYER_TIER if layers == 2 else next(t for t in TIERS if t >= length)
    key = (layers, dtype, tier)
    if key not in _models:
        path = _package(*key)
        _models[key] = (R.DecoderModel(R.load_plan(path, verify_weights=False)), K.read_plan(path))
    return _models[key]


def _seed(case: dict, seed: int) -> int:
    text = repr(sorted((k, v) for k, v in case.items() if k != "name")) + str(seed)
    return int.from_bytes(hashlib.sha256(text.encode()).digest()[:6], "little")


def _tokens(case: dict, seed: int, count: int) -> list[int]:
    generator = torch.Generator().manual_seed(_seed(case, seed))
    return torch.randint(0, _vocab(case["layers"]), (count,), generator=generator).tolist()


def _cache_rows(case: dict, seed: int) -> torch.Tensor:
    """The cached K and V rows before the step's position, [layers, 2, position, KV_WIDTH], spread
    as the projections of a normalized vector by N(0, 0.02) weights are."""
    generator = torch.Generator(device="cuda").manual_seed(_seed(case, seed))
    shape = (case["layers"], 2, case["position"], KV_WIDTH)
    rows = torch.randn(shape, generator=generator, device="cuda") * (0.02 * math.sqrt(HIDDEN))
    return rows.to(torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32)


def _hidden(seed: int) -> torch.Tensor:
    return torch.randn(HIDDEN, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)


class _Host:
    """The buffers of a host that drives the launch boundary itself."""

    def __init__(self, case: dict, seed: int):
        self.lib = R.library()
        model, plan = _model(case["layers"], case["dtype"], case["position"] + case["steps"])
        self.model, self.view = model, model.program_view()
        storage, layers, steps = plan["storage"], case["layers"], case["steps"]
        kind = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
        elem = kind.itemsize
        byte = lambda n: torch.zeros(max(int(n), 16), dtype=torch.uint8, device="cuda")  # noqa: E731
        self.kv = byte(storage["kv_bytes"])
        rows = self.kv.view(kind).view(layers, 2, plan["model"]["max_context"], KV_WIDTH)
        rows[:, :, : case["position"]] = _cache_rows(case, seed)
        self.written = rows[:, :, case["position"]: case["position"] + steps]
        self.logits = torch.zeros(_vocab(layers), dtype=torch.float32, device="cuda")
        words = self.lib.ti_exchange_words(C.byref(self.view.shape), layers, self.view.selection_slots)
        self.exchange = torch.zeros(words, dtype=torch.int64, device="cuda")
        self.tokens = torch.tensor(_tokens(case, seed, steps), dtype=torch.int32, device="cuda")
        self.others = [byte(HIDDEN * elem), byte(HIDDEN * elem), byte(storage["scratch_bytes"]), byte(storage["attention_bytes"]),
                       byte(storage["attention_partial_bytes"] + storage["ffn_partial_bytes"]),
                       byte(8 * max(1, self.view.selection_slots))]
        self.buffers = R.WorkerBuffers()
        b = self.buffers
        b.input, b.output, b.scratch, b.attention_scores, b.attention_partials, b.selection = (t.data_ptr() for t in self.others)
        b.kv, b.logits, b.exchange = self.kv.data_ptr(), self.logits.data_ptr(), self.exchange.data_ptr()
        b.epoch = 1
        self.advance = self.lib.ti_epochs_per_launch(layers)
        self.token = R.TokenInput(-1, self.tokens.data_ptr(), steps)
        self.position = case["position"]

    def launch(self) -> tuple:
        stream = torch.cuda.current_stream().cuda_stream
        code = self.lib.ti_enqueue_worker(stream, C.byref(self.view), C.byref(self.buffers), self.position, self.token,
                                          R.Selection())
        if code != 0:
            raise RuntimeError(self.lib.ti_last_error_message().decode())
        self.buffers.epoch += self.advance
        if self.buffers.epoch > 0xF0000000:  # a host that goes back to epoch 1 clears the exchange area first
            self.exchange.zero_()
            self.buffers.epoch = 1
        return self.logits, self.written


# ---------------------------------------------------------------- the contract

def prepare(case: dict, seed: int) -> dict:
    if case["kind"] == "step":
        return {"kind": "step", "host": _Host(case, seed)}
    if case["kind"] == "head":
        model, _ = _model(16, case["dtype"], 1)
        bits = _hidden(_seed(case, seed)).view(torch.int16).numpy().view("uint16")
        return {"kind": "head", "context": model.create_context(), "hidden": bits, "rounds": case["rounds"]}
    model, _ = _model(case["layers"], case["dtype"], case["prompt"] + case["new"])
    return {"kind": "request", "context": model.create_context(), "prompt": _tokens(case, seed, case["prompt"]),
            "new": case["new"]}


def run(state: dict):
    if state["kind"] == "step":
        logits, rows = state["host"].launch()
        return {"logits": logits, "kv": rows}
    ctx = state["context"]
    if state["kind"] == "head":
        ticket = ctx.enqueue_lm_head_step(state["hidden"], rounds=state["rounds"], logits=True)
        token = ctx.wait(ticket).generated[0]
        return {"token": token, "logits": ctx.collect(ticket)["logits"]}
    ctx.enqueue_reset()
    if state["new"] == 0:
        ticket = ctx.enqueue_prefill(state["prompt"], logits=True)
        ctx.wait(ticket)
        return {"logits": ctx.collect(ticket)["logits"]}
    ctx.enqueue_prefill(state["prompt"])
    ticket = ctx.enqueue_generate(state["new"], logits=True)
    tokens = torch.tensor(ctx.wait(ticket).generated)
    return {"tokens": tokens, "logits": ctx.collect(ticket)["logits"]}


def work(case: dict) -> dict:
    """Weights are read once per token that has to wait for the one before it (and once for a
    whole prompt), cache rows once per pass over them, new rows and logits written once.
    Products count two operations; attention those of the causal half."""
    elem = 2 if case["dtype"] == "bfloat16" else 4
    head = 128256 if case["kind"] == "head" else _vocab(case["layers"])
    head_bytes = head * HIDDEN * elem
    if case["kind"] == "head":
        return {"bytes": case["rounds"] * (head_bytes + 2 * HIDDEN * elem + 4 * head), "flops": case["rounds"] * 2 * head * HIDDEN}
    layers = case["layers"]
    layer_params = 2 * HIDDEN * HIDDEN + 2 * KV_WIDTH * HIDDEN + 3 * HIDDEN * FFN
    weights = layers * (layer_params + 2 * HIDDEN) * elem + HIDDEN * elem
    row = layers * 2 * KV_WIDTH * elem  # one position's K and V in every layer

    def attention(first, count):  # positions first .. first + count - 1, each over itself and those before it
        return layers * 4 * HIDDEN * (count * first + count * (count + 1) // 2)

    if case["kind"] == "step":
        p, n = case["position"], case["steps"]
        return {"bytes": weights + head_bytes + (p + n) * row + 4 * head,
                "flops": n * layers * 2 * layer_params + attention(p, n) + 2 * head * HIDDEN}
    n, new = case["prompt"], case["new"]
    decoded = sum(n + i + 1 for i in range(new))  # rows read or written by the new tokens' steps
    return {"bytes": (1 + new) * (weights + head_bytes) + (n + decoded) * row + 4 * head,
            "flops": (n + new) * layers * 2 * layer_params + attention(0, n + new) + (1 + new) * 2 * head * HIDDEN}


def tolerance(case: dict) -> dict:
    """Measured between a prefill by matrices and one position at a time, two evaluations that
    round at the same points and sum in other orders (100 to 1,001 positions): rel 0.004 and max 0.02
    through 2 layers, 0.010 and 0.05 through 16; the head alone flips single roundings of its
    logits.  fp32 results are 2.6e-7 off 64 bits."""
    if case["dtype"] == "float32":
        return {"rel": 2e-6, "max": 2e-5}
    if case["kind"] == "head":
        return {"rel": 2e-3, "max": 0.03}
    return {"rel": 1.5e-2, "max": 0.08} if case["layers"] == 2 else {"rel": 2.5e-2, "max": 0.2}


# ---------------------------------------------------------------- 64 bits

def _frequencies() -> torch.Tensor:
    """Llama-3 scaled rotary frequencies, in the 32 bits a package holds them in."""
    indices = torch.arange(0, DIM, 2, dtype=torch.float32)
    inverse = 1.0 / (500000.0 ** (indices / DIM))
    wavelength = 2 * math.pi / inverse
    low, high = 8192 / 1.0, 8192 / 4.0
    smooth = (8192 / wavelength - 1.0) / 3.0
    scaled = torch.where(wavelength > low, inverse / 32.0, inverse)
    blended = (1 - smooth) * scaled / 32.0 + smooth * scaled
    return torch.where((wavelength >= high) & (wavelength <= low), blended, scaled).cuda()


def _norm(x: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5)


def _forward(case: dict, tokens: list[int], cached: torch.Tensor | None):
    """Logits of the last of `tokens`, which follow the `cached` rows, and the K and V rows of all."""
    w = _stack_weights(case["layers"], case["dtype"])
    first = 0 if cached is None else cached.shape[2]
    n = len(tokens)
    x = w["embedding"][torch.tensor(tokens, device="cuda")].double()
    angles = (torch.arange(first, first + n, device="cuda", dtype=torch.float32)[:, None] * _frequencies()).double()
    cosine, sine = angles.cos()[:, None], angles.sin()[:, None]

    def rotate(v):
        a, b = v.chunk(2, dim=-1)
        return torch.cat((a * cosine - b * sine, b * cosine + a * sine), dim=-1)

    group, rows = HEADS // KV_HEADS, []
    for layer in range(case["layers"]):
        m = lambda v, name: v @ w[f"L{layer}.{name}"].double().T.contiguous()  # noqa: E731
        u = _norm(x)
        q = rotate(m(u, "Wq").view(n, HEADS, DIM))
        k = rotate(m(u, "Wk").view(n, KV_HEADS, DIM))
        v = m(u, "Wv").view(n, KV_HEADS, DIM)
        rows.append(torch.stack((k.reshape(n, KV_WIDTH), v.reshape(n, KV_WIDTH))))
        if cached is not None:
            k = torch.cat((cached[layer, 0].double().view(first, KV_HEADS, DIM), k))
            v = torch.cat((cached[layer, 1].double().view(first, KV_HEADS, DIM), v))
        kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
        out = torch.empty(n, KV_HEADS, group, DIM, dtype=torch.float64, device="cuda")
        block = 512
        for r in range(0, n, block):
            count, end = min(block, n - r), first + min(r + block, n)
            grouped = q[r:r + count].view(count, KV_HEADS, group, DIM).permute(1, 2, 0, 3).reshape(KV_HEADS, group * count, DIM)
            s = torch.bmm(grouped.contiguous(), kt[:, :, :end].contiguous()).view(KV_HEADS, group, count, end) / math.sqrt(DIM)
            s.masked_fill_(torch.arange(end, device="cuda") > torch.arange(first + r, end, device="cuda")[:, None], -math.inf)
            p = torch.softmax(s, dim=-1).view(KV_HEADS, group * count, end)
            a = torch.bmm(p, vt[:, :end].contiguous()).view(KV_HEADS, group, count, DIM)
            out[r:r + count] = a.permute(2, 0, 1, 3)
            del s, p
        x = x + m(out.view(n, HIDDEN), "Wo")
        z = _norm(x)
        y = torch.empty_like(x)
        for r in range(0, n, 4096):
            part = z[r:r + 4096]
            y[r:r + 4096] = m(torch.nn.functional.silu(m(part, "Wgate")) * m(part, "Wup"), "Wdown")
        x = x + y
    logits = (_norm(x[-1:]) @ w["embedding"].double().T.contiguous())[0]
    return logits, torch.stack(rows)


def exact(case: dict, seed: int):
    if case["kind"] == "head":
        w = _stack_weights(16, case["dtype"])["embedding"].double()
        logits = w @ _norm(_hidden(_seed(case, seed)).cuda().double())
        return {"token": None, "logits": logits}
    if case["kind"] == "step":
        logits, rows = _forward(case, _tokens(case, seed, case["steps"]), _cache_rows(case, seed))
        return {"logits": logits, "kv": rows}
    tokens = _tokens(case, seed, case["prompt"])
    # The greedy choice repeats the last token, by far (the embedding is tied and its rows long).
    logits, _ = _forward(case, tokens + tokens[-1:] * case["new"], None)
    return {"logits": logits} if case["new"] == 0 else {"tokens": None, "logits": logits}
