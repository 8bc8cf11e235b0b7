"""The calls whose speed matters to a user of this framework, over the sizes they are made at.

A case is one call (or one short chain of calls) through the package's public entry points. Six kinds:

  decide     one `DecisionEngine.forward_records` call: host packing, the decision forward, results on the host
  forward    `gemma.forward` on a packed batch that is already on the device: embedding, decoder layers, readout
  attention  `kernels.attention` ([B, S, H, D] with a key mask) in bf16 and fp32
  encoder    `kernels.flash_attention`, the packed bidirectional interface
  head       the Clef joint head: `clef_head.lexical_vectors` and `clef_head.forward`
  mlp        `kernels.mlp`, the fused norm -> gate|up -> down block

Decoder cases run the 9B and 27B shapes at full width and a reduced depth, so that three sets of weights are
made quickly and a pass reads all of them from memory, as a full-depth forward does; every layer of the full
depth does the same work.
"""

from __future__ import annotations

import math
from dataclasses import replace
from typing import Any

import numpy as np
import torch

from deciax_amd import clef_head, gemma, kernels
from deciax_amd.engine import DecisionEngine
from deciax_amd.schema import ByteTokenizer, encode

DEV = "cuda"
VOCAB = 32768  # rows of the embedding table: a forward reads only the rows its tokens name
BF16 = torch.bfloat16


def listed() -> list[dict[str, Any]]:
    return [
        # One short request through the engine, host work included: what `Decider.decide` waits for.
        dict(name="decide-one", kind="decide", model="gemma2-9b", layers=2, state=150, questions=1),
        # A handful of tokens (a token tokenizer's short request): weights stream once per call.
        dict(name="9b-1x97", kind="forward", model="gemma2-9b", layers=2, requests=1, lo=97, hi=97, questions=1),
        # One ordinary request, an odd length.
        dict(name="9b-1x517", kind="forward", model="gemma2-9b", layers=2, requests=1, lo=517, hi=517, questions=4),
        # One request with a long prompt (eight questions and their options).
        dict(name="9b-1x3300", kind="forward", model="gemma2-9b", layers=2, requests=1, lo=3300, hi=3300, questions=8),
        # The serving batch the benchmark times: ragged requests, log-uniform in [256, 16384].
        dict(name="9b-16-ragged", kind="forward", model="gemma2-9b", layers=2, requests=16, lo=256, hi=16384, questions=8),
        # The larger shape (head_dim 128, its weights beyond the last-level cache), a small batch.
        dict(name="27b-2x1000", kind="forward", model="gemma2-27b", layers=1, requests=2, lo=1000, hi=1000, questions=4),
        # Right-padded causal attention as a backbone without soft-capping calls it.
        dict(name="attn-bf16-4x2048", kind="attention", dtype="bf16", batch=4, seq=2048, hq=32, hkv=8, d=128, causal=True,
             window=0, cap=0.0),
        # Full-precision attention at the widest head, odd length, soft-capped.
        dict(name="attn-f32-2x701", kind="attention", dtype="f32", batch=2, seq=701, hq=8, hkv=4, d=256, causal=True,
             window=0, cap=50.0),
        # Encoder layer: bidirectional, packed q | k | v, head_dim 64.
        dict(name="encoder-8x1021", kind="encoder", batch=8, seq=1021, heads=12, window=0),
        # Joint head behind one request: a few questions, some twenty options.
        dict(name="head-1x600", kind="head", batch=1, seq=600, fields=6, opts=23, hidden=4096, width=1024, ff=2048,
             heads=16),
        # Joint head at the protocol's limits of fields and options, a batch of long requests.
        dict(name="head-8x4096", kind="head", batch=8, seq=4096, fields=64, opts=512, hidden=4096, width=1024, ff=2048,
             heads=16),
        # The gated MLP block by itself, fp32 out, some hundred rows.
        dict(name="mlp-200", kind="mlp", rows=200, d=3584, f=14336, act="gelu_tanh", out="f32"),
    ]


def draw(rng) -> dict[str, Any]:
    def log(lo: int, hi: int) -> int:
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decide", "forward", "forward", "forward", "attention", "attention", "encoder", "head", "head", "mlp"])
    if kind == "decide":
        return dict(kind=kind, model="gemma2-9b", layers=2, state=log(40, 6000), questions=rng.randint(1, 8))
    if kind == "forward":
        model = rng.choice(["gemma2-9b", "gemma2-9b", "gemma2-27b"])
        requests = rng.choice([1, 1, 2, 3, 5, 8])
        lo = log(24, 4096)
        return dict(kind=kind, model=model, layers=2 if model == "gemma2-9b" else 1, requests=requests, lo=lo,
                    hi=min(8192, int(lo * rng.uniform(1.0, 3.0))), questions=rng.randint(1, 8))
    if kind == "attention":
        dtype = rng.choice(["bf16", "f32"])
        d = rng.choice([64, 128, 256])
        hkv = rng.choice([2, 4, 8])
        return dict(kind=kind, dtype=dtype, batch=rng.randint(1, 4), seq=log(40, 2048 if dtype == "bf16" else 1024),
                    hq=hkv * rng.choice([1, 2, 4]), hkv=hkv, d=d, causal=rng.random() < 0.7,
                    window=rng.choice([0, 0, 128, 300]), cap=rng.choice([0.0, 50.0]))
    if kind == "encoder":
        return dict(kind=kind, batch=rng.randint(1, 12), seq=log(60, 2048), heads=rng.choice([4, 6, 12, 16]),
                    window=rng.choice([0, 64]))
    if kind == "head":
        fields = rng.randint(1, 64)
        return dict(kind=kind, batch=rng.randint(1, 6), seq=log(120, 4000), fields=fields,
                    opts=min(512, int(fields * rng.uniform(2.0, 8.0)) + 1), hidden=rng.choice([3584, 4096]),
                    width=rng.choice([512, 768, 1024]), ff=rng.choice([1024, 2048]), heads=rng.choice([8, 16]))
    model = rng.choice([(3584, 14336), (4608, 36864)])
    return dict(kind="mlp", rows=log(8, 3000), d=model[0], f=model[1], act=rng.choice(["gelu_tanh", "silu"]),
                out=rng.choice(["f32", "bf16"]))


# ------------------------------------------------------------------------------------------ inputs


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g: torch.Generator, shape: tuple[int, ...], std: float, dtype: torch.dtype = BF16) -> torch.Tensor:
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=g)


def _config(case: dict[str, Any]) -> gemma.GemmaConfig:
    return replace(gemma.CONFIGS[case["model"]], layers=case["layers"], vocab=VOCAB)


def _tensors(c: gemma.GemmaConfig, g: torch.Generator) -> dict[str, torch.Tensor]:
    """Random weights under the names `gemma.weights_from_host` takes."""
    h, d = c.hidden, c.head_dim
    t = {"embed": _normal(g, (c.vocab, h), 0.02), "final_norm": _normal(g, (h,), 0.1)}
    for i in range(c.layers):
        for name, shape in (("q", (c.heads * d, h)), ("k", (c.kv_heads * d, h)), ("v", (c.kv_heads * d, h)),
                            ("o", (h, c.heads * d)), ("gate", (c.intermediate, h)), ("up", (c.intermediate, h)),
                            ("down", (h, c.intermediate))):
            t[f"layers.{i}.{name}"] = _normal(g, shape, 0.02)
        for name in ("input_norm", "post_attn_norm", "pre_ffn_norm", "post_ffn_norm"):
            t[f"layers.{i}.{name}"] = _normal(g, (h,), 0.1)
    return t


def _lengths(case: dict[str, Any]) -> list[int]:
    """Request lengths of a case: part of its size, so the same for every seed."""
    r = np.random.Generator(np.random.PCG64(0))
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    return [int(round(math.exp(r.uniform(lo, hi)))) if hi > lo else case["lo"] for _ in range(case["requests"])]


def _requests(case: dict[str, Any], seed: int) -> tuple[list, list]:
    r = np.random.Generator(np.random.PCG64(seed))
    ids, options = [], []
    for n in _lengths(case):
        ids.append(r.integers(0, VOCAB, n).tolist())
        tail = min(n, 512)
        counts = [2 + (j * 3) % 7 for j in range(case["questions"])]
        pos = r.integers(n - tail, n, sum(counts))
        labels = r.integers(0, VOCAB, sum(counts))
        at, req = 0, []
        for k in counts:
            req.append([(int(p), int(t)) for p, t in zip(pos[at:at + k], labels[at:at + k])])
            at += k
        options.append(req)
    return ids, options


def _questions(n: int) -> dict[str, Any]:
    """n questions of the three kinds a request may ask, in turn."""
    kinds = [
        {"type": "noul", "instructions": "Does the message ask for an answer today?"},
        {"type": "choice", "instructions": "Which team should handle it?",
         "criteria": {"billing": "invoices and refunds", "support": "technical problems", "sales": None}},
        {"type": "score", "instructions": "How upset is the writer?", "criteria": ["calm", "annoyed", "angry"]},
    ]
    return {f"q{i}": kinds[i % 3] for i in range(n)}


def _record(case: dict[str, Any], seed: int):
    r = np.random.Generator(np.random.PCG64(seed))
    state = "".join(chr(c) for c in r.integers(97, 123, case["state"]))
    return encode(ByteTokenizer(VOCAB), {"message": state}, _questions(case["questions"]), 16384, vocab=VOCAB)


def _head_params(case: dict[str, Any], g: torch.Generator) -> dict[str, torch.Tensor]:
    h, w, ff = case["hidden"], case["width"], case["ff"]
    p: dict[str, torch.Tensor] = {}

    def mat(name: str, n: int, k: int, bias: bool = True) -> None:
        p[name + ".weight"] = _normal(g, (n, k), k ** -0.5, torch.float32)
        if bias:
            p[name + ".bias"] = _normal(g, (n,), 0.05, torch.float32)

    def ln(name: str, n: int) -> None:
        p[name + ".weight"] = 1 + _normal(g, (n,), 0.1, torch.float32)
        p[name + ".bias"] = _normal(g, (n,), 0.05, torch.float32)

    def att(name: str) -> None:
        p[name + ".in_proj_weight"] = _normal(g, (3 * w, w), w ** -0.5, torch.float32)
        p[name + ".in_proj_bias"] = _normal(g, (3 * w,), 0.05, torch.float32)
        mat(name + ".out_proj", w, w)

    ln("hidden_norm", h)
    mat("memory_projection", w, h)
    for name in ("option_context_projection", "option_lexical_projection", "option_question_projection", "global_projection"):
        mat(name, w, h, bias=False)
    mat("question_projection", w, h)
    for name in ("option_summary_norm", "field_norm", "option_norm"):
        ln(name, w)
    p["type_embedding.weight"] = _normal(g, (3, w), 0.2, torch.float32)
    mat("residual_scorer.0", ff, 4 * w)
    mat("residual_scorer.3", 1, ff)
    for i in range(2):
        n = f"evidence_layers.{i}"
        att(n + ".attention")
        for m in ("query_norm", "memory_norm", "feedforward_norm"):
            ln(f"{n}.{m}", w)
        mat(n + ".feedforward.0", ff, w)
        mat(n + ".feedforward.3", w, ff)
        n = f"layers.{i}"
        att(n + ".self_attn")
        att(n + ".multihead_attn")
        for m in ("norm1", "norm2", "norm3"):
            ln(f"{n}.{m}", w)
        mat(n + ".linear1", ff, w)
        mat(n + ".linear2", w, ff)
    p["prior_logit_scale"] = torch.tensor(2.0, device=DEV)
    p["joint_logit_scale"] = torch.tensor(2.5, device=DEV)
    p["residual_gate"] = torch.tensor(0.3, device=DEV)
    return p


def _head_arrays(case: dict[str, Any], seed: int) -> dict[str, np.ndarray]:
    """The collate arrays: full first request, shorter others (lengths and counts are part of the case's size, so
    the same for every seed), every field owning options in order."""
    size, r = (np.random.Generator(np.random.PCG64(x)) for x in (0, seed))
    b, s, q, o = case["batch"], case["seq"], case["fields"], case["opts"]
    lens = np.array([s] + [int(size.integers(max(s // 2, 64), s + 1)) for _ in range(b - 1)])
    mask = np.arange(s)[None, :] < lens[:, None]
    a = dict(mask=mask, question_spans=np.zeros((b, q, 2), np.int32), option_spans=np.zeros((b, o, 2), np.int32),
             lexical_spans=np.zeros((b, o, 2), np.int32), option_field=np.zeros((b, o), np.int32),
             option_mask=np.zeros((b, o), bool), question_mask=np.zeros((b, q), bool),
             types=r.integers(0, 3, (b, q)).astype(np.int32))
    for i in range(b):
        live_q = q if i == 0 else int(size.integers((q + 1) // 2, q + 1))
        live_o = o if i == 0 else int(size.integers(max(live_q, (o + 1) // 2), o + 1))
        a["question_mask"][i, :live_q] = True
        a["option_mask"][i, :live_o] = True
        a["option_field"][i, :live_o] = np.arange(live_o) * live_q // live_o
        for name, n, most in (("question_spans", live_q, 40), ("option_spans", live_o, 24)):
            width = r.integers(1, most, n)
            start = r.integers(0, lens[i] - width + 1)
            a[name][i, :n, 0], a[name][i, :n, 1] = start, start + width
        width = a["option_spans"][i, :, 1] - a["option_spans"][i, :, 0]
        ends = np.cumsum(width)
        a["lexical_spans"][i, :, 0], a["lexical_spans"][i, :, 1] = ends - width, ends
    a["lexical_ids"] = r.integers(0, VOCAB, (b, max(1, int(a["lexical_spans"].max())))).astype(np.int32)
    return a


def prepare(case: dict[str, Any], seed: int) -> dict[str, Any]:
    g = _gen(seed)
    kind = case["kind"]
    s: dict[str, Any] = {"case": case}
    if kind == "decide":
        c = _config(case)
        weights = gemma.weights_from_host(c, _tensors(c, g), device=DEV)
        s["engine"] = DecisionEngine(weights, ByteTokenizer(VOCAB), c.name)
        s["records"] = [_record(case, seed)]
    elif kind == "forward":
        c = _config(case)
        s["weights"] = gemma.weights_from_host(c, _tensors(c, g), device=DEV)
        s["batch"] = gemma.pack_batch(*_requests(case, seed), device=DEV)
        s["ws"] = gemma.Workspace(c, s["batch"].rows, s["batch"].vt_ld, torch.device(DEV))
    elif kind == "attention":
        dt = BF16 if case["dtype"] == "bf16" else torch.float32
        b, n, d = case["batch"], case["seq"], case["d"]
        s["q"], s["k"], s["v"] = (_normal(g, (b, n, h, d), 1.0, dt) for h in (case["hq"], case["hkv"], case["hkv"]))
        s["mask"] = _padding(b, n, seed)
    elif kind == "encoder":
        s["qkv"] = _normal(g, (case["batch"], case["seq"], 3 * case["heads"] * 64), 1.0)
        s["mask"] = _padding(case["batch"], case["seq"], seed)
    elif kind == "head":
        s["params"] = _head_params(case, g)
        s["embedding"] = _normal(g, (VOCAB, case["hidden"]), 1.0, torch.float32)
        s["hidden"] = _normal(g, (case["batch"], case["seq"], case["hidden"]), 1.0, torch.float32)
        s["arrays"] = _head_arrays(case, seed)
        s["live"] = torch.as_tensor(np.flatnonzero(s["arrays"]["option_mask"])).to(DEV)
    else:
        d, f = case["d"], case["f"]
        s["x"] = _normal(g, (case["rows"], d), 1.0)
        s["norm"] = _normal(g, (d,), 0.1)
        s["gate"], s["up"] = _normal(g, (f, d), 0.02), _normal(g, (f, d), 0.02)
        s["down"] = _normal(g, (d, f), 0.02)
        s["gate_up"] = kernels.pack_gate_up(s["gate"], s["up"])
    return s


def _padding(b: int, n: int, seed: int) -> torch.Tensor:
    """A right-padding key mask: the first row full, the others at least half."""
    r = np.random.Generator(np.random.PCG64(seed))
    lens = np.array([n] + [int(r.integers((n + 1) // 2, n + 1)) for _ in range(b - 1)])
    return torch.as_tensor(np.arange(n)[None, :] < lens[:, None]).to(DEV)


def run(s: dict[str, Any]) -> Any:
    case = s["case"]
    kind = case["kind"]
    if kind == "decide":
        return s["engine"].forward_records(s["records"])
    if kind == "forward":
        logits, probs = gemma.forward(s["weights"], s["batch"], s["ws"])
        return {"logits": logits, "probs": probs, "hidden": s["ws"].x[:s["batch"].rows]}
    if kind == "attention":
        return kernels.attention(s["q"], s["k"], s["v"], s["mask"], causal=case["causal"], window=case["window"],
                                 softcap=case["cap"])
    if kind == "encoder":
        return kernels.flash_attention(s["qkv"], s["mask"], heads=case["heads"], window=case["window"])
    if kind == "head":
        a = s["arrays"]
        lexical = clef_head.lexical_vectors(s["embedding"], a["lexical_ids"], a["lexical_spans"])
        logits = clef_head.forward(s["params"], s["hidden"], lexical, a, heads=case["heads"], routing_layers=2, layers=2)
        # padded options hold -1e9: the decoder reads the live ones
        return {"logits": logits, "live": logits.reshape(-1)[s["live"]]}
    return kernels.mlp(s["x"], s["norm"], s["gate_up"], s["down"], eps=1e-6, activation=case["act"],
                       out_dtype=torch.float32 if case["out"] == "f32" else BF16)


# ------------------------------------------------------------------------------------------ work and tolerance


def _pairs(n: int, causal: bool, window: int) -> int:
    i = np.arange(n, dtype=np.int64)
    lo = np.maximum(i - (window - 1 if causal else window), 0) if window > 0 else np.zeros(n, np.int64)
    hi = i if causal else (np.minimum(i + window, n - 1) if window > 0 else np.full(n, n - 1))
    return int((hi - lo + 1).sum())


def work(case: dict[str, Any]) -> dict[str, float]:
    kind = case["kind"]
    if kind in ("decide", "forward"):
        c = _config(case)
        lengths = _lengths(case) if kind == "forward" else [len(_record(case, 0).ids)]
        rows = sum(lengths)
        h, d = c.hidden, c.head_dim
        per_layer = h * c.qkv_width + c.heads * d * h + 3 * h * c.intermediate
        flops = 2.0 * rows * per_layer * c.layers
        for i in range(c.layers):
            w = c.window if c.sliding(i) else 0
            flops += 4.0 * c.heads * d * sum(_pairs(n, True, w) for n in lengths)
        # the weights, the tokens' embedding rows and the residual stream out
        return {"bytes": 2.0 * per_layer * c.layers + 2.0 * 2 * rows * h, "flops": flops}
    if kind == "attention":
        e = 2 if case["dtype"] == "bf16" else 4
        b, n, d = case["batch"], case["seq"], case["d"]
        return {"bytes": float(e * b * n * d * (2 * case["hq"] + 2 * case["hkv"])),
                "flops": 4.0 * case["hq"] * d * b * _pairs(n, case["causal"], case["window"])}
    if kind == "encoder":
        b, n, w = case["batch"], case["seq"], case["heads"] * 64
        return {"bytes": 2.0 * b * n * 4 * w, "flops": 4.0 * w * b * _pairs(n, False, case["window"])}
    if kind == "head":
        b, n, q, o = case["batch"], case["seq"], case["fields"], case["opts"]
        h, w, ff = case["hidden"], case["width"], case["ff"]
        rows = b * n * h * w + b * o * 2 * h * w + b * q * 2 * h * w + b * h * w          # projections
        rows += 2 * (b * (2 * o * w * w + 2 * n * w * w + 2 * o * n * w) + 2 * b * o * w * ff)   # evidence layers
        rows += 2 * (b * (4 * q * w * w + 2 * q * q * w) + b * (2 * q * w * w + 2 * n * w * w + 2 * q * n * w)
                     + 2 * b * q * w * ff)                                                # decision layers
        rows += b * o * (4 * w * ff + ff) + 2 * b * q * o * w                             # scorer and routing
        params = 6 * h * w + 2 * (4 * w * w + 2 * w * ff) + 2 * (8 * w * w + 2 * w * ff) + 4 * w * ff
        return {"bytes": 4.0 * (b * n * h + params), "flops": 2.0 * rows}
    rows, d, f = case["rows"], case["d"], case["f"]
    return {"bytes": 2.0 * (3 * d * f + rows * d) + rows * d * (4.0 if case["out"] == "f32" else 2.0),
            "flops": 6.0 * rows * d * f}


def tolerance(case: dict[str, Any]) -> Any:
    # bf16 paths: another summation order moves single roundings of the intermediate bf16 tensors, which travel
    # through what follows. fp32 paths: the summation order of 32-bit sums.
    kind = case["kind"]
    if kind in ("decide", "forward"):
        return {"rel": 1.5e-2}
    if kind == "attention":
        return {"rel": 8e-3} if case["dtype"] == "bf16" else {"rel": 1e-5}
    if kind == "encoder":
        return {"rel": 8e-3}
    if kind == "head":
        return {"rel": 5e-6}
    return {"rel": 5e-3} if case["out"] == "f32" else {"rel": 1e-2}


# ------------------------------------------------------------------------------------------ the same in 64 bits


def _rms(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * (1 + w.double())


def _mm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x @ w.double().t()


def _act(x: torch.Tensor, name: str) -> torch.Tensor:
    return torch.nn.functional.gelu(x, approximate="tanh") if name == "gelu_tanh" else torch.nn.functional.silu(x)


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, *, scale: float, cap: float, window: int, causal: bool,
            keep: torch.Tensor | None = None) -> torch.Tensor:
    """[n, H, D] queries against [m, Hkv, D] keys and values, double, one head and some thousand rows at a time."""
    n, hq, _ = q.shape
    m, hkv, _ = k.shape
    out = torch.empty_like(q)
    j = torch.arange(m, device=q.device)
    step = max(1, (1 << 27) // max(m, 1))
    for r0 in range(0, n, step):
        i = torch.arange(r0, min(n, r0 + step), device=q.device)[:, None]
        if causal:
            hide = (j > i) | ((j <= i - window) if window > 0 else torch.zeros_like(j, dtype=torch.bool))
        else:
            hide = ((j - i).abs() > window) if window > 0 else torch.zeros((i.shape[0], m), dtype=torch.bool, device=q.device)
        if keep is not None:
            hide = hide | ~keep
        for h in range(hq):
            g = h * hkv // hq
            t = q[r0:r0 + step, h] @ k[:, g].t() * scale
            if cap > 0:
                t = cap * torch.tanh(t / cap)
            t = t.masked_fill(hide, -1e30)
            out[r0:r0 + step, h] = torch.softmax(t, -1) @ v[:, g]
    return out


def _exact_forward(c: gemma.GemmaConfig, t: dict[str, torch.Tensor], ids: list, options: list) -> dict[str, Any]:
    lengths = [len(r) for r in ids]
    rows, d = sum(lengths), c.head_dim
    starts = np.concatenate([[0], np.cumsum(lengths)[:-1]]).tolist()
    flat = torch.as_tensor(np.concatenate([np.asarray(r) for r in ids])).to(DEV)
    pos = torch.cat([torch.arange(n, device=DEV) for n in lengths]).double()
    freq = pos[:, None] * c.rope_theta ** (-torch.arange(0, d, 2, device=DEV).double() / d)
    # the model holds its rotary tables and the embedding scale in bf16
    cos, sin = (f(freq).to(BF16).double()[:, None, :] for f in (torch.cos, torch.sin))
    scale = float(torch.tensor(math.sqrt(c.hidden)).to(BF16))

    def rope(x: torch.Tensor) -> torch.Tensor:
        a, b = x[..., :d // 2], x[..., d // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    x = t["embed"][flat].double() * scale
    for i in range(c.layers):
        p = {k.split(".", 2)[2]: v for k, v in t.items() if k.startswith(f"layers.{i}.")}
        h = _rms(x, p["input_norm"], c.eps)
        q = rope(_mm(h, p["q"]).view(rows, c.heads, d))
        k = rope(_mm(h, p["k"]).view(rows, c.kv_heads, d))
        v = _mm(h, p["v"]).view(rows, c.kv_heads, d)
        att = torch.cat([_attend(q[s:s + n], k[s:s + n], v[s:s + n], scale=c.query_pre_attn_scalar ** -0.5,
                                 cap=c.attn_softcap, window=c.window if i % 2 == 0 else 0, causal=True)
                         for s, n in zip(starts, lengths)])
        del q, k, v
        x = x + _rms(_mm(att.view(rows, -1), p["o"]), p["post_attn_norm"], c.eps)
        h = _rms(x, p["pre_ffn_norm"], c.eps)
        y = torch.empty_like(x)
        for r0 in range(0, rows, 16384):
            a = _act(_mm(h[r0:r0 + 16384], p["gate"]), c.activation) * _mm(h[r0:r0 + 16384], p["up"])
            y[r0:r0 + 16384] = _mm(a, p["down"])
        x = x + _rms(y, p["post_ffn_norm"], c.eps)
    where = torch.tensor([s + p for s, qs in zip(starts, options) for q in qs for p, _ in q], device=DEV)
    label = torch.tensor([t_ for qs in options for q in qs for _, t_ in q], device=DEV)
    z = (_rms(x[where], t["final_norm"], c.eps) * t["embed"][label].double()).sum(-1)
    z = c.final_softcap * torch.tanh(z / c.final_softcap)
    counts = [len(q) for qs in options for q in qs]
    probs = torch.cat([torch.softmax(part, 0) for part in z.split(counts)])
    return {"logits": z, "probs": probs, "hidden": x}


def _exact_head(case: dict[str, Any], s: dict[str, Any]) -> torch.Tensor:
    p = {k: v.double() for k, v in s["params"].items()}
    a = {k: torch.as_tensor(v).to(DEV) for k, v in s["arrays"].items()}
    heads, w = case["heads"], case["width"]
    owner = a["option_field"].long()

    def norm(x: torch.Tensor, n: str) -> torch.Tensor:
        return torch.nn.functional.layer_norm(x, x.shape[-1:], p[n + ".weight"], p[n + ".bias"], 1e-5)

    def dense(x: torch.Tensor, n: str) -> torch.Tensor:
        y = x @ p[n + ".weight"].t()
        return y + p[n + ".bias"] if n + ".bias" in p else y

    def means(x: torch.Tensor, spans: torch.Tensor) -> torch.Tensor:
        total = torch.cat([torch.zeros_like(x[:, :1]), x.cumsum(1)], 1)
        lo, hi = (spans[..., j].long() for j in (0, 1))
        pick = lambda i: total.gather(1, i[..., None].expand(*i.shape, x.shape[-1]))  # noqa: E731
        return (pick(hi) - pick(lo)) / (hi - lo).clamp(min=1)[..., None]

    def own(x: torch.Tensor) -> torch.Tensor:
        return x.gather(1, owner[..., None].expand(*owner.shape, x.shape[-1]))

    def mha(x: torch.Tensor, memory: torch.Tensor, keep: torch.Tensor, n: str) -> torch.Tensor:
        wq, wk, wv = p[n + ".in_proj_weight"].chunk(3)
        bq, bk, bv = p[n + ".in_proj_bias"].chunk(3)
        q, k, v = ((y @ m.t() + c).unflatten(-1, (heads, w // heads))
                   for y, m, c in ((x, wq, bq), (memory, wk, bk), (memory, wv, bv)))
        out = torch.stack([_attend(q[i], k[i], v[i], scale=(w // heads) ** -0.5, cap=0.0, window=0, causal=False,
                                   keep=keep[i]) for i in range(x.shape[0])])
        return dense(out.flatten(-2), n + ".out_proj")

    gelu = torch.nn.functional.gelu
    emb = s["embedding"].double()[a["lexical_ids"].long()]
    lexical = means(emb, a["lexical_spans"])
    h = norm(s["hidden"].double(), "hidden_norm")
    memory = dense(h, "memory_projection")
    last = a["mask"].sum(-1) - 1
    glob = h[torch.arange(h.shape[0], device=DEV), last]
    questions, contexts = means(h, a["question_spans"]), means(h, a["option_spans"])
    opts = dense(contexts, "option_context_projection") + dense(lexical, "option_lexical_projection")
    opts = opts + own(dense(questions, "option_question_projection"))
    for i in range(2):
        n = f"evidence_layers.{i}"
        opts = opts + mha(norm(opts, n + ".query_norm"), norm(memory, n + ".memory_norm"), a["mask"], n + ".attention")
        opts = opts + dense(gelu(dense(norm(opts, n + ".feedforward_norm"), n + ".feedforward.0")), n + ".feedforward.3")
    base = dense(questions, "question_projection")
    z = base @ opts.transpose(1, 2) / math.sqrt(w)
    owns = (owner[:, None, :] == torch.arange(base.shape[1], device=DEV)[None, :, None]) & a["option_mask"][:, None, :]
    summary = torch.softmax(z.masked_fill(~owns, -1e30), -1) @ opts
    fields = base + norm(summary, "option_summary_norm") + dense(glob, "global_projection")[:, None]
    fields = fields + p["type_embedding.weight"][a["types"].long()]
    for i in range(2):
        n = f"layers.{i}"
        x = norm(fields, n + ".norm1")
        fields = fields + mha(x, x, a["question_mask"], n + ".self_attn")
        fields = fields + mha(norm(fields, n + ".norm2"), memory, a["mask"], n + ".multihead_attn")
        fields = fields + dense(gelu(dense(norm(fields, n + ".norm3"), n + ".linear1")), n + ".linear2")
    f, o = own(norm(fields, "field_norm")), norm(opts, "option_norm")
    unit = torch.nn.functional.normalize
    prior = (unit(lexical, dim=-1) * unit(own(questions) + glob[:, None], dim=-1)).sum(-1)
    prior = prior * math.exp(min(float(p["prior_logit_scale"]), math.log(100.0)))
    cosine = (unit(f, dim=-1, eps=1e-8) * unit(o, dim=-1, eps=1e-8)).sum(-1)
    residual = dense(gelu(dense(torch.cat([f, o, f * o, (f - o).abs()], -1), "residual_scorer.0")), "residual_scorer.3")
    joint = math.exp(min(float(p["joint_logit_scale"]), math.log(100.0))) * cosine + residual[..., 0]
    return (prior + torch.sigmoid(p["residual_gate"]) * joint).masked_fill(~a["option_mask"], -1e9)


def exact(case: dict[str, Any], seed: int) -> Any:
    kind = case["kind"]
    if kind in ("decide", "forward"):
        c = _config(case)
        t = _tensors(c, _gen(seed))
        if kind == "forward":
            return _exact_forward(c, t, *_requests(case, seed))
        rec = _record(case, seed)
        got = _exact_forward(c, t, [list(rec.ids)], [[f.readout() for f in rec.fields]])
        return got["logits"], got["probs"]
    s = prepare(case, seed)
    if kind == "attention":
        return torch.stack([_attend(s["q"][i].double(), s["k"][i].double(), s["v"][i].double(), scale=case["d"] ** -0.5,
                                    cap=case["cap"], window=case["window"], causal=case["causal"], keep=s["mask"][i])
                            for i in range(case["batch"])])
    if kind == "encoder":
        b, n, w = case["batch"], case["seq"], case["heads"] * 64
        q, k, v = (x.double().unflatten(-1, (case["heads"], 64)) for x in s["qkv"].split(w, -1))
        out = torch.stack([_attend(q[i], k[i], v[i], scale=0.125, cap=0.0, window=case["window"], causal=False,
                                   keep=s["mask"][i]) for i in range(b)])
        return out.reshape(b, n, w)
    if kind == "head":
        logits = _exact_head(case, s)
        return {"logits": logits, "live": logits.reshape(-1)[s["live"]]}
    h = _rms(s["x"].double(), s["norm"], 1e-6)
    return _mm(_act(_mm(h, s["gate"]), case["act"]) * _mm(h, s["up"]), s["down"])
