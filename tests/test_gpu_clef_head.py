"""The Clef joint head on the GPU (deciax_amd/clef_head.py + csrc/head.hip).

Truth is the reference's own golden vectors (tests/golden/clef_head.npz =
tests/fixtures/clef_head.npz, Cloudflare's torch head), checked as tests/clef/test_head.py:11-29
checks the reference: the expected logits at atol 3e-6 / rtol 3e-5 and no leakage from padded
positions. Larger random shapes, with ragged spans and odd sizes, are checked against the oracle
(oracle/clef_head.py, itself pinned to the fixture)."""

from __future__ import annotations

import numpy as np
import pytest

from tests.conftest import rng, say
from tests.test_oracle_clef_head import load_fixture

pytestmark = pytest.mark.gpu


def _dev_params(params: dict) -> dict:
    import torch

    return {k: torch.as_tensor(np.ascontiguousarray(v, np.float32)).cuda() for k, v in params.items()}


def test_head_matches_reference_golden_vectors() -> None:
    import torch

    from deciax_amd import clef_head

    say("clef head: reference fixture")
    params, arrays, hidden, embedding, expected = load_fixture()
    p = _dev_params(params)
    lexical = clef_head.lexical_vectors(torch.as_tensor(embedding).cuda(), arrays["lexical_ids"],
                                        arrays["lexical_spans"])
    out = clef_head.forward(p, hidden, lexical, arrays, heads=4, routing_layers=2, layers=2).cpu().numpy()
    for i, e in expected.items():
        np.testing.assert_allclose(out[i, :len(e)], e, atol=3e-6, rtol=3e-5)
        assert (out[i, len(e):] == np.float32(-1e9)).all()
    changed = np.where(arrays["mask"][..., None], hidden, np.float32(10000.0))
    second = clef_head.forward(p, changed, lexical, arrays, heads=4, routing_layers=2, layers=2).cpu().numpy()
    np.testing.assert_allclose(out[:3], second[:3], atol=1e-6)


def _random_case(seed: int, batch: int, seq: int, hidden: int, width: int, ff: int, nq: int, no: int, ntypes: int,
                 routing_layers: int, layers: int):
    r = rng(seed)
    f = lambda *s, scale=0.2: (r.normal(size=s) * scale).astype(np.float32)  # noqa: E731
    p = {"hidden_norm.weight": 1 + f(hidden), "hidden_norm.bias": f(hidden),
         "memory_projection.weight": f(width, hidden), "memory_projection.bias": f(width),
         "option_context_projection.weight": f(width, hidden), "option_lexical_projection.weight": f(width, hidden),
         "option_question_projection.weight": f(width, hidden), "question_projection.weight": f(width, hidden),
         "question_projection.bias": f(width), "option_summary_norm.weight": 1 + f(width),
         "option_summary_norm.bias": f(width), "global_projection.weight": f(width, hidden),
         "type_embedding.weight": f(ntypes, width), "field_norm.weight": 1 + f(width), "field_norm.bias": f(width),
         "option_norm.weight": 1 + f(width), "option_norm.bias": f(width),
         "residual_scorer.0.weight": f(ff, 4 * width), "residual_scorer.0.bias": f(ff),
         "residual_scorer.3.weight": f(1, ff), "residual_scorer.3.bias": f(1),
         "prior_logit_scale": np.float32(2.0), "joint_logit_scale": np.float32(5.0),
         "residual_gate": np.float32(0.3)}

    def attn(n):
        p.update({n + ".in_proj_weight": f(3 * width, width), n + ".in_proj_bias": f(3 * width),
                  n + ".out_proj.weight": f(width, width), n + ".out_proj.bias": f(width)})

    def ln(n):
        p.update({n + ".weight": 1 + f(width), n + ".bias": f(width)})

    for i in range(routing_layers):
        n = f"evidence_layers.{i}"
        attn(n + ".attention")
        for m in ("query_norm", "memory_norm", "feedforward_norm"):
            ln(f"{n}.{m}")
        p.update({n + ".feedforward.0.weight": f(ff, width), n + ".feedforward.0.bias": f(ff),
                  n + ".feedforward.3.weight": f(width, ff), n + ".feedforward.3.bias": f(width)})
    for i in range(layers):
        n = f"layers.{i}"
        attn(n + ".self_attn")
        attn(n + ".multihead_attn")
        for m in ("norm1", "norm2", "norm3"):
            ln(f"{n}.{m}")
        p.update({n + ".linear1.weight": f(ff, width), n + ".linear1.bias": f(ff),
                  n + ".linear2.weight": f(width, ff), n + ".linear2.bias": f(width)})
    lens = r.integers(seq // 2, seq + 1, batch)
    mask = np.arange(seq)[None, :] < lens[:, None]
    a = {"mask": mask, "question_spans": np.zeros((batch, nq, 2), np.int32),
         "option_spans": np.zeros((batch, no, 2), np.int32), "option_field": np.zeros((batch, no), np.int32),
         "option_mask": np.zeros((batch, no), bool), "question_mask": np.zeros((batch, nq), bool),
         "types": r.integers(0, ntypes, (batch, nq)).astype(np.int32)}
    for b in range(batch):
        q_here = int(r.integers(1, nq + 1))
        a["question_mask"][b, :q_here] = True
        for q in range(q_here):
            s0 = int(r.integers(0, lens[b] - 4))
            a["question_spans"][b, q] = (s0, s0 + int(r.integers(1, 4)))
        o_here = int(r.integers(q_here, no + 1))
        a["option_mask"][b, :o_here] = True
        a["option_field"][b, :o_here] = np.sort(r.integers(0, q_here, o_here))
        a["option_field"][b, :q_here] = np.arange(q_here)  # every field owns an option
        for o in range(o_here):
            s0 = int(r.integers(0, lens[b] - 4))
            a["option_spans"][b, o] = (s0, s0 + int(r.integers(0, 4)))  # empty spans included
    hidden_x = f(batch, seq, hidden, scale=1.0)
    lexical = f(batch, no, hidden, scale=1.0)
    return p, a, hidden_x, lexical


@pytest.mark.parametrize("shape", [
    dict(batch=2, seq=300, hidden=64, width=32, ff=48, nq=5, no=17, ntypes=3, routing_layers=2, layers=2),
    dict(batch=3, seq=131, hidden=96, width=48, ff=80, nq=7, no=70, ntypes=4, routing_layers=1, layers=3),
])
def test_head_matches_oracle_random_shapes(shape: dict) -> None:
    from deciax_amd import clef_head
    from oracle import clef_head as oc

    say(f"clef head random {shape}")
    heads = 4
    p, a, hidden, lexical = _random_case(7 + shape["batch"], **shape)
    want = oc.forward(p, hidden, lexical, a, heads=heads, routing_layers=shape["routing_layers"],
                      layers=shape["layers"])
    got = clef_head.forward(_dev_params(p), hidden, lexical, a, heads=heads, routing_layers=shape["routing_layers"],
                            layers=shape["layers"]).cpu().numpy()
    live = a["option_mask"]
    np.testing.assert_allclose(got[live], want[live], atol=2e-5, rtol=2e-4)
    assert (got[~live] == np.float32(-1e9)).all()


def test_encoded_requests_through_head() -> None:
    """Requests encoded by deciax_amd.schema, laid out by `head_inputs` (the reference's collate,
    src/deciax/models/clef/input.py:140-182), with lexical vectors gathered on the GPU: the head's
    logits match the oracle fed the same arrays, and decode to the same answers."""
    import torch

    from deciax_amd import clef_head
    from deciax_amd.schema import ByteTokenizer, decode, encode, head_inputs
    from oracle import clef_head as oc

    say("clef head: encoded requests")
    tok = ByteTokenizer()
    questions = {"mood": {"type": "choice", "criteria": {"pos": "positive", "neg": "negative", "mix": None}},
                 "late": {"type": "noul"}, "stars": {"type": "score", "criteria": ["bad", "ok", "good"]}}
    records = [encode(tok, s, questions, 2048) for s in ("the parcel came late", {"ticket": 7, "text": "great"})]
    a = head_inputs(records, tok.pad_token_id)
    r = rng(11)
    batch, seq = a["input_ids"].shape
    hidden_dim = 64
    p, _, _, _ = _random_case(5, batch=batch, seq=seq, hidden=hidden_dim, width=32, ff=48, nq=3, no=8, ntypes=3,
                              routing_layers=1, layers=2)
    hidden = r.normal(size=(batch, seq, hidden_dim)).astype(np.float32)
    embedding = r.normal(size=(tok.vocab, hidden_dim)).astype(np.float32)
    lexical = clef_head.lexical_vectors(torch.as_tensor(embedding).cuda(), a["lexical_ids"], a["lexical_spans"])
    want_lex = oc.means(embedding[a["lexical_ids"]], a["lexical_spans"])
    np.testing.assert_allclose(lexical.cpu().numpy(), want_lex, atol=1e-5, rtol=1e-5)
    got = clef_head.forward(_dev_params(p), hidden, lexical, a, heads=4, routing_layers=1, layers=2).cpu().numpy()
    want = oc.forward(p, hidden, want_lex, a, heads=4, routing_layers=1, layers=2)
    live = a["option_mask"]
    np.testing.assert_allclose(got[live], want[live], atol=2e-5, rtol=2e-4)
    for i, record in enumerate(records):
        n = int(live[i].sum())
        ours, theirs = decode(record, got[i, :n], questions, "m"), decode(record, want[i, :n], questions, "m")
        assert ours["answers"]["mood"]["choice"] == theirs["answers"]["mood"]["choice"]
        assert ours["answers"]["late"]["noul"] == pytest.approx(theirs["answers"]["late"]["noul"], abs=2e-4)
        assert ours["answers"]["stars"]["score"] == pytest.approx(theirs["answers"]["stars"]["score"], abs=2e-4)


@pytest.mark.parametrize("m,n,k,pad", [
    (1, 1, 1, 0), (3, 17, 31, 0), (17, 1000, 1029, 3), (200, 1030, 95, 1), (513, 515, 100, 1),  # fp32 products, 32 x 32
    (601, 2047, 70, 0), (4097, 1025, 130, 4), (20000, 200, 36, 0),                              # and 64 x 32, 64 x 64 tiles
    (16, 16, 64, 0), (300, 1000, 96, 0),                                                        # split products
])
def test_linear_f32_tiles(m: int, n: int, k: int, pad: int) -> None:
    """Every tile shape at its edges, rows with and without 16-byte alignment, bias, GELU and accumulation, against
    the product in 64 bits. A sum of k fp32 products in any order is within k 2^-24 sum |x w| of it."""
    import torch

    from deciax_amd import kernels as K

    say(f"linear_f32 {m} x {n} x {k}, row padding {pad}")
    r = rng(m + n + k)
    x = torch.as_tensor(r.normal(size=(m, k + pad)).astype(np.float32)).cuda()[:, :k]
    w = torch.as_tensor(r.normal(size=(n, k + pad)).astype(np.float32)).cuda()[:, :k]
    b = torch.as_tensor(r.normal(size=n).astype(np.float32)).cuda()
    want = x.double() @ w.double().t()
    bound = (k + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs()) + 1e-30
    assert ((K.linear_f32(x, w).double() - want).abs() <= bound).all()
    base = torch.as_tensor(r.normal(size=(m, n)).astype(np.float32)).cuda()
    got = K.linear_f32(x, w, b, gelu=True, out=base.clone(), accumulate=True).double()
    act = torch.nn.functional.gelu(want + b.double())
    # GELU has slope at most 1.13; erff and the three roundings after it add a few ulp of the result
    assert ((got - base.double() - act).abs() <= 1.2 * bound + 2.0 ** -21 * (act.abs() + base.double().abs()) + 1e-6).all()


@pytest.mark.parametrize("m,n,k,pad,scale", [
    (1300, 2000, 100, 4, 1.0), (4097, 1025, 132, 0, 1.0), (1281, 2050, 64, 8, 1e-30),   # 128 x 64 tiles
    (4097, 2050, 100, 4, 1.0), (8200, 1025, 264, 0, 1.0),                               # 128 x 128 tiles
    (600, 2048, 68, 0, 1.0), (577, 2049, 80, 4, 1e30), (641, 2047, 1028, 0, 1.0),       # 32 x 32 tiles
    (1, 1, 64, 0, 1.0), (33, 31, 260, 4, 1.0), (65, 70, 2052, 0, 1.0), (5, 40, 6000, 8, 1.0),
])
def test_linear_f32_split_tiles(m: int, n: int, k: int, pad: int, scale: float) -> None:
    """The three-bf16 products at the edges of their tiles and of a 16-wide step, with bias, GELU and accumulation and
    rows that hold NaN past k, against 64 bits. The six products leave out up to 2^-24 |x w|, and the two accumulators
    take k / 16 and 5 k / 16 roundings, the second of terms 2^-8 the size: within the bound (k + 2) 2^-24 sum |x w| of an
    fp32 sum, and its 2-norm within that of torch's fp32 product."""
    import torch

    from deciax_amd import kernels as K

    say(f"linear_f32 split {m} x {n} x {k}, row padding {pad}, scale {scale}")
    r = rng(m + n + k)
    x = torch.as_tensor((r.normal(size=(m, k + pad)) * scale).astype(np.float32)).cuda()
    w = torch.as_tensor(r.normal(size=(n, k + pad)).astype(np.float32)).cuda()
    x[:, k:] = w[:, k:] = float("nan")
    x, w = x[:, :k], w[:, :k]
    b = torch.as_tensor((r.normal(size=n) * scale).astype(np.float32)).cuda()
    want = x.double() @ w.double().t()
    bound = (k + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs()) + 1e-38
    got = K.linear_f32(x, w).double()
    assert ((got - want).abs() <= bound).all()
    assert (got - want).norm() <= ((x @ w.t()).double() - want).norm()
    if scale != 1.0:
        return
    base = torch.as_tensor(r.normal(size=(m, n)).astype(np.float32)).cuda()
    got = K.linear_f32(x, w, b, gelu=True, out=base.clone(), accumulate=True).double()
    act = torch.nn.functional.gelu(want + b.double())
    assert ((got - base.double() - act).abs() <= 1.2 * bound + 2.0 ** -21 * (act.abs() + base.double().abs()) + 1e-6).all()


@pytest.mark.parametrize("m", [20, 600, 4100])
@pytest.mark.parametrize("scale", [1e-33, 1e-35, 1e-37])
def test_linear_f32_split_tiny_rows(m: int, scale: float) -> None:
    """Rows below the range in which three bf16 hold an fp32 number keep an fp32 sum's bound (k 2^-24 sum |x w|, a
    denormal's half unit per product), in every tile, beside rows of ordinary size and of zeros."""
    import torch

    from deciax_amd import kernels as K

    say(f"linear_f32 split, {m} rows, every other scaled by {scale}")
    r = rng(m)
    n, k = 1000, 260
    x = torch.as_tensor(r.normal(size=(m, k)).astype(np.float32)).cuda()
    w = torch.as_tensor(r.normal(size=(n, k)).astype(np.float32)).cuda()
    x[::2] *= scale
    x[5] = 0
    want = x.double() @ w.double().t()
    bound = (k + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + k * 2.0 ** -150
    got = K.linear_f32(x, w).double()
    assert ((got - want).abs() <= bound).all() and (got[5] == 0).all()
    ordinary = K.linear_f32(x[1::2].contiguous(), w).double()
    assert torch.equal(got[1::2], ordinary)


def test_linear_f32_split_not_finite() -> None:
    """Infinities, NaN and values past the largest bf16 give what fp32 products give."""
    import torch

    from deciax_amd import kernels as K

    say("linear_f32 split, values that are not finite")
    r = rng(5)
    m, n, k = 1300, 2000, 100
    x = torch.as_tensor(r.normal(size=(m, k)).astype(np.float32)).cuda()
    w = torch.as_tensor((r.normal(size=(n, k)) * 1e-3).astype(np.float32)).cuda()
    x[3, 5], x[700, 99], x[1299, 0], w[17, 50], w[1999, 3] = np.inf, -np.inf, np.nan, np.inf, np.nan
    x[40, 7] = x[1290, 64] = 3.395e38  # rounds to infinity in bf16
    want = x.double() @ w.double().t()
    got = K.linear_f32(x, w).double()
    torch.testing.assert_close(got.isnan(), want.isnan())
    torch.testing.assert_close(got.isinf(), want.isinf())
    live = want.isfinite()
    bound = (k + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert ((got - want).abs() <= bound)[live].all() and (got.sign() == want.sign())[want.isinf()].all()


@pytest.mark.parametrize("batch,rows,seq,n,d", [(1, 1, 1, 1, 1), (2, 50, 31, 7, 257), (3, 1000, 40, 20, 512)])
def test_span_means_gather_f32(batch: int, rows: int, seq: int, n: int, d: int) -> None:
    """Bit for bit the means of the gathered rows: empty and clipped spans, indices outside the table (clamped), rows
    in blocks of eight and the rest."""
    import torch

    from deciax_amd import kernels as K

    say(f"span_means_gather {batch} x {seq} of {rows} rows, {n} spans, width {d}")
    r = rng(rows + d)
    table = torch.as_tensor(r.normal(size=(rows, d)).astype(np.float32)).cuda()
    ids = torch.as_tensor(r.integers(-2, rows + 2, (batch, seq)).astype(np.int32)).cuda()
    lo = r.integers(-1, seq + 1, (batch, n))
    spans = torch.as_tensor(np.stack([lo, lo + r.integers(-1, 19, (batch, n))], -1).astype(np.int32)).cuda()
    copied = K.gather_rows_f32(table, ids.reshape(1, batch * seq), batch=1)
    got = K.span_means_gather_f32(table, ids, spans)
    assert torch.equal(got, K.span_means_f32(copied, spans, batch=batch))


def test_head_combine_scaled_f32() -> None:
    """The learned scalars on the device against the host's doubles, rounded once: capped and uncapped scales, both
    signs of the gate. Three products and two sums of fp32: 4 2^-24 of the terms' size."""
    import math

    import torch

    from deciax_amd import kernels as K

    say("head_combine_scaled")
    r = rng(3)
    n = 300
    prior, cosine, residual = (torch.as_tensor(r.normal(size=n).astype(np.float32)).cuda() for _ in range(3))
    mask = torch.as_tensor((r.random(n) < 0.8).astype(np.uint8)).cuda()
    for a, b, g in ((2.0, 2.5, 0.3), (4.605170, 7.0, -3.0), (80.0, -2.0, 40.0)):
        ps, js = (np.float32(math.exp(min(float(np.float32(v)), math.log(100.0)))) for v in (a, b))
        gate = np.float32(1.0 / (1.0 + math.exp(-float(np.float32(g)))))
        t = [torch.tensor(v, device="cuda") for v in (a, b, g)]
        got = K.head_combine_scaled_f32(prior, cosine, residual, mask, prior_logit_scale=t[0], joint_logit_scale=t[1],
                                        residual_gate=t[2]).double().cpu().numpy()
        p, c, x = (v.double().cpu().numpy() for v in (prior, cosine, residual))
        want = float(ps) * p + float(gate) * (float(js) * c + x)
        size = float(ps) * abs(p) + float(gate) * (float(js) * abs(c) + abs(x))
        live = mask.cpu().numpy().astype(bool)
        assert (abs(got - want) <= 4 * 2.0 ** -24 * size)[live].all() and (got[~live] == -1e9).all()


@pytest.mark.parametrize("kind", ["python", "host64", "device64", "device32", "device16"])
def test_head_scalars_keep_their_precision(kind: str, monkeypatch: pytest.MonkeyPatch) -> None:
    """Learned scalars in 64 bits are exponentiated in 64 bits wherever they are; those of fewer bits on the device are
    not read back. The two ways of combining agree to the roundings of their products and sums."""
    import math

    import torch

    from deciax_amd import clef_head
    from deciax_amd import kernels as K

    say(f"clef head, learned scalars: {kind}")
    p, a, hidden, lexical = _random_case(4, batch=2, seq=90, hidden=64, width=32, ff=48, nq=3, no=9, ntypes=3,
                                         routing_layers=1, layers=1)
    values = {"prior_logit_scale": 2.1, "joint_logit_scale": 4.3, "residual_gate": 0.7}  # none of them an fp32 number
    make = {"python": float, "host64": lambda v: torch.tensor(v, dtype=torch.float64),
            "device64": lambda v: torch.tensor(v, dtype=torch.float64, device="cuda"),
            "device32": lambda v: torch.tensor(v, device="cuda"),
            "device16": lambda v: torch.tensor(v, dtype=torch.bfloat16, device="cuda")}[kind]
    params = _dev_params(p)
    seen = {}
    features, combine = K.head_features_f32, K.head_combine_f32
    monkeypatch.setattr(K, "head_features_f32",
                        lambda *t, prior_scale, **kw: (seen.update(prior=prior_scale), features(*t, prior_scale=prior_scale, **kw))[1])
    monkeypatch.setattr(K, "head_combine_f32", lambda *t, **kw: (seen.update(kw), combine(*t, **kw))[1])
    got = clef_head.forward(params | {n: make(v) for n, v in values.items()}, hidden, lexical, a, heads=4, routing_layers=1,
                            layers=1)
    if kind.startswith("device") and kind != "device64":
        assert seen == {"prior": 1.0}
    else:
        assert seen == {"prior": math.exp(2.1), "joint_scale": math.exp(4.3), "gate": 1.0 / (1.0 + math.exp(-0.7))}
    if kind != "device16":
        want = clef_head.forward(params | {n: torch.tensor(v, device="cuda") for n, v in values.items()}, hidden, lexical, a,
                                 heads=4, routing_layers=1, layers=1)
        live = torch.as_tensor(a["option_mask"]).cuda()
        # scales of up to e^4.3 from scalars 2^-24 apart, times values of order one, and the roundings after them
        assert (got - want)[live].abs().max() <= 16 * 2.0 ** -24 * 4.3 * math.exp(4.3)
        assert torch.equal(got[~live], want[~live])


@pytest.mark.parametrize("batch,nq,nk,heads,dh", [
    (1, 1, 1, 1, 16), (2, 17, 65, 3, 32), (1, 6, 600, 16, 64), (2, 33, 130, 2, 48), (1, 5, 70, 2, 80), (1, 40, 64, 2, 96),
    (2, 20, 31, 2, 112), (1, 50, 515, 4, 128), (8, 40, 127, 40, 64), (1, 9, 40, 2, 24),
])
def test_mha_f32_forms(batch: int, nq: int, nk: int, heads: int, dh: int) -> None:
    """Matrix-core head dims, both workgroup forms and the general kernel (dh 24) against the masked softmax in 64
    bits, with holes in the mask and one batch row that keeps no key (the uniform average)."""
    import torch

    from deciax_amd import kernels as K

    say(f"mha_f32 {batch} x {nq} x {nk}, {heads} heads x {dh}")
    r = rng(nq + nk + dh)
    w = heads * dh
    q, k, v = (torch.as_tensor(r.normal(size=(batch * t, w)).astype(np.float32)).cuda() for t in (nq, nk, nk))
    mask = torch.as_tensor(r.random((batch, nk)) < 0.7).to(torch.uint8).cuda()
    mask[:, 0] = 1
    if batch > 1:
        mask[-1] = 0
    got = K.mha_f32(q, k, v, mask, batch=batch, heads=heads).double()
    split = lambda t: t.double().view(batch, -1, heads, dh).transpose(1, 2)  # noqa: E731
    s = split(q) @ split(k).transpose(-1, -2) / dh ** 0.5
    p = torch.softmax(s.masked_fill(~mask.bool()[:, None, None, :], -1e30), -1)
    want = (p @ split(v)).transpose(1, 2).reshape(batch * nq, w)
    # scores of dh products: relative 2^-24 (dh + 4) of sum |q k|, a few units; the weights inherit it
    err = (got - want).abs().max().item()
    assert err < 4 * 2.0 ** -24 * (dh + 16) * float((split(q).abs() @ split(k).abs().transpose(-1, -2)).max()) / dh ** 0.5, err


@pytest.mark.parametrize("nq,dh", [(3, 16), (40, 64), (5, 128), (700, 64)])
@pytest.mark.parametrize("nk", [1, 65, 127])
def test_mha_f32_infinite_last_value(nq: int, dh: int, nk: int) -> None:
    """An infinite value of the last key comes out infinite, in both workgroup forms: keys past the last add nothing."""
    import torch

    from deciax_amd import kernels as K

    say(f"mha_f32, infinite last value, {nq} x {nk} x {dh}")
    r = rng(nq + nk + dh)
    heads = 16
    q, k, v = (torch.as_tensor(r.normal(size=(t, heads * dh)).astype(np.float32)).cuda() for t in (nq, nk, nk))
    mask = torch.ones((1, nk), dtype=torch.uint8, device="cuda")
    want = K.mha_f32(q, k, v, mask, batch=1, heads=heads)
    v[nk - 1, 5], v[nk - 1, heads * dh - 1] = np.inf, -np.inf
    got = K.mha_f32(q, k, v, mask, batch=1, heads=heads)
    want[:, 5], want[:, -1] = np.inf, -np.inf
    assert torch.equal(got, want)


@pytest.mark.parametrize("heads,dh", [(16, 32), (16, 64), (8, 80), (8, 128)])
def test_mha_f32_rows_do_not_depend_on_the_launch(heads: int, dh: int) -> None:
    """A batch row alone and among eight, with its own keys and padded by masked ones: the same bits, in both workgroup
    forms."""
    import torch

    from deciax_amd import kernels as K

    say(f"mha_f32, one batch row alone and among eight, {heads} heads x {dh}")
    r = rng(heads + dh)
    nq, nk, w, lens = 130, 300, heads * dh, [300, 17, 64, 250, 299, 1, 128, 200]
    q, k, v = (torch.as_tensor(r.normal(size=(8, t, w)).astype(np.float32)).cuda() for t in (nq, nk, nk))
    mask = (torch.arange(nk, device="cuda")[None] < torch.tensor(lens, device="cuda")[:, None]).to(torch.uint8)
    flat = lambda t: t.reshape(-1, w).contiguous()  # noqa: E731
    got = K.mha_f32(flat(q), flat(k), flat(v), mask, batch=8, heads=heads).view(8, nq, w)
    for b, n in enumerate(lens):
        for few in (nq, 5):
            alone = K.mha_f32(flat(q[b, :few]), flat(k[b, :n]), flat(v[b, :n]), mask[b:b + 1, :n].contiguous(), batch=1, heads=heads)
            assert torch.equal(alone, got[b, :few]), f"batch row {b}, {few} queries"


@pytest.mark.parametrize("nq", [3, 600])
def test_mha_f32_weights_keep_fp32_precision(nq: int) -> None:
    """Scores that are exact (multiples of 1/8) from 0 to -70, one-hot values: each weight within 6 units in the last place
    of e^s / sum (a 2-ulp exponential, a sum of 64 positive terms in parts of a few, one quotient, the merge's factor).
    Rounding s log2(e) first would miss by |s| 2^-24: 35 units at -70."""
    import torch

    from deciax_amd import kernels as K

    say(f"mha_f32 weights, {nq} queries")
    heads, dh, nk = 16, 64, 64
    r = rng(nq)
    s = -np.sort(r.integers(0, 560, (nk,)) / 8.0)[::-1]
    s[-1] = 0.0
    q = torch.zeros((nq, heads, dh), device="cuda")
    k = torch.zeros((nk, heads, dh), device="cuda")
    q[:, :, 0] = 8.0
    k[:, :, 0] = torch.as_tensor(s.copy(), dtype=torch.float32, device="cuda")[:, None]
    v = torch.eye(64, device="cuda")[:, None, :].expand(nk, heads, dh)
    mask = torch.ones((1, nk), dtype=torch.uint8, device="cuda")
    got = K.mha_f32(*(t.reshape(-1, heads * dh).contiguous() for t in (q, k, v)), mask, batch=1, heads=heads)
    e = np.exp(s)
    want = torch.as_tensor(e / e.sum(), device="cuda")
    rel = ((got.view(nq, heads, dh).double() - want) / want).abs()
    assert rel.max() < 6 * 2.0 ** -23, float(rel.max())


@pytest.mark.parametrize("n,k,pad", [(1024, 1024, 0), (2047, 4096, 4), (1, 2048, 0), (96, 100, 0), (1030, 257, 0), (70, 63, 1)])
def test_linear_f32_rows_do_not_depend_on_m(n: int, k: int, pad: int) -> None:
    """A row has the same bits in every launch that holds it, whichever tiles its size takes: split products (rows of
    whole 16-byte chunks) and fp32 ones, with bias, GELU and accumulation. Values of other rows that are not finite change
    nothing either."""
    import torch

    from deciax_amd import kernels as K

    say(f"linear_f32 rows, {n} x {k}, row padding {pad}")
    r = rng(n + k)
    big = 9000
    x = torch.as_tensor(r.normal(size=(big, k + pad)).astype(np.float32)).cuda()[:, :k]
    w = torch.as_tensor(r.normal(size=(n, k + pad)).astype(np.float32)).cuda()[:, :k]
    b = torch.as_tensor(r.normal(size=n).astype(np.float32)).cuda()
    base = torch.as_tensor(r.normal(size=(big, n)).astype(np.float32)).cuda()
    run = lambda rows, xx=x: K.linear_f32(xx[rows], w, b, gelu=True, out=base[rows].clone(), accumulate=True)  # noqa: E731
    want = run(slice(0, big))
    for m in (1, 5, 33, 130, 600, 1300, 2100, 4200, 6500):
        assert torch.equal(run(slice(0, m)), want[:m]), f"first {m} rows"
        assert torch.equal(run(slice(big - m, big)), want[big - m:]), f"last {m} rows"
    dirty = x.clone()
    dirty[1::64, 0], dirty[2::64, k - 1], dirty[3::64, k // 2] = np.nan, np.inf, 3.395e38
    clean = torch.ones(big, dtype=torch.bool, device="cuda")
    for i in (1, 2, 3):
        clean[i::64] = False
    for m in (600, 2100, big):
        assert torch.equal(run(slice(0, m), dirty)[clean[:m]], want[:m][clean[:m]]), f"{m} rows beside others not finite"


def test_head_results_do_not_depend_on_the_batch() -> None:
    """Requests alone and in one padded batch (other lengths, option and field counts): the same logits, bit for bit."""
    import torch

    from deciax_amd import clef_head

    say("joint head, requests alone and in a batch")
    p, a, hidden, lexical = _random_case(3, batch=5, seq=700, hidden=1024, width=512, ff=1024, nq=20, no=90, ntypes=3,
                                         routing_layers=2, layers=2)
    params = {n: v * 0.2 if v.ndim == 2 else v for n, v in _dev_params(p).items()}
    kw = dict(heads=8, routing_layers=2, layers=2)
    want = clef_head.forward(params, hidden, lexical, a, **kw)
    for i in range(5):
        size = {"mask": int(a["mask"][i].sum()), "question": int(a["question_mask"][i].sum()),
                "types": int(a["question_mask"][i].sum()), "option": int(a["option_mask"][i].sum())}
        own = {n: v[i:i + 1, :size[n.split("_")[0]]] for n, v in a.items()}
        got = clef_head.forward(params, hidden[i:i + 1, :size["mask"]], lexical[i:i + 1, :size["option"]], own, **kw)
        assert got.isfinite().all() and torch.equal(got[0], want[i, :size["option"]]), f"request {i}"


@pytest.mark.parametrize("batch,fields", [(70000, 1), (1, 70000)])
def test_head_routing_beyond_a_grid_dimension(batch: int, fields: int) -> None:
    """More batch rows or fields than a launch's y or z dimension holds: a field that owns one option gets that option."""
    import torch

    from deciax_amd import kernels as K

    say(f"head routing, {batch} x {fields} fields")
    g = torch.Generator(device="cuda").manual_seed(1)
    options = torch.empty((batch * 2, 16), device="cuda").normal_(generator=g)
    base = torch.empty((batch * fields, 16), device="cuda").normal_(generator=g)
    owner = torch.tensor([[0, fields]], dtype=torch.int32, device="cuda").repeat(batch, 1)  # the second: no field's
    mask = torch.ones((batch, 2), dtype=torch.uint8, device="cuda")
    got = K.head_routing_f32(options, base, owner, mask, batch=batch)
    assert torch.equal(got[::fields], options[::2])
    if fields > 1:  # the others own none: the mean of all options
        torch.testing.assert_close(got[1:], options.mean(0).expand(fields - 1, 16), rtol=1e-6, atol=1e-6)
