"""The logits-to-token calls whose speed is measured: what a serving engine asks of this library.

Every case is one prepared call (`Context.prepare_sample`, `prepare_step`, `prepare_verify`,
`prepare_top2`, `prepare_logprobs`) launched once on logits that already sit in HBM, as a decode
loop launches it once a step.  The buffers, the row parameters and the sparse penalty entries are
what such a loop holds before the call.  Sizes and distributions are those of the library's five
workloads (lsamp/workloads.py), of its tests, and generic ones between them.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "mlx-swift-lm_amd"))

from lsamp import _ffi, workloads as W  # noqa: E402
from lsamp.api import Context  # noqa: E402

DEVICE = "cuda:0"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
MODES = {"residual": _ffi.VERIFY_RESIDUAL, "exact": _ffi.VERIFY_EXACT,
         "typical": _ffi.VERIFY_TYPICAL}

# What a case leaves unsaid.  `logits`: "flat" N(0, sigma^2); "boosted" the same with 32 tokens
# raised by 8; "peaked" with a Zipf(1.1) log-prior in a random order, as a trained model's head
# gives.  `pad`: rows are views of rows padded to a multiple of 64 tokens.
BASE = dict(semantics="cbv2", dtype="bf16", logits="peaked", sigma=3.0, pad=False,
            temperature=0.8, top_k=0, top_p=1.0, min_p=0.0, mixed=False,
            history=0, repetition=1.0, repetition_window=64, presence=0.0, frequency=0.0,
            mask=False, stats=False, logprobs=-1, mode="", window=0)


def _case(name, op, rows, vocab, **kw):
    return dict(BASE, op=op, rows=rows, vocab=vocab, **({"name": name} if name else {}), **kw)


def listed():
    return [
        # One chat stream, mlx-lm order: float32 logits, repetition penalty over the last 20
        # tokens, temperature and top-p.  Nothing but latency.
        _case("single_top_p", "sample", 1, 151936, semantics="mlxlm", dtype="f32",
              logits="boosted", temperature=0.7, top_p=0.9, history=512, repetition=1.1,
              repetition_window=20),
        # A few greedy streams of a model with a small vocabulary: the smallest call.
        _case("few_greedy", "sample", 4, 32000, temperature=0.0),
        # The ordinary batched decode step: penalties over long histories, joint top-k / top-p /
        # min-p.
        _case("decode_top_k", "sample", 64, 151936, top_k=50, top_p=0.95, min_p=0.05,
              history=2048, presence=0.5, frequency=0.3),
        # Continuous batching at full load, every request with its own parameters: greedy rows,
        # top-k rows and top-p rows side by side, the largest vocabulary.
        _case("mixed_batch", "sample", 256, 262144, logits="flat", sigma=4.0, mixed=True,
              history=4096, repetition=1.3, repetition_window=64),
        # A grammar-constrained batch: float32 logits, one packed token mask per row.
        _case("grammar", "sample", 64, 151936, dtype="f32", logits="flat", temperature=0.6,
              top_p=0.9, history=20, repetition=1.1, repetition_window=20, mask=True),
        # Many float32 rows with top-p alone: an engine that keeps its head in float32.
        _case("batch_f32_top_p", "sample", 128, 151936, dtype="f32", top_p=0.95),
        # float16 rows of an odd vocabulary, so no row but the first starts aligned; min-p alone,
        # with the row statistics that a monitoring engine reads.
        _case("ragged_min_p", "sample", 24, 40003, dtype="f16", temperature=1.0, min_p=0.05,
              stats=True),
        # A decode step whose clients asked for log-probabilities: the draw, the chosen token's
        # and the 20 best tokens' raw log-probability.
        _case("step_logprobs", "step", 64, 151936, top_p=0.95, history=2048, presence=0.5,
              logprobs=20),
        # Speculative decoding, textbook rule: 3 drafts and a bonus position a sequence.
        _case("verify_residual", "verify", 32, 151936, logits="flat", top_p=0.95, window=4,
              mode="residual"),
        # Speculative decoding as the engine's typical acceptance does it, with penalties.
        _case("verify_typical", "verify", 16, 151936, top_p=0.95, window=4, mode="typical",
              history=1024, frequency=0.3),
        # The two best tokens of every row: the speculation policy's margins.
        _case("top_two", "top2", 32, 151936),
        # Scoring a prompt: the log-probability of each of its tokens, and the 5 best beside it.
        _case("score_prompt", "logprobs", 192, 128256, logprobs=5),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["sample", "sample", "sample", "sample", "step", "verify", "top2", "logprobs"])
    vocab = rng.choice([32000, 128256, 151936, 262144, _log_int(rng, 4000, 262144),
                        _log_int(rng, 4000, 262144) | 1])
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    window = rng.randint(2, 5) if op == "verify" else 0
    mode = rng.choice(["residual", "exact", "typical"]) if op == "verify" else ""
    positions = 2 * window - 1 if mode == "residual" else max(1, window)
    # (half of the largest listed call's bytes, a third of its rows)
    most = int(67e6 / (positions * vocab * (4 if dtype == "f32" else 2)))
    rows = _log_int(rng, 1, max(1, min(256, most)))
    c = _case(None, op, rows, vocab, dtype=dtype, window=window, mode=mode,
              logits=rng.choice(["peaked", "flat", "boosted"]), sigma=round(rng.uniform(2, 4), 2),
              pad=op != "verify" and rng.random() < 0.5)
    if op == "top2":
        return c
    if op == "logprobs":
        return dict(c, logprobs=rng.choice([0, 1, 5, 20]))
    c["temperature"] = rng.choice([0.0, 0.6, 0.8, 1.0, round(rng.uniform(0.3, 1.3), 2)])
    kind = rng.choice(["top_k", "top_p", "min_p", "all", "none"])
    if kind in ("top_k", "all"):
        c["top_k"] = _log_int(rng, 1, 200)
    if kind in ("top_p", "all"):
        c["top_p"] = round(rng.uniform(0.7, 0.99), 3)
    if kind in ("min_p", "all"):
        c["min_p"] = round(rng.uniform(0.01, 0.2), 3)
    if rng.random() < 0.5:
        c["history"] = _log_int(rng, 16, 4096)
        if op == "verify":
            if mode != "residual":
                c["frequency"] = 0.3
        else:
            which = rng.choice(["repetition", "counts", "both"])
            if which != "counts":
                c["repetition"], c["repetition_window"] = 1.15, rng.choice([20, 64, 256])
            if which != "repetition":
                c["presence"], c["frequency"] = 0.5, 0.3
    if op == "sample":
        c["semantics"] = rng.choice(["cbv2", "cbv2", "mlxlm"])
        c["mixed"] = c["semantics"] == "cbv2" and rng.random() < 0.25
        c["mask"] = rng.random() < 0.25
    if op == "step":
        c["logprobs"] = rng.choice([-1, 0, 5, 20])
    return c


# ------------------------------------------------------------------------------------ inputs

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _zipf(vocab):
    p = torch.arange(1, vocab + 1, dtype=torch.float64, device=DEVICE) ** -1.1
    return p / p.sum()


def _logits(c, rows, g):
    """[rows, vocab] logits in the case's dtype, and each row's token order by rank (or None)."""
    v, order = c["vocab"], None
    stride = (v + 63) // 64 * 64 if c["pad"] else v
    out = torch.empty((rows, stride), dtype=DTYPES[c["dtype"]], device=DEVICE)
    if c["history"] or c["logits"] == "peaked":
        order = torch.empty((rows, v), dtype=torch.int64, device=DEVICE)
    for a in range(0, rows, 64):
        n = min(64, rows - a)
        x = torch.randn((n, stride), generator=g, device=DEVICE) * c["sigma"]
        if order is not None:
            perm = torch.rand((n, v), generator=g, device=DEVICE).argsort(1)
            order[a:a + n] = perm
            if c["logits"] == "peaked":
                prior = torch.log(_zipf(v)).float()
                x[:, :v].scatter_add_(1, perm, prior.expand(n, v).contiguous())
        if c["logits"] == "boosted":
            ids = torch.randint(0, v, (n, 32), generator=g, device=DEVICE)
            x.scatter_add_(1, ids, torch.full_like(ids, 8, dtype=torch.float32))
        out[a:a + n] = x.to(out.dtype)
    return out[:, :v], order


def _entries(c, rows, order, g):
    """Sparse penalty entries [n, 4] int32 (token, count, flags, bias) and the CSR bounds of a
    Zipf(1.1) history per row: output counts, and a flag on the tokens of the last window."""
    v, h, w = c["vocab"], c["history"], c["repetition_window"]
    ranks = torch.searchsorted(_zipf(v).cumsum(0), torch.rand((rows, h), generator=g,
                                                              device=DEVICE, dtype=torch.float64))
    tokens = order.gather(1, ranks.clamp_(max=v - 1))
    key = tokens + v * torch.arange(rows, device=DEVICE)[:, None]
    counted = c["presence"] != 0 or c["frequency"] != 0
    recent = key[:, max(0, h - w):] if c["repetition"] != 1.0 or not counted else key[:, :0]
    uniq, count = torch.unique(key if counted else recent, return_counts=True)
    entry = torch.zeros((len(uniq), 4), dtype=torch.int32, device=DEVICE)
    entry[:, 0] = (uniq % v).int()
    if counted:
        entry[:, 1] = count.int()
    if recent.numel():
        entry[:, 2] = torch.isin(uniq, recent).int() * _ffi.PEN_REPETITION
    if c["semantics"] == "mlxlm" and c["presence"] != 0:
        entry[:, 2] |= _ffi.PEN_PRESENCE
    bounds = torch.arange(rows + 1, device=DEVICE) * v
    return entry, torch.searchsorted(uniq, bounds).int()


def _params(c, rows, seed):
    """The resolved parameters of every row."""
    if c["semantics"] == "mlxlm":
        return [W.resolve_mlxlm(temperature=c["temperature"], top_p=c["top_p"], top_k=c["top_k"],
                                min_p=c["min_p"], repetition_penalty=c["repetition"],
                                repetition_context_size=c["repetition_window"],
                                presence_penalty=c["presence"] or None,
                                frequency_penalty=c["frequency"] or None)] * rows
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(rows):
        kw = dict(temperature=c["temperature"], top_p=c["top_p"], top_k=c["top_k"],
                  min_p=c["min_p"], repetition_penalty=c["repetition"])
        if c["mixed"]:
            kw.update(temperature=0.0 if rng.random() < 0.25 else rng.uniform(0.3, 1.2),
                      top_k=int(rng.choice([0, 20, 100])), top_p=rng.uniform(0.8, 1.0),
                      repetition_penalty=rng.uniform(1.0, c["repetition"]))
        kw = {k: v if k == "top_k" else float(np.float32(v)) for k, v in kw.items()}
        out.append(W.resolve_cbv2(repetition_context_size=c["repetition_window"],
                                  presence_penalty=c["presence"],
                                  frequency_penalty=c["frequency"], vocab=c["vocab"], **kw))
    return out


def _bitmask(c, rows, g):
    """Packed allowed-token masks, densities 0.1%, 2%, 30% and 100% by row; one row allows a
    single token."""
    words = (c["vocab"] + 31) // 32
    dense = torch.tensor([0.001, 0.02, 0.3, 2.0], device=DEVICE)[torch.arange(rows) % 4]
    allowed = torch.rand((rows, words * 32), generator=g, device=DEVICE) < dense[:, None]
    if rows > 1:
        allowed[-1] = False
    allowed[:, c["vocab"] - 291] = True
    bits = allowed.view(rows, words, 32).long() << torch.arange(32, device=DEVICE)
    return bits.sum(2).to(torch.int32)


def _nucleus_draw(logits, c, g):
    """One token a row from softmax(logits / T) cut at top-p: what a draft model proposed."""
    p, ids = torch.softmax(logits.float() / max(c["temperature"], 0.05), 1).sort(1, descending=True)
    run = p.cumsum(1)
    p = p * (run - p <= c["top_p"])
    u = torch.rand((len(p), 1), generator=g, device=DEVICE) * p.sum(1, keepdim=True)
    at = torch.searchsorted(p.cumsum(1), u).clamp_(max=c["vocab"] - 1)
    return ids.gather(1, at)[:, 0].int()


def _inputs(c, seed):
    g = _generator(seed)
    rows, v = c["rows"], c["vocab"]
    d = {}
    if c["op"] == "verify":
        wide = rows * c["window"]
        x, order = _logits(c, wide, g)
        d["target"] = x.view(rows, c["window"], v)
        draft = torch.empty((rows, c["window"] - 1, v), dtype=x.dtype, device=DEVICE)
        tokens = torch.empty((rows, c["window"] - 1), dtype=torch.int32, device=DEVICE)
        for j in range(c["window"] - 1):
            noise = torch.randn((rows, v), generator=g, device=DEVICE)
            draft[:, j] = (d["target"][:, j].float() + noise).to(x.dtype)
            tokens[:, j] = _nucleus_draw(draft[:, j], c, g)
        d["draft"], d["draft_tokens"] = draft, tokens
        d["uniforms"] = torch.rand((rows, c["window"]), generator=g, device=DEVICE)
        order = None if order is None else order[::c["window"]]
    else:
        d["logits"], order = _logits(c, rows, g)
        d["uniforms"] = torch.rand(rows, generator=g, device=DEVICE)
    if c["history"]:
        d["entries"], d["row_ptr"] = _entries(c, rows, order, g)
    if c["mask"]:
        d["bitmask"] = _bitmask(c, rows, g)
    if c["op"] == "logprobs":
        d["tokens"] = d["logits"].float().topk(8, dim=1).indices[
            torch.arange(rows, device=DEVICE),
            torch.randint(0, 8, (rows,), generator=g, device=DEVICE)].int()
    return d


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    rows, v = c["rows"], c["vocab"]
    wide = rows * (2 * c["window"] - 1) if c["window"] else rows
    ctx = Context(0, max_rows=wide, max_vocab=v)
    params = _params(c, rows, seed)
    entries = {k: d[k] for k in ("row_ptr", "entries") if k in d}
    if c["op"] in ("sample", "step"):
        kw = dict(entries, uniforms=d["uniforms"])
        if c["mask"]:
            kw.update(bitmask=d["bitmask"], mask_bits=v)
        if c["op"] == "sample":
            sem = _ffi.SEM_MLXLM if c["semantics"] == "mlxlm" else _ffi.SEM_CBV2
            call = ctx.prepare_sample(d["logits"], params, semantics=sem, want_stats=c["stats"],
                                      **kw)
        else:
            call = ctx.prepare_step(d["logits"], params, logprobs_top_k=c["logprobs"], **kw)
    elif c["op"] == "verify":
        kw = {}
        if entries:
            kw = dict(penalty_row_ptr=d["row_ptr"], penalty_entries=d["entries"],
                      scratch_cap=c["history"] + c["window"])
        call = ctx.prepare_verify(d["target"], d["draft"] if c["mode"] == "residual" else None,
                                  d["draft_tokens"], params, d["uniforms"], mode=MODES[c["mode"]],
                                  typical_delta=0.2 if c["mode"] == "typical" else 0.0, **kw)
    elif c["op"] == "top2":
        call = ctx.prepare_top2(d["logits"])
    else:
        call = ctx.prepare_logprobs(d["logits"], tokens=d["tokens"], top_k=c["logprobs"])
    return {"context": ctx, "call": call, "rows": rows, "stats": c["stats"]}


def run(state):
    call = state["call"]
    call.launch()
    out = call.outputs()
    if state["stats"]:
        raw = out.pop("stats")
        f = raw.view(torch.float32).view(-1, 12)
        out.update(max_value=f[:, 0], log_normalizer=f[:, 1], cut_value=f[:, 8],
                   kept_mass=f[:, 9], kept_entropy=f[:, 10],
                   kept=raw.view(torch.int32).view(-1, 12)[:, 2],
                   kept_weight=raw.view(torch.int64).view(-1, 6)[:, 2])
    return out


# ------------------------------------------------------------------------------- work, checks

def work(case):
    c = case
    size = 4 if c["dtype"] == "f32" else 2
    positions = 1
    if c["op"] == "verify":
        positions = 2 * c["window"] - 1 if c["mode"] == "residual" else c["window"]
    tokens = c["rows"] * c["vocab"] * positions
    total = tokens * size + c["rows"] * positions * 12
    if c["op"] not in ("top2", "logprobs"):
        total += c["rows"] * 32
    if c["history"]:
        counted = c["presence"] != 0 or c["frequency"] != 0
        n = c["history"] if counted else min(c["history"], c["repetition_window"])
        p = np.arange(1, c["vocab"] + 1, dtype=np.float64) ** -1.1
        distinct = float((1.0 - (1.0 - p / p.sum()) ** n).sum())
        total += int(c["rows"] * distinct * 16)
    if c["mask"]:
        total += c["rows"] * ((c["vocab"] + 31) // 32) * 4
    if c["logprobs"] > 0:
        total += c["rows"] * c["logprobs"] * 8
    # a comparison a token; a difference, an exponential and a sum where a mass is asked for
    return {"bytes": total, "flops": tokens * (1 if c["op"] == "top2" else 4)}


def tolerance(case):
    # Tokens, ids and kept sets are the same whatever the order of the sums.  Log-probabilities
    # and statistics are float32 values of float32 sums: 1e-7 from 64 bits, 3e-7 at most.
    if case["op"] == "logprobs" or case["logprobs"] >= 0 or case["stats"]:
        return {"rel": 5e-7, "max": 2e-6}
    return "exact"


def _filter_space(c, d, params):
    """Penalized, tempered and masked logits in 64 bits, with the parameters as columns."""
    x = d["logits"].double()
    rows, v = x.shape
    col = {k: torch.tensor([float(p[k]) for p in params], dtype=torch.float32,
                           device=DEVICE).double()[:, None] for k in params[0]}
    if "entries" in d:
        e = d["entries"]
        row = torch.repeat_interleave(torch.arange(rows, device=DEVICE), d["row_ptr"].diff())
        tok, count = e[:, 0].long(), e[:, 1].double()
        at = x[row, tok]
        rep, pres, freq = (col[k][row, 0] for k in ("repetition_penalty", "presence_penalty",
                                                    "frequency_penalty"))
        if c["semantics"] == "mlxlm" and c["dtype"] != "f32":
            low = DTYPES[c["dtype"]]  # those two penalties are rounded to the logits' type
            rep, pres = rep.to(low).double(), pres.to(low).double()
        flagged = (e[:, 2] & _ffi.PEN_REPETITION) != 0
        at = torch.where(flagged, torch.where(at < 0, at * rep, at / rep), at)
        at = torch.where(count > 0, at - freq * count - pres, at)
        x[row, tok] = at
    if c["semantics"] == "cbv2":
        x = x / col["temperature"]
    if "bitmask" in d:
        bits = d["bitmask"][:, :, None] >> torch.arange(32, device=DEVICE)
        allowed = (bits & 1).reshape(rows, -1)[:, :v] != 0
        x = torch.where(allowed, x, torch.full_like(x, -math.inf))
    return x, col


def _exact_rows(c, d, params):
    """Drawn tokens and statistics of one batch of rows in 64 bits (inverse CDF in token order)."""
    y, col = _filter_space(c, d, params)
    rows, v = y.shape
    top = y.max(1, keepdim=True).values
    mass = torch.exp(y - top)
    z = mass.sum(1, keepdim=True)
    key, ids = torch.sort(y, dim=1, descending=True, stable=True)
    m = torch.exp(key - top)
    before = m.cumsum(1) - m
    greedy = col["kind"] == _ffi.KIND_ARGMAX
    rank = torch.arange(v, device=DEVICE)[None, :]
    k = torch.where((col["top_k"] > 0) & (col["top_k"] < v), col["top_k"], torch.full_like(top, v))
    limit = torch.where(col["top_p"] < 1, col["top_p"], torch.full_like(top, 2.0)) * z
    if c["semantics"] == "mlxlm":  # the filters run one after the other; each keeps a prefix
        keep = (rank < k) & (before < limit)
        scale = 1.0 / col["temperature"].clamp(min=1e-30)
    else:
        keep = (rank < k) & (before <= limit)
        scale = torch.ones_like(top)
    keep &= key >= top + torch.log(col["min_p"])
    keep = torch.where(greedy, rank < 1, keep & (key > -math.inf))
    kept = torch.zeros_like(keep).scatter_(1, ids, keep)
    w = torch.where(kept, torch.exp((y - top) * torch.where(greedy, torch.ones_like(scale), scale)),
                    torch.zeros_like(y))
    run = w.cumsum(1)
    u = d["uniforms"].double()[:, None] * run[:, -1:]
    token = (run <= u).sum(1).clamp_(max=v - 1)
    p = w / run[:, -1:]
    return {"tokens": token.int(), "max_value": top[:, 0], "log_normalizer": torch.log(z[:, 0]),
            "cut_value": torch.where(kept, y, torch.full_like(y, math.inf)).min(1).values,
            "kept_mass": torch.where(kept, mass, torch.zeros_like(y)).sum(1),
            "kept_entropy": -torch.where(p > 0, p * torch.log(p), torch.zeros_like(p)).sum(1),
            "kept": kept.sum(1).int()}


def _take(d, params, a, n):
    """Rows a .. a + n of the inputs."""
    part = {k: d[k][a:a + n] for k in ("logits", "uniforms", "bitmask") if k in d}
    if "entries" in d:
        b = d["row_ptr"][a:a + n + 1]
        part["entries"], part["row_ptr"] = d["entries"][int(b[0]):int(b[-1])], b - b[0]
    return part, params[a:a + n]


def exact(case, seed):
    c = case
    if c["op"] == "verify":  # accepted counts and tokens: whole numbers
        return None
    d = _inputs(c, seed)
    rows = c["rows"]
    if c["op"] == "top2":
        x = d["logits"].double()
        values, ids = torch.sort(x, dim=1, descending=True, stable=True)
        return {"ids": ids[:, :2].int(), "values": values[:, :2]}
    out = {}
    if c["op"] != "logprobs":
        params = _params(c, rows, seed)
        parts = [_exact_rows(c, *_take(d, params, a, 16)) for a in range(0, rows, 16)]
        got = {k: torch.cat([p[k] for p in parts]) for k in parts[0]}
        out = {"tokens": got["tokens"], "row_flags": None}
        if c["stats"]:
            out.update({k: got[k] for k in got if k != "tokens"}, kept_weight=None)
    if c["logprobs"] >= 0:
        token = (d["tokens"] if c["op"] == "logprobs" else out["tokens"]).long()
        best, chosen = [], []
        for a in range(0, rows, 16):
            lp = torch.log_softmax(d["logits"][a:a + 16].double(), 1)
            best.append(torch.sort(lp, dim=1, descending=True, stable=True))
            chosen.append(lp.gather(1, token[a:a + 16, None])[:, 0])
        n = c["logprobs"]
        out["chosen"] = torch.cat(chosen)
        names = ("top_values", "top_ids")
        for k, name in enumerate(names):
            out[name] = torch.cat([b[k][:, :n] for b in best])
        out["top_ids"] = out["top_ids"].int()
        if c["op"] == "logprobs":
            out["row_flags"] = None
    return out
