"""Rows of top-p / min-p alone in the one-round fused kernel: drawn from the
slices' lists by the row's last arriver, or sent down the histogram path when
the lists cannot decide them.  Every batch mixes rows of each outcome: nuclei
of one token and of most of the row, one slice far above the others (its list
ends above the row's cut), ties longer than a list, few or no tokens left by
the mask, infinities and NaN.  Against the oracle, with the waits given up
(every slice but a row's last arriver leaves) and without."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from common import compare, rows_from_lists, run_gpu, run_oracle, to_torch_logits
from lsamp import _ffi
from lsamp import workloads as W
from lsamp.history import Cbv2RowState, TokenRing, csr, mlxlm_entries

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from lsamp.api import Context
    c = Context(0, max_rows=256, max_vocab=262144)
    yield c
    c.close()


def _bits(x, dtype):
    if dtype == _ffi.DTYPE_F32:
        return x.astype(np.float32)
    if dtype == _ffi.DTYPE_F16:
        return x.astype(np.float16).view(np.uint16)
    return W.f32_to_bf16_bits(x.astype(np.float32))


def _batch(rows, V, dtype, sem, seed, masked):
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 3, (rows, V))
    params, ents = [], []
    for r in range(rows):
        kind = r % 10
        if kind == 1:  # a few tokens hold everything
            x[r, rng.integers(0, V, 3)] += 25
        elif kind == 2:  # close to flat: most of the row is kept
            x[r] *= 0.25
        elif kind == 3:  # one slice far above a broad rest
            x[r, : V // 8] += 6
            x[r, rng.integers(0, V // 8)] += 16
        elif kind == 4:  # ties longer than any list
            x[r] = np.round(2 * x[r]) / 2
        elif kind == 5:
            x[r, rng.integers(0, V, 5)] = -np.inf
            x[r, rng.integers(0, V)] = np.nan
        elif kind == 6:
            x[r, [rng.integers(0, V), V - 1]] = np.inf
        elif kind == 7:
            x[r] = -np.inf
            x[r, rng.integers(0, V, 2)] = 1.0
        top_p = [0.9, 0.95, 0.5, 0.99, 1.0][r % 5]
        min_p = [0.0, 0.0, 0.02, 0.3, 0.05][(r // 2) % 5]
        T = [0.8, 1.0, 0.3, 1.7][(r // 3) % 4]
        kw = dict(temperature=T, top_p=top_p, min_p=min_p if top_p < 1 else max(min_p, 0.1))
        hist = rng.integers(0, V, 40).tolist() + np.argsort(-np.nan_to_num(x[r]))[:20].tolist()
        if sem == _ffi.SEM_CBV2:
            params.append(W.resolve_cbv2(presence_penalty=0.4, repetition_penalty=1.2, vocab=V, **kw))
            ents.append(Cbv2RowState([], hist, 64, True, True, vocab=V).entries())
        else:
            params.append(W.resolve_mlxlm(repetition_penalty=1.2, repetition_context_size=64, **kw))
            ring = TokenRing(64)
            ring.load_prompt(hist)
            ents.append(mlxlm_entries(repetition=ring))
    row_ptr, entries = csr(ents)
    cfg = dict(semantics=sem, dtype=dtype, rows=rows, vocab=V, logits=_bits(x, dtype),
               params=W._params(params), row_ptr=row_ptr, entries=entries, bitmask=None,
               mask_bits=0, uniforms=rng.random(rows, dtype=np.float32))
    if masked:
        allowed = rng.random((rows, (V + 31) // 32 * 32)) < \
            np.array([1.1, 0.3, 0.001, 0.0])[np.arange(rows) % 4][:, None]
        cfg["bitmask"] = np.packbits(allowed.reshape(rows, -1, 32)[:, :, ::-1], axis=2) \
            .view(">u4").reshape(rows, -1).astype(np.uint32)
        cfg["mask_bits"] = V
    return cfg


@pytest.mark.parametrize("rows,V,dtype,sem,masked", [
    (256, 4099, _ffi.DTYPE_BF16, _ffi.SEM_CBV2, False),    # one slice a row
    (128, 40003, _ffi.DTYPE_BF16, _ffi.SEM_MLXLM, False),  # two, unaligned rows
    (85, 9000, _ffi.DTYPE_F16, _ffi.SEM_CBV2, True),       # three
    (64, 65536, _ffi.DTYPE_F32, _ffi.SEM_CBV2, True),      # four
    (43, 9000, _ffi.DTYPE_F32, _ffi.SEM_MLXLM, False),     # five: min-p alone
    (32, 65536, _ffi.DTYPE_BF16, _ffi.SEM_CBV2, False),    # eight: min-p alone
    (256, 70001, _ffi.DTYPE_F32, _ffi.SEM_CBV2, False),    # past one round
])
def test_rows_from_lists(ctx, rows, V, dtype, sem, masked):
    cfg = _batch(rows, V, dtype, sem, rows + V, masked)
    o = run_oracle(cfg, threads=16)
    lib = _ffi.load_library()
    compare(cfg, run_gpu(ctx, cfg), o, label="lists")
    # rows of both outcomes; top-p rows go through lists of at most four slices
    launch, lists = ctx.last_launch(), rows_from_lists(ctx, rows)
    top_p = np.array([p["top_p"] < 1 for p in cfg["params"]])
    assert lists[~top_p].any() and lists[top_p].any() == (launch["slices"] <= 4)
    assert masked or not lists[6::10].any()  # (+inf logits, unless masked)
    assert launch["fused"] == (5 if dtype == _ffi.DTYPE_F32 and rows == 256 else 1)
    ctx.read_status()
    _ffi.check(lib.lsamp_test_set_spin_limit(0, 16), "lsamp_test_set_spin_limit")
    try:
        g = run_gpu(ctx, cfg)
    finally:
        _ffi.check(lib.lsamp_test_set_spin_limit(0, 0), "lsamp_test_set_spin_limit")
    ctx.read_status()
    compare(cfg, g, o, label="lists, waits given up")
    compare(cfg, run_gpu(ctx, cfg), o, label="lists again")
    assert ctx.read_status() == 0


@pytest.mark.parametrize("rows,V,dtype", [
    (7, 4099, _ffi.DTYPE_BF16),    # unaligned rows
    (64, 65536, _ffi.DTYPE_F32),   # one round
    (150, 40003, _ffi.DTYPE_F16),  # several rounds
    (150, 70001, _ffi.DTYPE_F32),  # past one round: split
])
def test_rows_without_filters(ctx, rows, V, dtype):
    """Every token is kept, so without statistics no histogram is built: the
    tokens are those of the call with statistics, which the oracle checks."""
    cfg = _batch(rows, V, dtype, _ffi.SEM_CBV2, rows + V, False)
    for r in range(rows):
        if r % 3:
            cfg["params"][r] = W._params([W.resolve_cbv2(
                temperature=[0.8, 1.0, 0.3, 1.7][r % 4], presence_penalty=0.4,
                repetition_penalty=1.2, vocab=V)])[0]
    full = run_gpu(ctx, cfg)
    compare(cfg, full, run_oracle(cfg, threads=16), label="no filters")
    for mode in (_ffi.MODE_AUTO, _ffi.MODE_SPLIT):
        ctx.set_mode(mode)
        try:
            out = ctx.sample(to_torch_logits(cfg), cfg["params"], semantics=cfg["semantics"],
                             vocab=V, row_ptr=cfg["row_ptr"], entries=cfg["entries"],
                             uniforms=cfg["uniforms"])
        finally:
            ctx.set_mode(_ffi.MODE_AUTO)
        assert np.array_equal(out["tokens"].cpu().numpy(), full["tokens"])
        assert np.array_equal(out["row_flags"].cpu().numpy().astype(np.uint32), full["row_flags"])
    assert ctx.read_status() == 0


def _sparse(V, ids, values):
    x = np.full(V, -np.inf)
    x[ids] = values
    return x


@pytest.mark.parametrize("rows,V,dtype", [
    (64, 65536, _ffi.DTYPE_F32), (64, 65536, _ffi.DTYPE_F16), (43, 9000, _ffi.DTYPE_F32),
    (256, 4099, _ffi.DTYPE_BF16)])
@pytest.mark.parametrize("sem", [_ffi.SEM_CBV2, _ffi.SEM_MLXLM])
def test_values_far_from_zero(ctx, rows, V, dtype, sem):
    """Rows whose surviving logits lie beyond the range in which a slice sums its
    mass (|x| / T past 2^20 log2 units; temperatures that divide such values
    exactly), and ordinary rows beside tokens filled with a very low finite
    value: some tokens, whole waves or whole slices."""
    rng = np.random.default_rng(V + dtype)
    x = rng.normal(0, 3, (rows, V))
    # (bins of 1/32 stay exact in float32 up to 2^19)
    far = 6e4 if dtype == _ffi.DTYPE_F16 else 2.5e5
    fill = {_ffi.DTYPE_F16: -65504.0, _ffi.DTYPE_BF16: -3.3895e38}.get(dtype, -3.4028235e38)
    T = np.full(rows, 0.8)
    for r in range(rows):
        kind, ids = r % 8, rng.choice(V, 3, replace=False)
        if kind == 0:  # three equal tokens far below
            x[r] = _sparse(V, ids, -far)
        elif kind == 1:  # and far above
            x[r] = _sparse(V, ids, far)
        elif kind == 2:  # a few hundred steps of the type's own spacing, far below
            ids = rng.choice(V, 300, replace=False)
            x[r] = _sparse(V, ids, -far + 0.0625 * rng.integers(0, 200, 300))
        elif kind == 3:  # most tokens filled low
            x[r, rng.random(V) < 0.97] = -1e9 if dtype != _ffi.DTYPE_F16 else fill
        elif kind == 4:  # a slice and more of them
            x[r, : V // 3] = fill
        elif kind == 5:  # every token but a few hundred
            keep = rng.choice(V, 300, replace=False)
            x[r] = np.where(np.isin(np.arange(V), keep), x[r], fill)
        elif kind == 6:  # the largest value far below, a cold row
            ids = rng.choice(V, 300, replace=False)
            x[r] = _sparse(V, ids, rng.normal(-3e4, 3, 300))
            T[r] = 2.0 ** -5
        if kind < 3:
            T[r] = 2.0 ** -5 if dtype == _ffi.DTYPE_F16 else 0.25
    params = []
    for r in range(rows):
        kw = dict(temperature=float(T[r]), top_p=[0.9, 0.97, 1.0][r // 8 % 3],
                  min_p=[0.0, 0.02, 0.05][r // 8 % 3])
        params.append(W.resolve_cbv2(vocab=V, **kw) if sem == _ffi.SEM_CBV2 else
                      W.resolve_mlxlm(**kw))
    with np.errstate(over="ignore"):
        cfg = dict(semantics=sem, dtype=dtype, rows=rows, vocab=V, logits=_bits(x, dtype),
                   params=W._params(params), row_ptr=None, entries=None, bitmask=None, mask_bits=0,
                   uniforms=rng.random(rows, dtype=np.float32))
    o = run_oracle(cfg, threads=16)
    g = run_gpu(ctx, cfg)
    compare(cfg, g, o, label="far")
    fin = np.isfinite(o["stats"]["log_normalizer"])
    gn, on = g["stats"]["log_normalizer"][fin], o["stats"]["log_normalizer"][fin]
    bad = np.abs(gn - on) > 2e-6 * (1 + np.abs(on))
    assert not bad.any(), (np.nonzero(fin)[0][bad], gn[bad], on[bad])
    assert ctx.read_status() == 0


@pytest.mark.parametrize("dtype", [_ffi.DTYPE_F32, _ffi.DTYPE_BF16])
@pytest.mark.parametrize("first", [True, False])
def test_mass_of_a_dominant_token_and_its_thread(ctx, dtype, first):
    """One token ahead of the 127 others of its thread, each just under 2^-25 of
    its mass (3.8e-6 together), and a rest that weighs nothing: top-p cuts inside
    the 127, where the row's mass decides how many stay (a running fp32 sum kept
    the dominant token alone).  Statistics against 64 bits."""
    rows, V = 256, 65536
    N = 4 if dtype == _ffi.DTYPE_F32 else 8
    rng = np.random.default_rng(dtype + first)
    x = rng.normal(-30, 1, (rows, V))
    mine = (np.arange(128) // N) * 512 * N + np.arange(128) % N  # thread 0 of a whole slice
    for r in range(rows):
        ids = mine + N * (r % 512)
        # 2^-25 is 17.33 nats; bf16 steps there are 1/8
        x[r, ids] = -(17.34 + 1e-3 * rng.random(128)) if N == 4 else -17.375
        x[r, ids[0 if first else 127]] = 0.0
    top_p = [np.float32(1) - np.float32(k * 2.0 ** -24) for k in (26, 30, 34, 38)]
    params = [W.resolve_cbv2(temperature=1.0, top_p=float(top_p[r % 4]), vocab=V)
              for r in range(rows)]
    cfg = dict(semantics=_ffi.SEM_CBV2, dtype=dtype, rows=rows, vocab=V, logits=_bits(x, dtype),
               params=W._params(params), row_ptr=None, entries=None, bitmask=None, mask_bits=0,
               uniforms=rng.random(rows, dtype=np.float32))
    o = run_oracle(cfg, threads=16)
    g = run_gpu(ctx, cfg)
    assert ctx.last_launch()["slices"] == 1 and rows_from_lists(ctx, rows).all()
    compare(cfg, g, o, label="dominant")
    assert (g["stats"]["kept"] > 16).all()
    y = W.bf16_bits_to_f32(cfg["logits"]) if N == 8 else cfg["logits"]
    z = np.log(np.exp(y.astype(np.float64)).sum(1))
    # (3.8e-6 of the mass in all; the sum's own error is below a tenth of it)
    assert np.abs(g["stats"]["log_normalizer"] - z).max() < 5e-7


@pytest.mark.parametrize("n", [12, 63, 65, 127, 300, 511, 513, 1025, 1800])
def test_ties_in_the_cut_bin(ctx, n):
    """Nuclei that end inside n equal tokens: the cut bin's keys are ranked by
    counting up to a work-group's threads and sorted past that."""
    rows, V = 64, 65536
    rng = np.random.default_rng(n)
    x = rng.normal(-12, 0.5, (rows, V))
    for r in range(rows):
        # (some in each of the row's four slices, so that no slice is flat)
        ids = rng.choice(V // 4, n + 1, replace=False) + V // 4 * (np.arange(n + 1) % 4)
        x[r, ids] = 2.0
        x[r, ids[0]] = 2.0 + [0.0, 1.5][r % 2]
    top_p = [0.3, 0.9, 0.97, 0.6]
    params = [W.resolve_cbv2(temperature=0.7, top_p=top_p[r % 4], vocab=V) for r in range(rows)]
    cfg = dict(semantics=_ffi.SEM_CBV2, dtype=_ffi.DTYPE_F16, rows=rows, vocab=V,
               logits=_bits(x, _ffi.DTYPE_F16), params=W._params(params), row_ptr=None, entries=None,
               bitmask=None, mask_bits=0, uniforms=rng.random(rows, dtype=np.float32))
    o = run_oracle(cfg, threads=16)
    g = run_gpu(ctx, cfg)
    assert rows_from_lists(ctx, rows).all()
    compare(cfg, g, o, label=f"{n} ties")


def test_keyed_draw_from_lists(ctx):
    """Philox keys: a row's uniform is its key's, drawn by the row's last arriver."""
    rows = 64
    cfg = _batch(rows, 65536, _ffi.DTYPE_BF16, _ffi.SEM_CBV2, 5, False)
    keys = np.array([O.rng_key(77, 1000 + r, 3) for r in range(rows)], np.uint64)
    u = np.array([O.rng_uniform(int(k), 0) for k in keys], np.float32)
    g = run_gpu(ctx, cfg, philox_keys=keys)
    top_p = np.array([p["top_p"] < 1 for p in cfg["params"]])
    assert rows_from_lists(ctx, rows)[top_p].any()
    compare(cfg, g, run_oracle(cfg, philox_keys=keys, threads=16), label="keys", uniforms=u)
