"""Prefill attention in the expanded form (keys and values per head, the rows
of a prompt in 64-row tiles): prompts at the edges of its tiles, several
prompts of unequal length in one step, a chunk after earlier positions, and
decode rows beside them, against the absorbed form of the same engine.

Both forms carry fp32 operands as bf16 pairs (relative error below 2^-17 per
operand, random) and read the same bf16 latent cache; one layer's appended
row may then round differently in the next layer's cache (2^-9 of an
element, rarely).  Logits agree to 2e-4 of their norm (measured 3e-5)."""
import numpy as np
import pytest

import mlamoe
from mlamoe import synth
from mlamoe.engine import Engine

pytestmark = pytest.mark.gpu

CFG = dict(n_layers=2, first_dense=2, H=256, NH=4, QKN=128, QKR=64, KVL=512, VHD=128, dense_inter=128, E=4,
           n_shared=1, K=2, I=64, vocab=300, router_sigmoid=0, norm_topk=0, routed_scaling=1.0, rms_eps=1e-6)


@pytest.fixture(scope="module")
def model():
    c = CFG
    return synth.model(4321, c["n_layers"], c["first_dense"], c["H"], c["NH"], c["QKN"], c["QKR"], c["KVL"], c["VHD"],
                       c["dense_inter"], c["E"], c["I"], c["n_shared"], c["vocab"])


def logits(model, steps, monkeypatch, expand_min, cfg=CFG):
    """Each step: a list of (slot, first position, rows).  All rows' logits,
    and each step's launches of the expanded and the absorbed attention per
    layer."""
    monkeypatch.setenv("MLAMOE_MLA_EXPAND_MIN", str(expand_min))
    rng = np.random.default_rng(5)
    toks = rng.integers(0, CFG["vocab"], (8, 2048)).astype(np.int32)
    out, forms = [], []
    with mlamoe.Context(0) as ctx:
        eng = Engine.from_host(ctx, cfg, model, mlamoe.rope_inv_freq(64, 10000.0), max_batch=8, max_seq=1200,
                               max_rows=2048)
        try:
            for st in steps:
                ctx.prof_reset()
                ctx.prof_enable(True)
                rows = [(s, p0 + i) for s, p0, n in st for i in range(n)]
                sl, ps = (np.array(a, np.int32) for a in zip(*rows))
                _, lg = eng.step_rows(sl, toks[sl, ps], ps, np.arange(len(rows)), want_logits=True)
                out.append(lg)
                ctx.prof_enable(False)
                n = [ctx.prof_query(k)[1] // cfg["n_layers"]
                     for k in ("mm_mla_attn_expanded", "mm_mla_attn", "mm_mla_attn_rows")]
                forms.append((n[0], n[1] + n[2]))
        finally:
            eng.close()
    return np.concatenate(out).astype(np.float64), forms


# with each step's launches per layer: expanded, absorbed
@pytest.mark.parametrize("steps,want", [
    ([[(0, 0, 128)]], [(1, 0)]), ([[(0, 0, 129)]], [(1, 0)]), ([[(3, 0, 161)]], [(1, 0)]), ([[(0, 0, 65)]], [(1, 0)]),
    ([[(1, 0, 1023)]], [(1, 0)]),
    ([[(0, 0, 300), (1, 0, 50), (2, 0, 128), (5, 0, 255)]], [(1, 1)]),      # unequal prompts (50: absorbed)
    # chunks, decode rows
    ([[(0, 0, 37)], [(0, 37, 200), (1, 0, 130)], [(0, 237, 1), (1, 130, 1), (2, 0, 140)]], [(0, 1), (1, 0), (1, 1)]),
    ([[(0, 0, 31)], [(0, 31, 66)], [(0, 97, 513)]], [(0, 1), (1, 0), (1, 0)]),
    ([[(0, 0, 1000), (1, 0, 1000)], [(0, 1000, 100), (1, 1000, 150)]], [(1, 0), (1, 0)]),
], ids=lambda v: "-".join("+".join(str(n) for _, _, n in st) if isinstance(st, list) else "%dx%d" % st for st in v))
def test_expanded_agrees_with_absorbed(model, monkeypatch, steps, want):
    a, forms = logits(model, steps, monkeypatch, 65)
    b, absorbed = logits(model, steps, monkeypatch, 0)
    assert forms == want and not any(e for e, _ in absorbed)
    err = np.linalg.norm(a - b) / np.linalg.norm(b)
    worst = np.max(np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1))
    print(f"{steps}: {err:.2e}, worst row {worst:.2e}", flush=True)
    assert err < 2e-4 and worst < 2e-3


def test_more_tiles_than_compute_units(monkeypatch):
    """16 heads: 16 row tiles give every CU one block, and the host puts the
    next 16 in reverse order.  18, 30 and 33 tiles: every row once."""
    c = dict(CFG, NH=16)
    m = synth.model(4323, c["n_layers"], c["first_dense"], c["H"], c["NH"], c["QKN"], c["QKR"], c["KVL"], c["VHD"],
                    c["dense_inter"], c["E"], c["I"], c["n_shared"], c["vocab"])
    for steps in ([[(0, 0, 1150), (1, 0, 898)]], [[(0, 0, 640), (1, 0, 640), (2, 0, 640)]], [[(0, 0, 1089)]]):
        a, forms = logits(m, steps, monkeypatch, 65, c)
        b, _ = logits(m, steps, monkeypatch, 0, c)
        assert forms == [(1, 0)]
        worst = np.max(np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1))
        assert np.linalg.norm(a - b) < 2e-4 * np.linalg.norm(b) and worst < 2e-3


def test_expanded_against_oracle(model, monkeypatch, oracle):
    """Every position of a 150-token prompt against the reference's forward."""
    got, forms = logits(model, [[(0, 0, 150)]], monkeypatch, 128)
    assert forms == [(1, 0)]
    toks = np.random.default_rng(5).integers(0, CFG["vocab"], (8, 2048)).astype(np.int32)[0, :150]
    ref = oracle.model_logits(CFG, model, toks, mlamoe.rope_inv_freq(64, 10000.0))
    err = np.max(np.abs(got - ref), axis=1) / np.max(np.abs(ref), axis=1)
    print(f"worst normwise logits error {err.max():.2e}", flush=True)
    assert err.max() < 2e-3              # the bar of the other prefill tests (bf16 cache, fp32 in the reference)


def test_scratch_cap_falls_back(model, monkeypatch):
    """Prompts whose expanded keys do not fit the attention scratch cap take
    the absorbed form: neither of two, the second, the first, both."""
    steps = [[(0, 0, 1000), (1, 0, 600)]]
    for blocks, want in ((32 + 19, (1, 0)), (40, (1, 1)), (31, (1, 1)), (18, (0, 1))):     # 32 keys of 4 heads each
        monkeypatch.setenv("MLAMOE_MLA_PART_MAX", str(blocks * 4 * 32768))
        a, forms = logits(model, steps, monkeypatch, 128)
        assert [(e, min(n, 1)) for e, n in forms] == [want]       # (absorbed rows go in groups within the cap)
    b, _ = logits(model, steps, monkeypatch, 0)
    assert np.linalg.norm(a - b) < 2e-4 * np.linalg.norm(b)


def test_no_room_for_the_expanded_keys(monkeypatch):
    """A step whose expanded keys the GPU has no room for takes the absorbed
    form.  64 heads: 512 rows take 134 MB of absorbed scratch, their expanded
    keys 33.5 MB per 512 positions."""
    c = dict(CFG, NH=64)
    m = synth.model(4322, c["n_layers"], c["first_dense"], c["H"], c["NH"], c["QKN"], c["QKR"], c["KVL"], c["VHD"],
                    c["dense_inter"], c["E"], c["I"], c["n_shared"], c["vocab"])
    toks = np.random.default_rng(7).integers(0, c["vocab"], 3072).astype(np.int32)
    out, forms = [], []
    for limit in (None, 150 << 20):
        if limit:
            monkeypatch.setenv("MLAMOE_WS_MAX", str(limit))
        with mlamoe.Context(0) as ctx:
            eng = Engine.from_host(ctx, c, m, mlamoe.rope_inv_freq(64, 10000.0), max_batch=1, max_seq=3072,
                                   init_seq=3072, max_rows=512)
            try:
                ctx.prof_enable(True)
                for p0 in range(0, 3072, 512):
                    ctx.prof_reset()
                    lg = eng.step_rows(np.zeros(512), toks[p0:p0 + 512], np.arange(p0, p0 + 512), np.arange(512),
                                       want_logits=True)[1]
                    forms.append(ctx.prof_query("mm_mla_attn_expanded")[1])
                assert not limit or ctx.workspace_bytes() <= limit
                ctx.prof_enable(False)
            finally:
                eng.close()
        out.append(lg.astype(np.float64))
    assert forms == [2] * 6 + [2] * 4 + [0] * 2
    assert np.linalg.norm(out[0] - out[1]) < 2e-4 * np.linalg.norm(out[0])


@pytest.mark.parametrize("first,n,bad", [(0, 150, 149), (0, 150, 100), (0, 150, 63), (37, 129, 40), (37, 129, 128),
                                         (0, 700, 350)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_row_that_is_not_finite(model, first, n, bad, value):
    """A row whose embedding is not finite gives NaN from its position on, and
    leaves the rows before it as they are: a key that a row does not see
    weighs nothing, whatever it holds."""
    m = dict(model, embed=model["embed"].copy())
    m["embed"][299] = synth.bf16_from_f32(np.full(CFG["H"], value, np.float32))
    toks = np.random.default_rng(6).integers(0, 299, first + n).astype(np.int32)
    out = []
    with mlamoe.Context(0) as ctx:
        eng = Engine.from_host(ctx, CFG, m, mlamoe.rope_inv_freq(64, 10000.0), max_batch=1, max_seq=1200, max_rows=2048)
        try:
            if first:
                eng.step_rows(np.zeros(first), toks[:first], np.arange(first), [])
            for t in (toks[first + bad], 299):
                toks[first + bad] = t
                ctx.prof_reset()
                ctx.prof_enable(True)
                out.append(eng.step_rows(np.zeros(n), toks[first:], np.arange(first, first + n), np.arange(n),
                                         want_logits=True)[1])
                assert ctx.prof_query("mm_mla_attn_expanded")[1] == CFG["n_layers"]
        finally:
            ctx.prof_enable(False)
            eng.close()
    assert np.array_equal(out[0][:bad], out[1][:bad])
    assert np.isfinite(out[0]).all() and np.isnan(out[1][bad:]).all()


def test_step_after_one_that_failed(model, monkeypatch):
    """A step that fails on its way (no room for its absorbed scratch either)
    leaves nothing queued that the next one's tables could reach."""
    toks = np.random.default_rng(8).integers(0, CFG["vocab"], 2048).astype(np.int32)
    out = []
    for limit in (None, 8 << 20):                  # 2,048 rows: 8 MB of expanded keys and their bits, 33 MB absorbed
        if limit:
            monkeypatch.setenv("MLAMOE_WS_MAX", str(limit))
        with mlamoe.Context(0) as ctx:
            eng = Engine.from_host(ctx, CFG, model, mlamoe.rope_inv_freq(64, 10000.0), max_batch=2, max_seq=2048,
                                   init_seq=2048, max_rows=2048)
            try:
                for _ in range(3 if limit else 0):
                    with pytest.raises(mlamoe.MMError, match="workspace"):
                        eng.step_rows(np.zeros(2048), toks, np.arange(2048), [])
                out.append(eng.step_rows(np.ones(130), toks[:130], np.arange(130), np.arange(130), want_logits=True)[1])
            finally:
                eng.close()
    assert np.array_equal(out[0], out[1])
