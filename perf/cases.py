"""The work this library does for its users, as cases that can be timed and
whose results can be compared: a MoE layer at decode, mid-size and prefill
token counts with bf16 and int8 experts, the dense projections, the absorbed
attention, one decode layer's attention half, the LM head, and the batched
engine's decode and prefill steps.

Shapes are DeepSeek-V2-Lite's, the ones bench.py and the tests run.  listed()
names the fixed cases, draw() gives more of the same ranges; prepare() makes a
case's inputs, weights and handles from a seed, run() is one pass through the
public entry points, exact() the same results in 64-bit torch.
"""
import ctypes as C
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mla-moe_amd"))

import mlamoe  # noqa: E402
from mlamoe.engine import Engine  # noqa: E402

H, E, K, I, NS = 2048, 64, 6, 1408, 2          # MoE geometry
S = NS * I                                     # the shared experts as one MLP
QKN, QKR, KVL, VHD = 128, 64, 512, 128         # MLA geometry
KVD = KVL + QKR
NH = 16
VOCAB, DENSE = 102400, 10944
LAYERS = 4                                     # engine cases: one dense layer, three MoE layers
EPS = 1e-6
STEP_ROWS = 2048                               # rows of one engine step at most
SCORED = 8                                     # rows per prompt whose logits a prefill step returns
# q_proj, kv_a_proj, kv_b_proj, o_proj: (outputs, inputs)
PROJ = {"q": (NH * (QKN + QKR), H), "kv_a": (KVD, H), "kv_b": (NH * (QKN + VHD), KVL), "o": (H, NH * VHD)}


def listed():
    return [
        # one token of interactive decoding through a MoE layer in the checkpoint's own bf16
        {"name": "ffn_bf16_t1", "kind": "ffn", "fmt": "bf16", "tokens": 1, "glm": False, "zipf": False},
        # a batch of decoding sequences with bf16 experts, for users who do not quantise
        {"name": "ffn_bf16_t64", "kind": "ffn", "fmt": "bf16", "tokens": 64, "glm": False, "zipf": False},
        # a prompt chunk of odd length with bf16 experts
        {"name": "ffn_bf16_t515", "kind": "ffn", "fmt": "bf16", "tokens": 515, "glm": False, "zipf": False},
        # the benchmark's decode batch with int8 experts, routed from the activations
        {"name": "ffn_i8_t64", "kind": "ffn", "fmt": "i8", "tokens": 64, "glm": False, "zipf": False},
        # a mixed step (decode rows and a short prompt) through the other router flavour:
        # sigmoid scores, selection bias, normalised and scaled weights
        {"name": "ffn_i8_glm_t181", "kind": "ffn", "fmt": "i8", "tokens": 181, "glm": True, "zipf": False},
        # the benchmark's prefill: a whole prompt, expert load skewed by a Zipf prior
        {"name": "ffn_i8_zipf_t2048", "kind": "ffn", "fmt": "i8", "tokens": 2048, "glm": False, "zipf": True},
        # the four projections of an attention layer over a prompt, activations cast to bf16
        {"name": "proj_cast_t512", "kind": "proj", "tokens": 512, "cast": True},
        # the absorbed attention of a decode batch over long latent caches
        {"name": "mla_b32_l4096", "kind": "mla", "batch": 32, "length": 4096, "heads": 16, "ragged": False},
        # the attention half of one decode layer for a single sequence: latency
        {"name": "attn_b1_l4096", "kind": "attn", "batch": 1, "length": 4096},
        # the LM head of a decode batch: norm, logits, greedy tokens
        {"name": "lm_head_b64", "kind": "lm", "batch": 64, "vocab": VOCAB},
        # a decode step of the engine with every slot taken, contexts of different lengths
        {"name": "step_i8_b64", "kind": "step", "fmt": "i8", "batch": 64, "length": 260},
        # an engine step that prefills waiting prompts, as the scheduler packs them
        {"name": "prefill_i8_r2047", "kind": "prefill", "fmt": "i8", "rows": 2047, "prompts": 2, "prior": 0},
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "ffn", "proj", "mla", "attn", "lm", "step", "prefill"])
    if kind == "ffn":
        fmt = rng.choice(["bf16", "i8"])
        return {"kind": kind, "fmt": fmt, "tokens": _between(rng, 1, 515 if fmt == "bf16" else 2048),
                "glm": rng.random() < 0.4, "zipf": rng.random() < 0.3}
    if kind == "proj":
        return {"kind": kind, "tokens": _between(rng, 1, 1024), "cast": rng.random() < 0.5}
    if kind == "mla":
        batch = _between(rng, 1, 64)
        return {"kind": kind, "batch": batch, "length": _between(rng, 16, min(32768, 131072 // batch)),
                "heads": rng.choice([16, 20]), "ragged": rng.random() < 0.5}
    if kind == "attn":
        batch = _between(rng, 1, 32)
        return {"kind": kind, "batch": batch, "length": _between(rng, 16, 4096)}
    if kind == "lm":
        return {"kind": kind, "batch": _between(rng, 1, 64), "vocab": rng.choice([VOCAB, rng.randint(30000, VOCAB)])}
    if kind == "step":
        fmt = rng.choice(["i8", "i8", "bf16"])
        batch = _between(rng, 1, 64 if fmt == "i8" else 8)
        return {"kind": kind, "fmt": fmt, "batch": batch, "length": _between(rng, 4, 260)}
    fmt = rng.choice(["i8", "i8", "bf16"])
    return {"kind": kind, "fmt": fmt, "rows": _between(rng, 65, STEP_ROWS if fmt == "i8" else 128),
            "prompts": rng.randint(1, 4), "prior": rng.choice([0, 0, rng.randint(1, 1024 if fmt == "i8" else 256)])}


# ---- inputs: torch tensors on the GPU, a function of (case, seed) ------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda") * std


def _weight(g, shape, std=0.02):
    return _normal(g, shape, std).to(torch.bfloat16)


def _norm_weight(g, n):
    return (1.0 + _normal(g, (n,), 0.1)).to(torch.bfloat16)


def _moe_weights(g, glm):
    w = dict(moe_gate=_weight(g, (E, H)), eg=_weight(g, (E, I, H)), eu=_weight(g, (E, I, H)),
             ed=_weight(g, (E, H, I)), sg=_weight(g, (S, H)), su=_weight(g, (S, H)), sd=_weight(g, (H, S)))
    w["moe_gate_bias"] = _normal(g, (E,), 0.1) if glm else None
    return w


def _front_weights(g):
    return dict(input_norm=_norm_weight(g, H), q_proj=_weight(g, PROJ["q"]), kv_a_proj=_weight(g, PROJ["kv_a"]),
                kv_a_norm=_norm_weight(g, KVL), kv_b=_weight(g, PROJ["kv_b"]), o_proj=_weight(g, PROJ["o"]))


def _inv_freq():
    """Plain RoPE frequencies of the rope dimensions, fp32."""
    return (1.0 / 10000.0 ** (np.arange(0, QKR, 2, dtype=np.float64) / QKR)).astype(np.float32)


def _zipf_prior(seed):
    rank = np.random.default_rng(seed).permutation(E)
    return torch.from_numpy((-1.1 * np.log1p(rank)).astype(np.float32)).cuda()


def _ffn_inputs(c, seed):
    g = _gen(seed)
    w = _moe_weights(g, c["glm"])
    return w, _normal(g, (c["tokens"], H)), _zipf_prior(seed) if c["zipf"] else None


def _proj_inputs(c, seed):
    g = _gen(seed)
    return {k: (_weight(g, shape), _normal(g, (c["tokens"], shape[1]))) for k, shape in PROJ.items()}


def _mla_lengths(c, seed):
    """Per-sequence context lengths: half to all of the longest, in an order of the seed's."""
    b, n = c["batch"], c["length"]
    if not c["ragged"]:
        return None
    lens = [max(1, n - (n // 2) * j // max(1, b - 1)) for j in range(b)]
    random.Random(seed).shuffle(lens)
    return torch.tensor(lens, dtype=torch.int32, device="cuda")


def _mla_inputs(c, seed):
    g, b, nh = _gen(seed), c["batch"], c["heads"]
    return (_weight(g, (nh * (QKN + VHD), KVL)), _normal(g, (b, c["length"], KVD)).to(torch.bfloat16),
            _normal(g, (b, nh, QKN + QKR)), _mla_lengths(c, seed))


def _attn_inputs(c, seed):
    g, b = _gen(seed), c["batch"]
    return _front_weights(g), _normal(g, (b, c["length"], KVD)).to(torch.bfloat16), _normal(g, (b, H))


def _lm_inputs(c, seed):
    g = _gen(seed)
    return _weight(g, (c["vocab"], H)), _norm_weight(g, H), _normal(g, (c["batch"], H))


def _model(seed):
    """A decoder's weights: the embedding, LAYERS layers (the first dense), the head."""
    g = _gen(seed)
    m = dict(embed=_weight(g, (VOCAB, H), 1.0), final_norm=_norm_weight(g, H), lm_head=_weight(g, (VOCAB, H)), layers=[])
    for n in range(LAYERS):
        w = _front_weights(g)
        w["post_norm"] = _norm_weight(g, H)
        if n == 0:
            w.update(gate=_weight(g, (DENSE, H)), up=_weight(g, (DENSE, H)), down=_weight(g, (H, DENSE)))
        else:
            w["moe"] = _moe_weights(g, False)
        m["layers"].append(w)
    return m


def _sequences(c, seed):
    """(tokens, first row of the timed step) of each slot: a decode step takes
    each sequence's last position, a prefill step a prompt's rows after its
    earlier chunk of `prior` positions."""
    rng = np.random.default_rng(seed)
    if c["kind"] == "step":
        b, n = c["batch"], c["length"]
        lens = [max(1, n - (3 * n // 4) * j // max(1, b - 1)) for j in range(b)]
        first = [n - 1 for n in lens]
    else:
        rows, left = [], c["rows"]
        for j in range(c["prompts"], 0, -1):        # unequal prompts, the longest first
            rows.append(left if j == 1 else max(1, left * 2 // (j + 1)))
            left -= rows[-1]
        first = [c["prior"]] * len(rows)
        lens = [c["prior"] + r for r in rows]
    return [(rng.integers(0, VOCAB, n).astype(np.int32), f) for n, f in zip(lens, first)]


def _wanted(seqs, lens):
    """Rows whose logits come back, of each sequence's lens[j] rows one after
    another: its last one after a decode step, its last SCORED after a prefill
    (a continuation is scored against its prompt's last positions)."""
    ends = np.cumsum(lens)
    return np.concatenate([np.arange(e - min(len(t) - first, SCORED), e) for e, (t, first) in zip(ends, seqs)]).astype(np.int32)


# ---- the handles a program keeps ----------------------------------------------


class _Dev:
    """A tensor as the binding's device buffer (pointer and shape)."""

    def __init__(self, t):
        self.t, self.ptr, self.shape = t, t.data_ptr(), tuple(t.shape)


def _dev(t):
    return None if t is None else _Dev(t)


_stream = None


def _program_stream():
    """The one stream that a program orders its work on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream.cuda_stream


class _Handles:
    """A context (and engine) closed with the state that holds it."""

    def __init__(self):
        self.ctx, self.engine = mlamoe.Context(0), None
        self.ctx.set_stream(_program_stream())

    def __del__(self):
        if self.engine is not None:
            self.engine.close()
        self.ctx.close()


def _load_moe(ctx, layer, w, fmt):
    flag = mlamoe.MM_LOAD_INT8 if fmt == "i8" else mlamoe.MM_LOAD_BF16
    ctx.moe_load_layer(layer, {k: _dev(t) for k, t in w.items()}, flag | mlamoe.MM_LOAD_DEVICE_PTRS)


def _moe_context(ctx, glm, layers=1):
    ctx.moe_init(H, E, NS, K, I, router_sigmoid=int(glm), norm_topk=int(glm), routed_scaling=1.8 if glm else 1.0,
                 n_layers=layers)


def _front_struct(w):
    return mlamoe.MlaFrontWeights(*[w[k].data_ptr() if k in w else None for k in mlamoe.FRONT_WEIGHTS])


def _build_engine(hs, m, fmt, slots, positions):
    ctx, lib = hs.ctx, mlamoe.lib()
    ctx.mla_init(NH, QKN, QKR, KVL, VHD, n_layers=LAYERS)
    ctx.mla_front_init(H, _inv_freq(), 0, EPS, EPS, 0)
    _moe_context(ctx, False, LAYERS)
    layers = []
    for n, w in enumerate(m["layers"]):
        ctx.mla_load_layer(n, _dev(w["kv_b"]), mlamoe.MM_LOAD_DEVICE_PTRS)
        layer = mlamoe.EngineLayer(_front_struct(w), w["o_proj"].data_ptr(), w["post_norm"].data_ptr())
        if "moe" in w:
            _load_moe(ctx, n, w["moe"], fmt)
        else:
            layer.dense_gate, layer.dense_up, layer.dense_down = (w[k].data_ptr() for k in ("gate", "up", "down"))
        layers.append(layer)
    cfg = mlamoe.EngineConfig(LAYERS, 1, H, DENSE, VOCAB, EPS, slots, positions,
                              mlamoe.MM_FWD_INT8 if fmt == "i8" else mlamoe.MM_FWD_BF16, positions, STEP_ROWS)
    h = C.c_void_p()
    mlamoe._check(lib.mm_engine_create(ctx.h, C.byref(cfg), C.byref(h)))
    hs.engine = Engine(ctx, h.value, cfg, [])
    for n, layer in enumerate(layers):
        mlamoe._check(lib.mm_engine_set_layer(h, n, C.byref(layer)))
    mlamoe._check(lib.mm_engine_set_head(h, m["embed"].data_ptr(), m["final_norm"].data_ptr(), m["lm_head"].data_ptr()))


def prepare(case, seed):
    hs = _Handles()
    ctx, kind = hs.ctx, case["kind"]
    st = {"kind": kind, "handles": hs, "ctx": ctx}

    def out(shape, dtype=torch.float32):
        return torch.zeros(shape, dtype=dtype, device="cuda")

    if kind == "ffn":
        w, x, prior = _ffn_inputs(case, seed)
        torch.cuda.synchronize()
        _moe_context(ctx, case["glm"])
        _load_moe(ctx, 0, w, case["fmt"])
        n = case["tokens"]
        st.update(tokens=n, flags=mlamoe.MM_FWD_INT8 if case["fmt"] == "i8" else mlamoe.MM_FWD_BF16, x=_Dev(x),
                  prior=_dev(prior), logits=_Dev(out((n, E))), out=_Dev(out((n, H))),
                  idx=_Dev(out((n, K), torch.int32)), w=_Dev(out((n, K))))
    elif kind == "proj":
        n = case["tokens"]
        st.update(tokens=n, flags=mlamoe.MM_MATMUL_X_BF16 if case["cast"] else 0,
                  mats={k: (_Dev(w), _Dev(x), _Dev(out((n, w.shape[0])))) for k, (w, x) in _proj_inputs(case, seed).items()})
    elif kind == "mla":
        kv_b, cache, q, lens = _mla_inputs(case, seed)
        torch.cuda.synchronize()
        nh = case["heads"]
        ctx.mla_init(nh, QKN, QKR, KVL, VHD)
        ctx.mla_load_layer(0, _Dev(kv_b), mlamoe.MM_LOAD_DEVICE_PTRS)
        st.update(batch=case["batch"], length=case["length"], cache=_Dev(cache), q=_Dev(q), lens=_dev(lens),
                  out=_Dev(out((case["batch"], nh * VHD))))
    elif kind == "attn":
        w, cache, x = _attn_inputs(case, seed)
        torch.cuda.synchronize()
        ctx.mla_init(NH, QKN, QKR, KVL, VHD)
        ctx.mla_front_init(H, _inv_freq(), 0, EPS, EPS, 0)
        ctx.mla_load_layer(0, _Dev(w["kv_b"]), mlamoe.MM_LOAD_DEVICE_PTRS)
        b, n = case["batch"], case["length"]
        st.update(batch=b, length=n, weights=w, front=_front_struct(w), o_proj=_Dev(w["o_proj"]), cache=_Dev(cache),
                  x=_Dev(x), pos=_Dev(torch.full((b,), n - 1, dtype=torch.int32, device="cuda")),
                  q=_Dev(out((b, PROJ["q"][0]))), rows=_Dev(out((b, KVD))), attn=_Dev(out((b, NH * VHD))), y=_Dev(out((b, H))))
    elif kind == "lm":
        w, norm, x = _lm_inputs(case, seed)
        b = case["batch"]
        st.update(batch=b, vocab=case["vocab"], w=_Dev(w), norm=_Dev(norm), x=_Dev(x), logits=_Dev(out((b, case["vocab"]))),
                  tokens=_Dev(out((b,), torch.int32)))
    else:
        m, seqs = _model(seed), _sequences(case, seed)
        torch.cuda.synchronize()
        _build_engine(hs, m, case["fmt"], len(seqs), max(len(t) for t, _ in seqs) + 8)
        for layer in m["layers"]:
            layer.pop("moe", None)                   # the library holds its own copy
        rows = [(s, t[p], p) for s, (t, first) in enumerate(seqs) for p in range(first)]
        for r0 in range(0, len(rows), STEP_ROWS):    # the positions before the timed step
            slots, toks, pos = zip(*rows[r0:r0 + STEP_ROWS])
            hs.engine.step_rows(slots, toks, pos, [])
        rows = [(s, t[p], p) for s, (t, first) in enumerate(seqs) for p in range(first, len(t))]
        slots, toks, pos = (np.array(a, np.int32) for a in zip(*rows))
        want = _wanted(seqs, [len(t) - first for t, first in seqs])
        st.update(model=m, slots=slots, toks=toks, pos=pos, want=want, next=np.zeros(want.size, np.int32),
                  logits=out((want.size, VOCAB)))
    torch.cuda.synchronize()
    return st


def run(st):
    ctx, kind = st["ctx"], st["kind"]
    if kind == "ffn":
        logits = None
        if st["prior"] is not None:
            ctx.router_logits_dev(0, st["tokens"], st["x"], st["logits"], st["prior"])
            logits = st["logits"]
        ctx.moe_forward_dev(0, st["tokens"], st["x"], st["out"], logits, st["idx"], st["w"], None, st["flags"])
        return {"out": st["out"].t, "experts": st["idx"].t, "weights": st["w"].t}
    if kind == "proj":
        for w, x, y in st["mats"].values():
            ctx.matmul_dev(y, x, w, w.shape[0], w.shape[1], st["tokens"], st["flags"])
        return {k: y.t for k, (_, _, y) in st["mats"].items()}
    if kind == "mla":
        ctx.mla_absorbed_decode_dev(0, st["batch"], st["q"], st["cache"], st["length"], st["length"], st["out"], st["lens"])
        return st["out"].t
    if kind == "attn":
        b, n = st["batch"], st["length"]
        ctx.mla_front_dev(b, st["x"], st["front"], st["pos"], st["q"], st["cache"], n, st["rows"])
        ctx.mla_absorbed_decode_dev(0, b, st["q"], st["cache"], n, n, st["attn"])
        ctx.matmul_dev(st["y"], st["attn"], st["o_proj"], H, NH * VHD, b)
        return {"q": st["q"].t, "row": st["rows"].t, "ctx": st["attn"].t, "y": st["y"].t}
    if kind == "lm":
        ctx.lm_head_dev(st["batch"], st["x"], st["norm"], EPS, st["w"], st["vocab"], H, st["logits"], st["tokens"])
        return {"logits": st["logits"].t, "tokens": st["tokens"].t}
    lib, h = mlamoe.lib(), st["handles"].engine.h
    nxt, toks, pos = st["next"], st["toks"], st["pos"]
    if kind == "step":
        st_ = lib.mm_engine_step(h, toks.size, toks.ctypes.data, pos.ctypes.data, nxt.ctypes.data, st["logits"].data_ptr())
    else:
        st_ = lib.mm_engine_step_rows(h, toks.size, st["slots"].ctypes.data, toks.ctypes.data, pos.ctypes.data,
                                      st["want"].size, st["want"].ctypes.data, nxt.ctypes.data, st["logits"].data_ptr())
    mlamoe._check(st_)
    return st["logits"]


# ---- what a pass cannot do without ---------------------------------------------


def _ffn_work(n, fmt):
    """One MoE layer over n tokens: the weights of the experts that n tokens
    choose (uniformly, K of E each) and of the shared one, read once."""
    touched = E * (1.0 - (1.0 - K / E) ** n)
    per = 1 if fmt == "i8" else 2
    nbytes = per * 3 * H * (touched * I + S) + 2 * E * H + 8 * n * H
    return nbytes, 2.0 * n * (3 * H * (K * I + S) + E * H)


def _attn_work(rows, keys, pairs):
    """Front, attention and o_proj of one layer over `rows` rows; `keys` cache
    rows read, `pairs` (row, key) pairs attended.  An attention pair costs
    the cheaper, unabsorbed form's products."""
    weights = sum(a * b for a, b in PROJ.values())
    return 2 * weights + 2 * KVD * keys, 2.0 * rows * weights + 2.0 * NH * pairs * (QKN + QKR + VHD)


def work(case):
    kind = case["kind"]
    if kind == "ffn":
        b, f = _ffn_work(case["tokens"], case["fmt"])
    elif kind == "proj":
        n = case["tokens"]
        b = sum(2 * a * k + 4 * n * (a + k) for a, k in PROJ.values())
        f = sum(2.0 * n * a * k for a, k in PROJ.values())
    elif kind == "mla":
        n, nh = case["batch"], case["heads"]
        keys = n * case["length"] * (0.75 if case["ragged"] else 1.0)
        b = 2 * KVD * keys + 2 * nh * (QKN + VHD) * KVL + 4 * n * nh * (QKN + QKR + VHD)
        f = 2.0 * nh * (keys * (KVD + KVL) + n * KVL * (QKN + VHD))
    elif kind == "attn":
        n = case["batch"]
        b, f = _attn_work(n, n * case["length"], 0)
        b, f = b + 8 * n * H, f + 2.0 * NH * n * case["length"] * (KVD + KVL)
    elif kind == "lm":
        n, v = case["batch"], case["vocab"]
        b, f = 2 * v * H + 4 * n * (H + v), 2.0 * n * v * H
    else:
        seqs = _sequences(case, 0)
        rows = sum(len(t) - first for t, first in seqs)
        keys = sum(len(t) for t, _ in seqs)
        pairs = sum((len(t) - first) * (len(t) + first + 1) // 2 for t, first in seqs)
        ab, af = _attn_work(rows, keys, pairs)
        fb, ff = _ffn_work(rows, case["fmt"])
        want = _wanted(seqs, [len(t) - first for t, first in seqs]).size
        b = LAYERS * ab + (LAYERS - 1) * fb + 6 * H * DENSE + 2 * VOCAB * H + 4 * want * VOCAB
        f = LAYERS * af + (LAYERS - 1) * ff + 6.0 * rows * H * DENSE + 2.0 * want * VOCAB * H
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    """About four times what the results are off their 64-bit values."""
    kind, fmt = case["kind"], case.get("fmt")
    if kind == "ffn":
        # int8: a hidden value near the middle of two steps may round to either
        return {"rel": 6e-6, "differ": 1e-3} if fmt == "bf16" else {"rel": 1e-3, "max": 0.05, "differ": 1e-3}
    if kind == "proj":
        return {"rel": 2e-6 if case["cast"] else 1e-5}   # fp32 activations travel as bf16 pairs
    if kind == "mla":
        return {"rel": 1.7e-5}
    if kind == "attn":
        return {"rel": 3e-5}                             # the appended cache row rounds to bf16
    if kind == "lm":
        return {"rel": 1e-5}
    # several layers: int8 activations turn a last-bit change into whole steps
    return {"rel": 0.03, "max": 0.5} if fmt == "i8" else {"rel": 3e-4}


# ---- the same results in 64 bits -------------------------------------------------


def _mm(x, w):
    return x @ w.double().T


def _swiglu(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _quant(x, single=True):
    """Per-row int8 in steps of max|x| / 127: (whole values, steps).  With
    `single` the step and the quotients are rounded to fp32, as the int8
    format defines them (many bf16 weights lie halfway between two steps)."""
    cut = (lambda v: v.float().double()) if single else (lambda v: v)
    x = x.double()
    s = cut(x.abs().amax(-1, keepdim=True) / 127)
    return torch.where(s > 0, cut(x / s).round().clamp(-127, 127), torch.zeros_like(x)), s


def _mlp(x, gate, up, down, fmt):
    if fmt != "i8":
        return _mm(_swiglu(_mm(x, gate), _mm(x, up)), down)
    (qx, sx), (qg, sg), (qu, su), (qd, sd) = (_quant(t) for t in (x, gate, up, down))
    hidden = _swiglu(qx @ qg.T * sx * sg.T, qx @ qu.T * sx * su.T)
    qh, sh = _quant(hidden, False)
    return qh @ qd.T * sh * sd.T


def _moe(x, w, fmt, glm, prior=None):
    logits = _mm(x, w["moe_gate"])
    if prior is not None:
        logits = logits + prior.double()
    scores = torch.sigmoid(logits) if glm else torch.softmax(logits, -1)
    choice = scores + w["moe_gate_bias"].double() if glm else scores
    idx = torch.sort(choice, dim=-1, descending=True, stable=True)[1][:, :K]
    weights = torch.gather(scores, 1, idx)
    if glm:
        weights = weights / weights.sum(-1, keepdim=True) * 1.8
    y = _mlp(x, w["sg"], w["su"], w["sd"], fmt)
    for e in range(E):
        rows, slot = torch.nonzero(idx == e, as_tuple=True)
        if rows.numel():
            y[rows] += weights[rows, slot, None] * _mlp(x[rows], w["eg"][e], w["eu"][e], w["ed"][e], fmt)
    return y, weights


def _rope(v, pos):
    """Adjacent pairs of the last dimension rotated by the fp32 angle pos * inv_freq."""
    ang = (pos[:, None].float() * torch.from_numpy(_inv_freq()).cuda()).double()
    shape = [v.shape[0]] + [1] * (v.dim() - 2) + [QKR // 2]
    c, s = torch.cos(ang).view(shape), torch.sin(ang).view(shape)
    a, b = v[..., 0::2], v[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)


def _front(x, w, pos):
    """q (RoPE applied) and the latent cache rows of rows x at positions pos."""
    xn = _rms(x, w["input_norm"])
    q = _mm(xn, w["q_proj"]).view(-1, NH, QKN + QKR)
    q = torch.cat((q[..., :QKN], _rope(q[..., QKN:], pos)), -1)
    comp = _mm(xn, w["kv_a_proj"])
    return q, torch.cat((_rms(comp[:, :KVL], w["kv_a_norm"]), _rope(comp[:, KVL:], pos)), -1)


def _attend(q, cache, kv_b, first):
    """Rows q [n, heads, 192] of positions first, first + 1, ... over one sequence's cache rows."""
    n, heads = q.shape[:2]
    w = kv_b.double().view(heads, QKN + VHD, KVL)
    c, pe = cache[:, :KVL], cache[:, KVL:]
    k, v = torch.einsum("lr,hdr->hld", c, w).split([QKN, VHD], -1)
    s = torch.einsum("nhd,hld->hnl", q[..., :QKN], k) + torch.einsum("nhd,ld->hnl", q[..., QKN:], pe)
    hidden = torch.arange(cache.shape[0], device="cuda")[None] > first + torch.arange(n, device="cuda")[:, None]
    scale = float(np.float32(1.0) / np.sqrt(np.float32(QKN + QKR)))
    s = torch.softmax((s * scale).masked_fill(hidden, -math.inf), -1)
    return torch.einsum("hnl,hld->nhd", s, v).reshape(n, heads * VHD)


def exact(case, seed):
    kind = case["kind"]
    if kind == "ffn":
        w, x, prior = _ffn_inputs(case, seed)
        out, weights = _moe(x.double(), w, case["fmt"], case["glm"], prior)
        return {"out": out, "experts": None, "weights": weights}
    if kind == "proj":
        cut = (lambda x: (x.view(torch.int32) & -65536).view(torch.float32)) if case["cast"] else (lambda x: x)
        return {k: _mm(cut(x).double(), w) for k, (w, x) in _proj_inputs(case, seed).items()}
    if kind == "mla":
        kv_b, cache, q, lens = _mla_inputs(case, seed)
        lens = [case["length"]] * case["batch"] if lens is None else lens.tolist()
        return torch.cat([_attend(q[b:b + 1].double(), cache[b, :n].double(), kv_b, n - 1) for b, n in enumerate(lens)])
    if kind == "attn":
        w, cache, x = _attn_inputs(case, seed)
        b, n = case["batch"], case["length"]
        q, rows = _front(x.double(), w, torch.full((b,), n - 1, device="cuda"))
        cache = cache.double()
        cache[:, -1] = rows.float().to(torch.bfloat16).double()
        ctx = torch.cat([_attend(q[j:j + 1], cache[j], w["kv_b"], n - 1) for j in range(b)])
        return {"q": q.reshape(b, -1), "row": rows, "ctx": ctx, "y": _mm(ctx, w["o_proj"])}
    if kind == "lm":
        w, norm, x = _lm_inputs(case, seed)
        return {"logits": _mm(_rms(x.double(), norm), w), "tokens": None}
    m, seqs = _model(seed), _sequences(case, seed)
    if case["fmt"] == "i8" and _wanted(seqs, [len(t) - first for t, first in seqs]).size < SCORED:
        return None    # int8 steps of several layers: a row's error is one of a wide spread
    toks = torch.from_numpy(np.concatenate([t for t, _ in seqs])).cuda().long()
    pos = torch.cat([torch.arange(len(t), device="cuda") for t, _ in seqs])
    ends = np.cumsum([len(t) for t, _ in seqs]).tolist()
    x = m["embed"][toks].double()
    for w in m["layers"]:
        q, rows = _front(x, w, pos)
        rows = rows.float().to(torch.bfloat16).double()
        ctx = torch.cat([_attend(q[e - len(t):e], rows[e - len(t):e], w["kv_b"], 0) for e, (t, _) in zip(ends, seqs)])
        x = x + _mm(ctx, w["o_proj"])
        xn = _rms(x, w["post_norm"])
        x = x + (_moe(xn, w["moe"], case["fmt"], False)[0] if "moe" in w else
                 _mlp(xn, w["gate"], w["up"], w["down"], "bf16"))
    want = torch.from_numpy(_wanted(seqs, [len(t) for t, _ in seqs])).cuda()
    return _mm(_rms(x[want], m["final_norm"]), m["lm_head"])
