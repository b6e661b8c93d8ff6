"""The bf16 MoE layer as grouped GEMMs (more than a few tokens) at the edges
of its tiles: 16-, 32- and 64-row tiles with remainders, experts with no row
and with every row, hidden sizes that are no multiple of the 64-wide K chunk,
column counts that are none of a tile's, no shared expert, more than 256
experts, several passes, and values that fp32 barely holds.

Bar: the weights and activations enter the products exactly (three bf16 parts
of every fp32 value), so only fp32 sums round: with n = H and I terms the
error of a sum of random terms is about sqrt(n) / 2 units of 2^-24 of its
norm, here below 2e-6 of the layer output's 2-norm (measured 3e-7)."""
import ctypes as C

import numpy as np
import pytest

import mlamoe
from mlamoe import synth

pytestmark = pytest.mark.gpu
TOL = 2e-6


def ref64(w, x, idx, wt, NS):
    f = lambda a: synth.bf16_to_f32(a).astype(np.float64)  # noqa: E731
    x = x.astype(np.float64)

    def mlp(v, g, u, d):
        a, b = v @ f(g).T, v @ f(u).T
        return (a / (1 + np.exp(-a)) * b) @ f(d).T
    out = mlp(x, w["sg"], w["su"], w["sd"]) if NS else np.zeros_like(x)
    for e in np.unique(idx):
        t, r = np.nonzero(idx == e)
        out[t] += wt[t, r, None].astype(np.float64) * mlp(x[t], w["eg"][e], w["eu"][e], w["ed"][e])
    return out


def run(H, E, K, I, NS, T, hot=False, scale=1.0, seed=0, chunk=None):
    w = synth.moe_layer(900 + seed, H, E, I, NS)
    x = synth.activations(901 + seed, T, H) * np.float32(scale)
    lg = synth.uniform_logits(902 + seed, T, E)
    if hot:                       # every token takes expert 1; expert 0 gets none
        lg[:, 1] += 9
        lg[:, 0] -= 9
    with mlamoe.Context(0) as ctx:
        ctx.moe_init(H, E, NS, K, I)
        ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_BF16)
        out, idx, wt, _ = ctx.moe_forward(0, x, logits=lg)
        again, *_ = ctx.moe_forward(0, x, logits=lg)
    assert np.array_equal(out, again)           # the counters were left clear
    ref = ref64(w, x, idx, wt, NS)
    err = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    print(f"H={H} E={E} K={K} I={I} NS={NS} T={T} hot={hot}: {err:.2e}", flush=True)
    assert err < TOL
    return out


@pytest.mark.parametrize("T", [5, 6, 9, 16, 17, 33, 64, 65, 131])
@pytest.mark.parametrize("hot", [False, True])
def test_row_tiles(T, hot):
    run(256, 8, 2, 128, 2, T, hot, seed=T)


@pytest.mark.parametrize("H,E,K,I,NS,T", [(264, 4, 2, 72, 1, 70), (72, 3, 1, 8, 0, 40), (1032, 6, 3, 136, 1, 9),
                                          (256, 300, 8, 64, 1, 37), (128, 160, 4, 64, 3, 90), (64, 2, 2, 200, 2, 300),
                                          # 16, 32 and 64 rows per tile where the sums move every 256 values
                                          (1032, 8, 2, 520, 1, 30), (1032, 8, 2, 520, 1, 64), (1032, 8, 2, 520, 1, 131)])
def test_shapes(H, E, K, I, NS, T):
    run(H, E, K, I, NS, T, seed=H + I)


@pytest.mark.parametrize("H,E,K,I,NS,T,grouped", [
    (256, 16, 4, 128, 2, 8, 0), (256, 16, 4, 128, 2, 9, 1),              # the GEMV stages' one pass, their second
    (1024, 4, 2, 2048, 0, 7, 0), (1024, 4, 2, 2048, 0, 8, 1),            # 126 and 151 MB of weights not read again
    (2048, 4, 4, 2048, 0, 4, 0), (2048, 4, 4, 2048, 0, 5, 1),            # 4 tokens stay with the GEMV
    (512, 65, 8, 2048, 4, 8, 0),                                         # more than 64 experts
    (2048, 4, 4, 2056, 0, 8, 0), (2056, 4, 4, 2048, 0, 8, 0), (2056, 4, 4, 2048, 0, 9, 1),    # rows of no whole lines
    (64, 65, 2, 64, 1, 16, 0), (64, 65, 2, 64, 1, 17, 1), (64, 64, 2, 64, 1, 9, 1), (512, 65, 2, 64, 1, 9, 1)])   # many narrow experts
def test_rule(H, E, K, I, NS, T, grouped):
    w, x = synth.moe_layer(940, H, E, I, NS), synth.activations(941, T, H)
    with mlamoe.Context(0) as ctx:
        ctx.moe_init(H, E, NS, K, I)
        ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_BF16)
        ctx.prof_enable(True)
        out, idx, wt, _ = ctx.moe_forward(0, x)
        ran = ctx.prof_query("mm_bf16_rows")[1]
        ctx.prof_enable(False)
    ref = ref64(w, x, idx, wt, NS)
    assert np.linalg.norm(out - ref) < TOL * np.linalg.norm(ref)
    assert ran == grouped


def test_passes_agree():
    """2,100 tokens (two passes) against the same rows alone: a row's result
    does not depend on the rows beside it."""
    H, E, K, I, NS, T = 64, 4, 2, 64, 1, 2100
    w, x = synth.moe_layer(950, H, E, I, NS), synth.activations(951, T, H)
    lg = synth.uniform_logits(952, T, E)
    with mlamoe.Context(0) as ctx:
        ctx.moe_init(H, E, NS, K, I)
        ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_BF16)
        out, *_ = ctx.moe_forward(0, x, logits=lg)
        part, *_ = ctx.moe_forward(0, x[2040:2060], logits=lg[2040:2060])
    assert np.array_equal(out[2040:2060], part)


def test_fixed_workspace():
    """The no-allocation entry point takes as many tokens per pass as its
    scratch holds: the same bits as the growing workspace."""
    H, E, K, I, NS, T = 1024, 8, 4, 512, 2, 700
    w, x = synth.moe_layer(960, H, E, I, NS), synth.activations(961, T, H)
    with mlamoe.Context(0) as ctx:
        ctx.moe_init(H, E, NS, K, I)
        ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_BF16)
        dx = ctx.to_device(x)
        a, b = ctx.empty((T, H), np.float32), ctx.empty((T, H), np.float32)
        mlamoe._check(mlamoe.lib().mm_moe_forward_noalloc_dev(ctx.h, 0, T, dx.ptr, a.ptr, None, None, None, None,
                                                              C.c_uint(mlamoe.MM_FWD_BF16)))
        assert ctx.workspace_bytes() == 0
        ctx.moe_forward_dev(0, T, dx, b)
        assert np.array_equal(a.download(), b.download())


@pytest.mark.parametrize("ws_max,gemv", [(16 << 20, False), (3 << 20, False), (1 << 19, True)])
def test_workspace_that_cannot_grow(monkeypatch, ws_max, gemv):
    """When the GPU has no room for a pass's workspace the call runs in
    shorter passes (the same bits), and without room for 5 tokens by the
    GEMV stages."""
    H, E, K, I, NS, T = 1024, 8, 4, 512, 2, 300
    w, x = synth.moe_layer(985, H, E, I, NS), synth.activations(986, T, H)
    outs = []
    for limit in (None, ws_max):
        if limit:
            monkeypatch.setenv("MLAMOE_WS_MAX", str(limit))
        else:
            monkeypatch.delenv("MLAMOE_WS_MAX", raising=False)
        with mlamoe.Context(0) as ctx:
            ctx.moe_init(H, E, NS, K, I)
            ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_BF16)
            ctx.prof_enable(True)
            out, idx, wt, _ = ctx.moe_forward(0, x)
            outs.append(out)
            grouped = ctx.prof_query("mm_bf16_rows")[1]
            ctx.prof_enable(False)
            assert ctx.workspace_bytes() <= ws_max if limit else ctx.workspace_bytes() > 16 << 20
            assert grouped == 1 if not limit else grouped == 0 if gemv else grouped > 1
    if gemv:
        ref = ref64(w, x, idx, wt, NS)
        assert np.linalg.norm(outs[1] - ref) < TOL * np.linalg.norm(ref)
    else:
        assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("inf", [False, True])
def test_large_and_infinite_activations(inf):
    """Activations near the largest fp32 value split without overflow; an
    infinite one gives infinity, as fp32 arithmetic does (weights positive
    where it meets them: infinity times zero is NaN in either)."""
    H, E, K, I, NS, T = 64, 2, 1, 64, 0, 20
    w = synth.moe_layer(970, H, E, I, NS)
    one = np.uint16(0x3f80)
    x = np.zeros((T, H), np.float32)
    if inf:
        for k in ("eg", "eu", "ed"):
            w[k] = np.full_like(w[k], one)             # g = u = sum x, out = I silu(g) u
        x[:, 0] = 2.0
        x[3, 0] = np.inf
        want = np.where(np.arange(T) == 3, np.inf, I * 4.0 / (1 + np.exp(-2.0)))
    else:
        for k in ("eg", "eu", "ed"):
            w[k] = np.zeros_like(w[k])
        w["eu"][:, 0, 0] = w["eg"][:, 0, 1] = one      # u[0] = x[0], g[0] = x[1]
        w["ed"][:, :, 0] = one                         # out = h[0]
        x[:, 0] = np.float32(8e36)
        x[:, 1] = 40.0                                 # silu(40) = 40
        want = np.full(T, 40.0 * np.float64(np.float32(8e36)))
    lg = synth.uniform_logits(971, T, E)
    with mlamoe.Context(0) as ctx:
        ctx.moe_init(H, E, NS, K, I)
        ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_BF16)
        out, idx, wt, _ = ctx.moe_forward(0, x, logits=lg)
    want = np.broadcast_to((wt[:, 0] * want)[:, None], out.shape)
    fin = np.isfinite(want)
    assert np.allclose(out[fin], want[fin], rtol=1e-6, atol=0)
    assert np.array_equal(out[~fin], want[~fin])


@pytest.mark.parametrize("where", ["eg", "eu", "ed", "sg", "su", "sd"])
def test_infinite_weights(where):
    """Infinite weights against activations exact in bf16, in two bf16 parts
    and in none: the infinities and NaN of 4 rows at a time (the GEMV, fp32
    products), and its values elsewhere."""
    H, E, K, I, NS, T = 64, 4, 2, 64, 1, 24
    r = np.random.default_rng(973)
    w = synth.moe_layer(974, H, E, I, NS)
    v = w[where].reshape(-1, w[where].shape[-1])
    v[r.integers(0, v.shape[0], 6), r.integers(0, v.shape[1], 6)] = np.array([0x7f80, 0xff80] * 3, np.uint16)
    x = synth.activations(975, T, H)
    kind = r.integers(0, 4, x.shape)                   # 0: one bf16, 1: two of them, 2: zero, 3: as drawn
    x[kind == 0] = (x[kind == 0].view(np.uint32) & 0xffff0000).view(np.float32)
    x[kind == 1] = (x[kind == 1].view(np.uint32) & 0xffffff00).view(np.float32)
    x[(kind == 2) & (r.random(x.shape) < 0.1)] = 0.0
    lg = synth.uniform_logits(976, T, E)
    with mlamoe.Context(0) as ctx:
        ctx.moe_init(H, E, NS, K, I)
        ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_BF16)
        out = ctx.moe_forward(0, x, logits=lg)[0]
        ref = np.concatenate([ctx.moe_forward(0, x[t:t + 4], logits=lg[t:t + 4])[0] for t in range(0, T, 4)])
    assert np.isinf(ref).any() or where in ("eg", "sg")     # (silu(-inf) is NaN: so are the rows it meets)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isfinite(out), fin) and np.array_equal(out[~fin], ref[~fin], equal_nan=True)
    assert np.linalg.norm(out[fin] - ref[fin]) <= 2 * TOL * np.linalg.norm(ref[fin])


@pytest.mark.parametrize("e", [-100, -110, -117])
def test_small_activations(e):
    """A value whose lower bf16 parts are subnormal: still the whole of it."""
    H, E, K, I, NS, T = 64, 2, 1, 64, 0, 20
    w = synth.moe_layer(977, H, E, I, NS)
    for k in ("eg", "eu", "ed"):
        w[k] = np.zeros_like(w[k])
    one = np.uint16(0x3f80)
    w["eu"][:, 0, 0] = w["eg"][:, 0, 1] = one          # u[0] = x[0], g[0] = x[1]
    w["ed"][:, :, 0] = np.uint16(0x7100)               # out = 2^99 h[0]: h's own parts are normal
    x = np.zeros((T, H), np.float32)
    x[:, 0] = np.ldexp(1.0 + np.random.default_rng(978).integers(1, 1 << 23, T) / (1 << 23), e).astype(np.float32)
    x[:, 1] = 2.0 ** 30                                # silu(2^30) = 2^30
    with mlamoe.Context(0) as ctx:
        ctx.moe_init(H, E, NS, K, I)
        ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_BF16)
        out, idx, wt, _ = ctx.moe_forward(0, x, logits=synth.uniform_logits(979, T, E))
    want = wt[:, 0].astype(np.float64) * x[:, 0] * 2.0 ** 129
    print(f"2^{e}: {np.max(np.abs(out / want[:, None] - 1)):.2e}", flush=True)
    assert np.max(np.abs(out / want[:, None] - 1)) < max(2.0 ** -22, 2.0 ** (-132 - e))


def test_rows_past_32_bit_offsets():
    """An intermediate size at which 64 hidden rows span 4 GB: the call takes
    the GEMV stages.  The experts' weights are zero but for a few rows."""
    H, E, K, I, NS, T = 8, 1, 1, 1 << 25, 0, 64
    r = np.random.default_rng(980)
    at = np.unique(np.r_[0, I - 1, r.integers(0, I, 12)])
    w = synth.moe_layer(980, H, E, 8, NS)
    for k, shape in (("eg", (E, I, H)), ("eu", (E, I, H)), ("ed", (E, H, I))):
        w[k] = np.zeros(shape, np.uint16)
    w["eg"][0, at], w["eu"][0, at] = synth.normal_bf16(r, (at.size, H)), synth.normal_bf16(r, (at.size, H))
    w["ed"][0][:, at] = synth.normal_bf16(r, (H, at.size))
    x = synth.activations(981, T, H)
    with mlamoe.Context(0) as ctx:
        ctx.moe_init(H, E, NS, K, I)
        ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_BF16)
        out, idx, wt, _ = ctx.moe_forward(0, x)
    few = dict(eg=w["eg"][:, at], eu=w["eu"][:, at], ed=w["ed"][:, :, at])
    ref = ref64(few, x, idx, wt, NS)
    assert np.linalg.norm(out - ref) < TOL * np.linalg.norm(ref)
