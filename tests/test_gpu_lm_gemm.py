"""GPU: the LM head's logits GEMM at the edges of its split: fewer 16-column
units than blocks, a ragged last unit, rows of y that are not 16-byte aligned,
one pass filled exactly and one unit past it, hidden sizes of fewer chunks
than a ring stage holds, or not a multiple of one; and the argmax partials it leaves.

Logits: x = hi + lo exactly up to 2^-17 relative per element and fp32 sums, so
1e-5 of the largest logit, the bar the LM head is held to elsewhere; tokens:
exactly the argmax of the returned logits (an integer rule)."""
import numpy as np
import pytest

import mlamoe
from mlamoe import synth

pytestmark = pytest.mark.gpu

UNIT, BLOCKS, PASS = 16, 256, 7


@pytest.fixture(scope="module")
def ctx():
    c = mlamoe.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("B,V,H", [
    (5, 1, 64), (64, 15, 128), (63, 17, 192), (17, UNIT * BLOCKS - 3, 64), (64, UNIT * BLOCKS + 1, 64),
    (33, UNIT * BLOCKS * PASS, 64), (6, UNIT * BLOCKS * PASS + 1, 320), (64, 2 * UNIT * BLOCKS * PASS + 6, 128)])
def test_lm_gemm_split_edges(ctx, B, V, H):
    print(f"lm gemm B={B} V={V} H={H}", flush=True)
    rng = np.random.default_rng(V + B)
    x = synth.normal_f32(rng, (B, H))
    norm = synth.bf16_from_f32(1.0 + synth.normal_f32(rng, (H,), 0.1))
    lm = synth.normal_bf16(rng, (V, H), 0.02)
    lm[V // 2] = lm[V - 1]                          # equal logits in two blocks: the lower index wins
    logits, tokens = ctx.lm_head(x, norm, 1e-6, lm)
    xn = ctx.rmsnorm(x, norm, 1e-6).astype(np.float64)
    ref = xn @ (lm.astype(np.uint32) << 16).view(np.float32).astype(np.float64).T
    assert np.abs(logits - ref).max() <= 1e-5 * np.abs(ref).max()
    assert np.array_equal(tokens, logits.argmax(1))
    assert np.array_equal(ctx.lm_head(x, norm, 1e-6, lm, want_logits=False)[1], tokens)


def test_lm_gemm_argmax_of_nan_and_inf(ctx):
    """NaN logits never win unless they are the first; infinities do."""
    rng = np.random.default_rng(3)
    B, V, H = 8, 5000, 128
    x = np.abs(synth.normal_f32(rng, (B, H))) + 0.1
    norm = synth.bf16_from_f32(np.ones(H, np.float32))
    lm = synth.normal_bf16(rng, (V, H), 0.02)
    lm[4000, 5], lm[17, 9], lm[3000, 1] = 0x7f80, 0x7fc0, 0xff80     # inf, NaN, -inf
    for first_nan in (False, True):
        if first_nan:
            lm[0, 0] = 0x7fc0
        logits, tokens = ctx.lm_head(x, norm, 1e-6, lm)
        assert np.isnan(logits[:, 17]).all() and np.array_equal(tokens, ctx.argmax(logits))
        if first_nan:
            assert (tokens == 0).all()
