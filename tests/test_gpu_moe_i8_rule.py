"""GPU: the int8 MoE at the edges of the rule that picks its GEMMs (tiled from
12 rows per expert on average): the last token count below it, the first that
meets it, and an even and a skewed routing there.  Same bars as the two paths
are held to by themselves (test_gpu_moe_i8)."""
import numpy as np
import pytest

import mlamoe
from mlamoe import synth
from test_gpu_moe_i8 import run_case

pytestmark = pytest.mark.gpu

E, K = 16, 4
T0 = 12 * E // K                          # tokens from which the tiled GEMMs are used


@pytest.mark.parametrize("T,skew", [(T0 - 1, False), (T0, False), (T0 + 1, True)])
def test_i8_gemm_rule(oracle, monkeypatch, T, skew):
    monkeypatch.delenv("MLAMOE_I8_TILED_MIN_T", raising=False)
    ctx = mlamoe.Context(0)
    try:
        logits = None
        if skew:                          # three experts take every token
            logits = np.random.default_rng(T).standard_normal((T, E)).astype(np.float32)
            logits[:, :3] += 20.0
        ctx.prof_enable(True)
        run_case(ctx, oracle, 256, E, K, 128, 2, T, 70 + T, logits=logits, check_all=False)
        tiled, decode = (ctx.prof_query(k)[1] for k in ("mm_i8_gemm_gu_dbg", "mm_i8_gu"))
        ctx.prof_enable(False)
        assert (tiled, decode) == ((1, 0) if T >= T0 else (0, 1))
    finally:
        ctx.close()


@pytest.mark.parametrize("H,I,T", [(256, 128, T0), (256, 128, 131), (512, 192, 255)])
def test_i8_gemm_rule_same_bits(monkeypatch, H, I, T):
    """The two GEMMs add integers and share the SwiGLU and the dequantisation,
    so a call that the rule makes tiled gives the decode-shaped GEMMs' bits."""
    w, x = synth.moe_layer(800 + T, H, E, I, 2), synth.activations(801 + T, T, H)
    outs = []
    for min_t in (None, "100000"):        # by the rule; decode-shaped at any length
        if min_t:
            monkeypatch.setenv("MLAMOE_I8_TILED_MIN_T", min_t)
        else:
            monkeypatch.delenv("MLAMOE_I8_TILED_MIN_T", raising=False)
        with mlamoe.Context(0) as ctx:
            ctx.moe_init(H, E, 2, K, I)
            ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_INT8)
            outs.append(ctx.moe_forward(0, x, flags=mlamoe.MM_FWD_INT8)[0])
    assert np.array_equal(outs[0], outs[1])
