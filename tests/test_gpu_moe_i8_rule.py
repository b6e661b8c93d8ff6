"""GPU: the int8 MoE at the edges of the rule that picks its GEMMs (tiled from
12 rows per expert on average and as many more as 480 MB of an expert's weights
are, at most 56): the last token count below it, the first that meets it, and
an even and a skewed routing there.  Same bars as the two paths are held to by
themselves (test_gpu_moe_i8)."""
import numpy as np
import pytest

import mlamoe
from mlamoe import synth
from test_gpu_moe_i8 import run_case

pytestmark = pytest.mark.gpu

SMALL = dict(H=256, E=16, K=4, I=128, NS=2)      # 0.1 MB per expert: 56 rows
LARGE = dict(H=2048, E=4, K=4, I=1024, NS=0)     # 6.3 MB: 12 rows and 76 of all experts' more


def first_tiled(c):
    rows = min(56 * c["E"], 12 * c["E"] + 480000000 // (3 * c["I"] * c["H"]))
    return -(-rows // c["K"])


@pytest.mark.parametrize("c,d,skew", [(SMALL, -1, False), (SMALL, 0, False), (SMALL, 1, True), (LARGE, -1, False),
                                      (LARGE, 0, False)])
def test_i8_gemm_rule(oracle, monkeypatch, c, d, skew):
    H, E, K, I, NS, T = c["H"], c["E"], c["K"], c["I"], c["NS"], first_tiled(c) + d
    monkeypatch.delenv("MLAMOE_I8_TILED_MIN_T", raising=False)
    ctx = mlamoe.Context(0)
    try:
        logits = None
        if skew:                          # three experts take every token
            logits = np.random.default_rng(T).standard_normal((T, E)).astype(np.float32)
            logits[:, :3] += 20.0
        ctx.prof_enable(True)
        run_case(ctx, oracle, H, E, K, I, NS, T, 70 + T, logits=logits, check_all=False)
        tiled, decode = (ctx.prof_query(k)[1] for k in ("mm_i8_gemm_gu_dbg", "mm_i8_gu"))
        ctx.prof_enable(False)
        assert (tiled, decode) == ((1, 0) if d >= 0 else (0, 1))
    finally:
        ctx.close()


@pytest.mark.parametrize("c,T", [(SMALL, first_tiled(SMALL)), (SMALL, 231), (dict(SMALL, H=512, I=192), 255),
                                 (LARGE, first_tiled(LARGE))])
def test_i8_gemm_rule_same_bits(monkeypatch, c, T):
    """The two GEMMs add integers and share the SwiGLU and the dequantisation,
    so a call that the rule makes tiled gives the decode-shaped GEMMs' bits."""
    H, E, K, I, NS = c["H"], c["E"], c["K"], c["I"], c["NS"]
    w, x = synth.moe_layer(800 + T, H, E, I, NS), synth.activations(801 + T, T, H)
    outs = []
    for min_t in (None, "100000"):        # by the rule; decode-shaped at any length
        if min_t:
            monkeypatch.setenv("MLAMOE_I8_TILED_MIN_T", min_t)
        else:
            monkeypatch.delenv("MLAMOE_I8_TILED_MIN_T", raising=False)
        with mlamoe.Context(0) as ctx:
            ctx.moe_init(H, E, NS, K, I)
            ctx.moe_load_layer(0, w, mlamoe.MM_LOAD_INT8)
            outs.append(ctx.moe_forward(0, x, flags=mlamoe.MM_FWD_INT8)[0])
    assert np.array_equal(outs[0], outs[1])
