"""GPU: the int8 MoE at the edges of the rule that picks its GEMMs (tiled from
12 rows per expert on average): the last token count below it, the first that
meets it, and an even and a skewed routing there.  Same bars as the two paths
are held to by themselves (test_gpu_moe_i8)."""
import numpy as np
import pytest

import mlamoe
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
