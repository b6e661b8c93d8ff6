"""The tiled bf16 GEMM (more than 64 rows, or inputs no multiple of 64) at the
edges of its tiles: every tile width (128, 64 and 32 columns, the last with K
split between waves), ragged rows, columns and K, the XCD rectangles that the
tile counts choose, outputs that start 4 bytes past an aligned address, and
two matrices over one input.

Operands are whole numbers whose sums stay below 2^24, so every order of
summation is exact: results must match bit for bit."""
import ctypes as C

import numpy as np
import pytest

import mlamoe
from mlamoe import synth

pytestmark = pytest.mark.gpu


def ints(rng, shape):
    return rng.integers(-8, 9, size=shape).astype(np.float32)


@pytest.fixture
def ctx():
    c = mlamoe.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("T,d,n", [
    (65, 31, 64), (128, 32, 72), (129, 33, 200), (300, 100, 136),       # 32-column tiles
    (513, 2501, 64), (1100, 1730, 128), (640, 4097, 264),              # 64 and 128 columns
    (2047, 2048, 192), (2100, 3648, 320), (37, 70, 264), (9000, 65, 576),
    (70, 40, 1096), (1920, 570, 1096), (2000, 2000, 1160)])           # 32, 64, 128 columns: every ring wraps, sums move
@pytest.mark.parametrize("flags", [0, mlamoe.MM_MATMUL_X_BF16])
def test_tiles_exact(ctx, T, d, n, flags):
    rng = np.random.default_rng(T + d + n)
    x, w = ints(rng, (T, n)), ints(rng, (d, n))
    want = (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.float32)
    print(f"tiles T={T} d={d} n={n} flags={flags}", flush=True)
    wb = synth.bf16_from_f32(w)
    assert np.array_equal(ctx.matmul(x, wb, flags), want)
    y0 = ints(rng, (T, d))
    assert np.array_equal(ctx.matmul(x, wb, flags | mlamoe.MM_MATMUL_ACCUMULATE, y0=y0), want + y0)


@pytest.mark.parametrize("T,d,n,bn", [(65, 8200, 72, 64),        # 129 tiles of 64 columns: one round, 257 of 32 two
                                      (100, 8192, 72, 32),       # 256 of 32: one round
                                      (200, 16400, 72, 128),     # 258 of 128: two rounds, 514 of 64 three
                                      (1920, 570, 72, 64)])
def test_column_widths(ctx, T, d, n, bn):
    """Shapes either side of a whole round of tiles per width; exact."""
    rng = np.random.default_rng(d)
    x, w = ints(rng, (T, n)), ints(rng, (d, n))
    print(f"widths T={T} d={d} n={n}: {bn} columns", flush=True)
    assert np.array_equal(ctx.matmul(x, synth.bf16_from_f32(w), mlamoe.MM_MATMUL_X_BF16), x @ w.T)


def test_unaligned_output(ctx):
    T, d, n = 140, 132, 128
    rng = np.random.default_rng(9)
    x, w = ints(rng, (T, n)), ints(rng, (d, n))
    dx, dw, dy = ctx.to_device(x), ctx.to_device(synth.bf16_from_f32(w)), ctx.empty((T * d + 2,), np.float32)
    ctx.fill(dy, T * d + 2, mlamoe.MM_FILL_F32_UNIFORM, 3)
    before = dy.download()
    mlamoe._check(mlamoe.lib().mm_matmul_bf16_dev(ctx.h, C.c_void_p(dy.ptr + 4), dx.ptr, dw.ptr, d, n, T, 0))
    y = dy.download()
    assert np.array_equal(y[1:-1].reshape(T, d), x @ w.T)
    assert y[0] == before[0] and y[-1] == before[-1]


@pytest.mark.parametrize("T", [70, 600])
def test_two_matrices(ctx, oracle, T):
    """The front's query and kv_a projections run as one launch over one
    input: both against the oracle."""
    H, NH, QKN, QKR, KVL, VHD, L = 2048, 16, 128, 64, 512, 64, 8
    w = synth.attn_layer(77, H, NH, QKN, QKR, KVL, VHD)
    x = synth.activations(78, T, H)
    inv = mlamoe.rope_inv_freq(QKR, 10000.0)
    ctx.mla_init(NH, QKN, QKR, KVL, VHD)
    ctx.mla_front_init(H, inv, 0, 1e-6, 1e-6, 0)
    pos = np.zeros(T, np.int32)                     # position 0: RoPE is the identity
    q, rows, _ = ctx.mla_front(x, w, pos, np.zeros((T, L, KVL + QKR), np.uint16))
    f = lambda a: synth.bf16_to_f32(a).astype(np.float64)  # noqa: E731
    xn = x / np.sqrt((x.astype(np.float64) ** 2).mean(1, keepdims=True) + 1e-6) * f(w["in_norm"])
    qr, cr = xn @ f(w["q_proj"]).T, xn @ f(w["kv_a"]).T
    cr[:, :KVL] /= np.sqrt((cr[:, :KVL] ** 2).mean(1, keepdims=True) + 1e-6)
    cr[:, :KVL] *= f(w["kv_a_norm"])
    # the bf16 pair of an fp32 input is off by up to 2^-18 of it
    for got, want in ((q, qr), (rows, cr)):
        assert np.linalg.norm(got - want) < 2.0 ** -18 * np.linalg.norm(want)


@pytest.mark.parametrize("T,d,n", [
    (128, 3, (1 << 24) + 72),       # 128 rows of x span 4 GB
    (2, 33, (1 << 26) + 8)])        # 32 rows of the weights do
def test_rows_past_32_bit_offsets(ctx, T, d, n):
    """Inner sizes at which a tile's rows span more than its loads' 32-bit
    offsets: the tile takes fewer rows, and no row is lost.  x and W hold
    whole numbers in a few columns, the first and the last among them, and
    zeros elsewhere."""
    print(f"long rows T={T} d={d} n={n}", flush=True)
    rng = np.random.default_rng(T + d)
    at = np.unique(np.r_[0, n - 1, n // 2, rng.integers(0, n, 12)])
    xs, ws = ints(rng, (T, at.size)), ints(rng, (d, at.size))

    def sparse(rows, values, kind, dtype):
        buf = ctx.empty((rows, n), dtype)
        ctx.fill(buf, rows * n, kind, 1, 0.0)          # deviation 0
        one = np.empty(1, dtype)
        for (r, j), v in np.ndenumerate(values):
            one[0] = v
            mlamoe._check(mlamoe.lib().mm_h2d(ctx.h, C.c_void_p(buf.ptr + (r * n + int(at[j])) * one.itemsize),
                                              one.ctypes.data, one.itemsize))
        return buf
    x = sparse(T, xs, mlamoe.MM_FILL_F32_NORMAL, np.float32)
    w = sparse(d, synth.bf16_from_f32(ws), mlamoe.MM_FILL_BF16_NORMAL, np.uint16)
    y = ctx.empty((T, d), np.float32)
    ctx.matmul_dev(y, x, w, d, n, T, mlamoe.MM_MATMUL_X_BF16)
    assert np.array_equal(y.download(), xs @ ws.T)
