"""Quantized matrices times many rows of f32 activations (gemm_rows.hip) at
the edges of its tiles: 32-token and 32-row tiles, 128-row workgroups, weight
chunks of two and four groups, K split and not, rows past the registers of the
activation pass."""
import numpy as np
import pytest

import qwenscriber_amd as qa
from oracle import oracle as o
from util import normal, quantized_matrix

pytestmark = pytest.mark.gpu

BIAS = {qa.FORMAT_Q4: 8, qa.FORMAT_Q5: 16, qa.FORMAT_Q8: 128}


def run_linear(ctx, fmt, rows, cols, scales, data, x):
    tokens = x.shape[0]
    m = ctx.matrix_upload(fmt, rows, cols, scales, data)
    xb, ob = ctx.to_device(x), ctx.buffer(tokens * rows * 4)
    ctx.linear(m, xb.ptr, cols, tokens, ob.ptr)
    out = ob.download(np.float32).reshape(tokens, rows)
    for b in (xb, ob):
        b.free()
    ctx.matrix_release(m)
    return out


def dequantized(fmt, rows, cols, scales, data):
    """The planes' values (codes and f16 scales are exact)."""
    groups = cols // 64
    s = np.frombuffer(scales.tobytes(), np.float16).astype(np.float64).reshape(rows, groups, 1)
    d = np.frombuffer(data.tobytes(), np.uint8).reshape(rows, groups, qa.DATA_BYTES[fmt])
    if fmt == qa.FORMAT_Q8:
        u = d.astype(np.int32)
    else:
        u = np.stack([d[..., :32] & 15, d[..., :32] >> 4], axis=-1).reshape(rows, groups, 64).astype(np.int32)
        if fmt == qa.FORMAT_Q5:
            u |= np.unpackbits(d[..., 32:], axis=-1, bitorder="little").astype(np.int32) << 4
    return ((u - BIAS[fmt]) * s).reshape(rows, cols)


def error_bound(x, w):
    """Of x times w^T: the values' and the sums' rounding, as the caller says."""
    tokens, cols = x.shape
    mass = np.abs(x).astype(np.float64) @ np.abs(w).T
    largest = np.abs(x).reshape(tokens, -1, 64).max(axis=2).astype(np.float64)
    floor = largest @ np.abs(w).reshape(w.shape[0], -1, 64).sum(axis=2).T
    return (cols // 64 + 24) * 2.0 ** -23 * mass + 2.0 ** -39 * floor + 1e-37


@pytest.mark.parametrize("fmt", [qa.FORMAT_Q4, qa.FORMAT_Q5, qa.FORMAT_Q8])
@pytest.mark.parametrize("rows,cols,tokens", [
    (48829, 256, 128),   # the least K and tokens; ragged last row tile
    (38760, 320, 129),   # a chunk of one group, one token past a tile
    (26880, 448, 159),   # seven groups
    (2048, 6144, 160),   # K split over slices
    (1600, 7808, 129),   # 122 groups in slices of whole chunks, the last one short
    (1480, 8256, 131),   # past the activation pass's registers (129 groups)
    (33, 1088, 44600),   # one row past a tile (q5; q4 and q8 on 16-token tiles)
    (513, 1088, 2900),   # one row past a workgroup's
])
def test_linear_many_tokens(ctx, fmt, rows, cols, tokens):
    if fmt == qa.FORMAT_Q5 and cols == 8256:
        pytest.skip("q5 rows of an odd number of groups end at 6144 values")
    _, scales, data = quantized_matrix(fmt, rows, cols, 5, rows + cols)
    x = normal(tokens * cols, 6, tokens).reshape(tokens, cols)
    # Tokens of very different magnitudes side by side.
    x[1] *= np.float32(1e-30)
    x[2] *= np.float32(1e25)
    x[3] = 0.0
    x[4, ::7] *= np.float32(3e4)
    got = run_linear(ctx, fmt, rows, cols, scales, data, x).astype(np.float64)
    w = dequantized(fmt, rows, cols, scales, data)
    want = x.astype(np.float64) @ w.T
    # Each product carries 2^-22 of its value (two f16 terms) or 2^-39 of its
    # group's largest (below the f16 range); a sum is rounded at most 9 times
    # within a group, once per group and slice, and twice at the end.
    bound = error_bound(x, w)
    worst = np.abs(got - want) / bound
    assert worst.max() <= 1.0, (worst.max(), np.unravel_index(worst.argmax(), worst.shape))


@pytest.mark.parametrize("fmt", [qa.FORMAT_Q4, qa.FORMAT_Q8])
def test_linear_many_tokens_non_finite(ctx, fmt):
    # An inf or NaN stays in its own token's outputs.
    rows, cols, tokens = 6300, 2048, 128
    _, scales, data = quantized_matrix(fmt, rows, cols, 8, 3)
    x = normal(tokens * cols, 9, 0).reshape(tokens, cols)
    clean = run_linear(ctx, fmt, rows, cols, scales, data, x)
    x[7, 100] = np.inf
    x[21, 5] = np.nan
    got = run_linear(ctx, fmt, rows, cols, scales, data, x)
    others = [t for t in range(tokens) if t not in (7, 21)]
    assert np.array_equal(got[others], clean[others])
    assert not np.isfinite(got[7]).any() and np.isnan(got[21]).all()


@pytest.mark.parametrize("fmt", [qa.FORMAT_Q4, qa.FORMAT_Q5, qa.FORMAT_Q8])
@pytest.mark.parametrize("outlier", [1e6, 1e12, 1e25])
def test_linear_many_tokens_outlier_group(ctx, fmt, outlier):
    # A group far above its row, under weights that are zero there, takes
    # nothing from the other groups' precision.
    rows, cols, tokens = 6400, 2048, 160
    values = normal(rows * cols, 10, 1, 0.02).reshape(rows, cols)
    values[:, 640:704] = 0.0
    scales, data = o.quantize_rows(fmt, values)
    x = normal(tokens * cols, 11, 2).reshape(tokens, cols)
    x[:, 650] = np.float32(outlier)
    got = run_linear(ctx, fmt, rows, cols, scales, data, x).astype(np.float64)
    w = dequantized(fmt, rows, cols, scales, data)
    assert not w[:, 640:704].any()
    worst = np.abs(got - x.astype(np.float64) @ w.T) / error_bound(x, w)
    assert worst.max() <= 1.0, worst.max()
