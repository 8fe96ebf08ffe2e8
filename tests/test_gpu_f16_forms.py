"""f16 products of more than 16 tokens (kernels.zig:82-112 linearF16): each
workgroup form the size rule chooses, at ragged rows and tokens and a K that
ends inside a chunk of steps, against float64."""
import numpy as np
import pytest

import qwenscriber_amd as qa
from util import normal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,tokens", [
    (1023, 320, 17),     # K split, 16 rows; a wavefront with two steps, the others one
    (2047, 1088, 37),    # 32 rows
    (6143, 1024, 23),    # 48 or 64 rows
    (4095, 2048, 50),    # 64 rows
    (1025, 1024, 402),   # 64 rows x 32 tokens
    (4097, 1600, 97),    # the same, a chunk of one step
    (12287, 2048, 40),   # 64 rows x 48 tokens
    (12289, 832, 65),    # 128 rows
    (4097, 1024, 401),   # 128 rows x 64 tokens
    (12290, 1024, 255),  # 256 rows x 64 tokens
])
def test_f16_linear_forms(ctx, rows, cols, tokens):
    w = normal(rows * cols, 51, rows).reshape(rows, cols).astype(np.float16)
    x = normal(tokens * cols, 52, tokens).reshape(tokens, cols)
    x[1] *= np.float32(1e-30)
    x[2] *= np.float32(1e25)
    x[3] = 0.0
    handle = ctx.matrix_upload(qa.FORMAT_F16, rows, cols, None, w.view(np.uint16).reshape(-1))
    bx, bo = ctx.to_device(x), ctx.buffer(tokens * rows * 4)
    try:
        ctx.linear(handle, bx.ptr, cols, tokens, bo.ptr)
        got = bo.download(np.float32).reshape(tokens, rows).astype(np.float64)
    finally:
        bx.free()
        bo.free()
        ctx.matrix_release(handle)
    wd = w.astype(np.float64)
    want = x.astype(np.float64) @ wd.T
    # Each product carries 2^-22 of its step's largest activation; a sum is
    # rounded once a 32-value MFMA, once a step, and a few times at the end.
    mass = np.abs(x).astype(np.float64) @ np.abs(wd).T
    largest = np.abs(x).reshape(tokens, -1, 64).max(axis=2).repeat(64, axis=1).astype(np.float64)
    bound = (5 * cols // 64 + 8) * 2.0 ** -24 * mass + 2.0 ** -22 * (largest @ np.abs(wd).T) + 1e-37
    worst = np.abs(got - want) / bound
    assert worst.max() <= 1.0, (worst.max(), np.unravel_index(worst.argmax(), worst.shape))
