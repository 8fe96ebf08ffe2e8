"""A few tokens of a small matrix, and a few sequences of a small decoder, on
the per-token GEMVs: at the ends of the token counts and sizes that go there,
and just past them."""
import numpy as np
import pytest

import qwenscriber_amd as qa
from oracle import oracle as o
from util import assert_close, normal, quantized_matrix

pytestmark = pytest.mark.gpu

SMALL = dict(hidden=256, layers=2, heads=4, kv_heads=2, head_dim=128, ffn=512, max_positions=64, eps=1e-6, theta=1e6)


@pytest.mark.parametrize("fmt,rows,cols,tokens", [
    (qa.FORMAT_Q4, 1, 64, 2), (qa.FORMAT_Q4, 127, 896, 16), (qa.FORMAT_Q4, 127, 896, 17),
    (qa.FORMAT_Q4, 2560, 2560, 16), (qa.FORMAT_Q4, 2600, 6144, 4), (qa.FORMAT_Q4, 2700, 6144, 4),
    (qa.FORMAT_Q4, 65, 320, 3),                                    # no fused GEMV for 320 values
    (qa.FORMAT_Q5, 1, 64, 2), (qa.FORMAT_Q5, 33, 192, 12), (qa.FORMAT_Q5, 33, 192, 13),
    (qa.FORMAT_Q5, 3255, 6144, 2), (qa.FORMAT_Q5, 8203, 3072, 2), (qa.FORMAT_Q5, 33000, 512, 3),
    (qa.FORMAT_Q8, 1, 64, 2), (qa.FORMAT_Q8, 33, 192, 12), (qa.FORMAT_Q8, 33, 192, 13),
    (qa.FORMAT_Q8, 1024, 3072, 2), (qa.FORMAT_Q8, 3255, 6144, 2), (qa.FORMAT_Q8, 31, 6208, 2),  # past the GEMV's rows
    # A wavefront a row: few rows x tokens there, more on the matrix cores.
    (qa.FORMAT_Q5, 3584, 896, 4), (qa.FORMAT_Q5, 3584, 896, 6), (qa.FORMAT_Q5, 12288, 128, 12),
    (qa.FORMAT_Q8, 3584, 896, 4), (qa.FORMAT_Q8, 3584, 896, 6), (qa.FORMAT_Q8, 12288, 128, 12),
    (qa.FORMAT_Q8, 1027, 2560, 8), (qa.FORMAT_Q8, 1027, 2560, 11),
])
def test_linear_few_tokens(ctx, fmt, rows, cols, tokens):
    _, scales, data = quantized_matrix(fmt, rows, cols, 3, rows)
    x = normal(tokens * cols, 4, tokens)
    want = o.linear_quantized(fmt, scales, data, rows, cols, x, tokens)
    m = ctx.matrix_upload(fmt, rows, cols, scales, data)
    xb, ob = ctx.to_device(x), ctx.buffer(tokens * rows * 4)
    ctx.linear(m, xb.ptr, cols, tokens, ob.ptr)
    assert_close(ob.download(np.float32), np.asarray(want).reshape(-1), rtol=1e-4, atol_rms=1e-5)
    ctx.matrix_release(m)


@pytest.mark.parametrize("fmt", [qa.FORMAT_Q4, qa.FORMAT_Q5, qa.FORMAT_Q8])
@pytest.mark.parametrize("tokens,offset", [(2, 0), (12, 0), (4, 512)])
def test_linear_few_tokens_in_place(ctx, fmt, tokens, offset):
    # The result over x, or over a part of it: every row is read before any is
    # written.
    rows = cols = 1024
    _, scales, data = quantized_matrix(fmt, rows, cols, 13, 0)
    x = normal(tokens * cols, 14, tokens)
    want = o.linear_quantized(fmt, scales, data, rows, cols, x, tokens)
    m = ctx.matrix_upload(fmt, rows, cols, scales, data)
    buf = ctx.to_device(np.concatenate([x, np.zeros(offset, np.float32)]))
    ctx.linear(m, buf.ptr, cols, tokens, buf.ptr + 4 * offset)
    assert_close(buf.download(np.float32)[offset:offset + tokens * rows], np.asarray(want).reshape(-1), rtol=1e-4, atol_rms=1e-5)
    ctx.matrix_release(m)


@pytest.mark.parametrize("fmt", [o.Q4, o.Q5, o.Q8])
@pytest.mark.parametrize("batch,vocab", [
    (3, 500), (8, 500),      # layers and lm_head per token
    (3, 140001),             # the lm_head on the matrix cores
    (9, 500),                # everything on the matrix cores
])
def test_decoder_few_sequences(ctx, fmt, batch, vocab):
    seed, config = 17, dict(SMALL, vocab=vocab)
    gpu = qa.Decoder(ctx, batch=batch, **config)
    ref = o.Decoder(seed, batch, fmt, o.CACHE_Q8, **config)
    try:
        gpu.init_synthetic(seed, fmt)
        for b in range(batch):
            gpu.prefill_random(b, 3 * b, seed)
            ref.prefill_random(b, 3 * b)
        tokens = [o.start_token(seed, b, vocab) for b in range(batch)]
        for step in range(4):
            gpu.forward(tokens, True)
            for b in range(batch):
                ref.forward(b, tokens[b], True)
                assert_close(gpu.logits(b), ref.logits(b), what=f"step {step} seq {b}")
            tokens = [int(o.argmax(ref.logits(b))) for b in range(batch)]
        ids = gpu.step(tokens)
        assert list(ids) == [ref.step(b, tokens[b]) for b in range(batch)]
    finally:
        gpu.close()
        ref.close()
