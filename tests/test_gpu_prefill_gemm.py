"""The prefill's 32-token-tile form (taken from 6e9 multiply-adds a layer),
teacher-forced against the oracle position by position: one layer of the 1.7B
shape, from an empty cache, and a second prompt that continues the first."""
import numpy as np
import pytest

from oracle import oracle as o
from test_gpu_prefill import PAD, make_pair, prompt, teacher_forced
from util import assert_close, normal

pytestmark = pytest.mark.gpu

LAYER = dict(hidden=2048, layers=1, heads=16, kv_heads=8, head_dim=128, ffn=6144, vocab=1000, max_positions=320,
             eps=1e-6, theta=1e6)


@pytest.mark.parametrize("fmt,cache,counts", [
    (o.Q4, "q8", (131, 120)),   # 120 positions: the fewest that this shape sends here
    (o.Q5, "f32", (129,)),
    (o.Q8, "q8", (160,)),
])
def test_prefill_gemm_against_oracle(ctx, fmt, cache, counts):
    gpu, ref = make_pair(ctx, LAYER, 1, 31, fmt, cache, [3])
    try:
        first = 3
        for k, count in enumerate(counts):
            pads = range(5, 5 + count // 2)
            tokens = prompt(count, LAYER["vocab"], pads, 40 + k)
            rows = normal(len(pads) * LAYER["hidden"], 41, k, 0.02).reshape(len(pads), LAYER["hidden"])
            rb = ctx.to_device(rows)
            try:
                got = gpu.prefill(0, tokens, PAD, rb.ptr, len(pads))
            finally:
                rb.free()
            want = teacher_forced(ctx, gpu, ref, 0, tokens, rows, first, LAYER, cache)
            first += count
            assert gpu.position(0) == first
            assert_close(gpu.logits(0), ref.logits(0), what=f"prompt {k} against the oracle (teacher-forced)")
            assert got == want
    finally:
        gpu.close()
        ref.close()
