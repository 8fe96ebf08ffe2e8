"""The prefill's 32-token-tile form (taken from 129 positions and 6e9
multiply-adds a layer), teacher-forced against the oracle position by position:
layers of the 1.7B shape and one wider, a prompt that continues another, and one
of more than a chunk."""
import numpy as np
import pytest

from oracle import oracle as o
from test_gpu_prefill import PAD, make_pair, prompt, teacher_forced
from util import assert_close, normal

pytestmark = pytest.mark.gpu

# Two layers: a layer's K slices pass to the next one's norm.
PAIR = dict(hidden=2048, layers=2, heads=16, kv_heads=8, head_dim=128, ffn=6144, vocab=1000, max_positions=560,
            eps=1e-6, theta=1e6)
# o and down with K whole at 512 positions: they add the residual themselves.
WIDE = dict(hidden=4096, layers=2, heads=16, kv_heads=8, head_dim=128, ffn=2048, vocab=1000, max_positions=520,
            eps=1e-6, theta=1e6)
LAYER = dict(hidden=2048, layers=1, heads=16, kv_heads=8, head_dim=128, ffn=6144, vocab=1000, max_positions=320,
             eps=1e-6, theta=1e6)


@pytest.mark.parametrize("config,fmt,cache,counts", [
    (PAIR, o.Q4, "q8", (540,)),   # q | k | v with K whole, then a second chunk on 16-token tiles
    (PAIR, o.Q8, "f32", (257, 270)),
    (WIDE, o.Q4, "q8", (512,)),
])
def test_prefill_gemm_layers_against_oracle(ctx, config, fmt, cache, counts):
    check_prompts(ctx, config, fmt, cache, counts)


@pytest.mark.parametrize("fmt,cache,counts", [
    (o.Q4, "q8", (131, 120)),   # 120 positions: on 16-token tiles, after the others' rows
    (o.Q5, "f32", (129,)),
    (o.Q8, "q8", (160,)),
])
def test_prefill_gemm_against_oracle(ctx, fmt, cache, counts):
    check_prompts(ctx, LAYER, fmt, cache, counts)


def check_prompts(ctx, config, fmt, cache, counts):
    gpu, ref = make_pair(ctx, config, 1, 31, fmt, cache, [3])
    try:
        first = 3
        for k, count in enumerate(counts):
            pads = range(5, 5 + count // 2)
            tokens = prompt(count, config["vocab"], pads, 40 + k)
            rows = normal(len(pads) * config["hidden"], 41, k, 0.02).reshape(len(pads), config["hidden"])
            rb = ctx.to_device(rows)
            try:
                got = gpu.prefill(0, tokens, PAD, rb.ptr, len(pads))
            finally:
                rb.free()
            want = teacher_forced(ctx, gpu, ref, 0, tokens, rows, first, config, cache)
            first += count
            assert gpu.position(0) == first
            assert_close(gpu.logits(0), ref.logits(0), what=f"prompt {k} against the oracle (teacher-forced)")
            assert got == want
    finally:
        gpu.close()
        ref.close()
