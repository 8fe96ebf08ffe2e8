"""The matrix-core convolution at the edges of its tiles: 64-channel
wavefronts and 256-channel workgroups, 32 and 64 positions, every number of
patch rounds, odd planes, and inputs of extreme or non-finite magnitude."""
import numpy as np
import pytest

from oracle import oracle as o
from test_gpu_frontend import f16_fast, run_conv
from util import assert_close, normal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,cout,cin,h,w", [
    (1, 64, 16, 1, 1),       # one position, one stage
    (2, 65, 16, 2, 2),       # a second wavefront of one channel
    (1, 257, 32, 7, 5),      # a second workgroup of one channel
    (1, 256, 16, 13, 11),    # 42 positions: 32 + 10
    (3, 33, 16, 9, 127),     # 64 positions to a row: two workgroups a row
    (5, 48, 48, 31, 3),      # two-column output: the patch is the whole plane
    (40, 300, 16, 33, 17),   # enough workgroups for the 64-position form
    (1, 16, 16, 64, 93),     # the most patch rounds
    (1, 250, 160, 9, 13),    # ten stages: two slices
    (2, 257, 176, 5, 7),     # eleven: a slice of six and one of five
    (1, 480, 480, 7, 25),    # thirty: six slices
])
def test_conv_tiles(ctx, batch, cout, cin, h, w):
    x = normal(batch * cin * h * w, 91, cin + w)
    wb = f16_fast(normal(cout * cin * 9, 92, cout, 1.0 / np.sqrt(9 * cin)))
    b = normal(cout, 93, 0, 0.1)
    got = run_conv(ctx, x, wb, b, batch, cout, cin, h, w)
    for i in range(0, batch, 7):
        want = o.conv3x3s2_gelu(x[i * cin * h * w:(i + 1) * cin * h * w], wb, b, cout, cin, h, w)
        assert_close(got[i], want, rtol=1e-5, atol_rms=1e-5, what=f"conv {cout}x{cin} {h}x{w} image {i}")


@pytest.mark.parametrize("scale", [1e-30, 1e30])
def test_conv_extreme_magnitudes(ctx, scale):
    # One image far from f16's range: the scale follows the input's largest.
    cin, cout, h, w = 32, 64, 9, 8
    x = (normal(cin * h * w, 94, 0) * np.float32(scale)).astype(np.float32)
    wb = f16_fast(normal(cout * cin * 9, 95, 0, 0.1))
    b = np.zeros(cout, np.float32)
    got = run_conv(ctx, x, wb, b, 1, cout, cin, h, w)[0]
    assert_close(got, o.conv3x3s2_gelu(x, wb, b, cout, cin, h, w), rtol=1e-5, atol_rms=1e-5)


def test_conv_non_finite_stays_local(ctx):
    # An inf or NaN reaches the positions whose taps read it, and no others.
    cin, cout, h, w = 16, 32, 16, 16
    x = normal(cin * h * w, 96, 0).reshape(cin, h, w)
    wb = f16_fast(normal(cout * cin * 9, 97, 0, 0.1))
    b = normal(cout, 98, 0, 0.1)
    clean = np.asarray(run_conv(ctx, x.reshape(-1), wb, b, 1, cout, cin, h, w)[0]).reshape(cout, 8, 8)
    bad = x.copy()
    bad[3, 5, 5], bad[9, 10, 2] = np.inf, np.nan
    got = np.asarray(run_conv(ctx, bad.reshape(-1), wb, b, 1, cout, cin, h, w)[0]).reshape(cout, 8, 8)
    touched = np.zeros((8, 8), bool)
    touched[2:4, 2:4] = True   # output rows and columns whose 3 x 3 taps cover 5
    touched[5, 1] = True       # ... and row 10, column 2
    assert np.array_equal(got[:, ~touched], clean[:, ~touched])
    assert np.isnan(got[:, 5, 1]).all() and not (got[:, 2:4, 2:4] == clean[:, 2:4, 2:4]).any()


def test_conv_images_of_different_magnitudes(ctx):
    # An image's result does not depend on the others': each has its own scale.
    cin, cout, h, w = 32, 64, 13, 11
    x = normal(6 * cin * h * w, 99, 0).reshape(6, cin, h, w)
    for i, factor in enumerate((1.0, 1e6, 1e-12, 1e12, 1.0, 1e-30)):
        x[i] *= np.float32(factor)
    x[4, 7, 5, 5] = np.float32(1e20)
    wb = f16_fast(normal(cout * cin * 9, 100, 0, 0.1))
    b = np.zeros(cout, np.float32)
    got = run_conv(ctx, x.reshape(-1), wb, b, 6, cout, cin, h, w)
    for i in (0, 1, 2, 3, 5):
        want = o.conv3x3s2_gelu(x[i].reshape(-1), wb, b, cout, cin, h, w)
        assert_close(got[i], want, rtol=1e-5, atol_rms=1e-5, what=f"image {i}")
        alone = run_conv(ctx, x[i].reshape(-1), wb, b, 1, cout, cin, h, w)
        assert np.array_equal(got[i], alone[0]), i


@pytest.mark.parametrize("outlier", [1e6, 1e9])
def test_conv_outlier_within_an_image(ctx, outlier):
    # A value far above its image: the positions that do not read it keep the
    # 2^-17 that two bf16 terms of each value kept.
    cin, cout, h, w = 32, 64, 16, 16
    x = normal(cin * h * w, 101, 0).reshape(cin, h, w)
    x[3, 5, 5] = np.float32(outlier)
    wb = f16_fast(normal(cout * cin * 9, 102, 0, 0.1))
    b = normal(cout, 103, 0, 0.1)
    got = np.asarray(run_conv(ctx, x.reshape(-1), wb, b, 1, cout, cin, h, w)[0]).reshape(cout, 8, 8)
    want = np.asarray(o.conv3x3s2_gelu(x.reshape(-1), wb, b, cout, cin, h, w)).reshape(cout, 8, 8)
    away = np.ones((8, 8), bool)
    away[2:4, 2:4] = False
    assert_close(got[:, away], want[:, away], rtol=2e-5, atol_rms=2e-5)


def test_conv_runs_of_images(ctx):
    # More images than their terms' scratch holds at once (38 of this shape):
    # the second run's images take their own scales.
    cin, cout, h, w, batch = 480, 32, 64, 50, 40
    two = normal(2 * cin * h * w, 104, 0).reshape(2, cin, h, w)
    two[1] *= np.float32(1e9)
    x = np.concatenate([two] * (batch // 2))
    wb = f16_fast(normal(cout * cin * 9, 105, 0, 1.0 / np.sqrt(9 * cin)))
    b = normal(cout, 106, 0, 0.1)
    got = run_conv(ctx, x.reshape(-1), wb, b, batch, cout, cin, h, w)
    for i in range(2):
        want = o.conv3x3s2_gelu(two[i].reshape(-1), wb, b, cout, cin, h, w)
        for k in (i, 36 + i, 38 + i):
            assert_close(got[k], want, rtol=1e-5, atol_rms=1e-5, what=f"image {k}")
