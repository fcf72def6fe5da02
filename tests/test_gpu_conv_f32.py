"""The fp32 conv, bit for bit the reference's operation order: every rows-per-wavefront variant (by row and channel
counts), ragged row counts, output channels that do not fill a 64-channel block, input channels in several chunks,
scattered rows (blocks with few offsets), and the shapes that keep the general kernel (Ci % 32 or Co % 4 not 0).
Tolerance: none."""
import math

import numpy as np
import pytest

import oracle_lib as orc
import sparse_hip as sh
import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    b = sh.Backend(0, sh.F32)
    yield b
    b.destroy()


@pytest.mark.parametrize("n,ci,co", [(1, 32, 4), (3, 32, 64), (17, 96, 100), (63, 64, 64), (65, 64, 132), (1000, 32, 36),
                                     (6999, 32, 64), (9001, 32, 64), (14648, 32, 64), (14645, 32, 320), (700, 40, 64),
                                     (700, 64, 30)])
def test_conv_f32_bit_identical(be, n, ci, co):
    rng = np.random.default_rng(n + ci + co)
    coords = np.ascontiguousarray(wl.make_coords(1)[:n])
    x = rng.standard_normal((n, ci), dtype=np.float32)
    w = (rng.standard_normal((co, 27, ci)) / math.sqrt(27 * ci)).astype(np.float32)
    b = (0.1 * rng.standard_normal(co)).astype(np.float32)
    rb = be.build_rulebook(coords)
    xb, yb = be.upload(x), be.alloc(n * co)
    step = 1 if n * co < 500000 else 61
    for bias in (b, None):
        be.conv(rb, xb, w, bias, yb, ci, co)
        exp = orc.Rulebook(coords).conv(x, w, bias, ci, co, rows=(0, n, step))
        assert np.array_equal(be.download(yb).reshape(n, co)[::step], exp)
    rb.free()


@pytest.mark.parametrize("n,ci,co,side", [(1, 32, 64, 1), (2, 96, 64, 2), (5, 64, 20, 3), (33, 64, 64, 8), (1000, 32, 64, 40),
                                          (8000, 96, 64, 70), (13000, 32, 64, 60), (14000, 64, 320, 120)])
def test_conv_f32_scattered_rows(be, n, ci, co, side):
    """Random voxels of a cube, repeated ones among them: blocks whose rows have neighbours at some offsets only."""
    rng = np.random.default_rng(n)
    coords = np.concatenate([np.zeros((n, 1), np.int64), rng.integers(0, side, (n, 3))], 1).astype(np.int32)
    x = rng.standard_normal((n, ci), dtype=np.float32)
    w = (rng.standard_normal((co, 27, ci)) / math.sqrt(27 * ci)).astype(np.float32)
    b = (0.1 * rng.standard_normal(co)).astype(np.float32)
    rb = be.build_rulebook(coords)
    xb, yb = be.upload(x), be.alloc(n * co)
    step = 1 if n * co < 500000 else 61
    be.conv(rb, xb, w, b, yb, ci, co)
    exp = orc.Rulebook(coords).conv(x, w, b, ci, co, rows=(0, n, step))
    assert np.array_equal(be.download(yb).reshape(n, co)[::step], exp)
    rb.free()
