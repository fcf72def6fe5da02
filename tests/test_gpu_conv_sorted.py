"""The AUTO policy's 16-bit conv (rows in their own order, and in mask order) where it can go wrong: the edges of its row
blocks, every block shape (16 to 256 channels; small sets and sets that fill the GPU), repeated coordinates, more rows
than one sort window, no memory for the order, and weights that are not finite.

Tolerance: both sides compute on the same rounded inputs, so they differ by their fp32 summation orders (some 1e-6 to
1e-5 here; 1e-4 allowed) and by the one rounding to the storage type.  Sums on either side of a tie round to
neighbouring values, one unit in the last place apart: of values with 8 (bf16) and 11 (fp16) significant bits that is
at most 2^-7 and 2^-10 of the value."""
import math

import numpy as np
import pytest

import oracle_lib as orc
import sparse_hip as sh
import workloads as wl

pytestmark = pytest.mark.gpu

TOL = {sh.BF16: 2.0 ** -7 + 1e-4, sh.F16: 2.0 ** -10 + 1e-4}


@pytest.fixture(scope="module")
def backends():
    bes = {dt: sh.Backend(0, dt) for dt in (sh.BF16, sh.F16)}
    yield bes
    for b in bes.values():
        b.destroy()


def err(got, exp):
    return float(np.max(np.abs(got - exp) / np.maximum(1.0, np.maximum(np.abs(got), np.abs(exp)))))


def weights(rng, ci, co, dtype):
    return sh.storage_round(rng.standard_normal((co, 27, ci)) / math.sqrt(27 * ci), dtype)


ORDER_WORK = 4e9  # rows x input x output channels of the convs on a rulebook, from which they take its rows in mask order


def reach_order(be, rb):
    """Runs convs on a rulebook until the next one takes its rows in mask order."""
    ci, co = (64, 64) if rb.n >= 4096 else (256, 1024)
    xb, yb = be.upload(np.ones((rb.n, ci), np.float32)), be.alloc(rb.n * co)
    w = be.keep(np.zeros((co, 27, ci), np.float32))
    for _ in range(math.ceil(ORDER_WORK / (rb.n * ci * co))):
        be.conv(rb, xb, w, None, yb, ci, co)
    be.synchronize()


def run(be, coords, x, w, b, ci, co):
    """One conv on a fresh rulebook, and again with the rows in mask order: the same bits."""
    n = coords.shape[0]
    rb = be.build_rulebook(coords)
    xb, yb, zb = be.upload(x), be.alloc(n * co), be.alloc(n * co)
    w, b = be.keep(w), None if b is None else be.keep(b)
    be.conv(rb, xb, w, b, zb, ci, co)
    reach_order(be, rb)
    be.conv(rb, xb, w, b, yb, ci, co)
    rb.free()
    assert np.array_equal(be.download_raw(yb), be.download_raw(zb))
    return be.download(yb).reshape(n, co)


def shell(n):
    return np.ascontiguousarray(wl.make_coords(1)[:n])


@pytest.mark.parametrize("n", [1, 15, 64, 65, 127, 129, 255, 257, 1000])
@pytest.mark.parametrize("ci,co", [(64, 16), (128, 32), (64, 64), (192, 64), (64, 128), (128, 192), (256, 256),
                                   (128, 384)])
def test_block_edges(backends, n, ci, co):
    dtype = sh.BF16 if n % 2 else sh.F16
    rng = np.random.default_rng(n * 7 + ci + co)
    coords = shell(n)
    x = sh.storage_round(rng.standard_normal((n, ci)), dtype)
    w, b = weights(rng, ci, co, dtype), (0.1 * rng.standard_normal(co)).astype(np.float32)
    y = run(backends[dtype], coords, x, w, b, ci, co)
    assert err(y, sh.storage_round(orc.Rulebook(coords).conv(x, w, b, ci, co), dtype)) <= TOL[dtype]


@pytest.mark.parametrize("n", [1, 31, 63, 64, 65, 127, 128, 129, 1000])
@pytest.mark.parametrize("ci,co", [(32, 16), (96, 32), (32, 64), (96, 128), (160, 192)])
def test_masked_block_edges(backends, n, ci, co):
    """The widths beside the sorted kernel's (odd multiples of 32), on the masked kernel."""
    dtype = sh.BF16 if n % 2 else sh.F16
    rng = np.random.default_rng(n * 7 + ci + co)
    coords = shell(n)
    x = sh.storage_round(rng.standard_normal((n, ci)), dtype)
    w, b = weights(rng, ci, co, dtype), (0.1 * rng.standard_normal(co)).astype(np.float32)
    y = run(backends[dtype], coords, x, w, b, ci, co)
    assert err(y, sh.storage_round(orc.Rulebook(coords).conv(x, w, b, ci, co), dtype)) <= TOL[dtype]


# Row counts that take each block shape at 256 and 128 channels (64 x 64 up to 256 x 256), sampled rows.
@pytest.mark.parametrize("ci,co,n", [(64, 256, 3000), (64, 256, 9000), (64, 256, 14648), (64, 512, 14648),
                                     (64, 1024, 6000), (64, 1024, 8100), (64, 1024, 9000), (64, 1024, 12000),
                                     (64, 1024, 14000), (64, 1024, 14648), (64, 128, 3000), (128, 128, 14648)])
def test_block_shapes(backends, ci, co, n):
    dtype = sh.BF16
    rng = np.random.default_rng(n + ci + co)
    coords = shell(n)
    coords = np.ascontiguousarray(coords[rng.permutation(n)])
    x = sh.storage_round(rng.standard_normal((n, ci)), dtype)
    w = weights(rng, ci, co, dtype)
    y = run(backends[dtype], coords, x, w, None, ci, co)
    step = 97
    exp = orc.Rulebook(coords).conv(x, w, None, ci, co, rows=(0, n, step))
    assert err(y[::step], sh.storage_round(exp, dtype)) <= TOL[dtype]


@pytest.mark.parametrize("ci,co", [(64, 64), (128, 128)])
def test_repeated_coordinates(backends, ci, co):
    """Every row of a repeated voxel has the last one as its centre neighbour."""
    dtype = sh.F16
    rng = np.random.default_rng(5)
    coords = shell(900)
    coords = np.ascontiguousarray(np.concatenate([coords, coords[::3], coords[::7]]))
    n = coords.shape[0]
    x = sh.storage_round(rng.standard_normal((n, ci)), dtype)
    w = weights(rng, ci, co, dtype)
    y = run(backends[dtype], coords, x, w, None, ci, co)
    assert err(y, sh.storage_round(orc.Rulebook(coords).conv(x, w, None, ci, co), dtype)) <= TOL[dtype]


@pytest.mark.parametrize("n,ci,co", [(1, 64, 64), (700, 64, 16), (1000, 128, 32), (5000, 64, 192), (9001, 128, 128),
                                     (14648, 64, 512)])
def test_no_memory_for_the_order(n, ci, co):
    """A conv on a built rulebook whose mask order cannot be allocated (every allocation fails) takes the rows in their own
    order.  A row's sums do not depend on which rows it shares blocks with: the same bits.  Tolerance: none."""
    dtype = sh.BF16 if n % 2 else sh.F16
    be = sh.Backend(0, dtype)
    rng = np.random.default_rng(n)
    coords = np.ascontiguousarray(shell(n)[rng.permutation(n)])
    x = rng.standard_normal((n, ci)).astype(np.float32)
    w, b = be.keep(weights(rng, ci, co, dtype)), be.keep((0.1 * rng.standard_normal(co)).astype(np.float32))
    xb, yb, zb = be.upload(x), be.alloc(n * co), be.alloc(n * co)
    wide = be.keep(np.zeros((1024, 27, 1024), np.float32))
    wx, wy = be.upload(np.zeros((n, 1024), np.float32)), be.alloc(n * 1024)
    be.conv(be.build_rulebook(coords), wx, wide, None, wy, 1024, 1024)  # its weights
    for out, starved in ((yb, False), (zb, True)):
        rb = be.build_rulebook(coords)
        be.profile(True)
        be.profile_read()
        if starved:
            be.trim(sh.TRIM_FREE_BUFFERS)
            be.fail_alloc(0)
        try:
            for _ in range(math.ceil(ORDER_WORK / (n * 1024 * 1024)) - 1):
                be.conv(rb, wx, wide, None, wy, 1024, 1024)
            assert be.profile_read()["map"][1] == 0  # not yet
            be.conv(rb, wx, wide, None, wy, 1024, 1024)
            be.conv(rb, xb, w, b, out, ci, co)
        finally:
            be.fail_alloc(-1)
        assert be.profile_read()["map"][1] == (0 if starved else 1)
        be.profile(False)
        rb.free()
    assert np.array_equal(be.download_raw(yb), be.download_raw(zb))
    be.destroy()


def test_more_rows_than_a_sort_window(backends):
    """419,340 rows (the sort takes 262,144 at a time), 64 -> 128: sampled rows in every part."""
    dtype = sh.BF16
    rng = np.random.default_rng(9)
    coords = wl.make_coords(2)
    n, ci, co = coords.shape[0], 64, 128
    x = sh.storage_round(rng.standard_normal((n, ci), dtype=np.float32), dtype)
    w = weights(rng, ci, co, dtype)
    y = run(backends[dtype], coords, x, w, None, ci, co)
    exp = orc.Rulebook(coords).conv(x, w, None, ci, co, rows=(0, n, 1009))
    assert err(y[::1009], sh.storage_round(exp, dtype)) <= TOL[dtype]


@pytest.mark.parametrize("c", [128, 256, 512])
def test_block_repeats_bit_for_bit(backends, c):
    """A whole ConvNeXt block on rulebooks built anew, in row order and in mask order, whose ties among rows of one bucket
    fall as the atomics do: the same bits each time."""
    dtype = sh.BF16
    be = backends[dtype]
    rng = np.random.default_rng(c)
    coords = np.ascontiguousarray(wl.make_coords(2)[:30000])
    n = coords.shape[0]
    x = be.upload(rng.standard_normal((n, c), dtype=np.float32))
    w, w0, w2 = (be.keep(np.ascontiguousarray(a, np.float32)) for a in
                 (weights(rng, c, c, dtype), rng.standard_normal((4 * c, c)) / math.sqrt(c),
                  rng.standard_normal((c, 4 * c)) / math.sqrt(4 * c)))
    got = []
    for _ in range(3):
        rb = be.build_rulebook(coords)
        for ordered in (False, True):
            if ordered:
                reach_order(be, rb)
            y = be.alloc(n * c)
            be.convnext_block(rb, x, w, None, None, None, w0, None, w2, None, y, c, 1e-6)
            got.append(be.download_raw(y))
        rb.free()
    for g in got[1:]:
        assert np.array_equal(g, got[0])


@pytest.mark.parametrize("algo", [sh.CONV_AUTO, sh.CONV_MASKED, sh.CONV_COMPACT])
@pytest.mark.parametrize("ci,co", [(64, 64), (128, 128), (192, 64), (320, 16), (96, 128)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_weights_that_are_not_finite(ci, co, bad, algo):
    """A weight of one offset that is not finite reaches only rows with a neighbour there, as in the reference, whichever
    schedule the policy and the shape lead to."""
    dtype = sh.BF16
    be = sh.Backend(0, dtype, conv_algo=algo)
    rng = np.random.default_rng(ci)
    coords = shell(700)
    x = sh.storage_round(rng.standard_normal((700, ci)), dtype)
    w = weights(rng, ci, co, dtype)
    w[3, 2, 5] = bad
    y = run(be, coords, x, w, None, ci, co)
    be.destroy()
    nbr = orc.Rulebook(coords).neighbors()
    has = nbr[:, 2] >= 0
    assert has.any() and not has.all()
    exp = sh.storage_round(orc.Rulebook(coords).conv(x, w, None, ci, co), dtype)
    other = np.arange(co) != 3
    assert err(y[:, other], exp[:, other]) <= TOL[dtype]
    assert not np.isfinite(y[has, 3]).any()
    assert err(y[~has, 3], exp[~has, 3]) <= TOL[dtype]
