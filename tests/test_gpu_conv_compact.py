"""The 16-bit COMPACT policy, whose kernel map is built as pair lists: both forms of the map against the oracle, whichever
is asked for first; convs on a built map when no memory is left (a compacted conv needs none; 64 -> 64, which takes the
row table where it fits, then walks the lists); the mesh extraction, which reads the row table; and features past the
2 GiB that AUTO's kernels address.

Tolerance where two schedules are compared: they differ by the order of their fp32 sums and one unit in the last place of
the storage type where those fall on either side of a tie (2^-7 of the value in bf16, 2^-10 in fp16; 1e-4 for the sums)."""
import math

import numpy as np
import pytest

import oracle_lib as orc
import sparse_hip as sh
import workloads as wl

pytestmark = pytest.mark.gpu

TOL = {sh.BF16: 2.0 ** -7 + 1e-4, sh.F16: 2.0 ** -10 + 1e-4}


def shell(n, repeated=0):
    coords = wl.make_coords(1)[:n - repeated]
    return np.ascontiguousarray(np.concatenate([coords, coords[:repeated]]))


@pytest.mark.parametrize("algo", [sh.CONV_AUTO, sh.CONV_COMPACT])
@pytest.mark.parametrize("lists_first", [False, True])
@pytest.mark.parametrize("n,repeated", [(1, 0), (63, 0), (256, 0), (257, 100), (1000, 0), (5003, 7)])
def test_both_forms_of_the_map(n, repeated, lists_first, algo):
    be = sh.Backend(0, sh.BF16, conv_algo=algo)
    coords = shell(n, repeated)
    rb = be.build_rulebook(coords)
    nbr = None if lists_first else be.neighbors(rb)
    counts, src, dst = be.pairs(rb)
    nbr = be.neighbors(rb) if nbr is None else nbr
    exp = orc.Rulebook(coords).neighbors()
    assert np.array_equal(nbr, exp)
    assert np.array_equal(counts, (exp >= 0).sum(0))
    at = 0
    for k in range(27):
        rows = np.flatnonzero(exp[:, k] >= 0)
        assert np.array_equal(dst[at:at + rows.size], rows) and np.array_equal(src[at:at + rows.size], exp[rows, k])
        at += rows.size
    assert be.rulebook_stats(rb)["pairs"] == at
    rb.free()
    be.destroy()


@pytest.mark.parametrize("dtype", [sh.BF16, sh.F16])
@pytest.mark.parametrize("n,ci,co", [(1, 64, 64), (1000, 64, 64), (257, 128, 128), (3000, 256, 256), (700, 64, 16)])
def test_built_map_needs_no_memory(n, ci, co, dtype):
    """Every allocation fails between the map and the conv.  64 -> 64 gives AUTO's bits where the rows fit."""
    rng = np.random.default_rng(n + co)
    coords = shell(n)
    x = rng.standard_normal((n, ci)).astype(np.float32)
    w = sh.storage_round(rng.standard_normal((co, 27, ci)) / math.sqrt(27 * ci), dtype)
    y = []
    for algo, starved in ((sh.CONV_AUTO, False), (sh.CONV_COMPACT, False), (sh.CONV_COMPACT, True)):
        be = sh.Backend(0, dtype, conv_algo=algo)
        wk = be.keep(w)
        xb, yb = be.upload(x), be.alloc(n * co)
        if starved:
            be.conv(be.build_rulebook(coords), xb, wk, None, yb, ci, co)  # the weights' device copy
        rb = be.build_rulebook(coords)
        if starved:
            be.trim(sh.TRIM_FREE_BUFFERS)
            be.fail_alloc(0)
        try:
            be.conv(rb, xb, wk, None, yb, ci, co)
        finally:
            be.fail_alloc(-1)
        y.append(be.download(yb))
        rb.free()
        be.destroy()
    if ci == 64 and co == 64:
        assert np.array_equal(y[0], y[1])
    else:
        assert np.array_equal(y[1], y[2])
    assert np.max(np.abs(y[2] - y[0]) / np.maximum(1.0, np.abs(y[0]))) <= TOL[dtype]


def test_mesh():
    rng = np.random.default_rng(0)
    coords = shell(5000)
    logits = rng.standard_normal((5000, 7)).astype(np.float32)
    mesh = []
    for algo in (sh.CONV_AUTO, sh.CONV_COMPACT):
        be = sh.Backend(0, sh.BF16, conv_algo=algo)
        mesh.append(be.flex_dual_grid_mesh(be.upload(logits), 5000, 7, 64, coords=coords))
        be.destroy()
    assert mesh[0][1].shape[0] > 0
    assert np.array_equal(mesh[0][0], mesh[1][0]) and np.array_equal(mesh[0][1], mesh[1][1])


def test_features_past_2_gib():
    """524,300 rows of 2,048 fp16 channels are more than the sorted conv's and the GEMM's loads address: the conv takes the
    compacted kernel, the linear the MFMA linear kernel.  Rows repeat a block of 1,000, and sampled outputs, among them
    rows whose sources lie past 2 GiB, are compared with 64-bit sums over their neighbours."""
    dtype, ci, co, n = sh.F16, 2048, 16, 524300
    rng = np.random.default_rng(1)
    c = np.ascontiguousarray(wl.make_coords(4)[:n])
    block = sh.storage_round(rng.standard_normal((1000, ci)), dtype)
    raw = np.concatenate([np.tile(block.astype(np.float16), (n // 1000, 1)), block[:n % 1000].astype(np.float16)])
    w = sh.storage_round(rng.standard_normal((co, 27, ci)) / math.sqrt(27 * ci), dtype)
    lw = sh.storage_round(rng.standard_normal((128, ci)) / math.sqrt(ci), dtype)
    be = sh.Backend(0, dtype, linear_algo=sh.LINEAR_KERNEL)
    xb, yb, zb = be.upload_raw(raw.view(np.uint16)), be.alloc(n * co), be.alloc(n * 128)
    rb = be.build_rulebook(c)
    be.conv(rb, xb, w, None, yb, ci, co)
    be.linear(xb, lw, None, zb, n, ci, 128)
    y, z = be.download(yb).reshape(n, co), be.download(zb).reshape(n, 128)
    rb.free()
    be.destroy()
    rows = np.unique(np.concatenate([np.arange(0, n, 3001), np.arange(n - 64, n)]))
    nbr = orc.Rulebook(c).neighbors()[rows]
    exp = np.zeros((rows.size, co))
    for k in range(27):
        has = nbr[:, k] >= 0
        exp[has] += block[nbr[has, k] % 1000].astype(np.float64) @ w[:, k].T.astype(np.float64)
    for got, want in ((y[rows], exp), (z[rows], block[rows % 1000].astype(np.float64) @ lw.T.astype(np.float64))):
        assert np.max(np.abs(got - want) / np.maximum(1.0, np.abs(want))) <= TOL[dtype]
