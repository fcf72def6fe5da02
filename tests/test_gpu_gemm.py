"""The linear slots' GEMM kernel (16-bit, Ci = 64 or Ci % 128 == 0, Co % 128 == 0; policy LINEAR_KERNEL) at the edges of
its row blocks and in each block shape, plain, with SiLU, and with the residual of the composed ConvNeXt tail; and widths
beside it, which keep fp32 weights.

Tolerance: against the oracle's linear on the same rounded inputs the fp32 sums differ by their order (some 1e-6; 1e-4
allowed) and the rounding to the storage type by one unit in the last place where they fall on either side of a tie
(2^-7 of the value in bf16, 2^-10 in fp16); SiLU's hardware exponential and reciprocal add about 2^-20."""
import math

import numpy as np
import pytest

import oracle_lib as orc
import sparse_hip as sh

pytestmark = pytest.mark.gpu

TOL = {sh.BF16: 2.0 ** -7 + 1e-4, sh.F16: 2.0 ** -10 + 1e-4}


@pytest.fixture(scope="module")
def backends():
    bes = {dt: sh.Backend(0, dt, linear_algo=sh.LINEAR_KERNEL) for dt in (sh.BF16, sh.F16)}
    yield bes
    for b in bes.values():
        b.destroy()


@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("n,ci,co", [(1, 64, 128), (63, 128, 256), (64, 192, 128), (129, 64, 384), (257, 320, 256),
                                     (5003, 64, 256), (20000, 64, 512), (33000, 64, 256), (131080, 64, 128),
                                     (5003, 512, 512), (41000, 64, 256), (131080, 64, 512), (524300, 64, 128)])
def test_linear_vs_oracle(backends, n, ci, co, silu):
    dtype = sh.F16 if n % 2 else sh.BF16
    be = backends[dtype]
    rng = np.random.default_rng(n + ci + co + silu)
    x = sh.storage_round(rng.standard_normal((n, ci), dtype=np.float32), dtype)
    w = sh.storage_round(rng.standard_normal((co, ci)) / math.sqrt(ci), dtype)
    b = (0.1 * rng.standard_normal(co)).astype(np.float32)
    xb, yb = be.upload(x), be.alloc(n * co)
    be.linear(xb, w, b, yb, n, ci, co, silu=silu)
    got = be.download(yb).reshape(n, co)
    rows = np.unique(np.concatenate([np.arange(min(n, 130)), np.arange(max(0, n - 130), n), rng.integers(0, n, 200)]))
    exp = sh.storage_round(orc.linear(x[rows], w, b, rows.size, ci, co, silu=silu), dtype)
    e = np.max(np.abs(got[rows] - exp) / np.maximum(1.0, np.abs(exp)))
    assert e <= TOL[dtype]


@pytest.mark.parametrize("algo", [sh.LINEAR_AUTO, sh.LINEAR_KERNEL])
@pytest.mark.parametrize("n,ci,co", [(1, 192, 128), (300, 192, 256), (257, 320, 128), (64, 448, 384)])
@pytest.mark.parametrize("dtype", [sh.BF16, sh.F16])
def test_weights_between_the_mfma_widths_stay_fp32(n, ci, co, dtype, algo):
    """Ci = 192, 320, 448: features 1, -1, 1, ... times weights 1 + 2^-12, 1, 1 + 2^-12, ... sum to ci / 2 * 2^-12, exact in
    fp32 in any order and in both storage types; weights rounded to 8 or 11 bits would give 0.  Tolerance: none."""
    be = sh.Backend(0, dtype, linear_algo=algo)
    x = np.tile(np.array([1, -1], np.float32), (n, ci // 2))
    w = np.tile(np.array([1 + 2.0 ** -12, 1], np.float32), (co, ci // 2))
    xb, yb = be.upload(x), be.alloc(n * co)
    be.linear(xb, w, None, yb, n, ci, co)
    assert np.all(be.download(yb) == ci // 2 * 2.0 ** -12)
    be.destroy()


@pytest.mark.parametrize("n", [1, 257, 12000, 12001])
def test_convnext_tail_256_vs_oracle(backends, n):
    """The ConvNeXt tail at C = 256 on both sides of the row count where the fused kernel takes over from row_norm and two
    GEMMs, and below it on the fused kernel too, which runs where the intermediates cannot be allocated (their allocation
    is made to fail) and where eps = 0.  Rounded where the slots store, the two routes differ by the order of fp32 sums: an
    intermediate one unit apart here and there (of 256 or 1,024 summed), then the last roundings of the second linear and
    the add, 2^-7 each in bf16 and 2^-10 in fp16; 2^-8 (2^-11) more for the intermediates."""
    c = 256
    dtype = sh.F16 if n % 2 else sh.BF16
    tol = 2.5 * TOL[dtype]
    be = backends[dtype]
    rng = np.random.default_rng(n)
    rnd = lambda a: sh.storage_round(a, dtype)
    x, res = rnd(rng.standard_normal((n, c))), rnd(rng.standard_normal((n, c)))
    gamma, beta = (1 + 0.1 * rng.standard_normal(c)).astype(np.float32), np.zeros(c, np.float32)
    w0, w2 = rnd(rng.standard_normal((4 * c, c)) / 16), rnd(rng.standard_normal((c, 4 * c)) / 32)
    b0, b2 = (0.1 * rng.standard_normal(4 * c)).astype(np.float32), (0.1 * rng.standard_normal(c)).astype(np.float32)
    rows = np.unique(np.concatenate([np.arange(min(n, 140)), np.arange(max(0, n - 140), n)]))
    e = rnd(orc.row_norm(x[rows], gamma, beta, rows.size, c, 1e-6))
    e = rnd(orc.linear(e, w0, b0, rows.size, c, 4 * c, silu=True))
    e = rnd(orc.add(res[rows], rnd(orc.linear(e, w2, b2, rows.size, 4 * c, c))))
    xb, rb, yb = be.upload(x), be.upload(res), be.alloc(n * c)

    def check(eps, allocs=-1):
        be.fail_alloc(allocs)
        try:
            be.convnext_mlp(xb, gamma, beta, w0, b0, w2, b2, rb, yb, n, c, eps)
        finally:
            be.fail_alloc(-1)
        got = be.download(yb).reshape(n, c)[rows]
        assert sh.LIB.trellis_sparse_hip_last_error(be.ptr) == b""
        assert np.max(np.abs(got - e) / np.maximum(1.0, np.abs(e))) <= tol

    check(1e-6)
    check(0.0)  # the rows' variances are near 1: the same result
    be.trim(sh.TRIM_FREE_BUFFERS)
    check(1e-6, allocs=0)
