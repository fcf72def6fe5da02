"""The linear slots' GEMM kernel (16-bit, Ci % 64 == 0, Co % 128 == 0; policy LINEAR_KERNEL) at the edges of its row
blocks and in each block shape, plain, with SiLU, and with the residual of the composed ConvNeXt tail.

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
                                     (5003, 64, 256), (20000, 64, 512), (33000, 64, 256), (131080, 64, 128)])
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
