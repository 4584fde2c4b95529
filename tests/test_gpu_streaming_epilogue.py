"""How the streaming kernel starts and ends a tile: K of one to five pairs of slices (as many as it requests ahead, fewer, more),
both tile widths, whole tiles and ragged ones at the lines where the dispatch takes them, and C as its rows in LDS are handed out -
row-major on and off 16-byte boundaries, by columns, read and not, with every step behind the product. int8, so that all of it is
exact and compared bit for bit with the product in int64; the values behind alpha = 0x01010101 use all 32 bits."""
import numpy as np
import pytest

import support
from gpu_support import run_fused_gemm
from support import GemmCase
from test_oracle_gemm import fused_expectation

pytestmark = pytest.mark.gpu

SHORT = (128, 256, 384, 512, 640)
# 136 tiles of 256 x 128, 208 of 256 x 256; 180 and 208 ragged ones (360 and 832 of 128 x 128, 70 and 81 per cent of a round), and a
# little below and above the line for 256 x 128 ones where C is read (280 and 306 of 512)
SIZES = ((4352, 1024, SHORT), (4096, 3328, SHORT), (2300, 2500, (528, 1040, 2064, 4112, 656)), (4001, 3300, (528, 2064, 1072, 1040, 4112)),
         (2500, 1790, (528, 2064, 528, 4112, 656)), (2300, 2070, (528, 2064, 656, 4112, 1040)))


def matrix(x, rows, run, ld):
    return np.lib.stride_tricks.as_strided(x, (rows, run), (ld * x.itemsize, x.itemsize))


@pytest.mark.parametrize("a_kc,b_kc", ((True, True), (True, False), (False, False), (False, True)))
@pytest.mark.parametrize("m,n,ks", SIZES)
def test_streamed_tiles_from_short_to_longer_k(gpu, m, n, ks, a_kc, b_kc):
    rng = np.random.default_rng(m + 2 * a_kc + b_kc)
    for i, k in enumerate(ks):
        by_columns, pad, beta = i % 4 == 2, (0, 3, 5, 4, 1)[i], (0, -77, 1, 0, 3)[i]
        lda, ldb = k if a_kc else -(-m // 16) * 16, k if b_kc else -(-n // 16) * 16
        rsc, csc = (1, m + pad) if by_columns else (n + pad, 1)
        case = GemmCase("i8", None, (1, 0x01010101, -3, 7, 2)[i], beta, m0=1, n0=1, k0=1, m1=m, n1=n, k1=k, rsa0=0, csa0=0,
                        rsa1=lda if a_kc else 1, csa1=1 if a_kc else lda, rsb0=0, csb0=0, rsb1=1 if b_kc else ldb, csb1=ldb if b_kc else 1,
                        rsc0=0, csc0=0, rsc1=rsc, csc1=csc)
        a, b, c = case.make_inputs(k + n)
        c[:] = rng.integers(-2 ** 31, 2 ** 31, size=c.size)
        x = matrix(a, m, k, lda) if a_kc else matrix(a, k, m, lda).T
        y = matrix(b, n, k, ldb).T if b_kc else matrix(b, k, n, ldb)
        rows = support.blocked_offsets(case.m1, case.n1, case.m0, case.n0, case.rsc0, case.csc0, case.rsc1, case.csc1)
        sums = (x.astype(np.float64) @ y.astype(np.float64)).astype(np.int64).reshape(rows.shape)
        plain = c.copy()
        plain[rows] = (case.alpha * sums + beta * c[rows].astype(np.int64)).astype(np.int32)
        bias = rng.integers(-1 << 12, 1 << 12, n).astype(np.int32) if i % 2 else None
        start = np.array([-1 << 30], np.int32) if i >= 3 else None
        act, rq = int(i == 3 or i == 2), None
        if i >= 2:
            rsq, csq = (1, m + 3) if i == 4 else (n + 4 * (i == 3), 1)
            rq = dict(q=np.full((m - 1) * rsq + (n - 1) * csq + 1, 0x55, np.int8), rsq=rsq, csq=csq, per_column=bool(i % 2),
                      scale=(rng.uniform(0.25, 2.0, n if i % 2 else 1) * 100.0 / 2.0 ** 31).astype(np.float32), zero=i, only=False, format=0)
        out = run_fused_gemm(gpu, "rc", case, a, b, c, bias, start, "device", activation=act, requant=rq)
        want = fused_expectation(case, plain, bias, start, activation=act, requant=rq)
        assert np.array_equal(out[0], want[0]), (k, vars(case))
        assert start is None or out[1][0] == want[1][0], k
        assert rq is None or np.array_equal(out[2], want[2]), k


@pytest.mark.parametrize("m,n,k", ((4096, 3328, 256), (4352, 1024, 384), (2300, 2500, 4112), (4001, 3300, 2064), (2304, 3584, 128)))
def test_int8_copies_in_dwords(gpu, m, n, k):
    """The loop of its own that such copies have where C is not read: whole tiles of both widths and ragged ones (rows and columns that
    end inside a tile, in a chunk and in a lane's dword's neighbour), with C and without, scalars of one and others, ReLU and none, one
    scale and one per column, with a bias and without, rows of the copy farther apart than they are long."""
    rng = np.random.default_rng(m + n)
    for i in range(4):
        alpha, act, only, per_column, pad = (1, 0x01010101, 1, -3)[i], i & 1, i >= 2, i in (1, 2), (0, 4, 8, 12)[i]
        case = GemmCase("i8", None, alpha, 0, m0=1, n0=1, k0=1, m1=m, n1=n, k1=k, rsa0=0, csa0=0, rsa1=k, csa1=1, rsb0=0, csb0=0, rsb1=1, csb1=k,
                        rsc0=0, csc0=0, rsc1=n + pad // 4, csc1=1)
        a, b, c = case.make_inputs(k + n + i)
        sums = (matrix(a, m, k, k).astype(np.float64) @ matrix(b, n, k, k).T.astype(np.float64)).astype(np.int64)
        rows = support.blocked_offsets(case.m1, case.n1, case.m0, case.n0, case.rsc0, case.csc0, case.rsc1, case.csc1)
        plain = c.copy()
        plain[rows] = (alpha * sums.reshape(rows.shape)).astype(np.int32)
        bias = rng.integers(-1 << 12, 1 << 12, n).astype(np.int32) if i != 3 else None
        spread = 2.0 ** 31 if abs(alpha) > 3 else 40.0 * 5461.0 * np.sqrt(k)
        rq = dict(q=np.full((m - 1) * (n + pad) + n, 0x55, np.int8), rsq=n + pad, csq=1, per_column=per_column,
                  scale=(rng.uniform(0.25, 2.0, n if per_column else 1) * 4000.0 / spread).astype(np.float32), zero=(0, -128, 127, 5)[i], only=only, format=0)
        out = run_fused_gemm(gpu, "rc", case, a, b, c, bias, None, "device", activation=act, requant=rq)
        want = fused_expectation(case, plain, bias, None, activation=act, requant=rq)
        assert np.array_equal(out[0], c if only else want[0]) and np.array_equal(out[2], want[2]), (i, vars(case))
