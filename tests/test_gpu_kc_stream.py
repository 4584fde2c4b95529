"""Decode batches against weights with K contiguous, streamed through LDS a line of every column at a time (skl_gemv_kcrows.hip,
skl_gemv_f4.hip): the sizes at which the ring, the row groups and the column groups begin and end."""
import numpy as np
import pytest

import ctypes as ct

import ofp4_support as f4
import skl_amd
import support
from gpu_support import run_fused_gemm, run_gemm
from support import GemmCase, run_oracle_gemm
from test_dispatch_rules import BF16, E4M3, F16, I8, streams_k_contiguous
from test_gpu_ofp4 import run as run_ofp4

pytestmark = pytest.mark.gpu


def _case(ta, m, n, k, alpha, beta, pad=0):
    """Row-major A, B with column j at j * (k + pad), row-major C."""
    return GemmCase(ta, None, alpha, beta, m0=1, n0=1, k0=1, m1=m, n1=n, k1=k, rsa0=0, csa0=0, rsa1=k + pad, csa1=1,
                    rsb0=0, csb0=0, rsb1=1, csb1=k + pad, rsc0=0, csc0=0, rsc1=n + 3, csc1=1)


KINDS = {"i8": I8, "bf16": BF16, "f16": F16, "f8e4m3": E4M3}


# K in bytes: one piece short of a line, one more than the ring holds for every wave, the last unit one piece long, fewer units
# than waves; N: one to four column groups (from 4097, 8193 and 12289 columns on), the last one and its last group ragged
@pytest.mark.parametrize("ta", ("i8", "bf16", "f16", "f8e4m3"))
@pytest.mark.parametrize("m,n,k_bytes", ((2, 9500, 112), (16, 4099, 4112), (17, 1031, 2064), (33, 12303, 1040), (48, 8193, 272), (33, 12303, 4112), (48, 8193, 2832),
                                         (65, 700, 1536), (96, 12305, 144), (5, 2051, 1 << 13)))
def test_edges(gpu, ta, m, n, k_bytes):
    k = k_bytes // (2 if ta in ("bf16", "f16") else 1)
    tiles = ta in ("bf16", "f16") and (m, k_bytes) in ((33, 1040), (48, 272))  # a short K of 16 bits: on the tile kernels
    assert streams_k_contiguous(KINDS[ta], m, n, k) != tiles
    for alpha, beta, pad in ((1, 0, 0), (-3, 2, 16)):
        case = _case(ta, m, n, k, alpha, beta, pad)
        a, b, c = case.make_inputs(m * 1009 + n + k)
        got = run_gemm(gpu, "rc", case, a, b, c, "device")
        if case.is_int:
            assert np.array_equal(got, run_oracle_gemm(case, a, b, c))
        else:
            support.assert_fp_gemm_close(case, a, b, c, got)
            assert np.array_equal(got.view(np.uint8), run_gemm(gpu, "rc", case, a, b, c, "device").view(np.uint8))


@pytest.mark.parametrize("ta", ("bf16", "f16"))
def test_rows_beyond_m_and_k_beyond_the_row_are_not_read(gpu, ta):
    """Padding between the rows of A and the columns of B is NaN: none of it reaches the product."""
    m, n, k, pad = 18, 4100, 1048, 24
    case = _case(ta, m, n, k, 1.0, 0.0, pad)
    a, b, c = case.make_inputs(77)
    want = run_gemm(gpu, "rc", case, a, b, c, "device")
    nan = np.uint16(0x7FFF)
    a, b = a.copy(), b.copy()
    for x, rows in ((a, m), (b, n)):
        bits = x.view(np.uint16)
        for i in range(rows):
            bits[i * (k + pad) + k:(i + 1) * (k + pad)] = nan
    got = run_gemm(gpu, "rc", case, a, b, c, "device")
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("ta", ("bf16", "f16"))
@pytest.mark.parametrize("act", (0, 2))
def test_fused_steps_follow_the_plain_call(gpu, ta, act):
    """16-bit kinds with bias and activation: the plain call's sums, then the steps (SiLU within 4 ulp of float64's)."""
    m, n, k = 19, 8200, 520
    case = _case(ta, m, n, k, 1.0, 0.0)
    a, b, c = case.make_inputs(5)
    plain = run_gemm(gpu, "rc", case, a, b, c, "device")
    bias = np.random.default_rng(9).uniform(-4, 4, n).astype(np.float32)
    got = run_fused_gemm(gpu, "rc", case, a, b, c, bias, None, "device", activation=act)[0]
    rows = np.arange(m)[:, None] * case.rsc1 + np.arange(n)[None, :]
    v = plain[rows] + bias[None, :]
    if act == 0:
        assert np.array_equal(got[rows], v)
    else:
        x = v.astype(np.float64)
        want = x / (1 + np.exp(-x))
        assert np.all(np.abs(got[rows] - want) <= 4 * 2.0 ** -23 * np.abs(want) + 1e-37)


def streamed_k(m, n, k, lds):
    fn = ct.CDLL(skl_amd.library_path()).skl_hip_gemv_f4_streamed_k
    fn.argtypes, fn.restype = [ct.c_size_t] * 5 + [ct.c_int, ct.c_size_t], ct.c_size_t
    return fn(m, n, k, k, k, lds != 0, lds)


# one to four column groups, the last one ragged, with one, two and four row groups and two workgroups' rows, the last row group ragged; K one
# block of scales beyond 2304, one beyond the 4096 k whose scales are fetched at once, and with a last part that is multiplied exactly behind
# the stream; columns of scales at every alignment
@pytest.mark.parametrize("m,n,k,streamed", ((1, 1040, 2336, 2336), (16, 4100, 4128, 4128), (17, 12300, 2336, 2336), (32, 8200, 2400, 2400), (31, 260, 14368, 12288),
                                            (33, 8200, 2368, 2368), (64, 4100, 2592, 2592), (65, 1040, 4128, 4096), (40, 12300, 2368, 2368), (128, 12300, 8192, 8192),
                                            (100, 8200, 10496, 8192), (70, 4100, 2592, 2592), (20, 1040, 2656, 2656), (24, 4100, 6464, 6464), (5, 12300, 2336, 2336)))
def test_streamed_4_bit_weights(gpu, m, n, k, streamed):
    """Inside the bound of the reference's fp8 GEMM test around the exact product of the decoded operands, without allowance, with block
    scales and without."""
    for alpha, beta in ((1.0, 0.0), (-1.5, 0.5)):
        case, a, b4, b8, scales, lds, c = f4.make_mx_problem(m + n + k, m, n, k, k, alpha, beta)
        assert streamed_k(m, n, k, lds) == streamed_k(m, n, k, 0) == streamed
        want, bound, oc = f4.mx_bound(case, a, b8, scales, lds, c, m, n, k, k)
        got = run_ofp4(gpu, case, a, b4, c, "device", m, n, k, k, scales, lds)
        assert np.all(np.abs(got[oc].astype(np.float64) - want) <= bound)
        want, bound, oc = f4.mx_bound(case, a, b8, np.full_like(scales, 127), lds, c, m, n, k, k)
        got = run_ofp4(gpu, case, a, b4, c, "device", m, n, k, k)
        assert np.all(np.abs(got[oc].astype(np.float64) - want) <= bound)


# K beyond what the scales' space holds, and more than 64 rows of a wide B up to K = 4096: the kernels with operands in registers
@pytest.mark.parametrize("m,n,k", ((3, 37, 65568), (128, 12290, 2336)))
def test_4_bit_weights_that_are_not_streamed(gpu, m, n, k):
    for alpha, beta in ((1.0, 0.0), (-1.5, 0.5)):
        case, a, b4, b8, scales, lds, c = f4.make_mx_problem(m + n + k, m, n, k, k, alpha, beta)
        assert streamed_k(m, n, k, lds) == 0
        want, bound, oc = f4.mx_bound(case, a, b8, scales, lds, c, m, n, k, k)
        got = run_ofp4(gpu, case, a, b4, c, "device", m, n, k, k, scales, lds)
        assert np.all(np.abs(got[oc].astype(np.float64) - want) <= bound)
