"""How the matrix-core kernels add up a long K: in how many parts, so that an fp32 sum keeps what many short chains of
roundings keep, and in the same parts with and without fused steps."""
import numpy as np
import pytest

import support
from gpu_support import run_fused_gemm, run_gemm
from support import GemmCase, rowmajor_case

pytestmark = pytest.mark.gpu


def operands(ta, m, n, k):
    rng = np.random.default_rng(m + 31 * n + 977 * k)
    gen = support.ETYPES[ta].gen
    return gen(rng, m * k).reshape(m, k), gen(rng, k * n).reshape(k, n)


def product(gpu, ta, a, b):
    """A * B, both row-major."""
    (m, k), n = a.shape, b.shape[1]
    case = rowmajor_case(ta, m, n, k, 1.0, 0.0)
    return run_gemm(gpu, "rc", case, np.ascontiguousarray(a).reshape(-1), np.ascontiguousarray(b).reshape(-1), np.zeros(m * n, np.float32), "device").reshape(m, n)


# 96 tiles of 128 x 128: six shares of 11 slices of 64 k; 64 of them with K of 4 KiB: 256 tiles of 64 x 64, each adding blocks of
# 256 k; 100 tiles of 64 x 64: four shares of 512 k, each of two blocks
@pytest.mark.parametrize("m,n,k,part", ((300, 4096, 4096, 704), (1024, 1024, 2048, 256), (640, 640, 2048, 512)))
@pytest.mark.parametrize("ta", ("bf16", "f16"))
def test_a_sum_is_made_of_parts(gpu, ta, m, n, k, part):
    """Bit for bit the sum, in order, of the parts' own products, which are too short to be parted."""
    a, b = operands(ta, m, n, k)
    got = product(gpu, ta, a, b)
    block = min(part, 256) if m > 300 else part
    total = None
    for k0 in range(0, k, part):
        share = None
        for k1 in range(k0, min(k0 + part, k), block):
            p = product(gpu, ta, a[:, k1:min(k1 + block, k0 + part)], b[k1:min(k1 + block, k0 + part)])
            share = p if share is None else share + p
        total = share if total is None else total + share
    assert np.array_equal(got.view(np.uint32), total.view(np.uint32))
    widen = support.ETYPES[ta].widen
    exact = widen(a) @ widen(b)
    # an instruction rounds about once per eight products, at the size of the chain so far; the sums of blocks and shares once each
    roundings = block / 8 + part / block + k / part
    assert np.linalg.norm(got - exact) <= 2.0 ** -24 / np.sqrt(3) * np.sqrt(roundings / 2) * np.linalg.norm(exact)


@pytest.mark.parametrize("ta,k", (("bf16", 2040), ("f16", 2047), ("bf16", 1984), ("f8e4m3", 4090)))
def test_fused_steps_on_the_sums_of_the_plain_call(gpu, ta, k):
    """144 tiles of 128 x 128 and a K around the 4 KiB from which it is shared: bias alone, ReLU and an 8-bit copy besides."""
    m = n = 1500
    a, b = operands(ta, m, n, k)
    case = rowmajor_case(ta, m, n, k, 1.0, 0.0)
    bias = np.random.default_rng(3).uniform(-4, 4, n).astype(np.float32)
    args = (gpu, "rc", case, a.reshape(-1), b.reshape(-1), np.zeros(m * n, np.float32), bias, None, "device")
    anchor = run_fused_gemm(*args)[0]
    assert np.array_equal(anchor, (product(gpu, ta, a, b) + bias).reshape(-1))
    assert np.array_equal(run_fused_gemm(*args, activation=1)[0], np.maximum(anchor, 0))
    rq = dict(q=np.zeros(m * n, np.int8), rsq=n, csq=1, scale=np.ones(1, np.float32), per_column=False, zero=0, only=False, format=0)
    assert np.array_equal(run_fused_gemm(*args, requant=rq)[0], anchor)


# B or A off the 16-byte rule: one row, a few, the most that count as few, and few columns; K beyond the fp8 kinds' exact products.
# `roundings`: one per eight products of a block, one per block unless their sum is compensated, one per share of K.
@pytest.mark.parametrize("ta,m,n,k,roundings", (("f8e4m3", 2, 1755, 3408, 16 + 1 + 7), ("f8e4m3", 89, 705, 3441, 64 + 1 + 7), ("f8e5m2", 1, 91, 2425, 16 + 1 + 5),
                                                ("f8e4m3", 300, 5, 4801, 16 + 1 + 9), ("bf16", 1, 1957, 593, 8 + 1 + 1), ("bf16", 4, 6614, 1401, 8 + 1 + 1),
                                                ("bf16", 9, 333, 4097, 8 + 4 + 16), ("f16", 16, 1157, 2817, 8 + 4 + 11)))
def test_few_rows_off_the_16_byte_rule_keep_exact_products_and_short_sums(gpu, ta, m, n, k, roundings):
    a, b = operands(ta, m, n, k)
    got = product(gpu, ta, a, b)
    widen = support.ETYPES[ta].widen
    exact = widen(a) @ widen(b)
    assert np.linalg.norm(got - exact) <= 2.0 ** -24 / np.sqrt(3) * np.sqrt(roundings / 2) * np.linalg.norm(exact)


@pytest.mark.parametrize("ta", ("bf16", "f16", "f8e4m3"))
def test_few_rows_with_infinities_and_nan(gpu, ta):
    """An infinite sum stays infinite, also when finite blocks of K follow it; opposite infinities and NaN give NaN."""
    m, n, k = 3, 33, 1025
    a, b = operands(ta, m, n, k)
    big = {"bf16": 0x7F80, "f16": 0x7C00}.get(ta)
    if big is None:
        a[:, 5], nan = 0x7F, True          # E4M3 has no infinity: NaN
    else:
        one = support.ETYPES[ta]
        b[5], b[700], nan = (0x3F80 if ta == "bf16" else 0x3C00), (0x3F80 if ta == "bf16" else 0x3C00), False
        a[0, 5], a[1, 5], a[1, 700] = big, big, big | 0x8000
    got = product(gpu, ta, a, b)
    if nan:
        assert np.isnan(got).all()
    else:
        assert np.isposinf(got[0]).all() and np.isnan(got[1]).all() and np.isfinite(got[2]).all()


def k_contiguous_product(gpu, ta, a, bt):
    """A * B with B stored column by column."""
    (m, k), n = a.shape, bt.shape[0]
    case = GemmCase(ta, None, 1.0, 0.0, m0=1, n0=1, k0=1, m1=m, n1=n, k1=k, rsa0=0, csa0=0, rsa1=k, csa1=1, rsb0=0, csb0=0, rsb1=1, csb1=k,
                    rsc0=0, csc0=0, rsc1=n, csc1=1)
    return run_gemm(gpu, "rc", case, a.reshape(-1), bt.reshape(-1), np.zeros(m * n, np.float32), "device").reshape(m, n)


# few rows: blocks of 128 bytes of K in eight waves; many: of 512 bytes in eight or four; fp8 with K beyond 4096 and beyond the
# exact products of the tile kernels, on a chip not full of workgroups
@pytest.mark.parametrize("ta,m,n,k", (("bf16", 2, 64, 14336), ("bf16", 4, 4112, 4096), ("f16", 16, 1024, 8192), ("bf16", 20, 3072, 8192), ("f16", 70, 4096, 4096),
                                      ("f8e4m3", 4, 4112, 8192), ("f8e4m3", 16, 8208, 14336), ("f8e5m2", 48, 9168, 8192), ("f8e4m3", 96, 8208, 4096)))
def test_k_contiguous_decode_batches_add_up_blocks(gpu, ta, m, n, k):
    rng = np.random.default_rng(m + n + k)
    gen, widen = support.ETYPES[ta].gen, support.ETYPES[ta].widen
    a, bt = gen(rng, m * k).reshape(m, k), gen(rng, n * k).reshape(n, k)
    got = k_contiguous_product(gpu, ta, a, bt)
    exact = widen(a) @ widen(bt).T
    line = 128 if ta.startswith("f8") else 64
    block, waves = (line if m <= 16 else 4 * line), (8 if m <= 32 else 4)
    roundings = block / 8 + k / waves / block + waves
    assert np.linalg.norm(got - exact) <= 2.0 ** -24 / np.sqrt(3) * np.sqrt(roundings / 2) * np.linalg.norm(exact)
