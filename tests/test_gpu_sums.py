"""How the matrix-core kernels add up a long K: in how many parts, so that an fp32 sum keeps what many short chains of
roundings keep, and in the same parts with and without fused steps."""
import numpy as np
import pytest

import support
from gpu_support import run_fused_gemm, run_gemm
from support import rowmajor_case

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
