"""Streaming kernels that no other test names one by one: ragged 256 x 128 tiles of every kind and layout, fp8 beyond the exact K on
256 x 128 tiles read across K, eight waves under a C that is read over several rounds. Each test asks the dispatch first which kernel
the problem takes, so that a line that moves fails here instead of leaving a kernel without its test."""
import numpy as np
import pytest

import support
from gpu_support import run_gemm
from test_dispatch_rules import BF16, E4M3, E5M2, F16, I8, RAGGED, route
from test_gpu_gemm import _dense_case
from test_gpu_gemm_in_place import ragged_large

pytestmark = pytest.mark.gpu

KINDS = {"i8": I8, "bf16": BF16, "f16": F16, "f8e4m3": E4M3, "f8e5m2": E5M2}
LAYOUTS = ((True, True), (True, False), (False, True), (False, False))
# one round of 256 x 128 tiles, the last ones 16 rows and columns wide; K in whole pairs of slices and eight or sixteen bytes, ending in
# an odd slice, and - where no operand has K contiguous - anywhere
RAGGED_K = [("i8", 528, 1, False), ("i8", 577, 1, False), ("i8", 4112, 0, True), ("bf16", 2056, 0.5, False), ("bf16", 2088, 0, True), ("bf16", 2049, 0.5, False),
            ("f16", 2088, 0.5, False), ("f16", 2056, 0, True), ("f8e4m3", 4112, 0.5, False), ("f8e4m3", 4240, 0, True), ("f8e4m3", 4097, 0.5, False),
            ("f8e5m2", 4240, 0.5, False)]


@pytest.mark.parametrize("a_rows,b_rows", LAYOUTS)
@pytest.mark.parametrize("ta,k,beta,relu", RAGGED_K)
def test_ragged_tiles_of_128_columns(gpu, ta, k, beta, relu, a_rows, b_rows):
    if k % 8 and (a_rows or not b_rows):
        pytest.skip("16 bytes along K that end inside: the bounds-checked kernels")
    pad = 32 // support.ETYPES[ta].dtype.itemsize
    assert route(KINDS[ta], 2320, 2832, k, a_rows, b_rows, pad=pad, beta=beta, act=int(relu)) == RAGGED + 128
    ragged_large(gpu, ta, 2320, 2832, k, a_rows, b_rows, beta, relu)


def against_fp64(gpu, ta, tb, m, n, k, a_kc, b_kc, alpha, beta, reference_mode=False):
    case = _dense_case(ta, m, n, k, a_kc, b_kc, alpha, beta, tb)
    rng = np.random.default_rng(m + n + k + 2 * a_kc + b_kc)
    a, b, c = case.make_inputs(int(rng.integers(1 << 30)))
    if ta.startswith("f8"):
        a = rng.integers(0x28, 0x48, size=a.size, dtype=np.uint8) | (rng.integers(0, 2, size=a.size, dtype=np.uint8) << 7)
        b = rng.integers(0x28, 0x48, size=b.size, dtype=np.uint8) | (rng.integers(0, 2, size=b.size, dtype=np.uint8) << 7)
    gpu.skl_hip_set_beta_zero_mode(int(reference_mode))
    try:
        got = run_gemm(gpu, "rc", case, a, b, c, "device")
    finally:
        gpu.skl_hip_set_beta_zero_mode(0)
    A, B, C, oc = case.dense(a, b, c)
    exact = alpha * (A @ B) + beta * C
    if case.is_int:
        assert np.array_equal(got[oc], (exact.astype(np.int64) & 0xFFFFFFFF).astype(np.uint32).view(np.int32))
        return
    gamma = 2.0 * np.expm1((k + 2) * np.log1p(2.0 ** -24))
    extra = support.FP8_MFMA_REL if ta.startswith("f8") and k > 2304 else 0.0
    bound = (gamma + extra) * abs(alpha) * (np.abs(A) @ np.abs(B)) + gamma * abs(beta) * np.abs(C)
    assert np.all(np.abs(got[oc] - exact) <= bound + np.abs(exact) * 2.0 ** -22)


@pytest.mark.parametrize("ta,tb", (("f8e4m3", None), ("f8e5m2", None), ("f8e4m3", "f8e5m2")))
@pytest.mark.parametrize("beta,reference_mode", ((0.5, False), (0.0, False), (0.0, True)))
def test_fp8_beyond_the_exact_k_read_across_k(gpu, ta, tb, beta, reference_mode):
    """256 x 128 tiles, K of 2432 elements: C read, not read, and looked through while the tile is multiplied."""
    assert route(KINDS[ta], 2048, 1664, 2432, False, True, kind_b=KINDS[tb or ta], beta=beta) == 128
    against_fp64(gpu, ta, tb, 2048, 1664, 2432, False, False, 1.5, beta, reference_mode)


@pytest.mark.parametrize("a_rows,b_rows", LAYOUTS)
@pytest.mark.parametrize("ta", ("i8", "bf16", "f8e4m3"))
def test_c_read_over_two_rounds_of_tiles(gpu, ta, a_rows, b_rows):
    """374 tiles of 256 x 256 whose last round stays one (eight waves), and 272 whose last 16 run as 32 of 256 x 128; the short fp8 K
    exact on both."""
    k = {"i8": 128, "bf16": 512, "f8e4m3": 256}[ta]
    for m, n in ((4352, 5632), (2048, 8704)):
        assert route(KINDS[ta], m, n, k, a_rows, b_rows, beta=1) == 256
        against_fp64(gpu, ta, None, m, n, k, a_rows, not b_rows, 3 if ta == "i8" else 1.5, -2 if ta == "i8" else 0.5)
