"""The matrix-core kernels that check bounds, on operands read where they lie: sizes at the edges of their tiles and of the
slices of K they keep under way, leading dimensions and bases off the 16-byte rule. What surrounds an operand - ahead of it,
behind it and in the gaps between its rows - is filled with the kind's largest or non-finite codes, so that an element taken
from there shows."""
import numpy as np
import pytest

import skl_amd
import support
from skl_amd import DeviceBuffer
from gpu_support import run_fused_gemm, run_gemm
from support import GemmCase, run_oracle_gemm
from test_oracle_gemm import fused_expectation

pytestmark = pytest.mark.gpu

POISON = {"i8": 127, "bf16": 0x7FC0, "f16": 0x7E00, "f8e4m3": 0x7F, "f8e5m2": 0x7E}
GUARD = 64


def in_place(gpu, ta, m, n, k, a_rows, b_rows, a_pad, b_pad, a_off, b_off, beta):
    """A row-major or by columns, B row-major or by columns, `pad` elements between rows, the base `off` elements off."""
    lda, ldb = (k if a_rows else m) + a_pad, (n if b_rows else k) + b_pad
    case = GemmCase(ta, None, 2 if ta == "i8" else 1.5, beta, m0=1, n0=1, k0=1, m1=m, n1=n, k1=k, rsa0=0, csa0=0,
                    rsa1=lda if a_rows else 1, csa1=1 if a_rows else lda, rsb0=0, csb0=0, rsb1=ldb if b_rows else 1,
                    csb1=1 if b_rows else ldb, rsc0=0, csc0=0, rsc1=n + 3, csc1=1)
    a, b, c = case.make_inputs(m + 31 * n + 977 * k + 7 * a_pad + 3 * b_pad + a_off)

    def poisoned(x, rows, run, ld):
        keep = np.zeros(x.size, bool)
        for r in range(rows):
            keep[r * ld:r * ld + run] = True
        x = x.copy()
        x[~keep] = POISON[ta]
        return x

    a, b = poisoned(a, m if a_rows else k, k if a_rows else m, lda), poisoned(b, k if b_rows else n, n if b_rows else k, ldb)
    guard = np.full(2 * GUARD, POISON[ta], a.dtype)
    es = a.itemsize
    da = DeviceBuffer.from_array(np.concatenate([guard[:GUARD // es + a_off], a, guard]))
    db = DeviceBuffer.from_array(np.concatenate([guard[:GUARD // es + b_off], b, guard]))
    dc = DeviceBuffer.from_array(c)
    getattr(gpu, f"skl_gemm_{ta}rc_{ta}rc_{case.ctag}rc_gfx950")(
        m, n, k, case.alpha, da.offset((GUARD // es + a_off) * es), case.rsa1, case.csa1, db.offset((GUARD // es + b_off) * es), case.rsb1, case.csb1,
        case.beta, dc, case.rsc1, 1)
    gpu.skl_hip_synchronize()
    skl_amd.check_error()
    got = dc.download(c.dtype, c.size)
    for d in (da, db, dc):
        d.free()
    if case.is_int:
        assert np.array_equal(got, run_oracle_gemm(case, a, b, c)), vars(case)
    else:
        support.assert_fp_gemm_close(case, a, b, c, got, extra_rel=support.FP8_MFMA_REL if ta.startswith("f8") else 0.0)


# one chunk, one tile less, exactly and more; K of a chunk, of one to eight slices of 128 bytes and what sticks out of them
SIZES = ((65, 63, 16), (64, 64, 127), (17, 130, 128), (129, 64, 257), (63, 129, 385), (128, 127, 520), (66, 200, 641), (300, 65, 1031))


@pytest.mark.parametrize("ta", ("i8", "bf16", "f8e4m3"))
@pytest.mark.parametrize("m,n,k", SIZES)
def test_operands_off_the_16_byte_rule_in_place(gpu, ta, m, n, k):
    for a_rows in (True, False):
        for b_rows in (True, False):
            for a_pad, b_pad, a_off, b_off in ((1, 0, 0, 0), (0, 3, 1, 5), (16, 16, 0, 0)):
                in_place(gpu, ta, m, n, k, a_rows, b_rows, a_pad, b_pad, a_off, b_off, (a_pad + b_rows) % 2)


@pytest.mark.parametrize("ta,k", (("f8e5m2", 2500), ("f8e4m3", 4097), ("f16", 1283), ("i8", 8191)))
def test_large_tiles_and_shared_k_off_the_16_byte_rule(gpu, ta, k):
    """Tiles of 128 x 128, the fp8 instructions' fragments of 32 bytes, and K shared between workgroups."""
    for a_rows, b_rows in ((True, False), (False, False), (True, True)):
        in_place(gpu, ta, 1025, 1031, k, a_rows, b_rows, 1, 2, 3, 0, 1)
        in_place(gpu, ta, 40, 333, k, a_rows, b_rows, 5, 0, 0, 1, 0)


def ragged_large(gpu, ta, m, n, k, a_rows, b_rows, beta, relu=False):
    """Operands on the 16-byte rule with poisoned gaps between their rows, against the product in fp64."""
    es = support.ETYPES[ta].dtype.itemsize
    pad = 32 // es
    lda, ldb = (k if a_rows else m) + pad, (n if b_rows else k) + pad
    case = GemmCase(ta, None, 2 if ta == "i8" else 1.5, beta, m0=1, n0=1, k0=1, m1=m, n1=n, k1=k, rsa0=0, csa0=0,
                    rsa1=lda if a_rows else 1, csa1=1 if a_rows else lda, rsb0=0, csb0=0, rsb1=ldb if b_rows else 1,
                    csb1=1 if b_rows else ldb, rsc0=0, csc0=0, rsc1=n, csc1=1)
    rng = np.random.default_rng(m + n + k + a_rows + 2 * b_rows)
    gen, widen = support.ETYPES[ta].gen, support.ETYPES[ta].widen
    a = np.full((m if a_rows else k, lda), POISON[ta], support.ETYPES[ta].dtype)
    b = np.full((k if b_rows else n, ldb), POISON[ta], support.ETYPES[ta].dtype)
    a[:, :lda - pad] = gen(rng, a.shape[0] * (lda - pad)).reshape(a.shape[0], -1)
    b[:, :ldb - pad] = gen(rng, b.shape[0] * (ldb - pad)).reshape(b.shape[0], -1)
    c = rng.integers(-100, 100, (m, n)).astype(case.cdtype)
    A, B = widen(a[:, :lda - pad]), widen(b[:, :ldb - pad])
    A, B = A if a_rows else A.T, B if b_rows else B.T
    exact = case.alpha * (A @ B) + beta * c
    if relu:
        got, _ = run_fused_gemm(gpu, "rc", case, a.reshape(-1)[:a.size - pad], b.reshape(-1)[:b.size - pad], c.reshape(-1), None, None, "device", activation=1)
        exact = np.maximum(exact, 0)
    else:
        got = run_gemm(gpu, "rc", case, a.reshape(-1)[:a.size - pad], b.reshape(-1)[:b.size - pad], c.reshape(-1), "device")
    got = got.reshape(m, n)
    if case.is_int:
        assert np.array_equal(got, (exact.astype(np.int64) & 0xFFFFFFFF).astype(np.uint32).view(np.int32))
        return
    gamma = 2.0 * np.expm1((k + 2) * np.log1p(2.0 ** -24))
    extra = support.FP8_MFMA_REL if ta.startswith("f8") else 0.0
    bound = (gamma + extra) * 1.5 * (np.abs(A) @ np.abs(B)) + gamma * abs(beta) * np.abs(c)
    assert np.all(np.abs(got - exact) <= bound + np.abs(exact) * 2.0 ** -22)


@pytest.mark.parametrize("ta,k", (("i8", 272), ("i8", 65), ("bf16", 264), ("bf16", 129), ("f8e4m3", 2416), ("f8e5m2", 2433)))
@pytest.mark.parametrize("a_rows,b_rows", ((True, True), (True, False), (False, True), (False, False)))
def test_streaming_kernel_on_ragged_tiles(gpu, ta, k, a_rows, b_rows):
    """One round of 256 x 128 tiles that reads C, every operand layout; a K that ends inside a slice, in an odd slice, and -
    where no operand has K contiguous - anywhere; the last tiles 16 rows and columns wide."""
    if k % 8 and (a_rows or not b_rows):
        pytest.skip("16 bytes along K that end inside: the bounds-checked kernels")
    ragged_large(gpu, ta, 2320, 2832, k, a_rows, b_rows, 1 if ta == "i8" else 0.5)


@pytest.mark.parametrize("ta,k,relu", (("i8", 4112, False), ("bf16", 2088, True), ("f8e4m3", 4240, False)))
@pytest.mark.parametrize("a_rows,b_rows", ((True, True), (False, True), (True, False)))
def test_streaming_kernel_on_ragged_wide_tiles(gpu, ta, k, relu, a_rows, b_rows):
    ragged_large(gpu, ta, 3856, 3104, k, a_rows, b_rows, 0, relu)


@pytest.mark.parametrize("ta", ("i8", "bf16", "f8e4m3"))
@pytest.mark.parametrize("m,n,k,block", ((70, 90, 200, 0), (64, 128, 96, 0), (257, 300, 160, 0), (1029, 1040, 160, 0), (72, 92, 80, 2), (132, 200, 96, 4), (1032, 1040, 96, 4),
                                         (40, 100, 4400, 0), (40, 101, 4400, 0)))
def test_fused_steps_of_the_bounds_checked_kernels(gpu, ta, m, n, k, block):
    """Tiles of 64 x 64 and 128 x 128 whose edges cut rows and columns, C row-major (`block` 0), by columns and in blocks of four rows,
    reading C; K whole and shared. The call with bias alone is the anchor: the steps make of its C what the rules say, bit for bit."""
    rng = np.random.default_rng(m + n + k)
    bias = rng.integers(-999, 999, n).astype(np.int32) if ta == "i8" else rng.uniform(-4, 4, n).astype(np.float32)
    start = np.array([-(1 << 31)], np.int32) if ta == "i8" else np.array([-np.inf], np.float32)
    for by_columns in ((False,) if block else (False, True)):
        if block:
            n1 = n // block
            case = GemmCase(ta, None, 2, -1, m0=4, n0=block, k0=1, m1=m // 4, n1=n1, k1=k, rsa0=k, csa0=0, rsa1=4 * k, csa1=1, rsb0=0, csb0=1, rsb1=n,
                            csb1=block, rsc0=block, csc0=1, rsc1=4 * block * n1 + 2, csc1=4 * block)
        else:
            case = GemmCase(ta, None, 1, 1, m0=1, n0=1, k0=1, m1=m, n1=n, k1=k, rsa0=0, csa0=0, rsa1=k, csa1=1, rsb0=0, csb0=0, rsb1=n, csb1=1,
                            rsc0=0, csc0=0, rsc1=1 if by_columns else n + 2, csc1=m + 1 if by_columns else 1)
        kind = "rcprc" if block else "rc"
        a, b, c = case.make_inputs(int(rng.integers(1 << 30)))
        anchor, _ = run_fused_gemm(gpu, kind, case, a, b, c, bias, None, "device")
        scales = (rng.uniform(0.5, 2.0, n) * 100.0 / float(np.abs(anchor.astype(np.float64)).max())).astype(np.float32)
        for rsq, csq, only in ((n + (-n) % 4, 1, False), (n + 5, 1, True), (1, m + 5, False)):
            rq = dict(q=np.full((m - 1) * rsq + (n - 1) * csq + 1, 0x55, np.int8), rsq=rsq, csq=csq, scale=scales, per_column=True, zero=3, only=only,
                      format=0 if ta == "i8" else 2)
            got, top, q = run_fused_gemm(gpu, kind, case, a, b, c, bias, start, "device", activation=1, requant=rq)
            want_c, want_top, want_q = fused_expectation(case, anchor, None, start, activation=1, requant=rq)
            assert np.array_equal(q, want_q) and top[0] == want_top[0], (by_columns, rsq, csq)
            assert np.array_equal(got.view(np.uint8), (c if only else want_c).view(np.uint8)), (by_columns, rsq, csq)


@pytest.mark.parametrize("ta,k", (("i8", 4112), ("bf16", 2056), ("f8e4m3", 4240)))
@pytest.mark.parametrize("c_form", ("rows", "columns", "blocks"))
def test_fused_steps_of_the_streaming_kernel_on_ragged_tiles(gpu, ta, k, c_form):
    """Bias per column, ReLU, maximum and an 8-bit copy - off the dword rule, by columns, and alone - where tiles of 256 x 256 end inside
    rows and columns, C row-major, by columns and in blocks of four. The call with bias alone is the anchor, which holds the product."""
    m, n = 3856, 3104
    rng = np.random.default_rng(k)
    bias = rng.integers(-999, 999, n).astype(np.int32) if ta == "i8" else rng.uniform(-4, 4, n).astype(np.float32)
    start = np.array([-(1 << 31)], np.int32) if ta == "i8" else np.array([-np.inf], np.float32)
    if c_form == "blocks":
        kind = "rcprc"
        case = GemmCase(ta, None, 1, 1, m0=4, n0=4, k0=1, m1=m // 4, n1=n // 4, k1=k, rsa0=k, csa0=0, rsa1=4 * k, csa1=1, rsb0=0, csb0=k, rsb1=1, csb1=4 * k,
                        rsc0=4, csc0=1, rsc1=4 * n + 4, csc1=16)
    else:
        kind = "rc"
        case = GemmCase(ta, None, 1, 0, m0=1, n0=1, k0=1, m1=m, n1=n, k1=k, rsa0=0, csa0=0, rsa1=k, csa1=1, rsb0=0, csb0=0, rsb1=1, csb1=k, rsc0=0, csc0=0,
                        rsc1=1 if c_form == "columns" else n, csc1=m + 1 if c_form == "columns" else 1)
    a, b, c = case.make_inputs(int(rng.integers(1 << 30)))
    anchor, _ = run_fused_gemm(gpu, kind, case, a, b, c, bias, None, "device")
    if c_form == "rows":
        widen = support.ETYPES[ta].widen
        A, B = widen(a[:m * k]).reshape(m, k), widen(b[:n * k]).reshape(n, k)
        exact = A @ B.T + bias
        if ta == "i8":
            assert np.array_equal(anchor.reshape(m, n), exact.astype(np.int64).astype(np.int32))
        else:
            gamma = 2.0 * np.expm1((k + 2) * np.log1p(2.0 ** -24))
            assert np.all(np.abs(anchor.reshape(m, n) - exact) <= gamma * (np.abs(A) @ np.abs(B).T + np.abs(bias)))
    scales = (rng.uniform(0.5, 2.0, n) * 100.0 / float(np.abs(anchor.astype(np.float64)).max())).astype(np.float32)
    forms = {"rows": ((n + 5, 1, False), (n + (-n) % 4, 1, True)), "columns": ((1, m + 5, False),), "blocks": ((n + 5, 1, False),)}[c_form]
    for rsq, csq, only in forms:
        rq = dict(q=np.full((m - 1) * rsq + (n - 1) * csq + 1, 0x55, np.int8), rsq=rsq, csq=csq, scale=scales, per_column=True, zero=3, only=only,
                  format=0 if ta == "i8" else 2)
        got, top, q = run_fused_gemm(gpu, kind, case, a, b, c, bias, start, "device", activation=1, requant=rq)
        want_c, want_top, want_q = fused_expectation(case, anchor, None, start, activation=1, requant=rq)
        assert np.array_equal(q, want_q) and top[0] == want_top[0], (rsq, csq, only)
        assert np.array_equal(got.view(np.uint8), (c if only else want_c).view(np.uint8)), (rsq, csq, only)
