"""The host side of the matrix-core dispatch, asked without a GPU: which problems go to the streaming kernel through copies
of A and B padded to whole tiles (skl_hip_gemm_mfma_padded_plan)."""
import ctypes as ct

import pytest

import skl_amd

I8, BF16, F16, E4M3, E5M2 = range(5)


class Requant(ct.Structure):  # skl_requant of skl_amd/csrc/skl_launch.h
    _fields_ = [("act", ct.c_int), ("q_per_column", ct.c_int), ("q_only", ct.c_int), ("q_zero", ct.c_int32), ("q", ct.c_void_p),
                ("rsq", ct.c_size_t), ("csq", ct.c_size_t), ("q_scale", ct.c_void_p), ("q_fmt", ct.c_int)]


class Canon(ct.Structure):  # skl_gemm_canon
    _fields_ = [("ta", ct.c_int), ("tb", ct.c_int), ("m", ct.c_size_t), ("n", ct.c_size_t), ("k", ct.c_size_t),
                ("a", ct.c_void_p), ("a_s1", ct.c_size_t), ("a_s0", ct.c_size_t), ("a_sk", ct.c_size_t),
                ("b", ct.c_void_p), ("b_s1", ct.c_size_t), ("b_s0", ct.c_size_t), ("b_sk", ct.c_size_t),
                ("c", ct.c_void_p), ("rsc0", ct.c_size_t), ("csc0", ct.c_size_t), ("rsc1", ct.c_size_t), ("csc1", ct.c_size_t),
                ("c_row_shift", ct.c_uint), ("c_col_shift", ct.c_uint), ("alpha", ct.c_double), ("beta", ct.c_double),
                ("bias", ct.c_void_p), ("max", ct.c_void_p), ("rq", Requant)]


def plan(kind, m, n, k, lda=None, ldb=None, act=0, q_fmt=None, b_rows=True):
    """The tile width of the padded plan for row-major A (lda) and B (row-major, or [n][k]); 0: no padded copies."""
    g = Canon(ta=kind, tb=kind, m=m, n=n, k=k, a=1 << 20, b=1 << 20, c=1 << 20, a_sk=1, c_row_shift=6, c_col_shift=6)
    g.a_s0 = lda or k
    g.a_s1 = 64 * g.a_s0
    ldb = ldb or (n if b_rows else k)
    g.b_s0, g.b_sk = (1, ldb) if b_rows else (ldb, 1)
    g.b_s1 = 64 * g.b_s0
    g.rsc0, g.csc0, g.rsc1, g.csc1 = n, 1, 64 * n, 64
    g.rq.act = act
    if q_fmt is not None:
        g.rq.q, g.rq.rsq, g.rq.csq, g.rq.q_scale, g.rq.q_fmt = 1 << 20, (n + 3) // 4 * 4, 1, 1 << 20, q_fmt
    fn = ct.CDLL(skl_amd.library_path()).skl_hip_gemm_mfma_padded_plan
    fn.argtypes = [ct.POINTER(Canon)] + [ct.POINTER(ct.c_size_t)] * 3
    padded = [ct.c_size_t(0) for _ in range(3)]
    cols = fn(ct.byref(g), *(ct.byref(x) for x in padded))
    if cols:
        mp, np_, kp = (x.value for x in padded)
        es = 2 if kind in (BF16, F16) else 1
        assert mp % 256 == 0 and np_ % cols == 0 and kp * es % 128 == 0 and mp >= m and np_ >= n and kp >= k
    return cols


@pytest.mark.parametrize("kind,same_fmt", ((I8, 0), (BF16, 2), (E4M3, 2)))
def test_fused_whole_tiles_copy_only_the_operand_that_needs_it(kind, same_fmt):
    """A fused problem of whole tiles with one operand off the 16-byte rule is not padded; nor with both off it when the
    8-bit copy goes out in dwords. The same problem without fused steps is, and so are ragged fused ones."""
    for lda, ldb in ((4097, None), (None, 4097)):
        assert plan(kind, 4096, 4096, 4096, lda, ldb, act=1, q_fmt=same_fmt) == 0
        assert plan(kind, 4096, 4096, 4096, lda, ldb, act=1) == 0
        assert plan(kind, 4096, 4096, 4096, lda, ldb) == 256
    assert plan(kind, 4096, 4096, 4096, 4097, 4097, act=1, q_fmt=same_fmt) == 0
    assert plan(kind, 4096, 4096 + 128, 4096, 4097, 4097 + 128, act=1, q_fmt=same_fmt) == 0
    assert plan(kind, 4096, 4096, 4096, 4097, 4097, act=1) == 0
    assert plan(kind, 4096, 3968, 4096, 4097, 3969, act=1) == 256  # both copied anyway, and 256 tiles of 256 columns
    assert plan(kind, 4001, 4099, 5003, act=1, q_fmt=same_fmt) == (0 if kind != I8 else 256)  # 272 tiles: a last round of 16
    assert plan(kind, 4001, 4099, 5003, ldb=4112, act=1, q_fmt=same_fmt) == (0 if kind == BF16 else 256)  # B read across K
    assert plan(kind, 4001, 4051, 5003, act=1, q_fmt=same_fmt) == 256
    assert plan(kind, 4001, 4051, 5008, lda=5008, ldb=4064, act=1, q_fmt=same_fmt) == 0  # aligned: ragged, read in place


@pytest.mark.parametrize("m", (1, 100, 256, 300, 2048, 51200))
@pytest.mark.parametrize("n", (1, 100, 130, 256, 6400))
def test_every_size_has_an_answer(m, n):
    for kind in range(5):
        for k in (1, 128, 2304, 2432, 5003):
            for act in (0, 1, 2):
                if kind or act < 2:
                    assert plan(kind, m, n, k, act=act) in (0, 128, 256)
                    assert plan(kind, m, n, k, lda=k + 1, ldb=k + 3, act=act, b_rows=False) in (0, 128, 256)


def in_place(kind, m, n, k, a=1 << 20, a_s0=None, a_sk=1, b_s0=1, b_sk=None, b_s1=None):
    g = Canon(ta=kind, tb=kind, m=m, n=n, k=k, a=a, b=1 << 20, c=1 << 20, c_row_shift=6, c_col_shift=6)
    g.a_s0, g.a_sk = a_s0 or k, a_sk
    g.b_s0, g.b_sk = b_s0, b_sk or n
    g.a_s1, g.b_s1 = 64 * g.a_s0, b_s1 or 64 * g.b_s0
    g.rsc0, g.csc0, g.rsc1, g.csc1 = n, 1, 64 * n, 64
    fn = ct.CDLL(skl_amd.library_path()).skl_hip_gemm_mfma_supported
    fn.argtypes = [ct.POINTER(Canon)]
    return fn(ct.byref(g))


@pytest.mark.parametrize("kind", range(5))
def test_operands_off_the_16_byte_rule_the_kernels_read_in_place(kind):
    """Any base and leading dimension, as long as a row along K, or a run along M / N, holds 16 bytes; strided along both
    dimensions, or whole tiles that a copy of the operand sends to the streaming kernel: not in place."""
    chunk = 8 if kind in (BF16, F16) else 16
    assert in_place(kind, 100, 100, chunk + 1) and in_place(kind, 100, 100, 999, a=(1 << 20) + 2)
    assert not in_place(kind, 100, 100, chunk - 1)
    assert in_place(kind, 100, chunk + 1, 100) and not in_place(kind, 100, chunk - 1, 100)
    assert not in_place(kind, 100, 100, 100, b_s0=2, b_sk=301)
    assert in_place(kind, 100, 2 * chunk + 1, 100, b_sk=64, b_s1=6400)  # one panel: its rows are on the rule
    assert not in_place(kind, 100, 64 + chunk + 1, 100, b_sk=65, b_s1=6501)  # blocks apart: a run's start has no bytes in front
    assert in_place(kind, 100, 64 + chunk, 100, b_sk=65, b_s1=6501)
    assert not in_place(kind, 4096, 4096, 4096, a_s0=4097) and in_place(kind, 4095, 4096, 4096, a_s0=4097)


def pays(kind, m, n, k, lda=None, ldb=None, b_rows=True):
    g = Canon(ta=kind, tb=kind, m=m, n=n, k=k, a=1 << 20, b=1 << 20, c=1 << 20, a_sk=1, c_row_shift=6, c_col_shift=6)
    g.a_s0 = lda or k
    ldb = ldb or (n if b_rows else k)
    g.b_s0, g.b_sk = (1, ldb) if b_rows else (ldb, 1)
    g.a_s1, g.b_s1 = 64 * g.a_s0, 64 * g.b_s0
    g.rsc0, g.csc0, g.rsc1, g.csc1 = n, 1, 64 * n, 64
    fn = ct.CDLL(skl_amd.library_path()).skl_hip_gemm_mfma_in_place_pays
    fn.argtypes = [ct.POINTER(Canon)]
    return fn(ct.byref(g))


@pytest.mark.parametrize("kind", (I8, BF16, E4M3))
def test_copies_padded_to_tiles_only_where_both_operands_need_them(kind):
    k = 4500 if kind != BF16 else 2500
    assert pays(kind, 4000, 4000, 5008, ldb=4000) and pays(kind, 4000, 4000, 5008, lda=5009)
    assert pays(kind, 4000, 4000, k + 1, lda=k + 1, ldb=4001)                          # B read across K
    assert not pays(kind, 4000, 4000, k + 1, b_rows=False)                             # 256 tiles, a full round
    assert pays(kind, 4000, 4000, k // 2 + 1, lda=k // 2 + 1, b_rows=False)            # short K
    assert pays(kind, 300, 300, k + 1, b_rows=False)                                   # six tiles
    assert not pays(kind, 4096, 4096, 4096, lda=4097) and pays(kind, 4096, 4096, 4096)  # whole tiles: one copy streams


def streams_k_contiguous(kind, m, n, k, pitch=None):
    """Whether a decode batch against weights with K contiguous, columns `pitch` apart, is the streaming kernel's."""
    g = Canon(ta=kind, tb=kind, m=m, n=n, k=k, a=1 << 20, b=1 << 20, c=1 << 20, a_sk=1, b_sk=1, c_row_shift=6, c_col_shift=6)
    g.a_s0, g.b_s0 = k, pitch or k
    g.a_s1, g.b_s1 = 64 * g.a_s0, 64 * g.b_s0
    g.rsc0, g.csc0, g.rsc1, g.csc1 = n, 1, 64 * n, 64
    fn = ct.CDLL(skl_amd.library_path()).skl_hip_gemv_kc_rows_supported
    fn.argtypes = [ct.POINTER(Canon)]
    return bool(fn(ct.byref(g)))


@pytest.mark.parametrize("kind", (E4M3, E5M2))
def test_fp8_decode_batches_that_only_the_streaming_kernel_multiplies_exactly(kind):
    """K up to 4096, or 8192 columns and more: however few workgroups there are."""
    for m, n, k in ((96, 9216, 14336), (16, 8208, 14336), (5, 8192, 16384), (96, 9168, 4096), (48, 1024, 4096), (96, 320, 4096), (70, 50000, 8192)):
        assert streams_k_contiguous(kind, m, n, k), (m, n, k)
    assert not streams_k_contiguous(kind, 48, 1024, 14336) and streams_k_contiguous(kind, 16, 1024, 14336)


def test_where_k_contiguous_decode_batches_leave_the_streaming_kernel():
    yes = ((BF16, 16, 32000, 8192), (BF16, 4, 20480, 4096), (BF16, 64, 11008, 4096), (BF16, 96, 50000, 2048), (F16, 16, 8208, 4096), (F16, 32, 4096, 8192),
           (I8, 16, 128, 14336), (I8, 48, 9168, 4096), (I8, 2, 32000, 8192), (I8, 64, 50000, 256))
    no = ((BF16, 64, 50000, 2048), (BF16, 16, 32000, 1024), (BF16, 2, 20480, 4096), (BF16, 64, 11008, 512), (BF16, 96, 8192, 14336), (F16, 48, 4096, 14336),
          (F16, 64, 448, 2688), (I8, 48, 2048, 8192), (I8, 2, 20480, 8192), (I8, 96, 1024, 8192))
    for case in yes:
        assert streams_k_contiguous(*case), case
    for case in no:
        assert not streams_k_contiguous(*case), case
    # columns that start inside lines take half as long again
    assert streams_k_contiguous(I8, 16, 256, 14336) and not streams_k_contiguous(I8, 16, 256, 14336, pitch=14352)


RAGGED = 1000


def route(kind, m, n, k, a_rows=True, b_rows=True, pad=0, beta=0, act=0, q=None, kind_b=None, lda=None):
    """The matrix-core kernel that takes a problem as it lies: 0 none, 1 the bounds-checked tiles, else the columns of the streaming
    kernel's tiles, RAGGED more where those are ragged. `pad` elements between rows; `q` the format of a row-major 8-bit copy."""
    g = Canon(ta=kind, tb=kind if kind_b is None else kind_b, m=m, n=n, k=k, a=1 << 20, b=1 << 20, c=1 << 20, c_row_shift=6, c_col_shift=6)
    lda, ldb = lda or (k if a_rows else m) + pad, (n if b_rows else k) + pad
    g.a_s0, g.a_sk = (lda, 1) if a_rows else (1, lda)
    g.b_s0, g.b_sk = (1, ldb) if b_rows else (ldb, 1)
    g.a_s1, g.b_s1 = 64 * g.a_s0, 64 * g.b_s0
    g.rsc0, g.csc0, g.rsc1, g.csc1 = n, 1, 64 * n, 64
    g.rq.act = act
    if q is not None:
        g.rq.q, g.rq.rsq, g.rq.csq, g.rq.q_scale, g.rq.q_fmt = 1 << 20, (n + 3) // 4 * 4, 1, 1 << 20, q
    scalar = ct.c_int32 if kind == I8 else ct.c_float
    scalar.from_buffer(g, Canon.beta.offset).value = beta
    if kind != I8:
        ct.c_uint32.from_buffer(g, Canon.beta.offset + 4).value = 1  # C is not read where beta is zero
    fn = ct.CDLL(skl_amd.library_path()).skl_hip_gemm_mfma_route
    fn.argtypes = [ct.POINTER(Canon)]
    return fn(ct.byref(g))


def test_whole_tiles_go_where_they_were_measured_to_be_faster():
    """A copy of whole numbers, a C that is read, SiLU: the streaming kernel; short plain products on half of the chip: not."""
    for kind, k in ((I8, 1024), (BF16, 512), (F16, 1024), (E4M3, 1024)):
        assert route(kind, 4096, 1024, k) == 1 and route(kind, 4096, 1024, 8192 if kind != E4M3 else 16384) == 128   # 128 tiles of 256 x 128
        assert route(kind, 4352, 1024, k) == 128 and route(kind, 4352, 1024, k, beta=1) == 128                       # 136
        assert route(kind, 4096, 3328, k, act=1, q=0 if kind == I8 else 2) == 256                                    # 208 of 256 x 256
    assert route(I8, 4096, 1024, 1024, beta=1) == 128 and route(BF16, 4096, 1024, 512, beta=1) == 128
    assert route(I8, 7424, 7168, 512, act=1, q=0) == 256 and route(I8, 7424, 7040, 512, act=1, q=0) == 128           # 812, and 1595 of 256 x 128
    assert route(I8, 7424, 7168, 512, act=1) == 256 and route(I8, 7424, 7040, 512, act=1) == 1                       # ReLU into C
    assert route(BF16, 7424, 7040, 512) == 1 and route(BF16, 7424, 7040, 1024) == 128                                # from 2 KiB of K on
    assert route(I8, 8192, 8192, 1024) == 256 and route(I8, 7424, 7168, 512) == 1
    assert route(E4M3, 8192, 12032, 640) == 256 and route(E4M3, 4352, 4608, 640) == 1                                # 1504 and 306 of 256 x 256
    for kind in (BF16, F16, E4M3):                                                                                   # GELU on 651 of 256 x 128, 2.5 rounds
        assert route(kind, 7936, 2688, 640, b_rows=False, act=3, q=2) == 128 and route(kind, 7936, 2688, 640, b_rows=False, act=3) == 1


@pytest.mark.parametrize("kind", (I8, BF16, F16, E4M3))
def test_whole_tiles_off_the_16_byte_rule_are_copied_only_to_stream(kind):
    """128 tiles of 256 x 128 with a short K run on the bounds-checked tiles, in place, whatever the leading dimension; with a C that is
    read, or more tiles, the copy of the operand lets the streaming kernel run. The padded plan follows the same lines."""
    k = 512 if kind in (BF16, F16) else 1024
    assert route(kind, 4096, 1024, k) == 1 and route(kind, 4096, 1024, k, lda=k + 1) == 1
    assert route(kind, 4352, 1024, k) == 128 and route(kind, 4352, 1024, k, lda=k + 1) == 0
    if kind != E4M3:
        assert route(kind, 4096, 1024, k, beta=1, lda=k + 1) == 0
    if kind == I8:
        assert plan(kind, 4090, 1020, k, lda=k + 1, ldb=1021) == 0 and plan(kind, 4346, 1020, k, lda=k + 1, ldb=1021) == 128
