"""Calls on a stream that finds no scratch memory left: which of them go on without a word, and that C is updated once."""
import numpy as np
import pytest

import skl_amd
import support

pytestmark = pytest.mark.gpu


def _streams_until_the_slots_are_gone(gpu, hip, ct):
    """Streams that hold scratch slots, and one more that finds none left."""
    streams = []
    da, dy = skl_amd.DeviceBuffer(4096 * 2049), skl_amd.DeviceBuffer(4 * 2048)
    for _ in range(34):
        stream = ct.c_void_p()
        assert hip.hipStreamCreate(ct.byref(stream)) == 0
        streams.append(stream)
        gpu.skl_hip_set_stream(stream.value)
        gpu.skl_gemm_i8_i8_i32_gfx950(1, 2048, 4096, 1, da, 4096, da, 2048, 0, dy, 2048)  # a GEMV: its workgroups meet in the stream's scratch
        assert gpu.skl_hip_synchronize() == 0
        if gpu.skl_hip_last_error() != 0:
            break
    else:
        pytest.fail("34 streams found a slot")
    da.free(), dy.free()
    return streams


@pytest.mark.parametrize("ta,m,n,k,beta,code", (("bf16", 40, 300, 1200, 1, 0),      # a K that is shared for speed alone: in one share, without a word
                                                ("f8e4m3", 64, 520, 1100, 0, 0),
                                                ("i8", 2048, 8448, 8192, 3, -5)))   # 33 tile columns of 256: the trailing ones would share K
def test_without_a_scratch_slot(gpu, ta, m, n, k, beta, code):
    """A stream beyond the 32 that hold scratch: the results of the others, each element of C updated once."""
    import ctypes as ct

    hip = ct.CDLL("libamdhip64.so.7")
    hip.hipStreamCreate.restype = hip.hipStreamDestroy.restype = ct.c_int
    rng = np.random.default_rng(m + n + k)
    gen = support.ETYPES[ta].gen
    a, b = gen(rng, m * k), gen(rng, k * n)
    ctype, acc = (np.int32, "i32") if ta == "i8" else (np.float32, "f32")
    c = rng.integers(-1000, 1000, m * n).astype(ctype)
    da, db, dc = (skl_amd.DeviceBuffer.from_array(x) for x in (a, b, c))
    scalar = int if ta == "i8" else float
    entry = getattr(gpu, f"skl_gemm_{ta}rc_{ta}rc_{acc}rc_gfx950")
    gpu.skl_hip_set_pointer_mode(1)
    streams = []

    def call():
        gpu.skl_hip_memcpy_h2d(dc, c, c.nbytes)
        entry(m, n, k, scalar(1), da, k, 1, db, n, 1, scalar(beta), dc, n, 1)
        assert gpu.skl_hip_synchronize() == 0
        return dc.download(ctype, c.size)

    try:
        want = call()
        skl_amd.check_error()
        streams = _streams_until_the_slots_are_gone(gpu, hip, ct)
        got = call()
        assert gpu.skl_hip_last_error() == code
        if ta == "i8":
            assert np.array_equal(got, want)
        else:
            widen = support.ETYPES[ta].widen
            exact = widen(a).reshape(m, k) @ widen(b).reshape(k, n) + beta * c.reshape(m, n)
            scale = np.abs(widen(a)).reshape(m, k) @ np.abs(widen(b)).reshape(k, n) + np.abs(beta * c.reshape(m, n))
            assert np.all(np.abs(got.reshape(m, n) - exact) <= (k + 2) * 2.0 ** -24 * scale)
    finally:
        gpu.skl_hip_set_stream(None)
        gpu.skl_hip_set_pointer_mode(0)
        for stream in streams:
            gpu.skl_hip_release_stream(stream.value)
            hip.hipStreamDestroy(stream)
        for d in (da, db, dc):
            d.free()
        gpu.skl_hip_last_error()
