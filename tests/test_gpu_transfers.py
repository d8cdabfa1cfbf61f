"""Copies between host and device: uploads that do not wait, downloads that come with the fault word."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from ojas_amd.backend import MiBackend

    backend = MiBackend(0)
    yield backend
    backend.close()


def test_staged_uploads_arrive_in_order(be):
    """Sizes off the 16-byte pieces, the largest that is staged and larger ones, offsets that are not aligned; more bytes than the
    staging memory holds between two waits, and the source overwritten as soon as the call returns."""
    print("staged uploads", flush=True)
    r = np.random.default_rng(0)
    sizes = [1, 3, 15, 16, 17, 255, 4095, 4096, 4097, 65536, 65537, (256 << 10) - 1, 256 << 10, (256 << 10) + 1, 700000] * 3
    made = []
    for i, n in enumerate(sizes):
        host = r.integers(-128, 128, n).astype(np.int8)
        made.append((host.copy(), be.upload(host, staged=True)))
        host[:] = 0
    for want, t in made:
        assert np.array_equal(be.download(t), want)
    base = be.upload(np.zeros(64, np.int8))
    for at in (1, 16, 40):
        piece = np.full(8, at, np.int8)
        be._check(be._lib.omx_upload_staged(be._ctx, be._p(base), C.c_uint64(at), C.c_void_p(piece.ctypes.data), C.c_uint64(8)))
    want = np.zeros(64, np.int8)
    for at in (1, 16, 40):
        want[at:at + 8] = at
    assert np.array_equal(be.download(base), want)
    with pytest.raises(Exception):
        be._check(be._lib.omx_upload_staged(be._ctx, None, C.c_uint64(0), C.c_void_p(want.ctypes.data), C.c_uint64(8)))


@pytest.mark.parametrize("n", [1, 7, 4095, 4096, 4097, 20000])
def test_downloads_report_a_fault_and_leave_the_destination(be, n):
    """Both sides of the size that travels with the fault word, from offsets of any alignment; a fault is reported once."""
    from ojas_amd.backend import NON_FINITE, OjasError

    print(f"download {n}", flush=True)
    host = np.random.default_rng(n).integers(-128, 128, n + 5).astype(np.int8)
    t = be.upload(host)
    back = np.zeros(n, np.int8)
    get = lambda: be._check(be._lib.omx_download(be._ctx, C.c_void_p(back.ctypes.data), be._p(t), C.c_uint64(5), C.c_uint64(n)))
    get()
    assert np.array_equal(back, host[5:])
    back[:] = 3
    be.silu_forward(be.upload(np.array([1.0, np.nan], np.float32)))
    with pytest.raises(OjasError) as e:
        get()
    assert e.value.code == NON_FINITE and "silu_forward" in str(e.value) and (back == 3).all()
    get()
    assert np.array_equal(back, host[5:])


def test_memory_of_others_is_copied_too(be):
    """Blocks that are not the context's own (another context's) take the runtime's copies, with the same results."""
    from ojas_amd.backend import MiBackend

    print("foreign memory", flush=True)
    other = MiBackend(0)
    try:
        there = other.upload(np.arange(100, dtype=np.int8))
        back, put = np.zeros(40, np.int8), np.full(16, 9, np.int8)
        be._check(be._lib.omx_download(be._ctx, C.c_void_p(back.ctypes.data), be._p(there), C.c_uint64(3), C.c_uint64(40)))
        assert np.array_equal(back, np.arange(3, 43))
        be._check(be._lib.omx_upload_staged(be._ctx, be._p(there), C.c_uint64(32), C.c_void_p(put.ctypes.data), C.c_uint64(16)))
        be.sync()
        after = other.download(there)
        assert (after[32:48] == 9).all() and after[48] == 48
    finally:
        other.close()
