"""Device-to-host copies of whole fields: below the staged copy's threshold of
4 MiB, just above it with a short last chunk, and at the headline size, where a
field set on the device comes back bit for bit; and from several threads at
once, of which one gets the pinned slots and the others the plain copy; and
into pinned and into device memory, which take the plain copy at any size."""
import ctypes as C
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import _cases as K

pytestmark = pytest.mark.gpu


def _event(N):
    import ipglasma_amd as I
    return I.Event(K.params("pPb", N=N, Ny=1), seed=3)


# 18 planes of N^2 doubles: 2.4, 5.3, 37.7 MB
@pytest.mark.parametrize("N", [128, 192, 512])
def test_field_round_trip(N):
    ev = _event(N)
    a = np.random.default_rng(N).normal(size=(N * N, 18))
    ev.set_field("Ux", a)
    np.testing.assert_array_equal(ev.field("Ux"), a)
    ev.close()


def test_field_round_trip_from_threads():
    import ipglasma_amd as I

    def go(k):
        ev = _event(256)
        a = np.random.default_rng(k).normal(size=(256 * 256, 18))
        right = 0
        for _ in range(5):
            ev.set_field("Ux", a)
            right += np.array_equal(ev.field("Ux"), a)
        ev.close()
        return right

    with ThreadPoolExecutor(4) as pool:
        # result() raises what a thread raised
        assert [f.result() for f in [pool.submit(go, k) for k in range(4)]] == [5] * 4
    I.release_cached_memory()  # hands the slots back; the next copy makes them again
    test_field_round_trip(192)


# 10 planes of N^2 doubles: 1.3 and 5.2 MB
@pytest.mark.parametrize("N", [128, 256])
@pytest.mark.parametrize("where", ["pinned", "device"])
def test_tmunu_into_memory_the_device_reaches(N, where):
    import _hipmem
    import ipglasma_amd as I
    ev = _event(N)
    while not ev.init():
        pass
    ev.run()
    if where == "device":
        out = _hipmem.DeviceArray((10, N * N), host=np.full((10, N * N), -1.0))
        assert I.lib().ipg_get_tmunu(ev._c, C.cast(out.ptr, C.POINTER(C.c_double))) == 0
        got = out.download()
    else:
        h = _hipmem.hip()
        h.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
        h.hipHostFree.argtypes = [C.c_void_p]
        p = C.c_void_p()
        assert h.hipHostMalloc(C.byref(p), 80 * N * N, 0) == 0
        d = C.cast(p, C.POINTER(C.c_double))
        out = np.ctypeslib.as_array(d, (10, N * N))
        out[:] = -1.0
        assert I.lib().ipg_get_tmunu(ev._c, d) == 0
        got = out.copy()
        h.hipHostFree(p)
    np.testing.assert_array_equal(got, ev.tmunu())
    ev.close()
