"""Large copies of the C ABI between the device and memory that is not pageable."""
import ctypes as C

import numpy as np
import pytest

from helpers import progress

pytestmark = pytest.mark.gpu
G = 4.0 / 3.0


@pytest.mark.parametrize("kind", ["device", "pinned"])
def test_large_copies_of_memory_the_runtime_knows(kind):
    """Arrays on the device, or pinned, in the place of the host arrays of
    large uploads and downloads go through the runtime at any size (CPU threads
    cannot copy device memory), before and after staging memory exists."""
    from test_zz_no_alloc import D2H, H2D, _hip

    from verona_amd import DeviceGrid, _lib
    progress(f"large copies {kind}")
    hip = _hip()
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.hipHostFree.argtypes = [C.c_void_p]
    n = 100
    rng = np.random.default_rng(2)
    P = np.asfortranarray(rng.standard_normal((5, n + 6, n + 6, n + 6)))
    assert P.nbytes > 24 << 20  # staged when pageable
    at = C.c_void_p()
    if kind == "device":
        assert hip.hipMalloc(C.byref(at), P.nbytes) == 0
    else:
        assert hip.hipHostMalloc(C.byref(at), P.nbytes, 0) == 0
    try:
        got = np.empty_like(P, order="F")
        with DeviceGrid(3, n, n, n, gamma=G) as dev:
            for k in range(3):
                assert hip.hipMemcpy(at, P.ctypes.data, P.nbytes, H2D) == 0
                _lib.check(dev.lib.vrn_upload(dev.h, _lib.SLOT["U"], C.cast(at, _lib._DP)), "upload")
                assert np.array_equal(dev.download("U"), P)
                dev.upload("U", P + k)
                _lib.check(dev.lib.vrn_download(dev.h, _lib.SLOT["U"], C.cast(at, _lib._DP)), "download")
                assert hip.hipMemcpy(got.ctypes.data, at, P.nbytes, D2H) == 0
                assert np.array_equal(got, P + k)
    finally:
        assert (hip.hipFree if kind == "device" else hip.hipHostFree)(at) == 0
