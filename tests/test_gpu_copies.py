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
    import torch

    from verona_amd import DeviceGrid, _lib
    progress(f"large copies {kind}")
    n = 100
    rng = np.random.default_rng(2)
    P = np.asfortranarray(rng.standard_normal((5, n + 6, n + 6, n + 6)))
    assert P.nbytes > 24 << 20  # staged when pageable
    flat = torch.from_numpy(P.ravel(order="F").copy())
    a = flat.cuda() if kind == "device" else flat.pin_memory()
    b = torch.empty_like(a)
    torch.cuda.synchronize()
    at = lambda t: C.cast(C.c_void_p(t.data_ptr()), _lib._DP)
    with DeviceGrid(3, n, n, n, gamma=G) as dev:
        for k in range(3):
            _lib.check(dev.lib.vrn_upload(dev.h, _lib.SLOT["U"], at(a)), "upload")
            assert np.array_equal(dev.download("U"), P)
            dev.upload("U", P + 1.0)
            _lib.check(dev.lib.vrn_download(dev.h, _lib.SLOT["U"], at(b)), "download")
            assert torch.equal(b, a + 1.0)
