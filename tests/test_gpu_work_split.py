"""Rules that choose a kernel's work split by size: results do not depend on it."""
import numpy as np
import pytest

from helpers import progress, state2, state3
from test_gpu_parity3d import G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4, 4, 4), (40, 4, 9), (7, 66, 5), (64, 64, 64), (130, 33, 47), (70, 9), (4, 130),
                                   (256, 251)])
@pytest.mark.parametrize("form", ["fp64", "fp64fast", "fp32"])
def test_automatic_march_segments(shape, form):
    """The automatic segments (1 cell and up on small grids) give the bits of
    one whole-length segment."""
    from verona_amd import DeviceGrid
    progress(f"march segments {shape} {form}")
    nd = len(shape)
    P = state3(*shape, seed=5) if nd == 3 else state2(*shape, seed=5)
    bc = ("periodic",) * (2 * nd) + ("none",) * (6 - 2 * nd)
    outs = []
    for whole in (False, True):
        with DeviceGrid(nd, *shape, *((1,) if nd == 2 else ()), gamma=G) as dev:
            if whole:
                r, x, s = dev.partition()
                dev.set_partition(r, x, max(8, max(shape)))
            dev.upload("P", P)
            dev.fill_ghosts(bc)
            dev.prim_to_cons()
            dev.set_step(ref_mode=False, rec="wenoz", riemann="hllc", integrator="rk3", precision=form, n_iter=50,
                         tol=1e-10, floor=1e-7, cfl=0.3, dx=1 / shape[0], dy=1 / shape[1],
                         dz=1 / shape[2] if nd == 3 else 1.0, bc=bc)
            for _ in range(2):
                dev.step()
            outs.append((dev.download("P"), dev.download("U")))
    for a, b in zip(*outs):
        assert np.array_equal(a, b, equal_nan=True)
