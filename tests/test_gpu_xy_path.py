"""Where the x direction runs inside the y march, and that switching it off
gives the same bits by another kernel."""
import numpy as np
import pytest

from helpers import progress, state2, state3

pytestmark = pytest.mark.gpu
G = 4.0 / 3.0


@pytest.mark.parametrize("rec", ["wenoz", "ppm", "minmod"])
@pytest.mark.parametrize("form", ["fp64", "fp64fast", "fp32"])
@pytest.mark.parametrize("shape", [(70, 9), (130, 12), (70, 9, 8), (20, 7, 6)])
def test_fused_and_separate_x_are_different_kernels(shape, form, rec):
    """3D FP64 forms, 2D fast form and 2D exact WENO-Z: the x-y march runs with
    the fusion on and the x and y sweeps with it off, the same bits; the other
    forms run the sweeps either way."""
    from verona_amd import DeviceGrid
    progress(f"x-y path {shape} {form} {rec}")
    nd = len(shape)
    fused = form != "fp32" and (nd == 3 or form == "fp64fast" or rec == "wenoz")
    P = (state2 if nd == 2 else state3)(*shape, seed=8)
    bc = ("outflow",) * (2 * nd) + ("none",) * (6 - 2 * nd)
    outs = []
    for on in (True, False):
        with DeviceGrid(nd, *shape, *((1,) if nd == 2 else ()), gamma=G) as dev:
            dev.set_xy_fusion(on)
            dev.upload("P", P)
            dev.fill_ghosts(bc)
            dev.prim_to_cons()
            dev.set_step(ref_mode=False, rec=rec, riemann="hllc", integrator="rk3", precision=form, n_iter=50, tol=1e-10,
                         floor=1e-7, cfl=0.3, bc=bc, **{k: 1 / n for k, n in zip(("dx", "dy", "dz"), shape)})
            dev.timing(1)
            for _ in range(2):
                dev.step()
            ran = dev.timing_report()
            outs.append((dev.download("P"), dev.download("U")))
        if fused and on:
            assert ran["xysweep"][0] == 6 and not {"xsweep", "ysweep"} & set(ran), ran
        else:
            assert ran["xsweep"][0] == ran["ysweep"][0] == 6 and "xysweep" not in ran, ran
    for a, b in zip(*outs):
        assert np.array_equal(a, b, equal_nan=True)
