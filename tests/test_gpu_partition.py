"""The work partition of the sweeps can be read, changed and put back."""
import pytest

from helpers import progress, state3

pytestmark = pytest.mark.gpu
G = 4.0 / 3.0


@pytest.mark.parametrize("form", ["fp64", "fp64fast", "fp32"])
def test_partition_read_back_and_set(form):
    """Setting what partition() gave leaves the chosen segments in use, at
    first and after another length: the marches of a small grid, which take
    segments of 1 cell there, keep their times (by segments of 8 cells they
    take two and a half times as long)."""
    from verona_amd import DeviceGrid
    from verona_amd._lib import VeronaHIPError
    progress(f"partition read back and set {form}")
    n, bc = 32, ("periodic",) * 6
    with DeviceGrid(3, n, n, n, G) as dev:
        dev.upload("P", state3(n, n, n, seed=5, jump=False))
        dev.fill_ghosts(bc)
        dev.prim_to_cons()
        dev.set_step(ref_mode=False, rec="wenoz", riemann="hllc", integrator="rk3", precision=form, n_iter=50, tol=1e-10,
                     floor=1e-7, cfl=0.1, dx=1 / n, dy=1 / n, dz=1 / n, bc=bc)

        def sweeps():
            best = 1e9
            for _ in range(5):
                dev.timing(2)
                for _ in range(3):
                    dev.step()
                best = min(best, sum(ms for k, (_, ms) in dev.timing_report().items() if k != "xsweep"))
                dev.timing(0)
            return best

        chosen = dev.partition()
        first = sweeps()
        dev.set_partition(*chosen)
        assert dev.partition() == chosen
        again = sweeps()
        dev.set_partition(chosen[0], chosen[1], 8)
        assert dev.partition() == (chosen[0], chosen[1], 8)
        eight = sweeps()
        dev.set_partition(*chosen)
        assert dev.partition() == chosen
        back = sweeps()
        for bad in (-1, 1, 7, 4097):
            with pytest.raises(VeronaHIPError):
                dev.set_partition(chosen[0], chosen[1], bad)
        assert dev.partition() == chosen
    progress(f"  us: chosen {1e3 * first:.1f}, set {1e3 * again:.1f}, 8 cells {1e3 * eight:.1f}, put back {1e3 * back:.1f}")
    assert max(again, back) < 1.25 * first < eight
