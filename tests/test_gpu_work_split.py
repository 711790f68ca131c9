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


@pytest.mark.parametrize("n", [1, 3, 63, 64, 65, 129, 8191, 8193, 65536])
def test_training_gradient_of_any_batch(n):
    """Slices of the batch that are empty, partly filled or longer than the
    samples a block holds at a time.  FP32 sums of at most 1024 + 64 terms
    against 64 bits: 1e-4 of the gradient's norm, as the other gradient test."""
    import mlp_ref
    from verona_amd.c2p import Con2PrimBatch, c4_states
    progress(f"training gradient n={n}")
    with Con2PrimBatch(1 << 17, G) as cp:
        X, T, ok = cp.features(*c4_states(1 << 17, seed=9, gamma=G))
        X, T = X[ok][:n], T[ok][:n]
        assert len(X) == n
        params = mlp_ref.he_init(13)
        loss, g = cp.grad(X, T, params, qat=False, q_ref=0.01)
    lr, gr = mlp_ref.loss_grad(params, X, T, qat=False, q_ref=0.01)
    assert abs(loss - lr) <= 1e-4 * lr
    assert np.linalg.norm(g - gr) <= 1e-4 * np.linalg.norm(gr)


@pytest.mark.parametrize("scale", [1e-290, 1e-300, 2e-304, 3e-307, 5e-310, 1e-322])
def test_ppm_fluxes_on_tiny_values(oracle, scale):
    """The division by six of PPM's interface values where its quotient or
    the remainder of the correction is subnormal: the oracle's bits."""
    from helpers import from_oracle3, to_oracle3
    from verona_amd import DeviceGrid
    progress(f"ppm on tiny values {scale}")
    P = state3(20, 12, 9, seed=41)
    rng = np.random.default_rng(41)
    P[2:] = scale * rng.standard_normal(P[2:].shape)
    P[3][rng.random(P[3].shape) < 0.3] = 0.0
    Po = to_oracle3(P)
    sl = (slice(None), slice(2, -3), slice(2, -3), slice(2, -3))
    with DeviceGrid(3, 20, 12, 9, G) as dev:
        dev.upload("P", P)
        for dim, slot in enumerate(["Fx", "Fy", "Fz"]):
            dev.upload(slot, np.zeros_like(P))
            dev.fluxes(dim, 1e-7, "ppm", "hll")
            a = dev.download(slot)[sl]
            b = from_oracle3(oracle.fluxes3(Po, G, 1e-7, dim, "ppm", "hll"))[sl]
            assert np.array_equal(a, b)


@pytest.mark.parametrize("rec,riemann", [("ppm", "hllc"), ("wenoz", "hll"), ("minmod", "hllc")])
@pytest.mark.parametrize("lengths", [[8], [62], [63, 9], [248], [249], [250, 8, 247], [300, 17, 1001], [2000]])
def test_tubes_split_over_workgroups(oracle, rec, riemann, lengths):
    """Tubes around the cells a wave (62) and a workgroup (248) hold, in
    ranges with halos, for step counts that leave a short last launch: the
    oracle's bits."""
    from test_gpu_tubes import _oracle_tubes
    from verona_amd.tubes import Tubes
    progress(f"split tubes {lengths} {rec} {riemann}")
    rng = np.random.default_rng(3)
    lengths = np.array(lengths)
    n = int(lengths.sum())
    x = np.concatenate([(np.arange(L) + 0.5) / L for L in lengths])
    rho = np.where(x < 0.4, 1.0, 0.3) * (1 + 0.1 * rng.standard_normal(n))
    u = np.where(x < 0.6, 2.0, 0.5) * (1 + 0.1 * rng.standard_normal(n))
    ux = 0.3 * np.sin(9 * x) + 0.02 * rng.standard_normal(n)
    dx = 1.0 / lengths
    dt = 0.3 * dx
    with Tubes(lengths) as tb:
        tb.upload(rho, u, ux, dt, dx)
        tb.set_method(rec, riemann, 50, 1e-10)
        for k in (1, 18, 4):
            tb.run(k)
        got = np.stack(tb.download())
    want = _oracle_tubes(oracle, lengths, rho, u, ux, dt, dx, 5.0 / 3.0, rec, riemann, 23)
    assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("rec,riemann", [("wenoz", "hll"), ("ppm", "hllc"), ("minmod", "hll")])
@pytest.mark.parametrize("shape", [(4, 4, 4), (63, 8, 9), (64, 15, 6), (9, 16, 70), (5, 40), (130, 12)])
def test_flux_regions(oracle, shape, rec, riemann):
    """Fluxes of the kernel boundary around the sizes of its waves (63 faces
    of a stream of rows; 8 columns of 7 faces): the oracle's bits on every
    face of the region, nothing written outside it."""
    from helpers import from_oracle3, to_oracle3
    from verona_amd import DeviceGrid
    progress(f"flux regions {shape} {rec} {riemann}")
    nd = len(shape)
    P = state3(*shape, seed=6) if nd == 3 else state2(*shape, seed=6)
    Po = to_oracle3(P)
    sl = (slice(None),) + (slice(2, -3),) * nd
    mark = np.full(P.shape, 123.0, order="F")
    with DeviceGrid(nd, *shape, *((1,) if nd == 2 else ()), gamma=G) as dev:
        dev.upload("P", P)
        for dim, slot in enumerate(["Fx", "Fy", "Fz"][:nd]):
            dev.upload(slot, mark)
            dev.fluxes(dim, 1e-7, rec, riemann)
            a = dev.download(slot)
            f = oracle.fluxes3 if nd == 3 else oracle.fluxes2
            b = from_oracle3(f(Po, G, 1e-7, dim, rec, riemann))
            assert np.array_equal(a[sl], b[sl])
            a[sl] = 123.0
            assert (a == 123.0).all()


def test_large_copies_from_two_threads():
    """Copies large enough for the pinned staging (and the ragged last slice
    of one), repeated, from two threads that want it at once, into fresh and
    into used arrays: every byte arrives."""
    import threading

    from verona_amd import DeviceGrid
    progress("large copies")
    errors = []

    def go(seed, n):
        rng = np.random.default_rng(seed)
        P = np.asfortranarray(rng.standard_normal((5, n + 6, n + 5, n + 7)))
        with DeviceGrid(3, n, n - 1, n + 1, gamma=G) as dev:
            out = np.empty(P.shape, order="F")
            for k in range(4):
                P[:, k, :, :] += 1.0
                dev.upload("U", P)
                dev.download("U", out=out)
                if not (np.array_equal(out, P) and np.array_equal(dev.download("U"), P)):
                    errors.append((seed, k))
    threads = [threading.Thread(target=go, args=a) for a in ((1, 95), (2, 90), (3, 61))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


@pytest.mark.parametrize("form", ["fp64", "fp64fast"])
@pytest.mark.parametrize("rec,riemann", [("wenoz", "hllc"), ("ppm", "hll"), ("minmod", "hllc")])
@pytest.mark.parametrize("shape,kind", [((4, 5), "periodic"), ((63, 9), "outflow"), ((64, 20), "none"), ((66, 17), "outflow"),
                                        ((131, 40), "periodic")])
def test_x_inside_the_2d_march(shape, kind, rec, riemann, form):
    """2D: the x direction inside the y march gives the bits of its own sweep,
    ghost cells included, around the widths of a wave."""
    from verona_amd import DeviceGrid
    progress(f"2D x-y march {shape} {kind} {rec} {riemann} {form}")
    P = state2(*shape, seed=8)
    bc = (kind,) * 4 + ("none",) * 2
    outs = []
    for on in (True, False):
        with DeviceGrid(2, *shape, gamma=G) as dev:
            dev.set_xy_fusion(on)
            dev.upload("P", P)
            dev.fill_ghosts(bc)
            dev.prim_to_cons()
            dev.set_step(ref_mode=False, rec=rec, riemann=riemann, integrator="rk3", precision=form, n_iter=50, tol=1e-10,
                         floor=1e-7, cfl=0.3, dx=1 / shape[0], dy=1 / shape[1], bc=bc)
            for _ in range(3):
                dev.step()
            outs.append((dev.download("P"), dev.download("U")))
    for a, b in zip(*outs):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("form", ["fp64", "fp64fast"])
@pytest.mark.parametrize("shape,rec,kind", [((129, 12), "wenoz", "periodic"), ((130, 7), "ppm", "outflow"),
                                            ((129, 9, 6), "ppm", "outflow"), ((130, 6, 5), "wenoz", "periodic"),
                                            ((131, 5, 7), "minmod", "outflow"), ((4, 5, 9), "wenoz", "periodic"),
                                            ((20, 7, 6), "ppm", "outflow"), ((21, 9, 13), "wenoz", "outflow"),
                                            ((22, 17, 11), "ppm", "periodic"), ((31, 6, 10), "minmod", "none"),
                                            ((33, 12, 9), "wenoz", "none"), ((62, 5, 5), "ppm", "outflow"),
                                            ((63, 8, 7), "wenoz", "periodic"), ((64, 9, 6), "ppm", "periodic"),
                                            ((65, 7, 9), "minmod", "outflow"), ((97, 10, 8), "wenoz", "outflow")])
def test_x_march_with_a_narrow_last_wave(shape, rec, kind, form):
    """x inside the y march gives the bits of its own sweep, ghost cells
    included, where a wave holds the ends of one to four rows and where only
    one to three columns of a row are left for it: the wave before then reads
    ghost columns that no pass has written by the boundary rule."""
    from verona_amd import DeviceGrid
    progress(f"narrow last wave {shape} {rec} {kind} {form}")
    nd = len(shape)
    P = (state2 if nd == 2 else state3)(*shape, seed=11)
    bc = (kind,) * (2 * nd) + ("none",) * (6 - 2 * nd)
    outs = []
    for on in (True, False):
        with DeviceGrid(nd, *shape, gamma=G) as dev:
            dev.set_xy_fusion(on)
            dev.upload("P", P)
            dev.fill_ghosts(bc)
            dev.prim_to_cons()
            dev.set_step(ref_mode=False, rec=rec, riemann="hllc", integrator="rk3", precision=form, n_iter=50, tol=1e-10,
                         floor=1e-7, cfl=0.3, bc=bc, **{k: 1 / n for k, n in zip(("dx", "dy", "dz"), shape)})
            for _ in range(3):
                dev.step()
            outs.append((dev.download("P"), dev.download("U")))
    for a, b in zip(*outs):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("shape", [(660, 7, 620), (700, 50, 8), (330, 8, 311)])
def test_segments_of_wide_grids(shape):
    """Grids of so many columns that a march's segments are the fixed ones
    (also cut to a short axis): the bits of short segments."""
    from verona_amd import DeviceGrid
    progress(f"wide grid {shape}")
    P = state3(*shape, seed=3)
    bc = ("outflow",) * 6
    outs = []
    for seg in (None, 8):
        with DeviceGrid(3, *shape, gamma=G) as dev:
            if seg:
                rows, xseg, _ = dev.partition()
                dev.set_partition(rows, xseg, seg)
            dev.upload("P", P)
            dev.fill_ghosts(bc)
            dev.prim_to_cons()
            dev.set_step(ref_mode=False, rec="minmod", riemann="hll", integrator="rk2", precision="fp64fast", n_iter=50,
                         tol=1e-10, floor=1e-7, cfl=0.3, bc=bc, **{k: 1 / n for k, n in zip(("dx", "dy", "dz"), shape)})
            dev.step()
            outs.append(dev.download("P"))
    assert np.array_equal(*outs, equal_nan=True)
