"""Batched tubes: whole tubes by persistent workgroups in the caller's launch
shape, and ranges of tubes with halos, each known to be the path that ran."""
import numpy as np
import pytest

from helpers import progress
from test_gpu_tubes import _oracle_tubes

pytestmark = pytest.mark.gpu
G1 = 5.0 / 3.0


def _batch():
    from verona_amd.tubes import shock_tube_batch
    return shock_tube_batch(48, lmin=40, lmax=700, seed=7)


@pytest.mark.parametrize("rec", ["minmod", "ppm", "wenoz"])
@pytest.mark.parametrize("riemann", ["hll", "hllc"])
def test_whole_tubes_in_every_form_and_shape(oracle, rec, riemann):
    """Whole tubes, eager and replayed graphs, in several launch shapes: the
    exact form gives the oracle's bits, the fast form the bits of its ranges
    and the oracle's values to 1e-12 relative L1 where both stay finite."""
    from verona_amd.tubes import Tubes
    progress(f"whole tubes {rec} {riemann}")
    lengths, rho, u, ux, dt, dx = _batch()
    O = _oracle_tubes(oracle, lengths, rho, u, ux, dt, dx, G1, rec, riemann, 24)
    with Tubes(lengths) as tb:
        tb.set_method(rec, riemann, 50, 1e-10)
        tb.set_split("always")
        assert tb.plan(24)[0] > 0 and tb.plan(24)[1] > len(lengths)
        tb.set_precision("fp64fast")
        tb.upload(rho, u, ux, dt, dx)
        tb.run(24)
        F = np.stack(tb.download())
        tb.set_split(False)
        assert tb.plan(24) == (0, 0)
        # a graph of one shape, captured and replayed, in both forms
        for block, grid, graph in [(64, 1, False), (128, 16, True), (128, 16, False), (1024, 3, False), (256, 48, True)]:
            for prec, want in (("fp64fast", F), ("fp64", O)):
                tb.set_precision(prec)
                tb.upload(rho, u, ux, dt, dx)
                for _ in range(3):
                    tb.run(8, block, grid, use_graph=graph)
                assert np.array_equal(np.stack(tb.download()), want, equal_nan=True), (block, grid, graph, prec)
    off = np.concatenate([[0], np.cumsum(lengths)])
    fin = lambda X: np.array([np.isfinite(X[:, off[t]:off[t + 1]]).all() for t in range(len(lengths))])
    both = fin(O) & fin(F)
    m = np.repeat(both, lengths)
    assert both.sum() >= 0.9 * fin(O).sum()
    for v in range(3):
        assert np.abs(F[v][m] - O[v][m]).sum() <= 1e-12 * np.abs(O[v][m]).sum()


@pytest.mark.parametrize("prec", ["fp64", "fp64fast"])
def test_ranges_and_whole_tubes_in_turn(prec):
    """Ranges swap the state buffers at each launch: a captured graph of whole
    tubes before and after them works on the current state."""
    from verona_amd.tubes import Tubes
    progress(f"ranges and whole tubes in turn {prec}")
    lengths, rho, u, ux, dt, dx = _batch()
    outs = []
    for turn in (False, True):
        with Tubes(lengths) as tb:
            tb.set_method("wenoz", "hllc", 50, 1e-10)
            tb.set_precision(prec)
            tb.upload(rho, u, ux, dt, dx)
            for k in range(9):
                tb.set_split("always" if turn and k % 3 == 1 else False)
                assert (tb.plan(4)[0] > 0) == (turn and k % 3 == 1)
                tb.run(4, 128, 16, use_graph=turn)
            outs.append(np.stack(tb.download()))
    assert np.array_equal(*outs, equal_nan=True)


def test_batches_left_whole(oracle):
    """Batches that fill the GPU one workgroup a tube are run whole without
    being told to."""
    from verona_amd.tubes import Tubes, shock_tube_batch
    progress("batches left whole")
    for n, lo, hi in ((4096, 256, 8192), (1280, 500, 500), (10000, 100, 300)):
        lengths, rho, u, ux, dt, dx = shock_tube_batch(n, lo, hi, seed=42)
        with Tubes(lengths) as tb:
            assert tb.plan(8) == (0, 0), (n, lo, hi)
            if n != 1280:
                continue
            tb.set_method("ppm", "hllc", 50, 1e-10)
            tb.upload(rho, u, ux, dt, dx)
            for _ in range(2):
                tb.run(4, 256, 1024, use_graph=True)
            G = np.stack(tb.download())
            for t in (0, 1, 640, 1279):
                c = slice(500 * t, 500 * (t + 1))
                O = _oracle_tubes(oracle, [500], rho[c], u[c], ux[c], dt[t:t + 1], dx[t:t + 1], G1, "ppm", "hllc", 8)
                assert np.array_equal(G[:, c], O, equal_nan=True), t


def test_autotune_measures_ranges_too(tmp_path):
    """autotune times ranges beside the launch shapes of whole tubes, sets the
    handle to the faster, also from its caches, and leaves the state alone; a
    handle kept to one path is tuned in that path alone."""
    import json

    from verona_amd import tubes
    from verona_amd.tubes import Tubes, shock_tube_batch
    progress("autotune and ranges")
    shapes = len(tubes.BLOCKS) * len(tubes.WAVES_PER_CU)
    f = tmp_path / "shapes.json"
    for n, L, ranges_win in ((2, 8000, True), (256, 1000, False)):
        lengths, rho, u, ux, dt, dx = shock_tube_batch(n, L, L, seed=3)
        outs = []
        for repeat in (0, 1, 2):
            with Tubes(lengths, gamma=1.61) as tb:
                tb.upload(rho, u, ux, dt, dx)
                tb.set_method("minmod", "hll", 50, 1e-10)
                if repeat == 2:
                    tubes._CACHE.clear()  # leaves the file
                shape = tb.autotune(probe_steps=1, cache_file=str(f))
                key = tb.signature() + ":ranges"
                if repeat == 0:
                    assert len(tb.autotune_trials) == shapes + 1
                    assert tb.autotune_trials[-1][0] < min(tb.autotune_trials[:-1])[0] or not ranges_win
                    assert json.loads(f.read_text())[key]["shape"] == list(tubes._CACHE[key])
                assert not hasattr(tb, "autotune_trials") or repeat == 0
                assert (tubes._CACHE[key] == ()) == (tb.plan(5, *shape) != (0, 0))
                if ranges_win:
                    assert tb.plan(5, *shape) != (0, 0) and shape == (128, 2 * tb.cu_count)
                tb.run(5, *shape)
                outs.append(np.stack(tb.download()))
                # another method is measured anew, ranges too, whatever won before
                if repeat == 0:
                    tb.set_method("ppm", "hllc", 50, 1e-10)
                    tb.autotune(probe_steps=1)
                    assert len(tb.autotune_trials) == shapes + 1
        assert np.array_equal(outs[0], outs[1], equal_nan=True) and np.array_equal(outs[0], outs[2], equal_nan=True)
    with Tubes([300, 500]) as tb:
        tb.set_method("minmod", "hll", 50, 1e-10)
        tb.upload(*(np.ones(800),) * 3, 1e-4, 1.0)
        tb.set_split("always")
        assert tb.autotune() == (128, 2 * tb.cu_count) and tb.autotune_trials == []
        tb.set_split(False)
        tb.autotune(probe_steps=1)
        assert len(tb.autotune_trials) == shapes and tb.plan(1) == (0, 0)


@pytest.mark.parametrize("n,length,shape,ranges", [(512, 500, (512, 512), False), (512, 500, (128, 512), True),
                                                   (256, 1000, (1024, 256), False), (256, 1000, (128, 512), True),
                                                   (64, 4000, (1024, 256), True), (1, 3000, (1024, 1), True)])
def test_ranges_only_where_faster_than_the_given_shape(n, length, shape, ranges):
    """Whether a batch runs in ranges depends on the launch shape that it is
    given: the faster path, measured, is the one that runs."""
    from verona_amd.tubes import Tubes, shock_tube_batch
    progress(f"{n} tubes of {length} in {shape}")
    lengths, rho, u, ux, dt, dx = shock_tube_batch(n, length, length, seed=5)
    with Tubes(lengths) as tb:
        tb.set_method("ppm", "hllc", 50, 1e-10)
        assert (tb.plan(32, *shape) != (0, 0)) == ranges
        ms = {}
        for mode in ("always", False):
            tb.set_split(mode)
            t = []
            for _ in range(4):
                tb.upload(rho, u, ux, dt, dx)
                t.append(tb.run(32, *shape, use_graph=False))
            ms[mode] = min(t)
        progress(f"  ranges {ms['always']:.3f} ms, whole tubes {ms[False]:.3f} ms")
        assert (ms["always"] < ms[False]) == ranges


def test_launches_of_very_many_steps():
    """Steps a launch stay where the ranges' halo (six cells a step, on both
    sides of a tube) fits an int, whatever the steps asked for; a run longer
    than one launch gives the bits of whole tubes."""
    from verona_amd.tubes import Tubes
    progress("very many steps")
    lengths = [40, 62]
    rng = np.random.default_rng(4)
    rho, u, ux = (1 + 0.1 * rng.standard_normal(102) for _ in range(3))
    dx = 1 / np.array(lengths)
    outs = []
    for on in (True, False):
        with Tubes(lengths) as tb:
            tb.set_split("always" if on else False)
            for n in (1, 4097, 2**31 - 1):
                k, ranges = tb.plan(n)
                assert (k > 0) == on and k <= n and 6 * k + max(lengths) < 2**31
            assert ranges == (2 if on else 0)
            tb.set_method("minmod", "hll", 50, 1e-10)
            tb.upload(rho, u, ux, 0.1 * dx, dx)
            tb.run(5000)
            outs.append(np.stack(tb.download()))
    assert np.isfinite(outs[0]).all() and np.array_equal(*outs)


@pytest.mark.parametrize("change", [dict(n_iter=1), dict(tol=1e-2)])
def test_graph_of_another_iteration_limit(change):
    """A captured graph holds the con2prim limit and tolerance it was captured
    with: other ones need another graph."""
    from verona_amd.tubes import Tubes
    progress(f"graph after {change}")
    lengths, rho, u, ux, dt, dx = _batch()
    outs = []
    with Tubes(lengths) as tb:
        tb.set_split(False)
        for graph in (True, False):
            for kw in ({}, change):
                tb.set_method("ppm", "hllc", **{"n_iter": 50, "tol": 1e-10, **kw})
                tb.upload(rho, u, ux, dt, dx)
                tb.run(6, 128, 16, use_graph=graph)
                outs.append(np.stack(tb.download()))
    assert np.array_equal(outs[0], outs[2], equal_nan=True)
    assert np.array_equal(outs[1], outs[3], equal_nan=True)
    assert not np.array_equal(outs[0], outs[1], equal_nan=True)
