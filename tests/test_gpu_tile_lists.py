"""Tile lists formed straight from the segments and through bins."""
import numpy as np
import pytest

import _oracle as O
from filsim_amd import abi, api, params
from helpers import random_segments, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,n,spread", [
    ((16, 16, 32), 1, 1.0),       # one row of tiles wide, one segment
    ((24, 16, 32), 63, 0.05),     # more than a tile's slab in few tiles
    ((64, 32, 48), 1023, 1.0),    # one segment short of a step
    ((64, 32, 48), 1025, 0.02),   # all in one row of tiles: long pool blocks
    ((144, 24, 32), 300, 1.0),    # 18 tiles a row: two wavefronts take two
    ((32, 40, 48), 4096, 1.0),    # most segments of the way without bins
    ((32, 40, 48), 4097, 1.0),    # fewest of the way through bins
    ((32, 40, 48), 5000, 0.02),   # crowded bins
    ((128, 128, 128), 2500, 0.3),  # rows times steps below the line
    ((320, 320, 320), 2500, 1.0),  # above it
])
def test_lists_match_vector_path(cuda, grid, n, spread):
    """Against the solver's vector path, which has no tile lists. FP64, other
    summation orders: 1e-12, the solver's parity bar, of |V| and of the larger
    of |W| and |V| / a. Three solves: the second must not see what the first
    left in the lists' pool, and segments that moved must change lists."""
    fp = params.fcm_params(grid)
    Y, F, T = random_segments(fp, n, seed=n + grid[0])
    Y *= spread
    shift = np.array(params.box(fp)) * 0.47
    with api.Fcm(fp, n) as fcm, api.Fcm(fp, n) as vec:
        vec.set_tuning(spread_mfma=0)
        for k in range(3):
            Yk = np.mod(Y + k * shift, params.box(fp))
            V, W = fcm.mobility_host(Yk, F, T)
            Vo, Wo = vec.mobility_host(Yk, F, T)
            top = max(np.linalg.norm(Wo), np.linalg.norm(Vo) / fp.a)
            assert rel(V, Vo) <= 1e-12, k
            assert np.linalg.norm(W - Wo) <= 1e-12 * top, k


@pytest.mark.parametrize("prec", [abi.FS_FP64, abi.FS_FP32])
def test_results_do_not_depend_on_capacity(cuda, prec):
    """A handle for 5,000 segments, which solves few segments without bins and
    many through them, against handles made for each count: the same bits, in
    turn, so that neither way sees what the other left (crowded tiles: both
    fill the lists' pool)."""
    fp = params.fcm_params((64, 32, 48))
    Y, F, T = random_segments(fp, 5000, seed=11)
    Y *= 0.5
    with api.Fcm(fp, 5000, precision=prec) as big:
        for n in (300, 5000, 4096, 4097, 300):
            V, W = big.mobility_host(Y[:n], F[:n], T[:n])
            with api.Fcm(fp, n, precision=prec) as own:
                Vo, Wo = own.mobility_host(Y[:n], F[:n], T[:n])
            assert np.array_equal(V, Vo) and np.array_equal(W, Wo), n


def test_binned_groups_equal_unbatched(cuda):
    """Two suspensions of more segments than the way without bins takes,
    stepped with fused stages and one after another: the same bits."""
    _groups_equal_unbatched((160,), (260, 270), (18, 20), (4097, 10**6))


@pytest.mark.parametrize("grid,nfil,nw,segments", [
    (50, (20, 24), (10, 12), (1, 4096)),       # without bins
    (150, (240, 250), (18, 20), (4097, 10**6)),  # through bins
])
def test_groups_on_cut_grids_equal_unbatched(cuda, grid, nfil, nw, segments):
    """The same on grids whose last tiles are cut off."""
    _groups_equal_unbatched((grid,), nfil, nw, segments)


def _groups_equal_unbatched(grids, nfil, nw, segments):
    solo, bat = [], []
    for seed in (1, 2):
        fp, sp, nws, props, st, info = params.sweep_point(
            seed, grids=grids, nfil_range=nfil, nw_range=nw,
            precision=abi.FS_FP32, tol=1e-4, dt=0.01)
        assert segments[0] <= info["segments"] <= segments[1]
        for group in (solo, bat):
            s = api.System(sp, nws, props)
            s.set_state(**st)
            group.append(s)
    batch = api.Batch(bat)
    batch.set_fused(True)
    assert batch.timestep(1) == [s.timestep(1) for s in solo]
    for a, b in zip(solo, bat):
        sa, sb = a.get_state(), b.get_state()
        for k in ("X", "U", "q", "lam"):
            assert np.array_equal(sa[k], sb[k]), k
    batch.close()


@pytest.mark.parametrize("ngd", [6, 8, 10, 12, 16, 20, 24])
def test_cut_tiles_match_vector_path(cuda, ngd):
    """Grids whose axes are no multiples of the tiles: cut by one to three
    axes, by 2 to 14 points, lines that are not 16-byte aligned, boxes narrower
    than a stencil and a tile. Bounds as above in FP64; FP32 1e-5, the bar of
    the solver's FP32 tests."""
    for grid in ((30, 36, 50), (40, 40, 40), (54, 30, 90), (36, 50, 48),
                 (32, 40, 54), (100, 32, 48), (30, 30, 60), (50, 90, 80)):
        if min(grid) < ngd + 4:
            continue
        fp = params.fcm_params(grid, ngd=ngd)
        n = 400
        Y, F, T = random_segments(fp, n, seed=sum(grid) + ngd)
        for prec, bar in ((abi.FS_FP64, 1e-12), (abi.FS_FP32, 1e-5)):
            with api.Fcm(fp, n, precision=prec) as fcm, \
                    api.Fcm(fp, n, precision=prec) as vec:
                vec.set_tuning(spread_mfma=0)
                V, W = fcm.mobility_host(Y, F, T)
                Vo, Wo = vec.mobility_host(Y, F, T)
            top = max(np.linalg.norm(Wo), np.linalg.norm(Vo) / fp.a)
            assert rel(V, Vo) <= bar, (grid, prec)
            assert np.linalg.norm(W - Wo) <= bar * top, (grid, prec)


@pytest.mark.parametrize("ngd", [12, 20, 24])
@pytest.mark.parametrize("grid", [(50, 90, 80), (54, 36, 90), (90, 100, 54)])
def test_cut_tiles_through_bins(cuda, grid, ngd):
    """More segments than the way without bins takes: one bin more on a cut
    axis (up to 100 bins a tile, two steps of 64), pool blocks of crowded
    tiles, and a second solve after the segments moved. Against the vector path
    or, where that has no tile for the grid, the FP64 oracle; bounds as
    above."""
    fp = params.fcm_params(grid, ngd=ngd)
    n = 4500
    Y, F, T = random_segments(fp, n, seed=sum(grid) + ngd)
    box = np.array(params.box(fp))
    Y[n // 2:] *= 0.3  # half of them crowded
    moved = [Y, np.mod(Y + 0.47 * box, box)]
    with api.Fcm(fp, n) as vec:
        try:
            vec.set_tuning(spread_mfma=0)
            ref = [vec.mobility_host(Yk, F, T) for Yk in moved]
        except abi.FsError:
            ref = [O.mobility(fp, Yk, F, T) for Yk in moved]
    for prec, bar in ((abi.FS_FP64, 1e-12), (abi.FS_FP32, 1e-5)):
        with api.Fcm(fp, n, precision=prec) as fcm:
            for k, (Vo, Wo) in enumerate(ref):
                V, W = fcm.mobility_host(moved[k], F, T)
                top = max(np.linalg.norm(Wo), np.linalg.norm(Vo) / fp.a)
                assert rel(V, Vo) <= bar, (prec, k)
                assert np.linalg.norm(W - Wo) <= bar * top, (prec, k)
