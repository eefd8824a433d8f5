"""What a full rebuild does in its short forms, against the oracle: the levels
of a small box in one workgroup (boxes on both sides of its limit, one to four
levels, with and without dilation), the leaves' bounds from the points' bounds
(and from the leaves where a point is negative, infinite or NaN), slots and the
subcell mapping of a tree whose leaves are all in use."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


def _check(gpu, pts, r, oracle=True):
    import oracle as O
    v = gpu.VolumeGVDB(0)
    v.Configure(*H.TREE)
    v.SetChannelDefault(16, 16, 1)
    v.AddChannel(0, gpu.T_FLOAT, 1)
    v.SetPoints(pts)
    v.RequestFullRebuild(True)
    v.RebuildTopology(len(pts), r, H.ZERO3)
    v.FinishTopology(False, True)
    # the bounds are those of the leaves
    i, leaf = v.info(), v.pool(0, 0)["mPos"]
    assert np.array_equal(i["obj_min"], leaf.min(0).astype(np.float32))
    assert np.array_equal(i["obj_max"], (leaf.max(0) + 8).astype(np.float32))
    if not oracle:
        v.close()
        return
    o = O.Oracle()
    assert o.rebuild_topology(pts, r) == 0
    o.finish_topology()
    H.assert_pools_equal(v, o)
    b = o.bounds()
    assert np.array_equal(i["obj_min"], b["obj_min"]) and np.array_equal(i["obj_max"], b["obj_max"])
    v.UpdateAtlas()
    assert o.update_atlas() == 0
    H.assert_pools_equal(v, o)
    assert np.array_equal(v.atlas_map(), o.atlas_map())
    v.close()


def _box(side, n, seed, lo=(0.0, 0.0, 0.0)):
    # n points in a box of `side` voxels, two of them at its corners
    g = np.random.default_rng(seed)
    p = np.asarray(lo) + np.asarray(side) * g.random((n, 3))
    p[0], p[1] = lo, np.asarray(lo) + np.asarray(side)
    return p.astype(np.float32)


# small boxes (one workgroup) and large ones (level by level), up to four levels
@pytest.mark.parametrize("r,side", [(2.0, (40, 20, 40)), (2.0, (480, 480, 480)), (2.0, (505, 500, 498)), (0.5, (500, 500, 500)),
                                    (0.5, (640, 640, 640)), (5.5, (70, 400, 33)), (2.0, (3000, 40, 40)), (1.0, (9, 9, 9))])
def test_levels_and_bounds(gpu, r, side):
    _check(gpu, _box(side, 3000, 5, (17.5, 33.0, 72.25)), r)


# one grid takes the one-workgroup form up to 3072 words (49,000 bricks with
# dilation, 36 a side), each further one of a batch adds 512
@pytest.mark.parametrize("side", [(262, 260, 262), (272, 270, 273), (277, 278, 276), (282, 283, 281), (300, 300, 300)])
def test_levels_around_the_one_grid_limit(gpu, side):
    _check(gpu, _box(side, 3000, 6, (17.5, 33.0, 72.25)), 2.0)


@pytest.mark.parametrize("grids,side", [(2, 285), (2, 305), (5, 320), (5, 345), (30, 470), (30, 510)])
def test_levels_of_a_batch_around_its_limit(gpu, grids, side):
    """The largest grid decides for the call; pools equal those of single calls."""
    sets = [_box((side, side, side) if k == 1 else (40 + 9 * k, 50, 60), 800, 7 + k, (17.5, 33.0, 72.25)) for k in range(grids)]
    vols = []
    for p in sets:
        v = gpu.VolumeGVDB(0)
        v.Configure(*H.TREE)
        v.SetPoints(p)
        v.RequestFullRebuild(True)
        vols.append(v)
    b = gpu.GridBatch(0, grids)
    b.RebuildTopology(vols, [len(p) for p in sets], 2.0)
    b.synchronize()
    for v, p in zip(vols, sets):
        one, _ = H.gpu_volume(gpu, p, 2.0, stop_after="topology")
        H.assert_pools_equal(v, one)
        one.close()
    b.close()
    for v in vols:
        v.close()


def test_bounds_at_the_root_corner_and_border(gpu):
    _check(gpu, _box((100, 100, 100), 500, 6), 3.0)   # dilation below zero
    # dilation past the root's far side, where the reference's walk ends
    # elsewhere: the bounds of the leaves that are there
    _check(gpu, _box((55.9, 55.9, 55.9), 500, 7, (8.0, 8.0, 8.0)), 2.0, oracle=False)
    _check(gpu, _box((30, 30, 30), 500, 7, (17.5, 33.0, 65.25)), 2.0, oracle=False)


@pytest.mark.parametrize("odd", ["negative", "inf", "nan", "one axis"])
def test_points_outside_the_build(gpu, odd):
    pts = _box((120, 90, 100), 800, 8, (20.0, 20.0, 20.0))
    if odd == "negative":
        pts[100] = (-5.0, 60.0, 300.0)
    elif odd == "inf":
        pts[100] = (60.0, np.inf, 60.0)
    elif odd == "nan":
        pts[100] = (np.nan, 5.0, 130.0)
    else:
        pts[100] = (60.0, -1.0, 60.0)
    if odd == "inf":
        # an infinite bound is no tree: refused as before
        v = gpu.VolumeGVDB(0)
        v.Configure(*H.TREE)
        v.SetPoints(pts)
        v.RequestFullRebuild(True)
        with pytest.raises(gpu.GVDBError):
            v.RebuildTopology(len(pts), 2.0, H.ZERO3)
        v.close()
        return
    # (a point that is none counts in the reference's topology: leaves only)
    _check(gpu, pts, 2.0, oracle=odd != "nan")


def test_subcell_mapping_and_tables(gpu):
    import oracle as O
    pts = _box((120, 90, 100), 3000, 9, (20.0, 20.0, 20.0))
    v, n = H.gpu_volume(gpu, pts, 2.0, stop_after="insert")
    assert np.array_equal(v.subcells()["mapping"], np.arange(len(v.pool(0, 0)), dtype=np.uint32))
    o, m = H.oracle_volume(O, pts, 2.0, stop_after="insert")
    a, b = v.subcells(), o.subcells(m)
    assert n == m
    for k in ("cnt", "off", "pos", "nid"):
        assert np.array_equal(np.asarray(a[k]).reshape(-1), np.asarray(b[k]).reshape(-1)), k
    v.close()
