"""GatherDensity over bricks with many points a voxel (the dense kernel) against
the oracle: blobs that fill bricks, fill part of them, or lie on a few voxels,
near the origin too (where the distances are float), at the radii of every
variant, FP32 and FP16, one grid, a batch and a graph replay; repeated gathers
after one insert (the list of dense bricks is reused); gathers recorded without
their insert, after a replayed insert and after a refused recording."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu

REL_TOL = 1e-5


def _points(kind, n, seed):
    g = np.random.default_rng(seed)
    sparse = 20.0 + 110.0 * g.random((600, 3))
    if kind == "full":         # several a voxel over 24^3 voxels
        p = 56.0 + 24.0 * g.random((n, 3))
    elif kind == "half":       # dense in half a brick
        p = np.array([64.0, 64.0, 64.0]) + np.array([8.0, 3.7, 8.0]) * g.random((n, 3))
    elif kind == "lattice":    # on voxels and halfway between: equal distances
        p = 60.0 + 0.5 * g.integers(0, 30, (n, 3))
    elif kind == "corner":     # the brick at the origin: float distances
        p = 0.02 + 7.9 * g.random((n, 3))
    else:                      # a few voxels
        p = np.array([75.2, 61.7, 66.1]) + 0.8 * g.standard_normal((n, 3))
    return np.concatenate([p, sparse]).astype(np.float32)


def _want(pts, r):
    import oracle as O
    o, m = H.oracle_volume(O, pts, r, precision=64)
    return o, m


CASES = [(k, n, r) for k, n in (("full", 60000), ("half", 9000), ("lattice", 30000), ("corner", 9000), ("few", 8000))
         for r in (1.0, 2.0, 2.25, 3.0, 4.5) if not (k == "corner" and r > 4.0)]


@pytest.mark.parametrize("kind,n,r", CASES)
def test_dense_bricks_match_oracle(gpu, kind, n, r):
    pts = _points(kind, n, 11)
    v, m = H.gpu_volume(gpu, pts, r)
    o, k = _want(pts, r)
    assert m == k
    info = o.atlas_info()
    _, rel, zeros = H.brick_density_errors(v.atlas(), o.atlas(64), o.atlas_map(), info["cnt"])
    assert zeros == 0 and rel <= REL_TOL
    a = v.atlas().copy()
    for _ in range(3):
        v.GatherDensity(4, len(pts), r, H.ZERO3, m, 0, 0, False)
        v.UpdateApron(0, 0.0)
        assert np.array_equal(v.atlas().view(np.uint32), a.view(np.uint32))
    v.close()


def test_dense_bricks_half_batch_and_graph(gpu):
    r = 2.0
    sets = [_points("full", 60000, 12), _points("few", 8000, 13), _points("half", 500, 14)]
    vols, one = [], []
    for p in sets:
        v, m = H.gpu_volume(gpu, p, r, atlas_type=gpu.T_HALF)
        one.append(v.atlas(0, np.float16).copy())
        vols.append(v)
    b = gpu.GridBatch(0, 3)
    n = [len(p) for p in sets]
    b.ClearChannel(vols, 0)
    lens = b.InsertPointsSubcell(vols, 4, n, r)
    b.GatherDensity(vols, 4, lens, r, 0)
    b.UpdateApron(vols, 0, 0.0)
    b.synchronize()
    for v, a in zip(vols, one):
        assert np.array_equal(v.atlas(0, np.float16).view(np.uint16), a.view(np.uint16))
    b.close()
    # a recording made of sparse points replays dense ones written in place
    p = sets[0]
    v, m = H.gpu_volume(gpu, p, r)
    want = v.atlas().copy()
    g = np.random.default_rng(3)
    thin = p.copy()
    thin[:60000] = (48.0 + 40.0 * g.random((60000, 3))).astype(np.float32)
    v.RequestFullRebuild(True)
    v.SetPoints(np.concatenate([p, thin]))
    v.RebuildTopology(2 * len(p), r, H.ZERO3)
    v.FinishTopology(False, True)
    v.UpdateAtlas()

    def chain():
        v.ClearChannel(0)
        ln = v.InsertPointsSubcell(4, len(p), r, H.ZERO3)
        v.GatherDensity(4, len(p), r, H.ZERO3, ln, 0, 0, False)
        v.UpdateApron(0, 0.0)

    v.SetPoints(thin)
    chain()
    v.synchronize()
    thin_atlas = v.atlas().copy()
    v.CaptureBegin()
    chain()
    gr = v.CaptureEnd()
    v.SetPoints(p)
    chain()
    v.synchronize()
    dense_atlas = v.atlas().copy()
    assert np.count_nonzero(dense_atlas) > 0 and want.shape[1:] == dense_atlas.shape[1:]
    for pts, a in ((thin, thin_atlas), (p, dense_atlas), (thin, thin_atlas), (p, dense_atlas)):
        v.SetPoints(pts)
        gr.launch()
        gr.synchronize()
        assert np.array_equal(v.atlas().view(np.uint32), a.view(np.uint32))
    gr.close()
    for x in vols + [v]:
        x.close()


def _thin_and_dense(gpu):
    """A grid over the union of two point sets of one size (one sparse, one
    with dense bricks), its buffers grown by a chain of each, and what the
    chain gives for each: (volume, {name: points}, {name: atlas}, {name: entries})."""
    r = 2.0
    dense = _points("full", 60000, 21)
    g = np.random.default_rng(22)
    thin = dense.copy()
    thin[:60000] = (48.0 + 40.0 * g.random((60000, 3))).astype(np.float32)
    sets = dict(thin=thin, dense=dense)
    v = gpu.VolumeGVDB(0)
    v.Configure(*H.TREE)
    v.SetChannelDefault(16, 16, 1)
    v.AddChannel(0, gpu.T_FLOAT, 1)
    v.SetPoints(np.concatenate([thin, dense]))
    v.RequestFullRebuild(True)
    v.RebuildTopology(2 * len(thin), r, H.ZERO3)
    v.FinishTopology(False, True)
    v.UpdateAtlas()
    atlas, entries = {}, {}
    for k in ("dense", "thin"):
        v.SetPoints(sets[k])
        v.ClearChannel(0)
        entries[k] = v.InsertPointsSubcell(4, len(thin), r, H.ZERO3)
        v.GatherDensity(4, len(thin), r, H.ZERO3, entries[k], 0, 0, False)
        v.UpdateApron(0, 0.0)
        v.synchronize()
        atlas[k] = v.atlas().view(np.uint32).copy()
    assert not np.array_equal(atlas["thin"], atlas["dense"])
    return v, sets, atlas, entries


def test_recorded_gather_follows_later_inserts(gpu):
    """GatherDensity and UpdateApron recorded alone, after an insert of sparse
    points: every replay gathers what the last insert binned, dense bricks too."""
    v, sets, atlas, entries = _thin_and_dense(gpu)
    n = len(sets["thin"])
    v.CaptureBegin()
    v.GatherDensity(4, n, 2.0, H.ZERO3, entries["thin"], 0, 0, False)
    v.UpdateApron(0, 0.0)
    gr = v.CaptureEnd()
    for k in ("dense", "thin", "dense", "dense"):
        v.SetPoints(sets[k])
        v.ClearChannel(0)
        assert v.InsertPointsSubcell(4, n, 2.0, H.ZERO3) == entries[k]
        gr.launch()
        gr.synchronize()
        assert np.array_equal(v.atlas().view(np.uint32), atlas[k]), k
    gr.close()
    v.close()


@pytest.mark.parametrize("wait", [True, False])
def test_eager_gather_after_a_replayed_insert(gpu, wait):
    """The chain recorded; an eager insert of sparse points; a replay over
    dense ones; then an eager gather (after the replay's wait or before it)."""
    v, sets, atlas, entries = _thin_and_dense(gpu)
    n = len(sets["thin"])
    v.CaptureBegin()
    v.InsertPointsSubcell(4, n, 2.0, H.ZERO3)
    gr = v.CaptureEnd()
    for _ in range(2):
        v.SetPoints(sets["thin"])
        ln = v.InsertPointsSubcell(4, n, 2.0, H.ZERO3)
        assert ln == entries["thin"]
        v.SetPoints(sets["dense"])
        v.ClearChannel(0)
        gr.launch()
        if wait:
            gr.synchronize()
            ln = entries["dense"]
        v.GatherDensity(4, n, 2.0, H.ZERO3, ln, 0, 0, False)
        v.UpdateApron(0, 0.0)
        v.synchronize()
        gr.synchronize()
        assert np.array_equal(v.atlas().view(np.uint32), atlas["dense"])
    gr.close()
    v.close()


def test_dense_bricks_after_a_refused_recording(gpu):
    """A grid's first gather inside a recording grows its buffers, so the
    recording is refused; the calls run directly afterwards all the same."""
    pts, r = _points("full", 60000, 23), 2.0
    want, _ = H.gpu_volume(gpu, pts, r)
    v, n = H.gpu_volume(gpu, pts, r, stop_after="insert")
    v.CaptureBegin()
    v.GatherDensity(4, len(pts), r, H.ZERO3, n, 0, 0, False)
    with pytest.raises(gpu.GVDBError) as e:
        v.CaptureEnd()
    assert e.value.code == gpu.ERR_STATE
    for _ in range(2):
        v.ClearChannel(0)
        v.GatherDensity(4, len(pts), r, H.ZERO3, n, 0, 0, False)
        v.UpdateApron(0, 0.0)
        v.synchronize()
        assert np.array_equal(v.atlas().view(np.uint32), want.atlas().view(np.uint32))
    v.close()
    want.close()
