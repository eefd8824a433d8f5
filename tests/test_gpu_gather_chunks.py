"""Gathers over bricks with more candidates than one pass of a workgroup
stages: level set, accumulated density and colours of a dense blob (up to
thousands of points in a brick) beside sparse points, at one and two subcells
of reach, against the oracle."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu

REL_TOL = 1e-5


def _blob(n, seed, spread):
    g = np.random.default_rng(seed)
    dense = np.array([101.3, 97.6, 103.2]) + spread * g.standard_normal((n, 3))
    sparse = 70.0 + 60.0 * g.random((400, 3))
    return np.clip(np.concatenate([dense, sparse]), 20.0, 200.0).astype(np.float32)


def _gpu(gpu, pts, r, clr):
    v = gpu.VolumeGVDB(0)
    v.Configure(*H.TREE)
    v.SetChannelDefault(16, 16, 1)
    v.AddChannel(0, gpu.T_FLOAT, 1)
    v.AddChannel(1, gpu.T_UCHAR4, 1)
    v.SetPoints(pts, clr)
    v.RequestFullRebuild(True)
    v.RebuildTopology(len(pts), r, H.ZERO3)
    v.FinishTopology(False, True)
    v.UpdateAtlas()
    v.ClearChannel(0)
    v.ClearChannel(1)
    n = v.InsertPointsSubcell(4, len(pts), r, H.ZERO3)
    return v, n


def _oracle(pts, r, clr):
    import oracle as O
    o = O.Oracle()
    assert o.rebuild_topology(pts, r) == 0
    o.finish_topology()
    assert o.update_atlas() == 0
    o.add_color_channel()
    o.clear_channel()
    rc, n = o.insert_points_subcell(pts, r, 4, colors=clr)
    assert rc == 0
    return o, n


# spread 1.5: every point within a few subcells; n around the 512 candidates
# of a pass, several passes, and past 65,536 / 255 points in a subcell
@pytest.mark.parametrize("r", [2.0, 4.0])
@pytest.mark.parametrize("n,spread", [(300, 1.5), (513, 1.0), (1100, 2.0), (9000, 1.5)])
def test_dense_blob(gpu, r, n, spread):
    pts = _blob(n, n, spread)
    clr = np.random.default_rng(n).integers(0, 1 << 32, len(pts), dtype=np.uint64).astype(np.uint32)
    clr[:n // 2] = 0xFFFFFFFF
    v, m = _gpu(gpu, pts, r, clr)
    o, k = _oracle(pts, r, clr)
    assert m == k
    v.GatherLevelSet(4, len(pts), r, H.ZERO3, m, 0, 1, False)
    o.gather_level_set(r, 4, 64)
    o.gather_color(4, False, exact=True)
    assert np.array_equal(v.atlas(1, np.uint32), o.color_atlas())
    info = o.atlas_info()
    _, rel, zeros = H.brick_density_errors(v.atlas(), o.atlas(64), o.atlas_map(), info["cnt"])
    assert zeros == 0 and rel <= REL_TOL
    # density into the level set: the maximum with r - |p - v| of the nearest
    # listed entry, which may be negative; colours averaged with the old ones
    v.GatherDensity(4, len(pts), r, H.ZERO3, m, 0, 1, True)
    o.gather_density(r, 4, 64, True)
    o.gather_color(4, True, exact=True)
    assert np.array_equal(v.atlas(1, np.uint32), o.color_atlas())
    a, b = v.atlas().astype(np.float64), o.atlas(64).astype(np.float64)
    assert np.max(np.abs(a - b)) <= 1e-5 * max(1.0, np.abs(b).max())
    v.close()
