"""HIP graphs of the per-frame chain ClearChannel -> InsertPointsSubcell ->
GatherDensity -> UpdateApron -> Render, one grid and a batch: a replay gives
the atlas and image of the same calls run eagerly, bit for bit; it re-reads
the point buffer (new positions written in place); it is refused once the
topology changes; a replay whose points leave the topology reports it; calls
outside the chain fail the recording."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu

R = 2.0
W = 96


def _grid(gpu, pts, centre):
    from gvdb_amd import workloads as Wk
    v = gpu.VolumeGVDB(0)
    v.Configure(*H.TREE)
    v.SetChannelDefault(16, 16, 1)
    v.AddChannel(0, gpu.T_FLOAT, 1)
    v.SetPoints(pts)
    v.RequestFullRebuild(True)
    v.RebuildTopology(len(pts), R, H.ZERO3)
    v.FinishTopology(False, True)
    v.UpdateAtlas()
    v.apply_scene(Wk.ea_scene(W, W, centre=centre, dist=300.0))
    v.AddRenderBuf(0, W, W, 16)
    return v


def _chain(gpu, v, n):
    v.ClearChannel(0)
    ln = v.InsertPointsSubcell(4, n, R, H.ZERO3)
    v.GatherDensity(4, n, R, H.ZERO3, ln, 0, 0, False)
    v.UpdateApron(0, 0.0)
    v.Render(gpu.SHADE_VOLUME, 0, 0)
    return ln


def _state(v):
    return v.atlas().view(np.uint32).copy(), v.ReadRenderBuf(0, W, W, 16).view(np.uint32).copy()


def _wipe(gpu, v):
    # overwrite what the chain writes: atlas and render buffer
    v.Compute(gpu.FUNC_FILL_F, 0, 1, (7.0, 0.0, 0.0), False, False, 0.0)
    v.Render(gpu.SHADE_TRILINEAR, 0, 0)


def test_graph_replay_one_grid(gpu):
    from gvdb_amd import workloads as Wk
    c = (128.0, 128.0, 128.0)
    pts = Wk.sphere_shell(40000, seed=41, radius=60.0, centre=c)
    n = len(pts)
    v = _grid(gpu, pts, c)
    ln0 = _chain(gpu, v, n)
    v.synchronize()
    a0, i0 = _state(v)
    assert ln0 > 0 and np.count_nonzero(a0) > 0
    v.CaptureBegin()
    _chain(gpu, v, n)
    g = v.CaptureEnd()
    _wipe(gpu, v)
    assert not np.array_equal(_state(v)[0], a0)
    for _ in range(3):      # replays with eager work between them
        g.launch()
        g.synchronize()
        a1, i1 = _state(v)
        assert np.array_equal(a1, a0) and np.array_equal(i1, i0)
        _wipe(gpu, v)
    # new positions in the same device buffer: the same points in another
    # order give the same atlas (the gather's max does not depend on order)
    rng = np.random.default_rng(5)
    v.SetPoints(pts[rng.permutation(n)])
    g.launch()
    g.synchronize()
    assert np.array_equal(_state(v)[0], a0)
    # other positions inside the topology: the replay equals the eager chain
    sub = pts[:n // 2]
    moved = np.concatenate([sub, sub[::-1] + np.float32(0.25)]).astype(np.float32)
    v.SetPoints(moved)
    g.launch()
    g.synchronize()
    a2, i2 = _state(v)
    assert not np.array_equal(a2, a0)
    ln_e = _chain(gpu, v, n)
    v.synchronize()
    a3, i3 = _state(v)
    assert ln_e > 0 and np.array_equal(a2, a3) and np.array_equal(i2, i3)
    # points outside every brick: the replay reports them
    v.SetPoints(pts + np.float32(400.0))
    g.launch()
    with pytest.raises(gpu.GVDBError) as e:
        g.synchronize()
    assert e.value.code == gpu.ERR_STATE
    # a new topology invalidates the graph
    v.SetPoints(pts)
    v.RequestFullRebuild(True)
    v.RebuildTopology(n, R, H.ZERO3)
    v.FinishTopology(False, True)
    v.UpdateAtlas()
    with pytest.raises(gpu.GVDBError) as e:
        g.launch()
    assert e.value.code == gpu.ERR_STATE
    g.close()
    v.close()


@pytest.mark.parametrize("side", [W, 400])     # four lanes a ray, one
def test_recorded_render_takes_the_committed_transfer_function(gpu, side):
    """A transfer function set and committed between replays is what the next
    replay draws with, as the recorded march reads the device table; ramps over
    the whole table and over a part of it."""
    from gvdb_amd import workloads as Wk
    c = (96.0, 96.0, 96.0)
    pts = Wk.sphere_shell(20000, seed=43, radius=40.0, centre=c)
    v = _grid(gpu, pts, c)
    _chain(gpu, v, len(pts))
    v.AddRenderBuf(0, side, side, 16)
    sc = Wk.ea_scene(side, side, centre=c, dist=200.0)
    tfs = [sc["tf"], (0.0, 1.0, (0.9, 0.1, 0.0, 0.2), (0.0, 0.7, 0.3, 1.0)),
           (0.25, 0.75, (0.0, 0.0, 1.0, 0.5), (1.0, 1.0, 0.0, 0.9))]

    def direct(tf):
        v.apply_scene(dict(sc, tf=tf))
        v.Render(gpu.SHADE_VOLUME, 0, 0)
        return v.ReadRenderBuf(0, side, side, 16).view(np.uint32).copy()

    direct(tfs[0])
    v.CaptureBegin()
    v.Render(gpu.SHADE_VOLUME, 0, 0)
    g = v.CaptureEnd()
    seen = []
    for k in (1, 0, 2, 1):
        v.apply_scene(dict(sc, tf=tfs[k]))
        g.launch()
        g.synchronize()
        img = v.ReadRenderBuf(0, side, side, 16).view(np.uint32).copy()
        assert np.array_equal(img, direct(tfs[k])), k
        seen.append(img)
    assert not np.array_equal(seen[0], seen[1]) and not np.array_equal(seen[1], seen[2])
    g.close()
    v.close()


def test_calls_outside_the_chain_fail_the_recording(gpu):
    from gvdb_amd import workloads as Wk
    c = (64.0, 64.0, 64.0)
    pts = Wk.sphere_shell(5000, seed=42, radius=30.0, centre=c)
    v = _grid(gpu, pts, c)
    _chain(gpu, v, len(pts))
    v.synchronize()
    v.CaptureBegin()
    v.ClearChannel(0)
    with pytest.raises(gpu.GVDBError):
        v.RebuildTopology(len(pts), R, H.ZERO3)
    with pytest.raises(gpu.GVDBError):
        v.CaptureEnd()
    # the grid works eagerly afterwards
    _chain(gpu, v, len(pts))
    v.synchronize()
    v.close()


def test_neighbour_table_of_a_recording_is_not_taken_as_built(gpu):
    """The chain recorded first on a new topology: refused where buffers had to
    grow, and not launched where they did not; the direct chain afterwards, and
    an UpdateApron by itself, build the neighbour table themselves."""
    from gvdb_amd import workloads as Wk
    c = (96.0, 96.0, 96.0)
    pts = Wk.sphere_shell(20000, seed=45, radius=40.0, centre=c)
    other = Wk.sphere_shell(20000, seed=46, radius=38.0, centre=(88.0, 104.0, 96.0))

    def direct(p):
        w = _grid(gpu, p, c)
        _chain(gpu, w, len(p))
        w.synchronize()
        s = _state(w)
        w.close()
        return s

    want, want2 = direct(pts), direct(other)
    v = _grid(gpu, pts, c)
    v.Render(gpu.SHADE_VOLUME, 0, 0)     # commits the transfer function
    v.synchronize()
    v.CaptureBegin()
    _chain(gpu, v, len(pts))
    with pytest.raises(gpu.GVDBError) as e:
        v.CaptureEnd()
    assert e.value.code == gpu.ERR_STATE
    _chain(gpu, v, len(pts))
    v.synchronize()
    assert all(np.array_equal(a, b) for a, b in zip(_state(v), want))
    # a topology of fewer bricks in the buffers there are
    v.SetPoints(other)
    v.RequestFullRebuild(True)
    v.RebuildTopology(len(other), R, H.ZERO3)
    v.FinishTopology(False, True)
    v.UpdateAtlas()
    v.CaptureBegin()
    _chain(gpu, v, len(other))
    g = v.CaptureEnd()
    _chain(gpu, v, len(other))
    v.synchronize()
    assert all(np.array_equal(a, b) for a, b in zip(_state(v), want2))
    _wipe(gpu, v)
    g.launch()
    g.synchronize()
    assert all(np.array_equal(a, b) for a, b in zip(_state(v), want2))
    g.close()
    v.close()


def _padded(v):
    return v.atlas().view(np.uint32).copy()


def test_aprons_and_recordings_use_their_own_boundary_layers(gpu):
    """UpdateApron after GatherDensity reads the layers the gather left; not
    those of a gather that is only recorded, nor from before a replay that wrote
    the atlas, nor, recorded alone, those current at the recording.  Each is
    compared with an UpdateApron that reads the bricks (after an operator that
    changes nothing: noise of amplitude 0)."""
    from gvdb_amd import workloads as Wk
    c = (96.0, 96.0, 96.0)
    pts = Wk.sphere_shell(20000, seed=47, radius=40.0, centre=c)
    n = len(pts)
    v = _grid(gpu, pts, c)
    ln = _chain(gpu, v, n)
    v.synchronize()

    def apron_from_bricks():
        v.Compute(gpu.FUNC_NOISE, 0, 1, (0.0, 0.0, 0.0), False, True, 0.0)
        v.UpdateApron(0, 0.0)
        v.synchronize()
        return _padded(v)

    def shrink():
        # interiors and aprons no longer the gather's
        v.Compute(gpu.FUNC_SMOOTH, 0, 1, (1.0, 0.0, 0.0), False, True, 0.0)

    # a gather and an apron recorded, not launched; then a direct apron
    shrink()
    v.CaptureBegin()
    v.GatherDensity(4, n, R, H.ZERO3, ln, 0, 0, False)
    v.UpdateApron(0, 0.0)
    both = v.CaptureEnd()
    v.UpdateApron(0, 0.0)
    v.synchronize()
    a = _padded(v)
    assert np.array_equal(a, apron_from_bricks())
    # an apron recorded alone right after a direct gather, replayed over other voxels
    v.GatherDensity(4, n, R, H.ZERO3, ln, 0, 0, False)
    v.CaptureBegin()
    v.UpdateApron(0, 0.0)
    alone = v.CaptureEnd()
    for _ in range(2):
        shrink()
        alone.launch()
        alone.synchronize()
        a = _padded(v)
        assert np.array_equal(a, apron_from_bricks())
    # the channel cleared by a replay between a direct gather and its apron
    v.CaptureBegin()
    v.ClearChannel(0)
    clear = v.CaptureEnd()
    v.GatherDensity(4, n, R, H.ZERO3, ln, 0, 0, False)
    clear.launch()
    clear.synchronize()
    v.UpdateApron(0, 0.0)
    v.synchronize()
    assert not _padded(v).any()
    # the recorded pair against the direct one
    both.launch()
    both.synchronize()
    a = _padded(v)
    v.GatherDensity(4, n, R, H.ZERO3, ln, 0, 0, False)
    v.UpdateApron(0, 0.0)
    v.synchronize()
    assert a.any() and np.array_equal(a, _padded(v)) and np.array_equal(a, apron_from_bricks())
    for g in (both, alone, clear):
        g.close()
    v.close()


def test_a_recorded_insert_counts_from_its_replay_on(gpu):
    """What an insert leaves for gathers and reads: the direct one's until a
    replay runs the recorded one (another radius here), with its own entry
    tables after every replay; none after a refused recording."""
    from gvdb_amd import workloads as Wk
    c = (96.0, 96.0, 96.0)
    pts = Wk.sphere_shell(20000, seed=48, radius=40.0, centre=c)
    sets = [pts, (c + (pts - c) * np.float32(0.98)).astype(np.float32)]
    n = len(pts)
    v = _grid(gpu, pts, c)
    v.CaptureBegin()
    v.InsertPointsSubcell(4, n, R, H.ZERO3)
    with pytest.raises(gpu.GVDBError):      # buffers had to grow
        v.CaptureEnd()
    with pytest.raises(gpu.GVDBError) as e:
        v.GatherLevelSet(4, n, R, H.ZERO3, 0, 0, 0, False)
    assert e.value.code == gpu.ERR_STATE

    def gather(p, r, ln=None):
        if ln is None:
            v.SetPoints(p)
            ln = v.InsertPointsSubcell(4, n, r, H.ZERO3)
        v.ClearChannel(0)
        v.GatherDensity(4, n, r, H.ZERO3, ln, 0, 0, False)
        v.UpdateApron(0, 0.0)
        v.synchronize()
        return _padded(v), ln

    want = {}
    for k, p in enumerate(sets):
        want[k], ln = gather(p, 1.0)
        want[k] = (want[k], ln, v.subcells())
    want2, ln2 = gather(pts, R)
    assert not np.array_equal(want[0][0], want[1][0]) and not np.array_equal(want[0][0], want2)
    v.CaptureBegin()
    v.InsertPointsSubcell(4, n, 1.0, H.ZERO3)
    g = v.CaptureEnd()
    assert np.array_equal(gather(None, R, ln2)[0], want2)      # not launched yet
    for k in (1, 0, 1):
        v.SetPoints(sets[k])
        g.launch()
        g.synchronize()
        a, ln, tables = want[k]
        assert np.array_equal(gather(None, 1.0, ln)[0], a)
        t = v.subcells()
        assert all(np.array_equal(t[x], tables[x]) for x in ("cnt", "off", "pos", "nid"))
        b, l2 = gather(pts, R)                                  # a direct insert takes over
        assert l2 == ln2 and np.array_equal(b, want2)
    g.close()
    v.close()


def test_call_outside_the_chain_fails_a_batch_recording(gpu):
    """A refused call in a batch's recording fails it and leaves no grid behind
    in it: batched and single calls run directly afterwards."""
    from gvdb_amd import workloads as Wk
    c = (64.0, 64.0, 64.0)
    sets = [Wk.sphere_shell(4000, seed=44 + k, radius=25.0 + k, centre=c) for k in range(3)]
    vols = [_grid(gpu, p, c) for p in sets]
    ns = [len(p) for p in sets]
    B = gpu.GridBatch(0, 3)
    lens = B.InsertPointsSubcell(vols, 4, ns, R)
    B.GatherDensity(vols, 4, lens, R, 0)
    B.synchronize()
    B.CaptureBegin()
    with pytest.raises(gpu.GVDBError):
        B.RebuildTopology(vols, ns, R)
    with pytest.raises(gpu.GVDBError):
        B.CaptureEnd()
    B.ClearChannel(vols, 0)
    assert np.array_equal(B.InsertPointsSubcell(vols, 4, ns, R), lens)
    B.synchronize()
    B.close()
    for v, n in zip(vols, ns):
        v.RequestFullRebuild(True)
        v.RebuildTopology(n, R, H.ZERO3)
        v.FinishTopology(False, True)
        v.UpdateAtlas()
        _chain(gpu, v, n)
        v.synchronize()
        v.close()


def test_graph_replay_batch(gpu):
    from gvdb_amd import workloads as Wk
    grids = [Wk.sphere_shell(4000 + 3000 * k, seed=50 + k, radius=20.0 + 8 * k, centre=(80.0 + 20 * k, 90.0, 100.0))
             for k in range(6)]
    c = (130.0, 90.0, 100.0)
    vols = [_grid(gpu, p, c) for p in grids]
    ns = [len(p) for p in grids]
    B = gpu.GridBatch(0, len(vols))

    def chain():
        B.ClearChannel(vols, 0)
        lens = B.InsertPointsSubcell(vols, 4, ns, R)
        B.GatherDensity(vols, 4, lens, R, 0)
        B.UpdateApron(vols, 0, 0.0)
        B.Render(vols, gpu.SHADE_VOLUME, 0, 0)

    chain()
    B.synchronize()
    ref = [_state(v) for v in vols]
    # the batched results equal the one-grid calls'
    for v, p, (a, i) in zip(vols, grids, ref):
        u = _grid(gpu, p, c)
        _chain(gpu, u, len(p))
        u.synchronize()
        au, iu = _state(u)
        assert np.array_equal(au, a) and np.array_equal(iu, i)
        u.close()
    B.CaptureBegin()
    chain()
    g = B.CaptureEnd()
    for v in vols:
        _wipe(gpu, v)
    for _ in range(2):
        g.launch()
        g.synchronize()
        for v, (a, i) in zip(vols, ref):
            a1, i1 = _state(v)
            assert np.array_equal(a1, a) and np.array_equal(i1, i)
        for v in vols:
            _wipe(gpu, v)
    g.close()
    B.close()
    for v in vols:
        v.close()
