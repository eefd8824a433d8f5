"""The march's launch variants give the same pixels bit for bit: four lanes
per ray (launches of few rays) against one lane per ray (the same view inside
a launch past the line, beside a larger image), at partial tiles, one pixel
and the line itself; and the transfer function evaluated as a ramp against the
same entries read from the table."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu

C = (64.0, 64.0, 64.0)
LINE = 98304      # rays of a launch that still take four lanes each


def _scene(W, mode, w, h, angs=(30.0, 20.0, 0.0)):
    sc = (W.ea_scene if mode == 7 else W.iso_scene)(w, h, centre=C, dist=190.0)
    return dict(sc, cam=dict(sc["cam"], angs=angs))


@pytest.mark.parametrize("mode", [7, 4])
@pytest.mark.parametrize("half", [False, True])
def test_four_lanes_per_ray_same_pixels(gpu, mode, half):
    from gvdb_amd import workloads as W
    pts = W.sphere_shell(30000, seed=31, radius=40.0, centre=C)
    t = gpu.T_HALF if half else None
    v, _ = H.gpu_volume(gpu, pts, 2.0, atlas_type=t)
    big, _ = H.gpu_volume(gpu, pts[:4000], 2.0, atlas_type=t)
    big.apply_scene(_scene(W, mode, 400, 400))
    big.AddRenderBuf(0, 400, 400, 16)
    b = gpu.GridBatch(0, 2)
    hits = 0
    for w, h, angs in ((1, 1, (0.0, 0.0, 0.0)), (3, 5, (30.0, 20.0, 0.0)), (97, 61, (0.0, 0.0, 0.0)),
                       (200, 136, (-133.0, 71.0, 0.0)), (256, LINE // 256, (90.0, 0.0, 0.0)),
                       (257, LINE // 256, (35.0, 30.0, 0.0))):
        sc = _scene(W, mode, w, h, angs)
        v.apply_scene(sc)
        v.AddRenderBuf(0, w, h, 16)
        v.Render(mode, 0, 0)
        one = v.ReadRenderBuf(0, w, h, 16).copy()
        b.Render([v, big], mode, 0, 0)
        b.synchronize()
        two = v.ReadRenderBuf(0, w, h, 16)
        assert np.array_equal(one.view(np.uint32), two.view(np.uint32)), (w, h)
        hits += np.count_nonzero(np.abs(one - np.asarray(sc["backclr"], np.float32)).max(-1))
    assert hits > 5000
    b.close()
    v.close()
    big.close()


@pytest.mark.parametrize("side", [100, 400])
def test_ramp_transfer_function_same_as_table(gpu, side):
    from gvdb_amd import workloads as W
    pts = W.sphere_shell(30000, seed=32, radius=40.0, centre=C)
    v, _ = H.gpu_volume(gpu, pts, 2.0)
    a, b = np.array([0.9, 0.1, 0.3, 0.013], np.float32), np.array([0.21, 0.7, 0.4, 0.77], np.float32)
    v.apply_scene(dict(_scene(W, 7, side, side), tf=(0.0, 1.0, a, b), vrange=(0.0, 0.1, 1.7)))
    v.AddRenderBuf(0, side, side, 16)
    v.Render(7, 0, 0)
    ramp = v.ReadRenderBuf(0, side, side, 16).copy()
    # the march reads entries up to 16300 of 16384: a second ramp past them
    # leaves what it reads as it was, and makes the table no single ramp
    L = gpu.load()
    assert L.gvdb_linear_transfer_func(v.h, 0.9985, 1.0, gpu._p(b), gpu._p(a)) == 0
    assert L.gvdb_commit_transfer_func(v.h) == 0
    v.Render(7, 0, 0)
    table = v.ReadRenderBuf(0, side, side, 16)
    assert np.count_nonzero(ramp[..., 3]) > 1000
    assert np.array_equal(ramp.view(np.uint32), table.view(np.uint32))
    v.close()
