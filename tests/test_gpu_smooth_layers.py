"""Smoothing of several iterations with the apron refreshed in between
(Compute, src/gvdb_volume_gvdb.cpp:4527-4552 of the reference) keeps the
bricks' boundary layers and writes one apron at the end; the result has to be
that of single iterations, bit by bit: atlases of a few bricks, of an odd number
of bricks, float and half, a boundary value, and a divisor that is no power of
two.  Noise and grow, which read no neighbour, likewise write only the last
apron."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("effect,params", [(113, (2.0, 0.0, 0.0)), (113, (0.3, 0.05, 0.0)), (114, (0.3, 0.0, 0.0)),
                                           (115, (0.05, 0.0, 0.0))])
@pytest.mark.parametrize("half,boundval,n,iters", [(False, 0.0, 3000, 2), (False, 0.75, 3000, 3), (True, 0.3, 3000, 4),
                                                   (False, 0.5, 2, 2), (True, 0.0, 60000, 5)])
def test_iterations_in_one_call_equal_single_calls(gpu, effect, params, half, boundval, n, iters):
    from gvdb_amd import workloads as W
    import gvdb_amd as G
    pts = W.sphere_shell(n, seed=17) if n > 2 else np.array([[60.5, 60.5, 60.5], [70.5, 73.5, 60.5]], np.float32)
    out = []
    for once in (True, False):
        v, _ = H.gpu_volume(gpu, pts, 2.0, atlas_type=G.T_HALF if half else None, boundval=boundval)
        if once:
            v.Compute(effect, 0, iters, params, True, True, boundval)
        else:
            for _ in range(iters):
                v.Compute(effect, 0, 1, params, True, True, boundval)
        v.synchronize()
        a = v.atlas(0, np.float16 if half else np.float32)
        out.append(a[H.used_brick_mask(a.shape, v.atlas_map(), v.atlas_info()["cnt"])].copy())
        v.close()
    a, b = (x.view(np.uint16 if half else np.uint32) for x in out)
    assert np.array_equal(a, b), "%d voxels differ" % int((a != b).sum())


def test_channel_created_again_smaller(gpu):
    """Channel 0 created again with fewer slots than the bricks had: the
    operator takes the slots there are; their neighbours lie past them."""
    from gvdb_amd import workloads as W
    pts = W.sphere_shell(3000, seed=17, radius=40.0, centre=(64.0, 64.0, 64.0))
    out = []
    for calls in ((3,), (1, 1, 1)):
        v, _ = H.gpu_volume(gpu, pts, 2.0, axiscnt=(16, 16, 8))
        used = v.atlas_info()["used"]
        assert 16 * 16 < used <= 16 * 16 * 8
        v.SetChannelDefault(16, 16, 1)
        v.AddChannel(0, gpu.T_FLOAT, 1)
        v.Compute(gpu.FUNC_FILL_F, 0, 1, (1.0, 0.0, 0.0), False, False, 0.0)
        for n in calls:
            v.Compute(gpu.FUNC_SMOOTH, 0, n, (2.0, 0.0, 0.0), True, True, 0.5)
        v.synchronize()
        out.append(v.atlas().view(np.uint32).copy())
        v.close()
    assert np.array_equal(out[0], out[1])


def _free_bytes(gpu):
    """Free device memory by the HIP runtime the library is linked to."""
    import ctypes
    gpu.load()
    with open("/proc/self/maps") as f:
        libs = sorted({x.split()[-1] for x in f if "libamdhip64" in x}, key=lambda x: "/opt/rocm" not in x)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(libs[0]).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_workspace_goes_back_when_the_atlas_grows(gpu):
    """A grid that has smoothed holds no more memory than one that has not,
    once its atlas had to grow (the workspace is the size of the old atlas)."""
    from gvdb_amd import workloads as W
    small, large = W.sphere_shell(120000, seed=18), W.sphere_shell(300000, seed=19, radius=170.0)
    used, held = {}, 0
    for smooth in (False, True, False, True):
        f0 = _free_bytes(gpu)
        v, _ = H.gpu_volume(gpu, small, 2.0)
        f1 = _free_bytes(gpu)
        if smooth:
            v.Compute(gpu.FUNC_SMOOTH, 0, 4, (2.0, 0.0, 0.0), True, True, 0.0)
            v.synchronize()
            held = f1 - _free_bytes(gpu)
        slots = v.atlas_info()["cnt"][2]
        v.SetPoints(large)
        v.RequestFullRebuild(True)
        v.RebuildTopology(len(large), 2.0, H.ZERO3)
        v.FinishTopology(False, True)
        v.UpdateAtlas()
        v.synchronize()
        assert v.atlas_info()["cnt"][2] > slots
        used[smooth] = f0 - _free_bytes(gpu)
        v.close()
    assert held > 20 << 20
    assert used[True] - used[False] < held / 4, (used, held)
