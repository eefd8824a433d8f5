"""The work a program of this library has it do, as measurable cases.

listed()            the cases, from the smallest call to the largest
draw(rng)           one more case of the same ranges
prepare(case, seed) points, grids, scene and buffers a program holds before the call
run(state)          one pass through the public entry points, and what it computed
work(case)          bytes and operations the pass cannot do without
exact(case, seed)   the voxel values of the pass in 64 bits, from the definitions

Every case uses the tree Configure(5, 4, 3, 3, 3) (8^3 bricks), subcell 4 and
apron 1, as the tests and the benchmark do.  Points lie in device memory
(SetDataGPU), and the atlas is created at a size that fits the grid
(SetChannelDefault).  Voxel results are returned as the grid's own atlas in
device memory (slots x 10 x 10 x 10, brick-major, as gvdb_amd_device.h lays it
out for user kernels), images as ReadRenderBuf returns them.
"""
import functools
import math
import os
import subprocess
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "gvdb-voxels_amd"))

import gvdb_amd as G  # noqa: E402
from gvdb_amd import workloads as W  # noqa: E402

ZERO3 = (0.0, 0.0, 0.0)
SUBCELL = 4
SMOOTH_P1 = 2.0      # centre weight of the smoothing case
DEV = "cuda" if torch.cuda.is_available() else "cpu"


# ------------------------------------------------------------------- cases --
def listed():
    return [
        # a preview or an interactive edit of a small scan: few points, a
        # small view; launches, host round trips and the readback count
        dict(name="frame_shell_10k", kind="frame", shape="shell", n=10000, span=240.0, radius=2.0, view="ea", side=256),
        # the small workload's frame: a scanned surface, rebuilt and marched
        dict(name="frame_shell_262k", kind="frame", shape="shell", n=262144, span=256.0, radius=2.0, view="ea", side=256),
        # the benchmark's step: the medium workload rebuilt and marched
        dict(name="frame_slab_4m_iso", kind="frame", shape="slab", n=4394304, span=400.0, radius=2.0, view="iso",
             side=1024),
        # points to density volume without a render (the volume goes on to
        # other kernels): the same points, FP32
        dict(name="splat_slab_4m", kind="splat", shape="slab", n=4394304, span=400.0, radius=2.0, dtype="float"),
        # an FP16 channel (half the memory per grid), ragged count, clumped points
        dict(name="splat_half_777k", kind="splat", shape="clusters", n=777777, span=360.0, radius=2.0, dtype="half"),
        # a wider falloff than the brick-local fast boxes take (7 voxels an axis)
        dict(name="splat_r3_300k", kind="splat", shape="shell", n=300001, span=240.0, radius=3.0, dtype="float"),
        # fluid surfacing: signed distance to the particles
        dict(name="levelset_500k", kind="levelset", shape="slab", n=500003, span=200.0, radius=2.0, dtype="float"),
        # coloured scan: density and mean colour channels
        dict(name="colour_250k", kind="colour", shape="shell", n=250007, span=240.0, radius=2.0, dtype="float"),
        # a particle simulation's frame over a persistent tree: the points
        # have moved, the topology is updated in place, then splatted
        dict(name="moving_400k", kind="moving", shape="slab", n=400009, span=180.0, radius=2.0, dtype="float"),
        # many small volumes (objects of a scene) per call, each with its view
        dict(name="batch_16", kind="batch", grids=16, n_lo=10000, n_hi=1000000, radius=2.0, side=256),
        # turning around a resident volume: the march alone
        dict(name="render_clusters_2m", kind="render", shape="clusters", n=2000000, span=440.0, radius=2.0, view="ea",
             side=512),
        # voxel post-processing: density smoothed in place
        dict(name="smooth_600k", kind="smooth", shape="shell", n=600011, span=300.0, radius=2.0, dtype="float", passes=4),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["frame", "frame", "splat", "splat", "levelset", "colour", "moving", "batch", "render", "smooth"])
    if kind == "batch":
        lo = int(_log(rng, 5000, 20000))
        return dict(kind=kind, grids=rng.randint(3, 16), n_lo=lo, n_hi=int(_log(rng, 4 * lo, 800000)), radius=2.0,
                    side=8 * rng.randint(16, 32) + rng.choice([0, 0, 3]))
    top = dict(frame=4000000, splat=4000000, levelset=700000, colour=1000000, moving=1000000, render=2000000,
               smooth=1000000)[kind]
    n = int(_log(rng, 8000, top)) | 1
    # 0.01 to 1 points per voxel of the box (a slab fills half of it, a shell
    # and clusters a part), the box between 60 and 440 voxels wide
    span = min(440.0, max(60.0, (n / _log(rng, 0.02, 1.0)) ** (1.0 / 3.0)))
    c = dict(kind=kind, shape=rng.choice(["shell", "slab", "clusters"]), n=n, span=round(span, 1), radius=2.0)
    if kind == "splat":
        c["radius"] = rng.choice([1.0, 1.5, 2.0, 2.0, 2.0, 2.25, 3.0])
        c["dtype"] = rng.choice(["float", "float", "half"])
    elif kind in ("levelset", "colour", "moving", "smooth"):
        c["dtype"] = rng.choice(["float", "float", "half"]) if kind == "smooth" else "float"
        if kind == "smooth":
            c["passes"] = rng.randint(1, 6)
    else:
        c["view"] = rng.choice(["ea", "iso"])
        c["side"] = rng.randint(100, 900)
    return c


# ------------------------------------------------------------------ points --
def _points(shape, n, span, seed, device=DEV):
    """n positions in a box `span` voxels wide whose corner is at (40, 24, 40):
    the tests' and benchmark's shell (a noisy sphere surface), slab (uniform,
    half as high as wide, with a dense plane below it) and Gaussian clusters."""
    g = torch.Generator(device=device)
    g.manual_seed(int(seed) * 7919 + 17)
    lo = torch.tensor([40.0, 24.0, 40.0], dtype=torch.float64, device=device)

    def rand(*s):
        return torch.rand(*s, generator=g, device=device, dtype=torch.float64)

    def randn(*s):
        return torch.randn(*s, generator=g, device=device, dtype=torch.float64)

    if shape == "shell":
        d = randn(n, 3)
        d /= d.norm(dim=1, keepdim=True)
        p = lo + span / 2 + d * (span / 2 - 8 + 1.5 * randn(n).clamp(-5, 5))[:, None]
    elif shape == "slab":
        m = n // 22
        s = rand(n, 3) * torch.tensor([span, span / 2, span], dtype=torch.float64, device=device)
        s[:, 1] += 10.0
        s[n - m:, 1] = 0.5
        p = lo + s
    else:
        # the same twelve blobs for every seed: the grids of a case stay alike in size
        k = 12
        f = np.random.default_rng(12)
        c = torch.from_numpy(span * (0.2 + 0.6 * f.random((k, 3)))).to(device)
        sg = torch.from_numpy(span * (0.02 + 0.05 * f.random(k))).to(device)
        lab = torch.randint(0, k, (n,), generator=g, device=device)
        p = lo + (c[lab] + sg[lab][:, None] * randn(n, 3)).clamp(0, span)
    return p.to(torch.float32).contiguous()


def _grid_sizes(case):
    """Point counts of a batch's grids (log-uniform) and their shapes."""
    g = np.random.default_rng(101)
    n = np.exp(np.log(case["n_lo"]) + np.log(case["n_hi"] / case["n_lo"]) * (np.arange(case["grids"]) + 0.5) /
               case["grids"]).astype(int)
    g.shuffle(n)
    kinds = [("shell", "slab", "clusters")[i % 3] for i in range(case["grids"])]
    spans = [float(min(300.0, max(60.0, (m / 0.06) ** (1.0 / 3.0)))) for m in n]
    return [(k, int(m), s) for k, m, s in zip(kinds, n, spans)]


def _inputs(case, seed):
    """Every point set of a case: [(points, ...)]."""
    if case["kind"] == "batch":
        return [_points(k, n, s, seed * 64 + i) for i, (k, n, s) in enumerate(_grid_sizes(case))]
    p = _points(case["shape"], case["n"], case["span"], seed)
    if case["kind"] != "moving":
        return [p]
    # the frame after: a drift and some diffusion
    g = torch.Generator(device=p.device)
    g.manual_seed(int(seed) + 5)
    q = p + 0.7 * torch.randn(p.shape, generator=g, device=p.device).clamp(-3, 3)
    q[:, 0] += 2.5
    q[:, 2] -= 1.25
    return [p, q.clamp_min(9.0).contiguous()]


@functools.lru_cache(maxsize=64)
def _bricks_of(key):
    case = dict(key)
    pts = _inputs(case, 1)
    if case["kind"] == "batch":
        return [len(_leaves(case, [p])) for p in pts]
    if case["kind"] == "moving":
        return [max(len(_leaves(case, pts)), len(_leaves(dict(case, kind="splat"), pts)))]
    return [len(_leaves(case, pts))]


def _bricks(case):
    """Bricks of each grid of a case (of one seed's points)."""
    return _bricks_of(tuple(sorted((k, v) for k, v in case.items() if k != "name")))


def _scene(view, side, span, height):
    c = (40.0 + span / 2, 24.0 + height / 2, 40.0 + span / 2)
    f = W.ea_scene if view == "ea" else W.iso_scene
    return f(side, side, centre=c, dist=2.1 * span)


# ----------------------------------------------------- the atlas as a tensor --
# A program that works on the volume on the device reaches it from its own
# kernels (ComputeKernel / RenderKernel); this one hands out the atlas address.
_PEEK = r"""
#include <hip/hip_runtime.h>
#include "gvdb_amd_device.h"
extern "C" __global__ void peek(const gvdb_device_view* v, unsigned char chan, void* out) {
    if (blockIdx.x + blockIdx.y + threadIdx.x + threadIdx.y) return;
    uint64_t* o = reinterpret_cast<uint64_t*>(out);
    o[0] = reinterpret_cast<uint64_t>(v->atlas);
    o[1] = uint64_t(v->atlas_cnt[0]) * v->atlas_cnt[1] * v->atlas_cnt[2];
    o[2] = uint64_t(v->brick_res);
}
"""


@functools.lru_cache(maxsize=None)
def _peek_kernel():
    with tempfile.TemporaryDirectory() as d:
        src, obj = os.path.join(d, "peek.hip"), os.path.join(d, "peek.hsaco")
        with open(src, "w") as f:
            f.write(_PEEK)
        subprocess.check_call([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--genco", "-O2",
                               "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                               "-w", "-I" + os.path.join(ROOT, "include"), src, "-o", obj])
        return G.module_function(G.module_load(obj), "peek")


class _Atlas:
    """The device array protocol over a grid's atlas; holds the grid."""

    def __init__(self, vol, chan, typestr):
        fn = _peek_kernel()
        vol.AddRenderBuf(3, 8, 8, 16)
        vol.RenderKernel(fn, chan, 3)
        ptr, slots, br = (int(x) for x in vol.ReadRenderBuf(3, 8, 8, 16).reshape(-1).view(np.uint64)[:3])
        self.owner = vol
        self.__cuda_array_interface__ = dict(shape=(slots, br, br, br), typestr=typestr, data=(ptr, False), version=3)


def _atlas(vol, chan=0, dtype="float"):
    return torch.as_tensor(_Atlas(vol, chan, {"float": "<f4", "half": "<f2", "rgba": "<i4"}[dtype]), device="cuda")


# ----------------------------------------------------------------- prepare --
def _atlas_z(bricks):
    """Layers of 16 x 16 atlas slots for about `bricks` bricks, with room to spare."""
    return int(bricks * 1.08) // 256 + 2


def _volume(pts, layers, dtype="float"):
    v = G.VolumeGVDB(0)
    v.Configure(5, 4, 3, 3, 3)
    v.SetChannelDefault(16, 16, layers)
    v.AddChannel(0, G.T_HALF if dtype == "half" else G.T_FLOAT, 1)
    v.SetDataGPU(pts.data_ptr(), pts.shape[0])
    return v


def _view(v, case, buf=0):
    v.apply_scene(_scene(case["view"], case["side"], case["span"], case["span"] / (2 if case["shape"] == "slab" else 1)))
    v.AddRenderBuf(buf, case["side"], case["side"], 4)
    return G.SHADE_VOLUME if case["view"] == "ea" else G.SHADE_TRILINEAR


def _rebuild(v, n, r):
    v.RequestFullRebuild(True)
    v.RebuildTopology(n, r, ZERO3)
    v.FinishTopology(False, True)
    v.UpdateAtlas()


def _fill(v, n, r, chan_clr=0):
    v.ClearChannel(0)
    ln = v.InsertPointsSubcell(SUBCELL, n, r, ZERO3)
    v.GatherDensity(SUBCELL, n, r, ZERO3, ln, 0, chan_clr, False)
    v.UpdateApron(0, 0.0)
    return ln


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return _prepare_batch(case, seed)
    pts = _inputs(case, seed)
    torch.cuda.synchronize()       # the grid's own stream reads them
    n, r = case["n"], case["radius"]
    v = _volume(pts[0], _atlas_z(_bricks(case)[0]), case.get("dtype", "float"))
    s = dict(case=case, pts=pts, v=v, n=n, r=r)
    if kind == "colour":
        g = torch.Generator(device="cuda")
        g.manual_seed(int(seed) + 3)
        v.AddChannel(1, G.T_UCHAR4, 1)
        s["rgba"] = torch.randint(0, 256, (n, 4), generator=g, device="cuda", dtype=torch.uint8)
        torch.cuda.synchronize()
        rc = G.load().gvdb_set_colors_gpu(v.h, s["rgba"].data_ptr(), n, 0, 4)
        assert rc == G.OK, rc
    if "view" in case:
        s["shade"] = _view(v, case)
    _rebuild(v, n, r)
    if kind == "moving":
        # the frame before, as the second call after Configure makes the tree
        # one that later calls update in place
        v.RebuildTopology(n, r, ZERO3)
        v.FinishTopology(False, True)
        v.UpdateAtlas()
        v.SetDataGPU(pts[1].data_ptr(), n)
    if kind in ("render", "smooth"):
        s["len"] = _fill(v, n, r)
    if kind == "moving":
        # sizes the atlas for the moved points
        v.RebuildTopology(n, r, ZERO3)
        v.FinishTopology(False, True)
        v.UpdateAtlas()
    if kind not in ("render",):
        s["atlas"] = _atlas(v, 0, case.get("dtype", "float"))
    if kind == "colour":
        s["colours"] = _atlas(v, 1, "rgba")
    return s


def _prepare_batch(case, seed):
    pts = _inputs(case, seed)
    torch.cuda.synchronize()
    vols = []
    for p, bricks, (kind, _, span) in zip(pts, _bricks(case), _grid_sizes(case)):
        v = _volume(p, _atlas_z(bricks))
        _view(v, dict(view="ea", side=case["side"], span=span, shape=kind))
        vols.append(v)
    s = dict(case=case, pts=pts, vols=vols, batch=G.GridBatch(0, len(vols)), n=[p.shape[0] for p in pts])
    for v, n in zip(vols, s["n"]):
        _rebuild(v, n, case["radius"])
    s["atlas"] = [_atlas(v) for v in vols]
    return s


# --------------------------------------------------------------------- run --
def run(s):
    case = s["case"]
    return globals()["_run_" + case["kind"]](s, case)


def _run_frame(s, case):
    v, n, r, side = s["v"], s["n"], s["r"], case["side"]
    _rebuild(v, n, r)
    ln = _fill(v, n, r)
    v.Render(s["shade"], 0, 0)
    return dict(image=v.ReadRenderBuf(0, side, side, 4), entries=ln, atlas=s["atlas"])


def _run_splat(s, case):
    _rebuild(s["v"], s["n"], s["r"])
    return dict(entries=_fill(s["v"], s["n"], s["r"]), atlas=s["atlas"])


def _run_levelset(s, case):
    v, n, r = s["v"], s["n"], s["r"]
    _rebuild(v, n, r)
    v.ClearChannel(0)
    ln = v.InsertPointsSubcell(SUBCELL, n, r, ZERO3)
    v.GatherLevelSet(SUBCELL, n, r, ZERO3, ln, 0, 0, False)
    v.UpdateApron(0, 3.0)
    return dict(entries=ln, atlas=s["atlas"])


def _run_colour(s, case):
    v = s["v"]
    _rebuild(v, s["n"], s["r"])
    v.ClearChannel(1)
    ln = _fill(v, s["n"], s["r"], 1)
    v.UpdateApron(1, 0.0)
    return dict(entries=ln, atlas=s["atlas"], colours=s["colours"])


def _run_moving(s, case):
    v, n, r = s["v"], s["n"], s["r"]
    v.RebuildTopology(n, r, ZERO3)       # in place: the tree of the frame before
    v.FinishTopology(False, True)
    v.UpdateAtlas()
    return dict(entries=_fill(v, n, r), atlas=s["atlas"])


def _run_render(s, case):
    v = s["v"]
    v.Render(s["shade"], 0, 0)
    return dict(image=v.ReadRenderBuf(0, case["side"], case["side"], 4))


def _run_smooth(s, case):
    v, n, r = s["v"], s["n"], s["r"]
    v.GatherDensity(SUBCELL, n, r, ZERO3, s["len"], 0, 0, False)
    v.UpdateApron(0, 0.0)
    v.Compute(G.FUNC_SMOOTH, 0, case["passes"], (SMOOTH_P1, 0.0, 0.0), True, True, 0.0)
    return dict(atlas=s["atlas"])


def _run_batch(s, case):
    b, vols, n, r, side = s["batch"], s["vols"], s["n"], case["radius"], case["side"]
    for v in vols:
        v.RequestFullRebuild(True)
    b.RebuildTopology(vols, n, r)
    b.FinishTopology(vols, False, True)
    b.UpdateAtlas(vols)
    b.ClearChannel(vols, 0)
    lens = b.InsertPointsSubcell(vols, SUBCELL, n, r)
    b.GatherDensity(vols, SUBCELL, lens, r, 0)
    b.UpdateApron(vols, 0, 0.0)
    b.Render(vols, G.SHADE_VOLUME, 0, 0)
    b.synchronize()
    return dict(images=[v.ReadRenderBuf(0, side, side, 4) for v in vols], entries=np.array(lens), atlas=s["atlas"])


# -------------------------------------------------------------------- work --
def work(case):
    """Points read once (12 B), every used brick's 1000 voxels written once,
    the image written once; a march and a smoothing pass read the volume once."""
    bricks = sum(_bricks(case))
    vox = 1000 * (2 if case.get("dtype") == "half" else 4)
    kind = case["kind"]
    images = case.get("grids", 1) * case.get("side", 0) ** 2 * 4
    if kind == "batch":
        n = sum(m for _, m, _ in _grid_sizes(case))
    else:
        n = case["n"]
    b = 12.0 * n + bricks * vox + images
    if kind == "render":
        b = bricks * 512 * 4 + images
    if kind == "colour":
        b += 4.0 * n + bricks * vox
    if kind == "smooth":
        b = 12.0 * n + bricks * vox * (1 + 2 * case["passes"])
    # about 30 candidate voxels a point, 8 operations each
    return dict(bytes=float(b), flops=0.0 if kind == "render" else 240.0 * n)


# ------------------------------------------------------------------- exact --
def _unique_bricks(lo, hi):
    """Unique brick coordinates of the boxes [lo, hi] (per point), in x-major order."""
    keys = []
    ext = (hi - lo).amax(0)
    for dx in range(int(ext[0]) + 1):
        for dy in range(int(ext[1]) + 1):
            for dz in range(int(ext[2]) + 1):
                b = lo + torch.tensor([dx, dy, dz], device=lo.device)
                b = b[(b <= hi).all(1)]
                keys.append(torch.unique((b[:, 0] << 40) | (b[:, 1] << 20) | b[:, 2]))
    return torch.unique(torch.cat(keys))


def _leaves(case, pts):
    """Brick keys (x << 40 | y << 20 | z) in atlas slot order: the points' own
    bricks sorted, then the sorted rest of the bricks [int(p) - r, int(p) + 2 r]
    touches; after an in-place update, those of them the moved points still
    touch within [int(p) - r, int(p) + r], then the new ones, sorted."""
    r = case["radius"]
    p = pts[0].long()
    own = _unique_bricks(p // 8, p // 8)
    # a radius below one voxel adds no bricks
    box = _unique_bricks((p.double() - r).long().clamp_min(0) // 8, (p.double() + 2 * r).long() // 8) if r >= 1 else own
    keys = torch.cat([own, box[~torch.isin(box, own)]])
    if case["kind"] == "moving":
        q = pts[1].long()
        now = _unique_bricks((q.double() - r).long().clamp_min(0) // 8, (q.double() + r).long() // 8)
        keys = torch.cat([keys[torch.isin(keys, now)], now[~torch.isin(now, keys)]])
    return keys


class _Dense:
    """A box of voxels in 64 bits around the bricks, and which of them a brick holds."""

    def __init__(self, keys, value):
        self.c = 8 * torch.stack([keys >> 40, (keys >> 20) & 0xFFFFF, keys & 0xFFFFF], 1)
        self.lo = self.c.amin(0) - 16
        self.dim = [int(x) for x in (self.c.amax(0) + 24 - self.lo)]
        dev = keys.device
        self.v = torch.full((self.dim[0] * self.dim[1] * self.dim[2],), float(value), dtype=torch.float64, device=dev)
        self.mask = torch.zeros_like(self.v, dtype=torch.bool)
        self.mask[self.index(8)] = True

    def flat(self, p):
        q = p - self.lo
        return (q[..., 0] * self.dim[1] + q[..., 1]) * self.dim[2] + q[..., 2]

    def index(self, side):
        """Flat indices of every brick's side^3 voxels (8: interior, 10: padded), z slowest."""
        a = torch.arange(side, device=self.c.device) - (side - 8) // 2
        z, y, x = torch.meshgrid(a, a, a, indexing="ij")
        off = self.flat(torch.stack([x, y, z], -1) + self.lo)
        return self.flat(self.c)[:, None, None, None] + off

    def atlas(self, bound, bricks):
        """The padded bricks, in an atlas created for about `bricks`: voxels no
        brick holds read `bound`, slots no brick has stay 0."""
        v = torch.where(self.mask, self.v, torch.full_like(self.v, bound))
        out = torch.zeros(256 * _atlas_z(bricks), 10, 10, 10, dtype=torch.float64, device=v.device)
        for k, i in enumerate(self.index(10).split(8192)):
            out[k * 8192:k * 8192 + len(i)] = v[i]
        return out


def _density(D, p, r):
    """max(0, max over points of r - |p - v|) on the voxels of the bricks."""
    w = int(math.floor(2 * r)) + 1
    for q in p.split(1 << 18):
        base = torch.ceil(q.double() - r).long()
        for dx in range(w):
            for dy in range(w):
                v = base[:, None, :] + torch.tensor([[dx, dy, z] for z in range(w)], device=p.device)[None]
                d = r - (q.double()[:, None, :] - v.double()).square().sum(-1).sqrt()
                keep = d > 0
                D.v.scatter_reduce_(0, D.flat(v)[keep], d[keep], "amax")
    D.v[~D.mask] = 0.0


def _levelset(D, p, r):
    """min(3, min of |p - v| - r over the points listed in the voxel's 4^3
    subcell: int(p - r) / 4 * 4 <= corner <= int(p + 1 + r) / 4 * 4 per axis)."""
    lo = ((p - r).to(torch.int32) // 4 * 4).long()
    hi = ((p + 1 + r).to(torch.int32) // 4 * 4).long()
    a = torch.arange(4, device=p.device)
    z, y, x = torch.meshgrid(a, a, a, indexing="ij")
    off = torch.stack([x, y, z], -1).reshape(-1, 3)
    steps = int(((hi - lo) // 4).amax()) + 1
    for k in range(steps ** 3):
        s = lo + 4 * torch.tensor([k % steps, k // steps % steps, k // steps // steps], device=p.device)
        on = (s <= hi).all(1)
        on[on.clone()] = D.mask[D.flat(s[on])]
        for sv, q in zip(s[on].split(1 << 18), p[on].double().split(1 << 18)):
            v = sv[:, None, :] + off[None]
            d = (q[:, None, :] - v.double()).square().sum(-1).sqrt() - r
            D.v.scatter_reduce_(0, D.flat(v).reshape(-1), d.reshape(-1), "amin")


def _smooth(D, passes):
    for _ in range(passes):
        v = D.v.view(D.dim)
        s = SMOOTH_P1 * v
        for ax in range(3):
            s = s + torch.roll(v, 1, ax) + torch.roll(v, -1, ax)
        D.v = torch.where(D.mask, (s / (SMOOTH_P1 + 6.0)).reshape(-1), torch.zeros_like(D.v))


def exact(case, seed):
    kind, r = case["kind"], case.get("radius")
    if kind == "render":
        return None
    pts = _inputs(case, seed)
    if kind == "batch":
        out = []
        for p, bricks in zip(pts, _bricks(case)):
            D = _Dense(_leaves(case, [p]), 0.0)
            _density(D, p, r)
            out.append(D.atlas(0.0, bricks))
        return dict(images=[None] * len(pts), entries=None, atlas=out)
    bricks = _bricks(case)[0]
    D = _Dense(_leaves(case, pts), 3.0 if kind == "levelset" else 0.0)
    if kind == "levelset":
        _levelset(D, pts[0], r)
        return dict(entries=None, atlas=D.atlas(3.0, bricks))
    _density(D, pts[-1], r)
    if kind == "smooth":
        _smooth(D, case["passes"])
        return dict(atlas=D.atlas(0.0, bricks))
    out = dict(atlas=D.atlas(0.0, bricks))
    out["entries"] = None
    if kind == "frame":
        out["image"] = None
    if kind == "colour":
        out["colours"] = None
    return out
