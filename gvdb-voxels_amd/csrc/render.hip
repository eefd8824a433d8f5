// render.hip -- hierarchical DDA ray march over the sparse tree.
//
// Follows rayCast (kernels/cuda_gvdb_raycast.cuh:543-611 of the reference)
// with the HDDA stepping of kernels/cuda_gvdb_dda.cuh:38-91, the
// emission-absorption brick march rayDeepBrick (:485-533) and the trilinear
// isosurface march raySurfaceTrilinearBrick (:281-300) with getGradient
// (:132-141) and Phong + shadow ray (kernels/cuda_gvdb_module.cu:38-57).
// Samples are exact software trilinear reads of the brick-major atlas; the
// reference's texture unit is replaced because its filter weights are
// quantised.  One 64-thread workgroup renders one pixel tile (8x8 by
// default; 16x4, 32x2 or 64x1 when the autotuner finds them faster; 4x4 with
// four lanes per ray when a launch has few rays).
//
// What bounds it: small images the serial chain of their longest wave (steps,
// fetches, accumulation), large ones L1 lookups and vector issue together
// (isosurface 1024^2 over 4.4 M slab points, 0.51 ms: 299 M cache-line lookups,
// 0.49 ms at one a cycle and CU, 262 M vector instructions of a wave, 0.43 ms;
// emission-absorption 512^2 of 2 M clustered points, 1.20 ms: 0.77 and 0.55).
// Hence, with the same arithmetic:
// the walk and the march are decoupled (ray_cast), so lanes do not wait for
// each other at brick borders; a level's facts, the child list and the exit
// time stay in registers and LDS instead of being re-read through per-lane
// indices at every cell; divisions by powers of two are products; a ramp
// transfer function is computed, not looked up (64 lanes' lookups touch 64
// lines).  Measured, ms before -> now: emission-absorption 256^2 of a
// 10 k-point shell 0.36 -> 0.20, 512^2 of 2 M clustered points 1.78 -> 1.17,
// 2048^2 of a 500 k slab 6.97 -> 4.0; isosurface 1024^2 0.82 -> 0.52.
#include "kernels.h"
#include "tree_device.h"
#include <hip/hip_fp16.h>
#include <cmath>

// Contraction is off in this file: the walk performs the reference's FP32
// operations one by one (no fused multiply-adds), so every ray takes the
// steps of a plain IEEE single-precision evaluation of rayCast, also where a
// step sits on a rounding edge (far from the origin the 1e-3 epsilon is a
// few ulps).
#pragma clang fp contract(off)

namespace gvdb {

struct f3 { float x, y, z; };
__device__ inline f3 mk3(float a, float b, float c) { return f3{a, b, c}; }
__device__ inline f3 operator+(f3 a, f3 b) { return mk3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ inline f3 operator-(f3 a, f3 b) { return mk3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ inline f3 operator*(f3 a, float s) { return mk3(a.x * s, a.y * s, a.z * s); }
__device__ inline float dot3(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ inline f3 norm3(f3 a) { float il = 1.0f / sqrtf(dot3(a, a)); return a * il; }

template <typename AT>
__device__ inline float ldv(const AT* a, u64 o);
template <>
__device__ inline float ldv<float>(const float* a, u64 o) { return a[o]; }
template <>
__device__ inline float ldv<__half>(const __half* a, u64 o) { return __half2float(a[o]); }

// Trilinear sample at atlas coordinate (x, y, z) = p + mValue, the sum formed
// in FP32 as the reference's tex3D call forms it (far from the atlas origin
// the position carries that sum's rounding), read from the padded brick
// whose first voxel is atlas voxel (cx, cy, cz) and whose data starts at
// `b`: an unnormalised linear fetch (texel centres at integer + 0.5) with
// exact weights, blended as a + f (b - a) along x, then y, then z.  Split
// into the fetch (four x-adjacent pairs, one 8-byte load each for FP32) and
// the blend, so the loads of several samples can be in flight together.
// A march sample (p in [0, res)) has its lower taps at padded indices 0..8;
// indices are clamped into the brick, so a fetch at any position stays
// inside it.
struct Taps {
    float c[8];   // c000 c100 c010 c110 c001 c101 c011 c111
    float fx, fy, fz;
};

template <typename AT>
__device__ inline void ld_pair(const AT* p, float& a, float& b);
template <>
__device__ inline void ld_pair<float>(const float* p, float& a, float& b) {
    float2 v;
    __builtin_memcpy(&v, p, sizeof(v));
    a = v.x;
    b = v.y;
}
template <>
__device__ inline void ld_pair<__half>(const __half* p, float& a, float& b) {
    __half2 v;
    __builtin_memcpy(&v, p, sizeof(v));
    a = __low2float(v);
    b = __high2float(v);
}

struct Corner {
    int c[3];      // atlas voxel of the padded brick's first voxel (mValue - apron)
    float o[3];    // mValue as floats: atlas position = p + o
    float base;    // 111 c: index of that voxel in rows of 10 and layers of 100 (BR = 10)
};

// BR: the padded brick side when known (10: 8^3 bricks, apron 1, and an atlas
// under 2^17 voxels a side), so the tap offsets are constants and the local
// index 100 z + 10 y + x comes from the atlas voxel in floats (whole numbers
// below 2^24: exact); 0: taken from the tree.
template <typename AT, int BR>
__device__ inline void tri_fetch(const AT* b, int br_rt, const Corner& K, float x, float y, float z, Taps& T) {
    const int br = BR ? BR : br_rt;
    const float ux = x - 0.5f, uy = y - 0.5f, uz = z - 0.5f;
    const float fx0 = floorf(ux), fy0 = floorf(uy), fz0 = floorf(uz);
    T.fx = ux - fx0;
    T.fy = uy - fy0;
    T.fz = uz - fz0;
    unsigned at;
    if constexpr (BR != 0) {
        const float f = __builtin_fmaf(fz0, float(BR * BR), __builtin_fmaf(fy0, float(BR), fx0 - K.base));
        // (f < 0 or past the brick: a sample past a face, fetched but never used)
        at = unsigned(__builtin_amdgcn_fmed3f(f, 0.0f, float((BR - 2) * (BR * BR + BR + 1))));
    } else {
        const int ix = min(max(int(fx0) - K.c[0], 0), br - 2), iy = min(max(int(fy0) - K.c[1], 0), br - 2),
                  iz = min(max(int(fz0) - K.c[2], 0), br - 2);
        at = unsigned((iz * br + iy) * br + ix);
    }
    const AT* o = b + at;
    const int sy = br, sz = br * br;
    ld_pair<AT>(o, T.c[0], T.c[1]);
    ld_pair<AT>(o + sy, T.c[2], T.c[3]);
    ld_pair<AT>(o + sz, T.c[4], T.c[5]);
    ld_pair<AT>(o + sz + sy, T.c[6], T.c[7]);
}

__device__ inline float tri_blend(const Taps& T) {
    const float* c = T.c;
    float c00 = c[0] + T.fx * (c[1] - c[0]), c10 = c[2] + T.fx * (c[3] - c[2]);
    float c01 = c[4] + T.fx * (c[5] - c[4]), c11 = c[6] + T.fx * (c[7] - c[6]);
    float c0 = c00 + T.fy * (c10 - c00), c1 = c01 + T.fy * (c11 - c01);
    return c0 + T.fz * (c1 - c0);
}

// The same sample where the lower tap may be the brick's last padded voxel
// (the gradient's tap half a voxel past a march sample): that tap's weight
// is 1 and its upper neighbour (outside the brick) is weighted 0, so the
// fetch takes the pair below and moves the upper value down.
template <typename AT>
__device__ inline float tri_edge(const AT* b, int br, const Corner& K, float x, float y, float z) {
    Taps T;
    tri_fetch<AT, 0>(b, br, K, x, y, z, T);
    float* c = T.c;
    if (int(floorf(x - 0.5f)) - K.c[0] == br - 1)
        for (int k = 0; k < 8; k += 2) c[k] = c[k + 1];
    if (int(floorf(y - 0.5f)) - K.c[1] == br - 1) {
        c[0] = c[2]; c[1] = c[3]; c[4] = c[6]; c[5] = c[7];
    }
    if (int(floorf(z - 0.5f)) - K.c[2] == br - 1)
        for (int k = 0; k < 4; k++) c[k] = c[k + 4];
    return tri_blend(T);
}

// getColorF (kernels/cuda_gvdb_raycast.cuh:206-209): the colour channel's
// voxel at the integer part of the atlas position, bytes / 255
__device__ inline float4 color_at(const uint32_t* cb, int br, const Corner& K, float x, float y, float z) {
    const int ix = min(max(int(x) - K.c[0], 0), br - 1), iy = min(max(int(y) - K.c[1], 0), br - 1),
              iz = min(max(int(z) - K.c[2], 0), br - 1);
    const uint32_t c = cb[(iz * br + iy) * br + ix];
    return make_float4(float(c & 0xFFu) / 255.0f, float((c >> 8) & 0xFFu) / 255.0f, float((c >> 16) & 0xFFu) / 255.0f,
                       float(c >> 24) / 255.0f);
}

// x / d where `inv` is 1 / d when d is a power of two (the product is then
// the quotient, both exact roundings of one number) and 0 otherwise.
__device__ inline float div_by(float x, float d, float inv) { return inv != 0.0f ? x * inv : x / d; }

// What the walk needs of a level, in LDS: a lane's level is its own, so
// indexing the kernel's arguments by it would be a memory load each time.
struct LevelInfo {
    const Node* nodes;
    const u64* clists;
    float vdel, inv;  // width of a cell (a child's range), a power of two of at least 1, and 1 / it
    int logdim;
};

// L lanes hold one ray (64 / L rays per workgroup).  The rays' level stacks
// and the bricks their walks have found ahead live in LDS.
static const int QUEUE = 8;   // (4: 256^2 0.250 ms, 8: 0.231 ms; 2: 0.316 ms)
template <int L>
struct RenderShared {
    LevelInfo lev[MAXLEV];
    uint2 queue[QUEUE][64 / L];     // leaf index, entry time
    int nodeid[MAXLEV][64 / L];     // (all MAXLEV levels: 9.5 KB a workgroup for L = 1, 2.6 KB for L = 4)
    float tMax[MAXLEV][64 / L];
};

__device__ inline bool inside(f3 p, float r0) {
    // (a NaN fails, or, alone on its axis, gives taps that are NaN and pass no test)
    return fminf(fminf(p.x, p.y), p.z) >= 0.0f && fmaxf(fmaxf(p.x, p.y), p.z) < r0;
}

// The march through one brick: its data, the corner, the next sample's
// position in the brick and its number.
template <typename AT>
struct March {
    const AT* b;
    u64 slot;             // offset of the brick in every channel
    Corner K;
    f3 p, vmin;
    int it;
};

template <typename AT>
__device__ inline void march_enter(March<AT>& M, const RenderArgs& A, const AT* atlas, const Node* nodes0, int id, float tin,
                                   f3 pos, f3 dir) {
    const Node* n = nodes0 + id;
    const int np[3] = {n->mPos[0], n->mPos[1], n->mPos[2]}, v[3] = {n->mValue[0], n->mValue[1], n->mValue[2]};
    // the slot's coordinates v / brick side as products with its rounded-up
    // reciprocal (exact while v * brick side < 2^32; -1, a leaf without a
    // slot, is slot 0 as the division makes it)
    auto side = [&](int x) { return __umulhi(unsigned(max(x, 0)), A.br_inv); };
    u64 slot = (u64(side(v[2])) * unsigned(A.t.atlas_cnt[1]) + side(v[1])) * unsigned(A.t.atlas_cnt[0]) + side(v[0]);
    M.slot = slot * unsigned(A.t.brick_vox);
    M.b = atlas + M.slot;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        M.K.c[a] = v[a] - A.t.apron;
        M.K.o[a] = float(v[a]);
    }
    M.K.base = float((M.K.c[2] * 10 + M.K.c[1]) * 10 + M.K.c[0]);
    M.vmin = mk3(float(np[0]), float(np[1]), float(np[2]));
    const float dstep = A.s.steps[0];
    const float tx = dstep * ceilf(div_by(tin, dstep, A.step_inv));
    M.p = pos + dir * tx - M.vmin;
    M.it = 0;
}

// Lanes of a ray.
template <int L>
__device__ inline uint32_t group_mask(bool p, int g0) {
    return uint32_t(__ballot(p) >> g0) & ((1u << L) - 1u);
}
// the value of lane U of the group on all of its lanes (a quad permutation)
template <int L, int U>
__device__ inline float group_get(float v) {
    static_assert(L == 4 && U < 4, "groups are quads");
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), U * 0x55, 0xF, 0xF, true));
}

// Entry i of the transfer function.  A table that is one linear ramp (set over
// its whole range by LinearTransferFunc) is evaluated as the host filled it,
// the same products and sums; another one is read.
__device__ inline float4 tf_at(const RenderArgs& A, int i) {
    if (!A.tf_ramp) return A.tf[i];
    const float x = float(i) * (1.0f / float(TF_SIZE));
    return make_float4(A.tf_a[0] + x * A.tf_d[0], A.tf_a[1] + x * A.tf_d[1], A.tf_a[2] + x * A.tf_d[2],
                       A.tf_a[3] + x * A.tf_d[3]);
}

// One step of rayDeepBrick (emission-absorption): U samples fetched ahead
// (positions advanced one step at a time, as the reference does), then
// accumulated in order under the reference's loop conditions; a sample past
// the end is fetched but never used.  Returns whether the brick goes on.
template <typename AT, int U, int BR>
__device__ inline bool deep_step(const RenderArgs& A, March<AT>& M, f3 wpt, float clr[4]) {
    const int br = BR ? BR : A.t.brick_res;
    const float r0 = float(A.t.res[0]);
    const float minval = A.s.cutoff[0], alphacut = A.s.cutoff[1];
    static_assert(MAX_ITER % U == 0, "the sample count ends between batches");
    const bool first = M.it < MAX_ITER;
    Taps T[U];
    bool ok[U];
    f3 q = M.p;
#pragma unroll
    for (int u = 0; u < U; u++) {
        ok[u] = first && inside(q, r0);
        tri_fetch<AT, BR>(M.b, br, M.K, q.x + M.K.o[0], q.y + M.K.o[1], q.z + M.K.o[2], T[u]);
        q = q + wpt;
    }
    float raw[U];
    bool any = false;
#pragma unroll
    for (int u = 0; u < U; u++) {
        raw[u] = tri_blend(T[u]);
        any = any || (ok[u] && raw[u] >= minval);
    }
    bool live = true;
    if (any) {
        const float extinct = A.s.extinct[0], albedo = A.s.extinct[1], dstep = A.s.steps[0];
        const float th = A.s.thresh[0], vr = A.s.thresh[2] - A.s.thresh[1];
        float4 val[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const float x = fminf(1.0f, fmaxf(0.0f, div_by(raw[u] - th, vr, A.vr_inv)));
            val[u] = tf_at(A, int(x * 16300.0f));
        }
        f3 p = M.p;
#pragma unroll
        for (int u = 0; u < U; u++) {
            live = live && clr[3] > alphacut && ok[u];
            if (live && raw[u] >= minval) {
                // the reference's products, left to right; the colour channel's
                // factor only when there is one (a factor of 1 changes nothing)
                float w = expf(extinct * val[u].w * dstep);
                float kx = val[u].x * clr[3] * (1.0f - w) * albedo, ky = val[u].y * clr[3] * (1.0f - w) * albedo,
                      kz = val[u].z * clr[3] * (1.0f - w) * albedo;
                if (A.clr) {
                    const float4 h = color_at(A.clr + M.slot, br, M.K, p.x + M.K.o[0], p.y + M.K.o[1], p.z + M.K.o[2]);
                    kx = kx * h.x;
                    ky = ky * h.y;
                    kz = kz * h.z;
                }
                clr[0] += kx;
                clr[1] += ky;
                clr[2] += kz;
                clr[3] *= w;
            }
            p = p + wpt;
        }
    }
    live = live && clr[3] > alphacut;
#pragma unroll
    for (int u = 0; u < U; u++) live = live && ok[u];
    M.p = q;
    M.it += U;
    return live;
}

// One lane's sample: table colour, exp(extinct * alpha * step), colour-channel factor.
struct EaSample {
    float x, y, z, w, hx, hy, hz;
};

// Accumulates samples U..L-1 of the batch under the reference's loop conditions.
template <int L, int U>
__device__ inline void ea_accumulate(const EaSample& s, uint32_t okm, uint32_t actm, bool colour, float albedo,
                                     float alphacut, float clr[4], bool& live) {
    if constexpr (U < L) {
        const float w = group_get<L, U>(s.w);
        float kx = group_get<L, U>(s.x), ky = group_get<L, U>(s.y), kz = group_get<L, U>(s.z);
        live = live && clr[3] > alphacut && ((okm >> U) & 1u);
        if (live && ((actm >> U) & 1u)) {
            const float e = 1.0f - w;
            kx = kx * clr[3] * e * albedo;
            ky = ky * clr[3] * e * albedo;
            kz = kz * clr[3] * e * albedo;
            if (colour) {
                kx = kx * group_get<L, U>(s.hx);
                ky = ky * group_get<L, U>(s.hy);
                kz = kz * group_get<L, U>(s.hz);
            }
            clr[0] += kx;
            clr[1] += ky;
            clr[2] += kz;
            clr[3] *= w;
        }
        ea_accumulate<L, U + 1>(s, okm, actm, colour, albedo, alphacut, clr, live);
    }
}

// The same step with L lanes per ray: lane k of the group holds sample k of
// the batch (M.p and M.it are its own), so a batch costs a lane one fetch,
// blend, table read and exp; every lane then accumulates the batch in order.
template <typename AT, int L, int BR>
__device__ inline bool deep_step_split(const RenderArgs& A, March<AT>& M, f3 wpt, int g0, float clr[4]) {
    const int br = BR ? BR : A.t.brick_res;
    const float r0 = float(A.t.res[0]);
    const float minval = A.s.cutoff[0], alphacut = A.s.cutoff[1];
    const bool ok = M.it < MAX_ITER && inside(M.p, r0);
    const uint32_t okm = group_mask<L>(ok, g0);
    Taps T;
    tri_fetch<AT, BR>(M.b, br, M.K, M.p.x + M.K.o[0], M.p.y + M.K.o[1], M.p.z + M.K.o[2], T);
    const float raw = tri_blend(T);
    const bool act = ok && raw >= minval;
    const uint32_t actm = group_mask<L>(act, g0);
    bool live = true;
    if (actm) {
        EaSample v{0, 0, 0, 1, 1, 1, 1};
        if (act) {
            const float th = A.s.thresh[0], vr = A.s.thresh[2] - A.s.thresh[1];
            const float x = fminf(1.0f, fmaxf(0.0f, div_by(raw - th, vr, A.vr_inv)));
            const float4 val = tf_at(A, int(x * 16300.0f));
            v.x = val.x;
            v.y = val.y;
            v.z = val.z;
            v.w = expf(A.s.extinct[0] * val.w * A.s.steps[0]);
            if (A.clr) {
                const float4 h = color_at(A.clr + M.slot, br, M.K, M.p.x + M.K.o[0], M.p.y + M.K.o[1], M.p.z + M.K.o[2]);
                v.hx = h.x;
                v.hy = h.y;
                v.hz = h.z;
            }
        }
        ea_accumulate<L, 0>(v, okm, actm, A.clr != nullptr, A.s.extinct[1], alphacut, clr, live);
    }
#pragma unroll
    for (int k = 0; k < L; k++) M.p = M.p + wpt;
    M.it += L;
    return live && clr[3] > alphacut && okm == (1u << L) - 1u;
}

// One step of raySurfaceTrilinearBrick: U samples (L = 1) or L samples, one
// per lane of the ray; 0: the brick goes on, 1: it ends, 2: a sample reached
// the threshold and M.p is its position.
template <typename AT, int U, int L, int BR>
__device__ inline int surf_step(const RenderArgs& A, March<AT>& M, f3 wpt, int g0) {
    const int br = BR ? BR : A.t.brick_res;
    const float r0 = float(A.t.res[0]);
    const float th = A.s.thresh[0];
    if constexpr (L > 1) {
        const bool ok = M.it < MAX_ITER && inside(M.p, r0);
        const uint32_t out = group_mask<L>(!ok, g0);
        Taps T;
        tri_fetch<AT, BR>(M.b, br, M.K, M.p.x + M.K.o[0], M.p.y + M.K.o[1], M.p.z + M.K.o[2], T);
        // samples at or above the threshold before the first one outside
        const uint32_t h = group_mask<L>(tri_blend(T) >= th, g0) & (out ? (out & (0u - out)) - 1u : (1u << L) - 1u);
        if (h) {
            const int u = g0 + __ffs(h) - 1;
            M.p = mk3(__shfl(M.p.x, u, 64), __shfl(M.p.y, u, 64), __shfl(M.p.z, u, 64));
            return 2;
        }
#pragma unroll
        for (int k = 0; k < L; k++) M.p = M.p + wpt;
        M.it += L;
        return out ? 1 : 0;
    } else {
        static_assert(MAX_ITER % U == 0, "the sample count ends between batches");
        const bool first = M.it < MAX_ITER;
        Taps T[U];
        bool ok[U];
        f3 q = M.p;
#pragma unroll
        for (int u = 0; u < U; u++) {
            ok[u] = first && inside(q, r0);
            tri_fetch<AT, BR>(M.b, br, M.K, q.x + M.K.o[0], q.y + M.K.o[1], q.z + M.K.o[2], T[u]);
            q = q + wpt;
        }
        int r = 0;
        f3 p = M.p;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int e = !ok[u] ? 1 : (tri_blend(T[u]) >= th ? 2 : 0);
            if (r == 0 && e != 0) { r = e; M.p = p; }
            p = p + wpt;
        }
        if (r == 0) M.p = q;
        M.it += U;
        return r;
    }
}

// getGradient at the atlas position of the hit, the hit's colour.
template <typename AT, int L, int BR>
__device__ inline void surf_hit(const RenderArgs& A, const March<AT>& M, int s, f3& hit, f3& nrm, float hclr[4]) {
    const int br = BR ? BR : A.t.brick_res;
    hit = M.p + M.vmin;
    const f3 P = mk3(M.p.x + M.K.o[0], M.p.y + M.K.o[1], M.p.z + M.K.o[2]);
    f3 g;
    if constexpr (L > 1) {
        // lane k of the ray takes axis k (adding or subtracting 0 leaves the
        // other components as they are)
        const float hx = s == 0 ? 0.5f : 0.0f, hy = s == 1 ? 0.5f : 0.0f, hz = s == 2 ? 0.5f : 0.0f;
        const float d = tri_edge<AT>(M.b, br, M.K, P.x - hx, P.y - hy, P.z - hz) -
                        tri_edge<AT>(M.b, br, M.K, P.x + hx, P.y + hy, P.z + hz);
        g = mk3(group_get<L, 0>(d), group_get<L, 1>(d), group_get<L, 2>(d));
    } else {
        float d[3];
#pragma nounroll
        for (int a = 0; a < 3; a++) {
            const float hx = a == 0 ? 0.5f : 0.0f, hy = a == 1 ? 0.5f : 0.0f, hz = a == 2 ? 0.5f : 0.0f;
            const float e = tri_edge<AT>(M.b, br, M.K, P.x - hx, P.y - hy, P.z - hz) -
                            tri_edge<AT>(M.b, br, M.K, P.x + hx, P.y + hy, P.z + hz);
            if (a == 0) d[0] = e;
            if (a == 1) d[1] = e;
            if (a == 2) d[2] = e;
        }
        g = mk3(d[0], d[1], d[2]);
    }
    nrm = norm3(g);
    if (A.clr) {
        const float4 h = color_at(A.clr + M.slot, br, M.K, P.x, P.y, P.z);
        hclr[0] = h.x; hclr[1] = h.y; hclr[2] = h.z; hclr[3] = h.w;
    }
}

// The walk's state at the current node: HDDA as the reference's, with the
// node's child list, level facts and exit time in registers.
struct Walk {
    f3 tDel, tSide;
    float tx, tmax, inv;
    int p[3];
    int lev, logdim, it;
    const u64* cl;     // the node's child list, or null
};

// Sets the walk up in node `id` of level `lev` at time w.tx (Prepare of the
// reference's HDDA: cell widths are powers of two of at least 1, so the
// division by one is the product with its reciprocal, and |width / dir| of
// one level is that of another times their ratio).
template <int L>
__device__ inline void walk_enter(Walk& w, const RenderShared<L>& S, int lev, int id, f3 pos, f3 dir) {
    const LevelInfo I = S.lev[lev];
    const Node* n = I.nodes + id;
    const int np[3] = {n->mPos[0], n->mPos[1], n->mPos[2]};
    const u64 list = n->mChildList;
    const float inv = I.inv, k = I.vdel * w.inv;
    w.lev = lev;
    w.logdim = I.logdim;
    w.inv = inv;
    w.tDel = w.tDel * k;
    const float pf[3] = {(pos.x + w.tx * dir.x - float(np[0])) * inv, (pos.y + w.tx * dir.y - float(np[1])) * inv,
                         (pos.z + w.tx * dir.z - float(np[2])) * inv};
    const float td[3] = {w.tDel.x, w.tDel.y, w.tDel.z}, ds[3] = {dir.x > 0 ? 1.0f : -1.0f, dir.y > 0 ? 1.0f : -1.0f,
                                                                dir.z > 0 ? 1.0f : -1.0f};
    float ts[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float fl = floorf(pf[a]);
        ts[a] = ((fl - pf[a] + 0.5f) * ds[a] + 0.5f) * td[a] + w.tx;
        w.p[a] = int(fl);
    }
    w.tSide = mk3(ts[0], ts[1], ts[2]);
    // the child list (usually of the node's own level)
    const int clev = int((list >> 8) & 0xFF);
    const LevelInfo& C = S.lev[clev < MAXLEV ? clev : 0];
    w.cl = list == ID_UNDEFL ? nullptr : C.clists + ((list >> 16) << (3 * C.logdim));
}

// One iteration of rayCast's loop: the brick of the cell the walk stands in
// (>= 0; the walk steps past it), -1 for another cell or a descent, -2 at the
// end of the walk.  tin: the brick's entry time.
template <int L>
__device__ inline int walk_step(Walk& w, RenderShared<L>& S, int top, int ray, float eps, f3 pos, f3 dir, float& tin) {
    const int res = 1 << w.logdim;
    const int plo = min(min(w.p[0], w.p[1]), w.p[2]), phi = max(max(w.p[0], w.p[1]), w.p[2]);
    if (!(w.it < MAX_ITER && w.lev <= top && plo >= 0 && phi <= res)) return -2;
    int child = -1;
    if (phi < res && w.cl) child = int(w.cl[(((w.p[2] << w.logdim) + w.p[1]) << w.logdim) + w.p[0]] >> 16);
    const bool b0 = (w.tSide.x < w.tSide.y) & (w.tSide.x <= w.tSide.z);
    const bool b1 = (w.tSide.y < w.tSide.z) & (w.tSide.y <= w.tSide.x);
    const bool b2 = (w.tSide.z < w.tSide.x) & (w.tSide.z <= w.tSide.y);
    const float ty = b0 ? w.tSide.x : (b1 ? w.tSide.y : w.tSide.z);
    w.it++;
    int brick = -1, lev = w.lev;
    bool enter = false;
    if (child >= 0 && lev > 1) {
        lev--;
        S.nodeid[lev][ray] = child;
        w.tx += eps;
        w.tmax = ty - eps;
        S.tMax[lev][ray] = w.tmax;
        enter = true;
    } else {
        brick = child;
        tin = w.tx + eps;
        w.tx = ty;
        w.tSide = w.tSide + mk3((b0 ? 1.0f : 0.0f) * w.tDel.x, (b1 ? 1.0f : 0.0f) * w.tDel.y, (b2 ? 1.0f : 0.0f) * w.tDel.z);
        w.p[0] += b0 ? (dir.x > 0 ? 1 : -1) : 0;
        w.p[1] += b1 ? (dir.y > 0 ? 1 : -1) : 0;
        w.p[2] += b2 ? (dir.z > 0 ? 1 : -1) : 0;
    }
    // up to the level whose node the walk is still in; its Prepare depends on
    // the time alone, so only the last node is entered
    while (lev <= top && w.tx > w.tmax) {
        lev++;
        enter = true;
        if (lev <= top) w.tmax = S.tMax[lev][ray];
    }
    w.lev = lev;
    if (enter && lev <= top) walk_enter<L>(w, S, lev, S.nodeid[lev][ray], pos, dir);
    return brick;
}

// rayCast.  MODE 0: deep (EA), MODE 1: trilinear surface.
// The rays of a wave do not wait for each other at brick borders: the walks
// run ahead and queue the bricks they find (all rays with room step together
// until none lacks a brick), and each pass of the loop takes one batch of
// samples of every ray's own brick.
template <int MODE, typename AT, int U, int L, int BR>
__device__ inline void ray_cast(const RenderArgs& A, const AT* atlas, bool on, f3 pos, f3 dir, f3& hit, f3& nrm,
                                float clr[4], RenderShared<L>& S) {
    const Tree& t = A.t;
    const int lane = threadIdx.x & 63, ray = lane / L, s = lane & (L - 1), g0 = lane & ~(L - 1);
    const int top = t.top_lev;
    const float eps = t.epsilon;
    float h0 = (t.bmin[0] - pos.x) / dir.x, h1 = (t.bmax[0] - pos.x) / dir.x;
    float h2 = (t.bmin[1] - pos.y) / dir.y, h3 = (t.bmax[1] - pos.y) / dir.y;
    float h4 = (t.bmin[2] - pos.z) / dir.z, h5 = (t.bmax[2] - pos.z) / dir.z;
    float t0 = fmaxf(fmaxf(fminf(h0, h1), fminf(h2, h3)), fminf(h4, h5));
    float t1 = fminf(fminf(fmaxf(h0, h1), fmaxf(h2, h3)), fmaxf(h4, h5));
    t0 = (t0 < 0) ? 0.0f : t0;
    bool alive = on && !(t1 < t0 || t1 < 0) && top > 0;   // a top node without cells: nothing to step through
    bool walking = alive, have = false, found = false;
    Walk w;
    w.it = 0;
    w.tx = t0 + eps;
    w.tmax = t1 - eps;
    w.inv = 1.0f;
    w.tDel = mk3(fabsf(1.0f / dir.x), fabsf(1.0f / dir.y), fabsf(1.0f / dir.z));
    S.nodeid[top][ray] = 0;
    S.tMax[top][ray] = w.tmax;
    if (alive) walk_enter<L>(w, S, top, 0, pos, dir);
    const f3 wpt = dir * A.s.steps[0];
    March<AT> M;
    uint32_t qh = 0, qn = 0;
    for (;;) {
        while (__any(alive && !have && qn == 0 && walking)) {
            if (alive && walking && qn < QUEUE) {
                float tin = 0.0f;
                const int b = walk_step<L>(w, S, top, ray, eps, pos, dir, tin);
                if (b == -2) walking = false;
                if (b >= 0) {
                    S.queue[(qh + qn) & (QUEUE - 1)][ray] = make_uint2(uint32_t(b), __float_as_uint(tin));
                    qn++;
                }
            }
        }
        if (alive && !have) {
            alive = qn > 0;
            if (alive) {
                const uint2 e = S.queue[qh][ray];
                qh = (qh + 1) & (QUEUE - 1);
                qn--;
                march_enter<AT>(M, A, atlas, S.lev[0].nodes, int(e.x), __uint_as_float(e.y), pos, dir);
                if constexpr (L > 1) {
                    // lane s starts at sample s (positions advanced one step at a time)
#pragma unroll
                    for (int k = 1; k < L; k++) {
                        const f3 q = M.p + wpt;
                        if (s >= k) M.p = q;
                    }
                    M.it = s;
                }
                have = true;
            }
        }
        if (!__any(alive)) break;
        if (have) {
            if (MODE == 0) {
                bool more;
                if constexpr (L > 1) more = deep_step_split<AT, L, BR>(A, M, wpt, g0, clr);
                else more = deep_step<AT, U, BR>(A, M, wpt, clr);
                if (!more) {
                    have = false;
                    clr[0] = fminf(clr[0], 1.0f); clr[1] = fminf(clr[1], 1.0f); clr[2] = fminf(clr[2], 1.0f);
                    clr[3] = fmaxf(clr[3], 0.0f);
                    // at or under the cutoff no later brick adds anything
                    if (clr[3] <= 0 || !(clr[3] > A.s.cutoff[1])) {
                        if (clr[3] <= 0) clr[3] = 0;
                        alive = false;
                    }
                }
            } else {
                const int r = surf_step<AT, U, L, BR>(A, M, wpt, g0);
                if (r) have = false;
                if (r == 2) {
                    found = true;
                    alive = false;
                }
            }
        }
    }
    if (MODE == 1 && found) surf_hit<AT, L, BR>(A, M, s, hit, nrm, clr);
}

__device__ inline f3 mmult(const float* m, f3 v) {
    return mk3(v.x * m[0] + v.y * m[4] + v.z * m[8] + m[12], v.x * m[1] + v.y * m[5] + v.z * m[9] + m[13],
               v.x * m[2] + v.y * m[6] + v.z * m[10] + m[14]);
}

template <int MODE, typename AT, int U, int L, int BR>
__device__ inline void k_render_body(const RenderArgs& A, uint32_t bid, RenderShared<L>& S) {
    if (int(threadIdx.x) < A.t.levels) {
        const int l = threadIdx.x;
        const float vdel = float(A.t.range[l] >> A.t.logdim[l]);
        S.lev[l] = LevelInfo{A.t.nodes[l], A.t.clists[l], vdel, 1.0f / vdel, A.t.logdim[l]};
    }
    __syncthreads();
    // the workgroup's ray packet: a tile_w x (64 / L / tile_w) pixel tile
    const int tw = A.tile_w, sh = __builtin_ctz(unsigned(tw));
    const int tiles_x = (A.s.width + tw - 1) >> sh;
    const int tile = int(bid);
    const unsigned ray = threadIdx.x / unsigned(L);
    const int x = (tile % tiles_x) * tw + int(ray & unsigned(tw - 1));
    const int y = (tile / tiles_x) * ((64 / L) >> sh) + int(ray >> sh);
    const bool on = x < A.s.width && y < A.s.height;
    const AT* atlas = reinterpret_cast<const AT*>(A.atlas);
    f3 rpos = mmult(A.s.invxform, mk3(A.s.campos[0], A.s.campos[1], A.s.campos[2]));
    float fx = float(x + 0.5f) / float(A.s.width), fy = float(y + 0.5f) / float(A.s.height);
    f3 v = mk3(fx * A.s.camu[0] + fy * A.s.camv[0] + A.s.cams[0], fx * A.s.camu[1] + fy * A.s.camv[1] + A.s.cams[1],
               fx * A.s.camu[2] + fy * A.s.camv[2] + A.s.cams[2]);
    f3 rdir = norm3(mmult(A.s.invxrot, v));
    float res[4];
    if (MODE == 0) {
        float clr[4] = {0, 0, 0, 1};
        f3 hit = mk3(0, 0, NOHIT), nrm = mk3(0, 0, 0);
        ray_cast<0, AT, U, L, BR>(A, atlas, on, rpos, rdir, hit, nrm, clr, S);
        float a = 1.0f - clr[3];
        for (int k = 0; k < 3; k++) res[k] = A.s.backclr[k] + a * (clr[k] - A.s.backclr[k]);
        res[3] = a;
    } else {
        float clr[4] = {1, 1, 1, 1};
        f3 hit = mk3(NOHIT, NOHIT, NOHIT), nrm = mk3(0, 0, 0);
        // the primary ray, then the shadow ray, through the same code
        f3 pos = rpos, dir = rdir;
        float diff = 0.0f;
        bool cast = on;
#pragma nounroll
        for (int pass = 0; pass < 2; pass++) {
            f3 h2 = mk3(NOHIT, NOHIT, NOHIT), n2 = mk3(0, 0, 0);
            float c2[4] = {1, 1, 1, 1};
            ray_cast<1, AT, U, L, BR>(A, atlas, cast, pos, dir, h2, n2, c2, S);
            if (pass == 0) {
                hit = h2;
                nrm = n2;
                for (int k = 0; k < 4; k++) clr[k] = c2[k];
                cast = cast && hit.z != NOHIT;
                const f3 lp = mk3(A.s.light_pos[0], A.s.light_pos[1], A.s.light_pos[2]);
                dir = norm3(lp - hit);
                diff = 0.9f * fmaxf(0.0f, dot3(nrm, dir));
                pos = hit + nrm * A.s.shadow[1];
                if (!(A.s.shadow[0] > 0) || !__any(cast)) break;
            } else if (cast && h2.z != NOHIT) {
                diff = diff * (1.0f - A.s.shadow[0]);
            }
        }
        if (hit.z == NOHIT) {
            for (int k = 0; k < 4; k++) res[k] = A.s.backclr[k];
        } else {
            const float amb = 0.1f;
            for (int k = 0; k < 3; k++) res[k] = clr[k] * (diff + amb);
            res[3] = 1.0f;
        }
    }
    if (!on || (L > 1 && (threadIdx.x & (L - 1)))) return;
    u64 pix = u64(y) * A.s.width + x;
    if (A.out_float) {
        reinterpret_cast<float4*>(A.out)[pix] = make_float4(res[0], res[1], res[2], res[3]);
    } else {
        uchar4 c;
        c.x = (unsigned char)(res[0] * 255.0f);
        c.y = (unsigned char)(res[1] * 255.0f);
        c.z = (unsigned char)(res[2] * 255.0f);
        c.w = (unsigned char)(res[3] * 255.0f);
        reinterpret_cast<uchar4*>(A.out)[pix] = c;
    }
}

// One 64-thread workgroup per pixel tile; several grids' images in one launch.
// Occupancy asked of the compiler: four waves per SIMD (128 VGPRs) hold the
// taps of four samples, but for 17 to 20 words of the isosurface's FP32 form;
// five spill there (isosurface 1024^2 0.52 -> 1.2 ms) and three gain nothing.
// One sample or two, or one per lane, are compiled for five (two samples spill 3
// to 17 words); with one lane per ray the 9.5 KB of LDS allow 17 waves a CU.
template <int MODE, typename AT, int U, int L, int BR>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(U == 4 ? 4 : 5))) void k_render(RenderArgs a0,
                                                                                                    MultiMap m) {
    __shared__ RenderShared<L> S;
    if (m.G <= 1) {
        k_render_body<MODE, AT, U, L, BR>(a0, blockIdx.x, S);
        return;
    }
    const int g = multi_grid(m, blockIdx.x);
    k_render_body<MODE, AT, U, L, BR>(multi_rec<RenderArgs>(m, g), blockIdx.x - multi_first(m)[g], S);
}

// Launches of up to this many rays take four lanes per ray: with one, they
// are at most 1.5 waves per SIMD (256 CUs, 4 SIMDs) and last as long as their
// longest wave's chain of samples.  Measured (ms, one lane / four): 100^2
// emission-absorption 0.239 / 0.196, 256^2 0.218 / 0.200, 300^2 isosurface
// 0.330 / 0.295; past the line the walks repeated on four lanes cost more:
// 512^2 1.17 / 1.35, isosurface 1024^2 0.52 / 0.80.
static const u64 SPLIT_RAYS = 98304;
static const int SPLIT = 4;

// Samples fetched ahead per brick step and the ray-packet shape come from
// the launch-shape knobs (tune.cpp): defaults are the measured winners, the
// autotuner re-picks them for the caller's scene; brick sides other than 10 and
// atlases of 2^17 voxels a side take them too (4^3 bricks, 500 k points of a
// shell, one sample / four: emission-absorption 512^2 0.51 / 0.41 ms,
// isosurface 1024^2 0.65 / 0.49).
template <int MODE, typename AT>
static void launch_as(bool ten, bool split, int u, dim3 grid, hipStream_t s, const RenderArgs& a0, const MultiMap& m) {
    if (!ten && u == 4) hipLaunchKernelGGL((k_render<MODE, AT, 4, 1, 0>), grid, dim3(64), 0, s, a0, m);
    else if (!ten && u == 2) hipLaunchKernelGGL((k_render<MODE, AT, 2, 1, 0>), grid, dim3(64), 0, s, a0, m);
    else if (!ten) hipLaunchKernelGGL((k_render<MODE, AT, 1, 1, 0>), grid, dim3(64), 0, s, a0, m);
    else if (split) hipLaunchKernelGGL((k_render<MODE, AT, 1, SPLIT, 10>), grid, dim3(64), 0, s, a0, m);
    else if (u == 4) hipLaunchKernelGGL((k_render<MODE, AT, 4, 1, 10>), grid, dim3(64), 0, s, a0, m);
    else if (u == 2) hipLaunchKernelGGL((k_render<MODE, AT, 2, 1, 10>), grid, dim3(64), 0, s, a0, m);
    else hipLaunchKernelGGL((k_render<MODE, AT, 1, 1, 10>), grid, dim3(64), 0, s, a0, m);
}

// The index arithmetic of BR = 10 (tri_fetch): 111 times the side below 2^24.
static bool ten_sided(const Tree& t) {
    for (int a = 0; a < 3; a++)
        if ((long long)t.atlas_cnt[a] * 10 >= (1 << 17)) return false;
    return t.brick_res == 10 && t.apron == 1;
}

// 1 / d when d is a power of two (of a size whose inverse is one too), else 0.
static float pow2_inverse(float d) {
    int e = 0;
    const float m = std::frexp(d, &e);
    return std::fabs(m) == 0.5f && e > -100 && e < 100 ? 1.0f / d : 0.0f;
}

// One launch per variant of the kernel: bit 0 isosurface, 1 half, 2 not ten_sided.
static int variant_of(const RenderArgs& a) {
    return (a.shading == SHADE_VOLUME ? 0 : 1) | (a.atlas_type == T_HALF ? 2 : 0) | (ten_sided(a.t) ? 0 : 4);
}
// Do the images of `variant` (if any) go with four lanes per ray?
static bool split_of(const RenderArgs* a, int G, int variant) {
    u64 rays = 0;
    for (int g = 0; g < G; g++)
        if (variant_of(a[g]) == variant) rays += u64(a[g].s.width) * u64(a[g].s.height);
    return !(variant & 4) && rays <= SPLIT_RAYS;
}

bool render_reads_knobs(const RenderArgs* a, int G) {
    for (int g = 0; g < G; g++)
        if (variant_of(a[g]) % 2 == variant_of(a[0]) % 2 && !split_of(a, G, variant_of(a[g]))) return true;
    return false;
}

hipError_t launch_render_multi(const RenderArgs* a, int G, Arena* ar, hipStream_t s) {
    for (int g = 0; g < G; g++)
        if (a[g].shading != SHADE_VOLUME && a[g].shading != SHADE_TRILINEAR) return hipErrorInvalidValue;
    for (int variant = 0; variant < 8; variant++) {
        const int mode = variant & 1;
        const bool half = variant & 2, ten = !(variant & 4);
        std::vector<RenderArgs> sel;
        for (int g = 0; g < G; g++)
            if (variant_of(a[g]) == variant) sel.push_back(a[g]);
        if (sel.empty()) continue;
        const bool split = split_of(sel.data(), int(sel.size()), variant);
        const int per = split ? 64 / SPLIT : 64;
        const int tw = split ? 4 : knob(mode ? KNOB_RENDER_TILE_ISO : KNOB_RENDER_TILE_EA), th = per / tw;
        std::vector<uint32_t> nb;
        for (RenderArgs& r : sel) {
            r.tile_w = tw;
            r.br_inv = uint32_t((0x100000000ull + unsigned(r.t.brick_res) - 1) / unsigned(r.t.brick_res));
            r.step_inv = pow2_inverse(r.s.steps[0]);
            r.vr_inv = pow2_inverse(r.s.thresh[2] - r.s.thresh[1]);
            nb.push_back(uint32_t(((r.s.width + tw - 1) / tw) * ((r.s.height + th - 1) / th)));
        }
        MultiLaunch L;
        hipError_t e = multi_setup(ar, sel.data(), nb.data(), int(sel.size()), s, L);
        if (e != hipSuccess) return e;
        if (L.blocks == 0) continue;
        const int u = knob(mode ? KNOB_RENDER_UNROLL_ISO : KNOB_RENDER_UNROLL_EA);
        if (mode == 0 && half) launch_as<0, __half>(ten, split, u, dim3(L.blocks), s, sel[0], L.map);
        else if (mode == 0) launch_as<0, float>(ten, split, u, dim3(L.blocks), s, sel[0], L.map);
        else if (half) launch_as<1, __half>(ten, split, u, dim3(L.blocks), s, sel[0], L.map);
        else launch_as<1, float>(ten, split, u, dim3(L.blocks), s, sel[0], L.map);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace gvdb
