// compute.hip -- Compute(effect, ...) operators on float and half atlas
// channels (src/gvdb_volume_gvdb.cpp:4527-4552; kernels/cuda_gvdb_operators.cuh
// :148-455 of the reference).
//
// The reference launches 8x8x8 blocks over the 3D atlas texture.  Its
// "packed" operators (smooth, noise, grow) give each block one atlas brick:
// the block reads the brick's padded 10^3 voxels into shared memory and
// writes the 8^3 interior, so bricks never read each other's writes.  Here
// one 512-thread workgroup does the same for CB bricks of the brick-major
// atlas, over the bricks that hold leaves.  The "unpacked" fill writes every
// atlas voxel of [1, min(8 * blocks, res) - 1] per axis, apron voxels
// included, as the reference's indexing does.
#include "kernels.h"
#include "tree_device.h"
#include <hip/hip_fp16.h>
#include <algorithm>

#pragma clang fp contract(off)

namespace gvdb {

namespace {
template <typename AT> __device__ inline float ldv(const void* a, u64 o);
template <> __device__ inline float ldv<float>(const void* a, u64 o) { return static_cast<const float*>(a)[o]; }
template <> __device__ inline float ldv<__half>(const void* a, u64 o) {
    return __half2float(static_cast<const __half*>(a)[o]);
}
template <typename AT> __device__ inline void stv(void* a, u64 o, float v);
template <> __device__ inline void stv<float>(void* a, u64 o, float v) { static_cast<float*>(a)[o] = v; }
template <> __device__ inline void stv<__half>(void* a, u64 o, float v) { static_cast<__half*>(a)[o] = __float2half(v); }

// Bob Jenkins' one-at-a-time final mix and its compound forms, and the
// [0, 1) float built from the low 23 bits (random(float3),
// kernels/cuda_gvdb.cuh:135-164).
__device__ inline uint32_t oaat(uint32_t x) {
    x += (x << 10u);
    x ^= (x >> 6u);
    x += (x << 3u);
    x ^= (x >> 11u);
    x += (x << 15u);
    return x;
}
__device__ inline float random3(float a, float b, float c) {
    const uint32_t h = oaat(uint32_t(__float_as_int(a)) ^ oaat(uint32_t(__float_as_int(b))) ^
                            oaat(uint32_t(__float_as_int(c))));
    return __int_as_float(int((h & 0x007FFFFFu) | 0x3F800000u)) - 1.0f;
}
}  // namespace

// CB brick slots per workgroup: thread t owns interior voxel (t & 7, t >> 3 & 7,
// t >> 6) + 1 of each.  The padded bricks go through LDS, in whole 16-byte
// pieces where they come from or go to the atlas.  The operators are bound by
// the bytes they move (17 k bricks, FP32: 0.040 ms a pass at 3.4 TB/s for the
// padded bricks in and out).
//
// A smoothing of several iterations with the apron refreshed in between needs
// no apron in between: only the face neighbours are read.  Its iterations (from
// / to: the atlas or a.cells) keep the 512 interior voxels of every brick in
// a.cells and hand the boundary layers to the next iteration in two buffers in
// turn, and the apron is written once, after the last one.  17 k bricks, FP32,
// four iterations: four passes of 0.040 ms and four aprons of 0.027 ms before,
// 0.105 ms of passes and one apron of 0.019 ms now.
static const int CB = 4;
static const int BRICK = 1000;   // voxels of a padded 8^3 brick
static const int CELLS = 512;
static const int LAYERS = CB * 6 / 8;   // boundary layers per wave
static_assert(CB * 6 % 8 == 0, "whole layers per wave");

template <typename AT>
__device__ inline float apply_op(const ComputeArgs& a, const AT* b, int at, u64 slot, int lx, int ly, int lz) {
    float v = ldv<AT>(b, at);
    if (a.op == OP_SMOOTH) {
        // v = (p1 c + the six face neighbours) / (p1 + 6.0) + p2, the division
        // and the sum with p2 in double as the reference's double literal makes
        // them (the division a product where p1 + 6 is a power of two)
        v *= a.p1;
        v += ldv<AT>(b, at - 1);
        v += ldv<AT>(b, at + 1);
        v += ldv<AT>(b, at - 10);
        v += ldv<AT>(b, at + 10);
        v += ldv<AT>(b, at - 100);
        v += ldv<AT>(b, at + 100);
        const double q = a.inv != 0.0 ? double(v) * a.inv : double(v) / (double(a.p1) + 6.0);
        v = float(q + double(a.p2));
    } else if (a.op == OP_NOISE) {
        if (double(v) > 0.01) {
            const int sx = int(slot % u64(a.t.atlas_cnt[0]));
            const int sy = int((slot / u64(a.t.atlas_cnt[0])) % u64(a.t.atlas_cnt[1]));
            const int sz = int(slot / (u64(a.t.atlas_cnt[0]) * a.t.atlas_cnt[1]));
            v += random3(float(sx * 10 + lx), float(sy * 10 + ly), float(sz * 10 + lz)) * a.p1;
        }
    } else if (a.op == OP_GROW) {
        if (v != 0.0f) v = float(double(v) + double(a.p1) * 10.0);
        if (double(v) < 0.01) v = 0.0f;
    }
    return v;
}

// Boundary layers by slot in ApronArgs' order: voxel (u, w) of layer f is
// (z, y), (z, x) or (y, x) for the x, y and z layers; `edge` is its place along
// the layer's own axis.
__device__ inline int layer_voxel(int f, int u, int w, int edge) {
    if (f < 2) return (w * 10 + u) * 10 + edge;
    return f < 4 ? (w * 10 + edge) * 10 + u : (edge * 10 + w) * 10 + u;
}

// What the voxel beyond layer f of a slot comes from, in a.links[8 slot + f]:
// the neighbour's slot (its layers; below a.slots) or LINK_BOUND.  LINK_OWN:
// the slot holds no live brick, its apron stays as the atlas has it.
static const int LINK_BOUND = -1, LINK_OWN = -2;

__device__ inline int link_of(const ComputeArgs& a, u64 slot, int f) {
    const int leaf = a.t.amap[slot].mLeafNode;
    if (leaf < 0 || leaf >= a.leaves) return LINK_OWN;
    const long long* base = a.base + u64(leaf) * 27;
    if (base[13] != (long long)(slot * BRICK)) return LINK_OWN;
    const int step = f < 2 ? 1 : (f < 4 ? 3 : 9);
    const long long o = base[(f & 1) ? 13 + step : 13 - step];
    return o < 0 ? LINK_BOUND : int(u64(o) / u64(BRICK));
}

template <typename AT, bool FROM_CELLS, bool TO_CELLS>
__global__ __launch_bounds__(512) void k_compute_packed(ComputeArgs a) {
    __shared__ __align__(16) AT b[CB * BRICK];
    const u64 slot0 = u64(blockIdx.x) * CB;
    const int nb = min(CB, a.slots - int(slot0));
    const int pieces = nb * BRICK * int(sizeof(AT)) / 16;
    AT* const atlas = static_cast<AT*>(a.atlas);
    AT* const cells = static_cast<AT*>(a.cells);
    const int t = threadIdx.x;
    const int lx = (t & 7) + 1, ly = ((t >> 3) & 7) + 1, lz = (t >> 6) + 1;
    const int at = (lz * 10 + ly) * 10 + lx;
    // of the boundary layers, wave i takes LAYERS from LAYERS i on, a voxel per lane
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, u = lx, w = (lane >> 3) + 1;
    if (FROM_CELLS) {
        AT c[CB];
#pragma unroll
        for (int k = 0; k < CB; k++)
            if (k < nb) c[k] = cells[(slot0 + k) * CELLS + t];
        // a wave per layer: its link is one scalar load, and all are on their
        // way before the first is used
        const AT* faces = static_cast<const AT*>(a.faces_in);
        int l[LAYERS];
#pragma unroll
        for (int r = 0; r < LAYERS; r++) {
            const int q = wave * LAYERS + r;
            l[r] = q < nb * 6 ? a.links[(slot0 + q / 6) * 8 + q % 6] : LINK_BOUND;
        }
        AT g[LAYERS];
#pragma unroll
        for (int r = 0; r < LAYERS; r++) {
            const int q = wave * LAYERS + r, k = q / 6, f = q - k * 6;
            if (l[r] >= 0) g[r] = faces[u64(l[r]) * FACE_VALS + u64((f ^ 1) * 64 + lane)];
            else if (l[r] == LINK_BOUND) stv<AT>(&g[r], 0, a.boundval);
            else g[r] = atlas[(slot0 + k) * BRICK + layer_voxel(f, u, w, (f & 1) ? 9 : 0)];
        }
#pragma unroll
        for (int k = 0; k < CB; k++)
            if (k < nb) b[k * BRICK + at] = c[k];
#pragma unroll
        for (int r = 0; r < LAYERS; r++) {
            const int q = wave * LAYERS + r, k = q / 6, f = q - k * 6;
            b[k * BRICK + layer_voxel(f, u, w, (f & 1) ? 9 : 0)] = g[r];
        }
    } else {
        const uint4* src = reinterpret_cast<const uint4*>(atlas + slot0 * BRICK);
        for (int i = t; i < pieces; i += 512) reinterpret_cast<uint4*>(b)[i] = src[i];
        // the first of several iterations also looks the neighbours up
        if (TO_CELLS && t < nb * 8 && (t & 7) < 6) a.links[slot0 * 8 + t] = link_of(a, slot0 + (t >> 3), t & 7);
    }
    __syncthreads();
    float v[CB];
#pragma unroll
    for (int k = 0; k < CB; k++)
        if (k < nb) v[k] = apply_op<AT>(a, b + k * BRICK, at, slot0 + k, lx, ly, lz);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < CB; k++)
        if (k < nb) {
            stv<AT>(b, k * BRICK + at, v[k]);
            if (TO_CELLS) stv<AT>(cells, (slot0 + k) * CELLS + t, v[k]);
            else if (FROM_CELLS) stv<AT>(atlas, (slot0 + k) * BRICK + at, v[k]);
        }
    if (FROM_CELLS && !TO_CELLS && !a.faces_out) return;
    __syncthreads();
    if (!FROM_CELLS && !TO_CELLS) {
        uint4* dst = reinterpret_cast<uint4*>(atlas + slot0 * BRICK);
        for (int i = t; i < pieces; i += 512) dst[i] = reinterpret_cast<const uint4*>(b)[i];
    }
    if (!a.faces_out) return;
    AT* out = static_cast<AT*>(a.faces_out) + slot0 * FACE_VALS;
#pragma unroll
    for (int r = 0; r < LAYERS; r++) {
        const int q = wave * LAYERS + r, k = q / 6, f = q - k * 6;
        if (q < nb * 6) out[q * 64 + lane] = b[k * BRICK + layer_voxel(f, u, w, (f & 1) ? 8 : 1)];
    }
}

// Atlas voxels [lo, hi] (inclusive) per axis, in atlas coordinates.
template <typename AT>
__global__ __launch_bounds__(256) void k_compute_fill(ComputeArgs a) {
    const u64 nx = u64(a.hi[0] - a.lo[0] + 1), ny = u64(a.hi[1] - a.lo[1] + 1), nz = u64(a.hi[2] - a.lo[2] + 1);
    const u64 n = nx * ny * nz;
    for (u64 i = u64(blockIdx.x) * 256 + threadIdx.x; i < n; i += u64(gridDim.x) * 256) {
        const int x = a.lo[0] + int(i % nx), y = a.lo[1] + int((i / nx) % ny), z = a.lo[2] + int(i / (nx * ny));
        float v = a.p1;
        if (a.p3 < 0) {
            v = sinf(float(double(uint32_t(x) * 12u) / (3.141592 * 30.0)));
            v += sinf(float(double(uint32_t(y) * 12u) / (3.141592 * 30.0)));
            v += sinf(float(double(uint32_t(z) * 12u) / (3.141592 * 30.0)));
        }
        stv<AT>(a.atlas, atlas_offset(a.t, x, y, z), v);
    }
}

template <typename AT>
static void launch_packed(const ComputeArgs& a, hipStream_t s) {
    const dim3 grid(unsigned((a.slots + CB - 1) / CB)), wg(512);
    if (a.from_cells && a.to_cells) hipLaunchKernelGGL((k_compute_packed<AT, true, true>), grid, wg, 0, s, a);
    else if (a.from_cells) hipLaunchKernelGGL((k_compute_packed<AT, true, false>), grid, wg, 0, s, a);
    else if (a.to_cells) hipLaunchKernelGGL((k_compute_packed<AT, false, true>), grid, wg, 0, s, a);
    else hipLaunchKernelGGL((k_compute_packed<AT, false, false>), grid, wg, 0, s, a);
}

hipError_t launch_compute(const ComputeArgs& a, hipStream_t s) {
    const bool half = a.atlas_type == T_HALF;
    if (a.op == OP_FILL) {
        for (int k = 0; k < 3; k++)
            if (a.hi[k] < a.lo[k]) return hipSuccess;
        const u64 n = u64(a.hi[0] - a.lo[0] + 1) * u64(a.hi[1] - a.lo[1] + 1) * u64(a.hi[2] - a.lo[2] + 1);
        const unsigned g = unsigned(std::min<u64>((n + 255) / 256, 65536));
        if (half) hipLaunchKernelGGL(k_compute_fill<__half>, dim3(g), dim3(256), 0, s, a);
        else hipLaunchKernelGGL(k_compute_fill<float>, dim3(g), dim3(256), 0, s, a);
        return hipGetLastError();
    }
    if (a.slots <= 0) return hipSuccess;
    if (a.t.brickwid != 8 || a.t.brick_res != 10) return hipErrorInvalidValue;
    if (half) launch_packed<__half>(a, s);
    else launch_packed<float>(a, s);
    return hipGetLastError();
}

}  // namespace gvdb
