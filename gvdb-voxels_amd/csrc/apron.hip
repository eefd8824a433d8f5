// apron.hip -- UpdateApron as neighbour-face copies.
//
// The reference (gvdbUpdateApronF, kernels/cuda_gvdb_operators.cuh:72-131)
// maps every apron voxel of a brick back to index space and walks the tree
// from the top node to find the brick that holds it, reading that brick's
// interior voxel or writing the boundary value when no brick covers it.  All
// apron voxels in one of the 26 directions around a brick fall inside the same
// neighbour brick, so here each brick does the 26 walks once (k_neighbors),
// and the copy kernel moves the 488 apron voxels of a brick from the
// neighbours' interior faces, edges and corners.
#include "kernels.h"
#include "tree_device.h"
#include <hip/hip_fp16.h>
#include <mutex>
#include <cstring>
#include <algorithm>

namespace gvdb {

__device__ inline void dir_of(int d, int& dx, int& dy, int& dz) {
    // d in [0,27) without the centre 13: dx fastest
    dx = d % 3 - 1;
    dy = (d / 3) % 3 - 1;
    dz = d / 9 - 1;
}

// 32 lanes per brick (27 directions used), two bricks per wave: the mask of
// present neighbours comes from one ballot, written by the brick's lane 0.
__device__ inline void k_neighbors_body(const NbrArgs& a, uint32_t bid, uint32_t) {
    const Tree& t = a.t;
    int* nbr = a.nbr;
    const u64 g = u64(bid) * 256 + threadIdx.x;
    const int b = int(g >> 5), d = int(g & 31);
    const bool valid = b < a.n && d < 27;
    int v = -1;
    if (a.bcnt) {
        if (b < a.n && d < a.spb) a.bcnt[u64(b) * u64(a.spb) + u64(d)] = 0;
        if (g < 96) a.lenparts[g] = 0;
        if (g == 0) *a.orphans = 0;
    }
    if (valid) {
        const Node* n = t.nodes[0] + b;
        int dx, dy, dz;
        dir_of(d, dx, dy, dz);
        if (a.bt.tab) {
            // the brick table at the brick's coordinates plus the direction
            // (d = 13: the brick itself, -1 when the table does not hold it)
            const int sh = __builtin_ctz(unsigned(t.brickwid));
            v = tab_leaf(a.bt, (n->mPos[0] >> sh) + dx, (n->mPos[1] >> sh) + dy, (n->mPos[2] >> sh) + dz);
            if (d == 13 && v != b) v = -1;
        } else if (d == 13) {
            // the brick itself, or -1 when the walk from the top node does not reach it
            v = pos_leaf(t, n->mPos[0], n->mPos[1], n->mPos[2]) == b ? b : -1;
        } else {
            int w = t.brickwid;
            // a voxel centre inside the neighbour box: local coordinate -1, 0 or w
            float px = float(n->mPos[0]) + float(dx < 0 ? -1 : (dx > 0 ? w : 0)) + 0.5f;
            float py = float(n->mPos[1]) + float(dy < 0 ? -1 : (dy > 0 ? w : 0)) + 0.5f;
            float pz = float(n->mPos[2]) + float(dz < 0 ? -1 : (dz > 0 ? w : 0)) + 0.5f;
            v = point_leaf(t, px, py, pz);
        }
        const u64 e = u64(b) * 27 + u64(d);
        nbr[e] = v;
        if (a.base) {
            // atlas offset of the neighbour's padded brick (d = 13: the brick's own)
            const int m = d == 13 ? b : v;
            const Node* mn = t.nodes[0] + (m >= 0 ? m : 0);
            const bool live = m >= 0 && (d != 13 || mn->mFlags) && mn->mValue[0] >= 0;
            a.base[e] = live ? (long long)(slot_of(t, mn->mValue) * u64(t.brick_vox)) : -1ll;
        }
    }
    const u64 bal = __ballot(valid && v >= 0);
    if (a.mask && valid && d == 0) {
        const uint32_t m = uint32_t(bal >> (threadIdx.x & 32)) & 0x7FFFFFFu;
        a.mask[b] = m;
        if (a.bt.tab) {
            // beside the brick's index in the table (its own entry: v is b here
            // when the table holds the brick), for the insert's one-read lookup
            const Node* n = t.nodes[0] + b;
            const int sh = __builtin_ctz(unsigned(t.brickwid));
            const unsigned x = unsigned((n->mPos[0] >> sh) - a.bt.lo[0]), y = unsigned((n->mPos[1] >> sh) - a.bt.lo[1]),
                           z = unsigned((n->mPos[2] >> sh) - a.bt.lo[2]);
            if (x < unsigned(a.bt.dim[0]) && y < unsigned(a.bt.dim[1]) && z < unsigned(a.bt.dim[2]))
                reinterpret_cast<uint32_t*>(a.bt.tab)[2 * tab_index(a.bt, x, y, z) + 1] = m;
        }
    }
}

GVDB_MULTI(k_neighbors, NbrArgs, 256)

hipError_t launch_neighbors_multi(const NbrArgs* a, int G, Arena* ar, hipStream_t s) {
    std::vector<uint32_t> nb(G);
    for (int g = 0; g < G; g++) nb[g] = a[g].n > 0 ? uint32_t((u64(a[g].n) * 32 + 255) / 256) : 0;
    MultiLaunch L;
    hipError_t e = multi_setup(ar, a, nb.data(), G, s, L);
    if (e != hipSuccess || L.blocks == 0) return e;
    L.map.xcd = knob(KNOB_XCD_ORDER);
    hipLaunchKernelGGL(k_neighbors, dim3(L.blocks), dim3(256), 0, s, a[0], L.map);
    return hipGetLastError();
}

template <typename AT>
__device__ inline float ld(const AT* a, u64 o);
template <>
__device__ inline float ld<float>(const float* a, u64 o) { return a[o]; }
template <>
__device__ inline float ld<__half>(const __half* a, u64 o) { return __half2float(a[o]); }
template <typename AT>
__device__ inline void st(AT* a, u64 o, float v);
template <>
__device__ inline void st<float>(float* a, u64 o, float v) { a[o] = v; }
template <>
__device__ inline void st<__half>(__half* a, u64 o, float v) { a[o] = __float2half(v); }
// uchar4 channels move as 32-bit words; the value travels through the body as
// a float holding those bits (moved, never computed with), and the boundary
// value arrives already packed (apron_bound)
template <>
__device__ inline float ld<uint32_t>(const uint32_t* a, u64 o) { return __uint_as_float(a[o]); }
template <>
__device__ inline void st<uint32_t>(uint32_t* a, u64 o, float v) { a[o] = __float_as_uint(v); }

// UpdateApron<uchar4>'s boundary value, make_uchar4(boundval, ...) (kernels/
// cuda_gvdb_operators.cuh:143-146): each byte is boundval converted to an
// unsigned char, truncated and clamped to [0, 255] (NaN: 0), packed into the
// bits of a float
static float apron_bound_u8x4(float b) {
    const float c = b > 0.f ? (b < 255.f ? b : 255.f) : 0.f;   // NaN fails b > 0
    const uint32_t u = uint32_t(c) * 0x01010101u;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// Apron voxel a of a padded brick of side br = w + 2: the two z faces
// (br^2 each), then per interior z layer its ring (br^2 - w^2: the y = 0 and
// y = br - 1 rows, then x = 0 / x = br - 1 of each row between).
__host__ __device__ constexpr void apron_decode(int a, int w_, int& x, int& y, int& z) {
    const unsigned w = unsigned(w_), br = w + 2, face = br * br, ring = br * br - w * w, u = unsigned(a);
    if (u < 2 * face) {
        z = u < face ? 0 : int(br) - 1;
        const unsigned r = u < face ? u : u - face;
        y = int(r / br);
        x = int(r - unsigned(y) * br);
    } else {
        const unsigned s = u - 2 * face;
        z = int(s / ring) + 1;
        const int r = int(s - unsigned(z - 1) * ring);
        if (r < int(br)) { x = r; y = 0; }
        else if (r < 2 * int(br)) { x = r - int(br); y = int(br) - 1; }
        else { const int q = r - 2 * int(br); y = (q >> 1) + 1; x = (q & 1) ? int(br) - 1 : 0; }
    }
}

// Where apron voxel a of a brick w wide lies (own: its index in the padded
// brick) and where its value is: direction d of the neighbour, and the index
// in that neighbour's padded brick (faces = false) or among its six face
// layers (true: the face towards this brick, x faces first).
__host__ __device__ constexpr void apron_source(int a, int w, bool faces, int& own, int& d, int& src) {
    int x = 0, y = 0, z = 0;
    apron_decode(a, w, x, y, z);
    const int br = w + 2;
    const int dx = x == 0 ? -1 : (x == br - 1 ? 1 : 0), dy = y == 0 ? -1 : (y == br - 1 ? 1 : 0),
              dz = z == 0 ? -1 : (z == br - 1 ? 1 : 0);
    own = (z * br + y) * br + x;
    d = (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1);
    const int sx = (x - 1) - dx * w, sy = (y - 1) - dy * w, sz = (z - 1) - dz * w;   // interior voxel of the neighbour
    if (faces)
        src = dx ? (dx < 0 ? 1 : 0) * 64 + sz * 8 + sy
                 : (dy ? (dy < 0 ? 3 : 2) * 64 + sz * 8 + sx : (dz < 0 ? 5 : 4) * 64 + sy * 8 + sx);
    else
        src = ((sz + 1) * br + sy + 1) * br + sx + 1;
}

// The same for 8^3 bricks as a table: own | d << 10 | src << 15.
static const int APRON8 = 488;
struct ApronTable {
    uint32_t e[2][APRON8];
};
static constexpr ApronTable make_apron_table() {
    ApronTable t{};
    for (int f = 0; f < 2; f++)
        for (int a = 0; a < APRON8; a++) {
            int own = 0, d = 0, src = 0;
            apron_source(a, 8, f != 0, own, d, src);
            t.e[f][a] = uint32_t(own) | uint32_t(d) << 10 | uint32_t(src) << 15;
        }
    return t;
}
static __constant__ ApronTable apron_table = make_apron_table();

// A run of up to RUN consecutive bricks b0.. of one grid.  The sources of the
// run's 26 directions a brick (offset of the neighbour's faces or padded
// brick, -1: none; 13: the brick's own offset) come in one load and one
// barrier.  8^3 bricks: thread a owns apron voxel a of every brick of the run,
// its place and its source looked up once, so a voxel costs an LDS read, a
// load and a store, and the loads of eight bricks are in flight together
// (decoding every voxel, and for faces a second lookup behind it, took most of
// the time: 73 k bricks, FP32, 0.156 -> 0.126 ms).  What is left is the writes:
// every row of a brick has apron voxels at both ends, so all of its cache
// lines are written for half of their bytes.  Ends with a barrier, so the next
// run may reuse the LDS.
template <typename AT, int RUN>
__device__ inline void apron_run(const ApronArgs& ap, uint32_t b0, long long* base) {
    const int nb = min(RUN, int(uint32_t(ap.n) - b0));
    AT* atlas = reinterpret_cast<AT*>(ap.atlas);
    const AT* from = ap.faces ? reinterpret_cast<const AT*>(ap.faces) : atlas;
    for (int i = threadIdx.x; i < nb * 27; i += 512) {
        const u64 e = u64(b0) * 27 + u64(i);
        long long o = ap.base[e];
        if (ap.faces && o >= 0 && i % 27 != 13)
            o = (ap.by_slot ? (long long)(u64(o) / u64(ap.t.brick_vox)) : (long long)ap.nbr[e]) * FACE_VALS;
        base[i] = o;
    }
    __syncthreads();
    const int w = ap.t.brickwid;
    if (w == 8) {
        if (threadIdx.x < APRON8) {
            const uint32_t t = apron_table.e[ap.faces ? 1 : 0][threadIdx.x];
            const int own = int(t & 1023u), d = int((t >> 10) & 31u), src = int(t >> 15);
            for (int k0 = 0; k0 < nb; k0 += 8) {
                float v[8];
                long long at[8];
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    at[k] = k0 + k < nb ? base[(k0 + k) * 27 + 13] : -1ll;
                    const long long o = at[k] >= 0 ? base[(k0 + k) * 27 + d] : -1ll;
                    v[k] = ap.boundval;
                    if (o >= 0) v[k] = ld<AT>(from, u64(o) + u64(src));
                }
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (at[k] >= 0) st<AT>(atlas, u64(at[k]) + u64(own), v[k]);
            }
        }
    } else {
        const int br = ap.t.brick_res;
        const int per = 2 * br * br + w * (br * br - w * w);
        for (int v = threadIdx.x; v < nb * per; v += 512) {
            const int k = v / per;
            if (base[k * 27 + 13] < 0) continue;
            int own = 0, d = 0, src = 0;
            apron_source(v - k * per, w, ap.faces != nullptr, own, d, src);
            const long long o = base[k * 27 + d];
            st<AT>(atlas, u64(base[k * 27 + 13]) + u64(own), o >= 0 ? ld<AT>(from, u64(o) + u64(src)) : ap.boundval);
        }
    }
    __syncthreads();
}

// Several grids: RUN bricks of one grid per workgroup (the apron-run knob:
// 1, 2, 4 or 8), one after the other, so the grid lookup and the record
// loads before the first brick are paid once per run (a brick alone is one
// voxel per thread).
template <typename AT, int RUN>
__global__ __launch_bounds__(512) void k_apron_runs(ApronArgs, MultiMap m) {
    __shared__ long long base[RUN * 27];
    const uint32_t bi = m.xcd ? xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x;
    const int g = multi_grid(m, bi);
    const uint32_t* first = multi_first(m);
    const ApronArgs& a = multi_rec<ApronArgs>(m, g);
    const uint32_t b0 = (bi - first[g]) * uint32_t(RUN);
    if (b0 < uint32_t(a.n)) apron_run<AT, RUN>(a, b0, base);
}

// Several grids, persistent: a fixed number of workgroups (about as many as
// the device holds at once) take runs of QRUN bricks from one device counter
// until the queue is empty.  A run's grid is looked up only when it falls
// outside the workgroup's previous grid; every workgroup leaves when the
// counter passes the last run.
static const int QRUN = 8;
static const uint32_t APRON_QUEUE_WORKGROUPS = 256 * 4;   // 4 per CU of 256
template <typename AT>
__global__ __launch_bounds__(512) void k_apron_queue(ApronArgs, MultiMap m, uint32_t* counter, uint32_t nruns) {
    __shared__ uint32_t s_run;
    __shared__ long long base[QRUN * 27];
    const uint32_t* first = multi_first(m);
    int g = -1;
    uint32_t lo = 0, hi = 0;
    for (;;) {
        if (threadIdx.x == 0) s_run = atomicAdd(counter, 1u);
        __syncthreads();
        const uint32_t run = s_run;
        __syncthreads();                   // read before thread 0 takes the next run
        if (run >= nruns) break;
        if (g < 0 || run < lo || run >= hi) {
            g = multi_grid(m, run);
            lo = first[g];
            hi = first[g + 1];
        }
        const ApronArgs& a = multi_rec<ApronArgs>(m, g);
        const uint32_t b0 = (run - lo) * uint32_t(QRUN);
        if (b0 < uint32_t(a.n)) apron_run<AT, QRUN>(a, b0, base);
    }
}

template <typename AT>
static void launch_apron_runs(int run, dim3 grid, hipStream_t s, const ApronArgs& a0, const MultiMap& m) {
    switch (run) {
    case 1: hipLaunchKernelGGL((k_apron_runs<AT, 1>), grid, dim3(512), 0, s, a0, m); break;
    case 2: hipLaunchKernelGGL((k_apron_runs<AT, 2>), grid, dim3(512), 0, s, a0, m); break;
    case 8: hipLaunchKernelGGL((k_apron_runs<AT, 8>), grid, dim3(512), 0, s, a0, m); break;
    default: hipLaunchKernelGGL((k_apron_runs<AT, 4>), grid, dim3(512), 0, s, a0, m); break;
    }
}

// One grid: runs of RUN consecutive bricks per workgroup, the record by value.
template <typename AT, int RUN>
__global__ __launch_bounds__(512) void k_apron_flat(ApronArgs a0, MultiMap m) {
    __shared__ long long base[RUN * 27];
    const uint32_t bi = m.xcd ? xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x;
    const uint32_t b0 = bi * uint32_t(RUN);
    if (b0 < uint32_t(a0.n)) apron_run<AT, RUN>(a0, b0, base);
}

template <typename AT>
static void launch_apron_seq(int run, dim3 grid, hipStream_t s, const ApronArgs& a0, const MultiMap& m) {
    switch (run) {
    case 2: hipLaunchKernelGGL((k_apron_flat<AT, 2>), grid, dim3(512), 0, s, a0, m); break;
    case 4: hipLaunchKernelGGL((k_apron_flat<AT, 4>), grid, dim3(512), 0, s, a0, m); break;
    case 8: hipLaunchKernelGGL((k_apron_flat<AT, 8>), grid, dim3(512), 0, s, a0, m); break;
    case 16: hipLaunchKernelGGL((k_apron_flat<AT, 16>), grid, dim3(512), 0, s, a0, m); break;
    case 32: hipLaunchKernelGGL((k_apron_flat<AT, 32>), grid, dim3(512), 0, s, a0, m); break;
    default: hipLaunchKernelGGL((k_apron_flat<AT, 1>), grid, dim3(512), 0, s, a0, m); break;
    }
}

template <typename AT>
static void launch_apron_as(bool queue, bool runs, int run, uint32_t nwg, uint32_t* ctr, const MultiLaunch& L,
                            hipStream_t s, const ApronArgs& a0) {
    if (queue)
        hipLaunchKernelGGL(k_apron_queue<AT>, dim3(nwg), dim3(512), 0, s, a0, L.map, ctr, L.blocks);
    else if (runs) launch_apron_runs<AT>(run, dim3(L.blocks), s, a0, L.map);
    else launch_apron_seq<AT>(run, dim3(L.blocks), s, a0, L.map);
}

hipError_t launch_apron_multi(const ApronArgs* a, int G, Arena* ar, hipStream_t s) {
    // one launch per channel type: 0 float, 1 half, 2 uchar4
    for (int kind = 0; kind < 3; kind++) {
        std::vector<ApronArgs> sel;
        std::vector<uint32_t> nb;
        for (int g = 0; g < G; g++) {
            if (a[g].t.apron != 1) return hipErrorInvalidValue;
            const int k = a[g].atlas_type == T_HALF ? 1 : (a[g].atlas_type == T_UCHAR4 ? 2 : 0);
            if (k != kind || a[g].n <= 0) continue;
            sel.push_back(a[g]);
            if (kind == 2) {
                sel.back().boundval = apron_bound_u8x4(a[g].boundval);
                sel.back().faces = nullptr;
            }
        }
        if (sel.empty()) continue;
        // one grid: runs of `run` consecutive bricks per workgroup (1: a
        // workgroup per brick); several: runs of one grid's bricks, or the
        // persistent queue over runs of QRUN bricks
        const bool runs = sel.size() > 1;
        const bool queue = runs && knob(KNOB_APRON_QUEUE) == 1;
        const int run = queue ? QRUN : (runs ? knob(KNOB_APRON_RUN) : knob(KNOB_APRON_RUN_ONE));
        for (const ApronArgs& x : sel) nb.push_back(uint32_t((x.n + run - 1) / run));
        MultiLaunch L;
        hipError_t e = multi_setup(ar, sel.data(), nb.data(), int(sel.size()), s, L);
        if (e != hipSuccess) return e;
        if (L.blocks == 0) continue;
        // without the compact layers a brick reads rows of its neighbours' lines:
        // each XCD takes a contiguous part, so those stay in its L2 (17 k bricks
        // 0.0365 -> 0.0273 ms; with them the order does not matter)
        bool rows = true;
        for (const ApronArgs& x : sel) rows = rows && !x.faces;
        L.map.xcd = rows ? 1 : knob(KNOB_XCD_ORDER);
        uint32_t* ctr = nullptr;
        const uint32_t nwg = std::min<uint32_t>(L.blocks, APRON_QUEUE_WORKGROUPS);
        if (queue) {
            // the counter starts at zero: a copy recorded on the stream (also
            // inside a graph), from the argument staging
            const uint32_t zero = 0;
            ctr = ar ? static_cast<uint32_t*>(ar->push(&zero, sizeof(zero), s, e)) : nullptr;
            if (!ctr) return e != hipSuccess ? e : hipErrorInvalidValue;
        }
        if (kind == 1) launch_apron_as<__half>(queue, runs, run, nwg, ctr, L, s, sel[0]);
        else if (kind == 2) launch_apron_as<uint32_t>(queue, runs, run, nwg, ctr, L, s, sel[0]);
        else launch_apron_as<float>(queue, runs, run, nwg, ctr, L, s, sel[0]);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// ------------------------------------------- UpdateApron without allocation
// The neighbour table of gvdb_update_apron_noalloc.  Every device that loads
// this code object holds its own copy until the process ends.  In host code
// the name stands for no device address: noalloc_scratch() looks up the
// current device's copy with hipGetSymbolAddress, and only that address is
// handed to kernels.
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

static const int NOALLOC_DEVICES = 64;

hipError_t noalloc_scratch(int device, void** ptr) {
    static std::mutex mu;
    static void* addr[NOALLOC_DEVICES] = {};
    *ptr = nullptr;
    if (device < 0 || device >= NOALLOC_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[device]) {
        int cur = 0;
        hipError_t e = hipGetDevice(&cur);
        if (e != hipSuccess) return e;
        if (cur != device && (e = hipSetDevice(device)) != hipSuccess) return e;
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        addr[device] = p;
    }
    *ptr = addr[device];
    return hipSuccess;
}

hipError_t launch_apron_noalloc(const Tree& t, void* sp, const void* faces, void* atlas, int atlas_type,
                                float boundval, int bricks, hipStream_t s) {
    if (bricks <= 0) return hipSuccess;
    if (!sp || bricks > NOALLOC_MAX_BRICKS || t.apron != 1) return hipErrorInvalidValue;
    // offsets first (8-byte entries), then the leaf indices
    long long* base = static_cast<long long*>(sp);
    int* nbr = reinterpret_cast<int*>(static_cast<char*>(sp) + size_t(bricks) * 27 * 8);
    const MultiMap one{1, nullptr, nullptr, knob(KNOB_XCD_ORDER), {}, {}};
    // every entry of both tables is written by the neighbour pass before the
    // copy reads it, so nothing from an earlier call is read
    const NbrArgs na{t, nbr, bricks, nullptr, base};
    hipLaunchKernelGGL(k_neighbors, dim3(uint32_t((u64(bricks) * 32 + 255) / 256)), dim3(256), 0, s, na, one);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid(uint32_t((bricks + 7) / 8));
    MultiMap order = one;   // as launch_apron_multi orders the workgroups
    if (!faces || atlas_type == T_UCHAR4) order.xcd = 1;
    if (atlas_type == T_UCHAR4) {
        const ApronArgs aa{t, base, nbr, nullptr, atlas, atlas_type, apron_bound_u8x4(boundval), bricks};
        hipLaunchKernelGGL((k_apron_flat<uint32_t, 8>), grid, dim3(512), 0, s, aa, order);
        return hipGetLastError();
    }
    const ApronArgs aa{t, base, nbr, faces, atlas, atlas_type, boundval, bricks};
    if (atlas_type == T_HALF) hipLaunchKernelGGL((k_apron_flat<__half, 8>), grid, dim3(512), 0, s, aa, order);
    else hipLaunchKernelGGL((k_apron_flat<float, 8>), grid, dim3(512), 0, s, aa, order);
    return hipGetLastError();
}

}  // namespace gvdb
