// Grid SDF construction on gfx950: the signed distance of a triangle mesh at every node of a cubic
// Lagrange grid (Discregrid::MeshDistance::signedDistanceCached evaluated by
// CubicLagrangeDiscreteGrid::addFunction, environment_body.cpp:66-73).
//
// Distance: the closest point of every triangle (Voronoi-region test of the triangle's vertices,
// edges and face; Ericson, "Real-Time Collision Detection", 5.1.5), the smallest squared distance
// winning (the first triangle on ties). Sign: negative where (x - closest point) points against the
// angle-weighted pseudonormal of the closest feature (Baerentzen & Aanaes 2005): the vertex normal
// sum of incident face normals weighted by the incident angles, the edge normal sum of the normals
// of the faces sharing the edge, or the face normal. Zero-area triangles are left out.
//
// A wave per grid node walks a tree of bounds over the triangles in Morton order (k_grid_nodes); up to 512
// triangles are scanned instead (k_grid_scan). What bounds
// it: the FP32 tests of a few hundred tree nodes and triangles a grid node and the round trips to L2 between
// the batches. On the 20,480-triangle ball and 24^3 cells (104,625 nodes) 963 us, where the scan of
// 128-triangle tiles through LDS that it replaces took 12.4 ms.
#include <algorithm>
#include <cmath>
#include <vector>

#include "abi_util.h"
#include "grid_sdf.h"
#include "scan_sort.h"
#include "sdf.h"

namespace sbs {

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kRun = 16;  // grid nodes a wave takes (6,500 waves for 24^3 cells: six a SIMD)
// Each of at most 16 levels leaves at most 48 children of one batch waiting while the walk goes deeper.
constexpr uint32_t kStack = 1024, kList = 256;
constexpr uint32_t kMaxTriangles = 1u << 30;
// Meshes that are scanned instead, and grids whose nodes take eight lanes each in the scan (k_grid_scan).
constexpr uint32_t kScanTriangles = 512;
constexpr uint64_t kSplitNodes = 131072;

struct grid_params {
    uint32_t res[3];
    double dmin[3], cell[3];
};

// The nearest triangle so far: squared distance and index in Morton order. The nearest is the smallest
// (squared distance, original index) pair, so the visiting order does not change the result: it equals
// the scan of every triangle in original order keeping the first nearest.
struct nearest {
    double d2 = DBL_MAX;
    uint32_t t = 0xffffffffu, o = 0xffffffffu;
};

// A grid node for the walk's tests: its position relative to the mesh's center in FP32, and the distance
// `limit` beyond which nothing can be nearer than (or as near as) the best so far. The tests bound
// distances from below in FP32; limit is the best distance widened by 1e-5 of itself and by 4e-6 of the
// coordinates, which is several times what their roundings add up to, and by 1e-18: a limit of which the square
// is a normal number, beside which what is lost where squares and products are denormal does not count (a ball
// of 1e-18 had wrong values without it). Beyond 1e19 squares are infinite, and nothing is left out.
struct seeker {
    float x, y, z, margin, limit;
    __device__ __forceinline__ void set(mesh_dev const& mesh, const double p[3])
    {
        x = float(p[0] - mesh.center[0]);
        y = float(p[1] - mesh.center[1]);
        z = float(p[2] - mesh.center[2]);
        margin = fmaf(4e-6f, mesh.reach + fabsf(x) + fabsf(y) + fabsf(z), 1e-18f);
        limit = INFINITY;
    }
    __device__ __forceinline__ void bound(double d2) { limit = float(sqrt(d2)) * (1.0f + 1e-5f) + margin; }
    // squared distance to the node's box
    __device__ __forceinline__ float box2(float4 lo, float4 hi) const
    {
        float const ex = fmaxf(fmaxf(lo.x - x, x - hi.x), 0.0f), ey = fmaxf(fmaxf(lo.y - y, y - hi.y), 0.0f),
                    ez = fmaxf(fmaxf(lo.z - z, z - hi.z), 0.0f);
        return fmaf(ex, ex, fmaf(ey, ey, ez * ez));
    }
    // Whether the node's triangles can be that near: the distance to their box, then to the slab that
    // holds them along their mean normal. The box of a patch that faces the seeker obliquely reaches much
    // nearer than the patch (ball of 20,480 triangles: 45 leaves a node with the boxes alone, 30 with the
    // slabs).
    __device__ __forceinline__ bool may_hold(const float4* node) const
    {
        float4 const lo = node[0], hi = node[1], sl = node[2];
        float const h = fmaf(x, lo.w, fmaf(y, hi.w, z * sl.x));
        float const gap = fmaxf(sl.y - h, h - sl.z);
        return !(box2(lo, hi) > limit * limit) && !(gap > limit);
    }
    // Whether a triangle can be: no point of it is nearer than its nearest corner along the direction to
    // its centroid (about ten triangles a node are left for the FP64 closest point). A square below 1e-37 counts
    // as that: the root of a denormal is none, and nearer than 1e-18 the result is below the margin.
    __device__ __forceinline__ bool may_be(float4 a, float4 b, float4 c) const
    {
        float const ax = a.x - x, ay = a.y - y, az = a.z - z, bx = b.x - x, by = b.y - y, bz = b.z - z,
                    cx = c.x - x, cy = c.y - y, cz = c.z - z;
        float const wx = ax + bx + cx, wy = ay + by + cy, wz = az + bz + cz;
        float const r = __builtin_amdgcn_rsqf(fmaxf(fmaf(wx, wx, fmaf(wy, wy, wz * wz)), 1e-37f));
        float const m = fminf(fminf(fmaf(ax, wx, fmaf(ay, wy, az * wz)), fmaf(bx, wx, fmaf(by, wy, bz * wz))),
                              fmaf(cx, wx, fmaf(cy, wy, cz * wz)));
        return !(m * r > limit);
    }
};

// Triangle t's exact closest point against the best so far. MORTON: t counts in Morton order, not in their own.
template <bool MORTON>
__device__ __forceinline__ void visit(mesh_dev const& mesh, uint32_t t, const double p[3], nearest& best)
{
#pragma clang fp contract(off)
    double c[9], q[3];
    for (int k = 0; k < 9; ++k) c[k] = mesh.corners[9 * std::size_t(t) + k];
    int feat;
    tri_closest_point(p, c, q, &feat);
    double const e0 = p[0] - q[0], e1 = p[1] - q[1], e2 = p[2] - q[2];
    double const d2 = e0 * e0 + e1 * e1 + e2 * e2;
    uint32_t const o = MORTON ? mesh.orig[t] : t;
    if (d2 < best.d2 || (d2 == best.d2 && o < best.o)) best = nearest{d2, t, o};
}

// Every lane gets the nearest of its `lanes` neighbours.
__device__ __forceinline__ void wave_nearest(nearest& best, int lanes = 64)
{
    for (int o = lanes / 2; o > 0; o >>= 1) {
        nearest const b{__shfl_xor(best.d2, o, 64), uint32_t(__shfl_xor(best.t, o, 64)), uint32_t(__shfl_xor(best.o, o, 64))};
        if (b.d2 < best.d2 || (b.d2 == best.d2 && b.o < best.o)) best = b;
    }
}

// The signed distance from the nearest triangle t: its closest point again, the pseudo-normal of the feature
// that holds it (an edge's is the sum of its triangles' unit normals in original order).
template <bool MORTON>
__device__ __forceinline__ double signed_distance(mesh_dev const& mesh, mesh_normals const& nm, const double p[3],
                                                  uint32_t t)
{
#pragma clang fp contract(off)
    if (t == 0xffffffffu) return DBL_MAX;
    double c[9], q[3], nrm[3] = {0.0, 0.0, 0.0};
    for (int k = 0; k < 9; ++k) c[k] = mesh.corners[9 * std::size_t(t) + k];
    uint32_t const o = MORTON ? mesh.orig[t] : t;
    int feat;
    tri_closest_point(p, c, q, &feat);
    const uint32_t* tv = mesh.tri + 3 * std::size_t(o);
    if (feat < 3) {
        for (int d = 0; d < 3; ++d) nrm[d] = nm.vnormal[3 * std::size_t(tv[feat]) + d];
    } else if (feat < 6) {
        uint32_t const v = tv[feat - 3], w = tv[feat == 5 ? 0 : feat - 2];
        for (uint32_t i = nm.face_off[v], e = nm.face_off[v + 1]; i < e; ++i) {
            uint32_t const f = nm.faces[i];
            const uint32_t* fv = mesh.tri + 3 * std::size_t(f);
            if (fv[0] != w && fv[1] != w && fv[2] != w) continue;
            for (int d = 0; d < 3; ++d) nrm[d] = nrm[d] + nm.fnormal[3 * std::size_t(f) + d];
        }
    } else {
        for (int d = 0; d < 3; ++d) nrm[d] = nm.fnormal[3 * std::size_t(o) + d];
    }
    double const e0 = p[0] - q[0], e1 = p[1] - q[1], e2 = p[2] - q[2];
    double const s = e0 * nrm[0] + e1 * nrm[1] + e2 * nrm[2];
    double const d = sqrt(e0 * e0 + e1 * e1 + e2 * e2);
    return s < 0.0 ? -d : d;
}

// One wave walks the tree for one grid node, kRun consecutive nodes one after the other. The walk takes up
// to 16 tree nodes off a stack in LDS and tests their 64 children at once, one a lane, each with FP32
// bounds; children that may hold something go back on the stack, triangles that may be the nearest to a
// list whose exact FP64 closest points the lanes then share. (A lane per grid node walked 64 different
// paths: 4.3 ms on the 20,480-triangle ball and 24^3 cells, 0.96 ms so.) The first bound is exact distances
// to 64 triangles that are neighbours in Morton order: those of the last node's nearest one, for a run's
// first node those of the nearest box. out: the nearest triangle (in Morton order; ~0: none).
__global__ void __launch_bounds__(kBlock) k_grid_nodes(mesh_dev mesh, grid_params gp, uint64_t n,
                                                       uint32_t* __restrict__ out)
{
    constexpr uint32_t kWaves = kBlock / 64;
    __shared__ uint32_t stack_lds[kWaves][kStack], list_lds[kWaves][kList];
    uint32_t const wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint64_t const l0 = (uint64_t(blockIdx.x) * kWaves + wave) * kRun;
    if (l0 >= n) return;
    uint32_t const cnt = uint32_t(n - l0 < kRun ? n - l0 : kRun);
    uint32_t* const stack = stack_lds[wave];
    uint32_t* const list = list_lds[wave];
    uint64_t const below = (uint64_t(1) << lane) - 1;
    grid_dims const dims(gp.res);
    static_assert(kScanTriangles >= 64, "a tree has three levels at least");
    uint32_t const top = mesh.levels - 1;
    constexpr uint32_t start = 2;
    uint32_t mine = 0xffffffffu;  // lane r: the nearest of node l0 + r
    uint32_t block = 0;  // of 64 triangles
    for (uint32_t r = 0; r < cnt; ++r) {
        double p[3];
        grid_node_position(dims, gp.dmin, gp.cell, l0 + r, p);
        seeker at;
        at.set(mesh, p);
        if (r == 0) {  // a node two levels up is one block of 64 triangles
            float md = INFINITY;
            for (uint32_t i = lane; i < mesh.level_count[start]; i += 64) {
                const float4* node = mesh.node + 3 * (std::size_t(mesh.level_off[start]) + i);
                float const d = at.box2(node[0], node[1]);
                if (d < md) md = d, block = i;
            }
            for (int o = 32; o > 0; o >>= 1) {
                float const d = __shfl_xor(md, o, 64);
                uint32_t const i = __shfl_xor(block, o, 64);
                if (d < md || (d == md && i < block)) md = d, block = i;
            }
        }
        nearest best;
        if (64 * block + lane < mesh.m) visit<true>(mesh, 64 * block + lane, p, best);
        wave_nearest(best);
        at.bound(best.d2);
        uint32_t sp = 0, candidates = 0;
        auto push = [&](uint32_t* to, uint32_t& count, bool want, uint32_t value) {
            uint64_t const mask = __ballot(want);
            if (want) to[count + __popcll(mask & below)] = value;
            count += __popcll(mask);
            __builtin_amdgcn_wave_barrier();
        };
        auto drain = [&] {
            for (uint32_t i = lane; i < candidates; i += 64) visit<true>(mesh, list[i], p, best);
            candidates = 0;
            __builtin_amdgcn_wave_barrier();
        };
        {
            const float4* node = mesh.node + 3 * (std::size_t(mesh.level_off[top]) + min(lane, mesh.level_count[top] - 1));
            bool const want = lane < mesh.level_count[top] && at.may_hold(node);
            push(stack, sp, want, __float_as_uint(node[2].w));
        }
        while (sp > 0) {
            uint32_t const take = min(sp, 16u), e = lane >> 2;
            sp -= take;
            uint32_t const info = e < take ? stack[sp + e] : 0u;
            __builtin_amdgcn_wave_barrier();
            bool const valid = e < take && (lane & 3u) <= ((info >> 29) & 3u), leaf = info >> 31;
            uint32_t const child = (info & 0x1fffffffu) * (leaf ? kTreeArity : 1u) + (lane & 3u);
            bool hold = false, candidate = false;
            uint32_t next = child;
            if (valid && leaf) {
                const float4* c = mesh.corners32 + 3 * std::size_t(child);
                candidate = child / 64 != block && at.may_be(c[0], c[1], c[2]);
            } else if (valid) {
                const float4* node = mesh.node + 3 * std::size_t(child);
                hold = at.may_hold(node);
                next = __float_as_uint(node[2].w);
            }
            push(stack, sp, hold, next);
            push(list, candidates, candidate, next);
            if (candidates > kList - 64) drain();
        }
        drain();
        wave_nearest(best);
        block = best.t < mesh.m ? best.t / 64 : 0;
        if (lane == r) mine = best.t;
    }
    if (lane < cnt) out[l0 + lane] = mine;
}

// A mesh of few triangles, in their own order: SPLIT lanes take a grid node, each scans every SPLIT-th triangle, with
// the walk's FP32 test before an exact closest point, and the nearest of theirs is the node's. With one lane the
// triangles' reads are the wave's, through the scalar cache. What bounds it: the chain of exact closest points a
// lane computes in grids of few nodes, the arithmetic of all lanes in large ones. A call in us, scanned and with
// the tree (whose making alone is 25 launches, and whose walk keeps a wave busy a node): 12 triangles and 24^3
// cells 205 and 410, 40^3 460 and 1,010, 64^3 1,330 and 3,330; a ball of 320 triangles and 12^3 cells 195 and 380 to
// 520, 24^3 295 and 500, 40^3 670 and 1,280. A ball of 1,280: 24^3 515 and 565, 64^3 3,260 and 4,745; a double cone of
// 400: 24^3 420 and 595, 40^3 1,220 and 1,410; of 800: 655 and 750, but 1,980 and 1,630; a ball of 5,120: 1,310 and
// 840. So 512 triangles, below which the scan is never the slower one. Eight lanes a node or one: a ball of 320
// triangles, 12^3 cells 195 and 315, 24^3 (105,000 nodes) 295 and 335, 40^3 (472,000) 800 and 670; a double cone of 400,
// 420 and 590, then 1,160 and 1,220; 64^3 (1.9M) 4,350 and 3,230.
template <uint32_t SPLIT>
__global__ void __launch_bounds__(kBlock) k_grid_scan(mesh_dev mesh, mesh_normals nm, grid_params gp, uint64_t n,
                                                      double* __restrict__ out)
{
    uint64_t const l = (uint64_t(blockIdx.x) * kBlock + threadIdx.x) / SPLIT;
    if (l >= n) return;
    double p[3];
    grid_node_position(grid_dims(gp.res), gp.dmin, gp.cell, l, p);
    seeker at;
    at.set(mesh, p);
    nearest best;
    for (uint32_t t = SPLIT == 1 ? 0u : threadIdx.x % SPLIT; t < mesh.m; t += SPLIT) {
        const float4* c = mesh.corners32 + 3 * std::size_t(t);
        if (!at.may_be(c[0], c[1], c[2])) continue;
        double const before = best.d2;
        visit<false>(mesh, t, p, best);
        if (best.d2 < before) at.bound(best.d2);
    }
    wave_nearest(best, int(SPLIT));
    if (threadIdx.x % SPLIT == 0) out[l] = signed_distance<false>(mesh, nm, p, best.t);
}

__global__ void __launch_bounds__(kBlock) k_grid_signs(mesh_dev mesh, mesh_normals nm, grid_params gp, uint64_t n,
                                                       const uint32_t* __restrict__ nearest_of, double* __restrict__ out)
{
    uint64_t const l = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (l >= n) return;
    double p[3];
    grid_node_position(grid_dims(gp.res), gp.dmin, gp.cell, l, p);
    out[l] = signed_distance<true>(mesh, nm, p, nearest_of[l]);
}

// ---------------------------------------------------------------- the tree

// Morton codes of the triangles' centroids, 10 bits per axis over the mesh's box (lo, scale = 1024 / extent).
struct morton_box {
    double lo[3], scale[3];
};

__global__ void k_tree_keys(const double* __restrict__ pos, const uint32_t* __restrict__ tri, uint32_t m, morton_box box,
                            uint32_t* __restrict__ key, uint32_t* __restrict__ orig)
{
    uint32_t const t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= m) return;
    uint32_t code = 0;
    for (int d = 0; d < 3; ++d) {
        double const c = (pos[3 * std::size_t(tri[3 * t]) + d] + pos[3 * std::size_t(tri[3 * t + 1]) + d] +
                          pos[3 * std::size_t(tri[3 * t + 2]) + d]) / 3.0;
        uint32_t x = uint32_t(fmin(1023.0, fmax(0.0, (c - box.lo[d]) * box.scale[d])));
        x = (x | (x << 16)) & 0x30000ffu;
        x = (x | (x << 8)) & 0x300f00fu;
        x = (x | (x << 4)) & 0x30c30c3u;
        x = (x | (x << 2)) & 0x9249249u;
        code |= x << d;
    }
    key[t] = code;
    orig[t] = t;
}

// The triangles' corners in Morton order, and relative to the mesh's center in FP32 (the walk's margin covers
// the rounding).
__global__ void k_tree_corners(mesh_dev mesh, const double* __restrict__ pos, double* __restrict__ corners,
                               float4* __restrict__ corners32)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;  // of 3 m
    if (i >= 3 * mesh.m) return;
    uint32_t const v = mesh.tri[3 * std::size_t(mesh.orig[i / 3]) + i % 3];
    double const x = pos[3 * std::size_t(v)], y = pos[3 * std::size_t(v) + 1], z = pos[3 * std::size_t(v) + 2];
    corners[3 * std::size_t(i)] = x;
    corners[3 * std::size_t(i) + 1] = y;
    corners[3 * std::size_t(i) + 2] = z;
    corners32[i] = make_float4(float(x - mesh.center[0]), float(y - mesh.center[1]), float(z - mesh.center[2]), 0.0f);
}

__device__ __forceinline__ float wave_min(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
    return v;
}

// Workgroups of k_tree_level: a wave makes one node after another, so that a level of 2^28 nodes (2^30 triangles)
// still has fewer than 2^32 threads.
constexpr uint32_t kMaxLevelBlocks = 1u << 20;
constexpr uint32_t level_blocks(uint32_t nodes)
{
    uint32_t const blocks = (nodes + kBlock / 64 - 1) / (kBlock / 64);
    return blocks < kMaxLevelBlocks ? blocks : kMaxLevelBlocks;
}
static_assert(uint64_t(kMaxLevelBlocks) * kBlock < (uint64_t(1) << 32) &&
                  (uint64_t(kMaxTriangles) / kTreeArity + uint64_t(kMaxLevelBlocks) * (kBlock / 64)) < (uint64_t(1) << 32),
              "threads and node indices fit 32 bits");

// A wave makes a node of tree level `level`: the box of its children (triangles at level 0), and the slab that
// holds its corners along the mean normal of its triangles, for patches of up to 256 triangles (larger ones
// bend too far for one). sum: the nodes' summed unit normals.
__device__ __forceinline__ void tree_node(mesh_dev const& mesh, uint32_t level, uint32_t i, float4* __restrict__ node,
                                          float4* __restrict__ sum)
{
    uint32_t const lane = threadIdx.x & 63;
    uint32_t const n = level ? mesh.level_count[level - 1] : mesh.m, below = level ? mesh.level_off[level - 1] : 0u;
    uint32_t const j0 = i * kTreeArity, have = min(kTreeArity, n - j0), j = j0 + min(lane, have - 1);
    float4 l, h, u;
    if (level == 0) {
        float4 const a = mesh.corners32[3 * std::size_t(j)], b = mesh.corners32[3 * std::size_t(j) + 1],
                     c = mesh.corners32[3 * std::size_t(j) + 2];
        l = make_float4(fminf(a.x, fminf(b.x, c.x)), fminf(a.y, fminf(b.y, c.y)), fminf(a.z, fminf(b.z, c.z)), 0.0f);
        h = make_float4(fmaxf(a.x, fmaxf(b.x, c.x)), fmaxf(a.y, fmaxf(b.y, c.y)), fmaxf(a.z, fmaxf(b.z, c.z)), 0.0f);
        float const ex = b.x - a.x, ey = b.y - a.y, ez = b.z - a.z, fx = c.x - a.x, fy = c.y - a.y, fz = c.z - a.z;
        u = make_float4(ey * fz - ez * fy, ez * fx - ex * fz, ex * fy - ey * fx, 0.0f);
        float const ln = sqrtf(u.x * u.x + u.y * u.y + u.z * u.z);
        float const inv = ln > 0.0f && isfinite(ln) ? 1.0f / ln : 0.0f;
        u = make_float4(inv > 0.0f && isfinite(inv) ? u.x * inv : 0.0f, inv > 0.0f && isfinite(inv) ? u.y * inv : 0.0f,
                        inv > 0.0f && isfinite(inv) ? u.z * inv : 0.0f, 0.0f);
    } else {
        const float4* o = node + 3 * (std::size_t(below) + j);
        l = o[0];
        h = o[1];
        u = sum[below + j];
    }
    // of the children, held by the first lanes
    bool const mine = lane < have;
    float const lx = wave_min(l.x), ly = wave_min(l.y), lz = wave_min(l.z);
    float const hx = -wave_min(-h.x), hy = -wave_min(-h.y), hz = -wave_min(-h.z);
    u = mine ? u : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int o = 2; o > 0; o >>= 1) {
        u.x += __shfl_xor(u.x, o, 64);
        u.y += __shfl_xor(u.y, o, 64);
        u.z += __shfl_xor(u.z, o, 64);
    }
    u = make_float4(__shfl(u.x, 0, 64), __shfl(u.y, 0, 64), __shfl(u.z, 0, 64), 0.0f);
    float const ln = sqrtf(u.x * u.x + u.y * u.y + u.z * u.z);
    bool const slab = ln > 1e-3f && isfinite(ln) && level < 4;
    float const gx = slab ? u.x / ln : 0.0f, gy = slab ? u.y / ln : 0.0f, gz = slab ? u.z / ln : 0.0f;
    float s0 = INFINITY, s1 = INFINITY;  // lowest, and the highest negated
    if (slab) {
        std::size_t const per = 3 * std::size_t(kTreeArity) << (2 * level), end = 3 * std::size_t(mesh.m);
        for (std::size_t k = i * per + lane; k < (i + 1) * per && k < end; k += 64) {
            float4 const c = mesh.corners32[k];
            float const e = c.x * gx + c.y * gy + c.z * gz;
            s0 = fminf(s0, e);
            s1 = fminf(s1, -e);
        }
        s0 = wave_min(s0);
        s1 = wave_min(s1);
    }
    if (lane == 0) {
        // where its children are: bit 31 a leaf, bits 29-30 their count less one, the rest the leaf's
        // index or the first child's place in the node array
        uint32_t const info = (level == 0 ? 0x80000000u | i : below + j0) | (have - 1) << 29;
        float4* const o = node + 3 * (std::size_t(mesh.level_off[level]) + i);
        o[0] = make_float4(lx, ly, lz, gx);
        o[1] = make_float4(hx, hy, hz, gy);
        o[2] = make_float4(gz, slab ? s0 : -INFINITY, slab ? -s1 : INFINITY, __uint_as_float(info));
        sum[mesh.level_off[level] + i] = u;
    }
}

__global__ void __launch_bounds__(kBlock) k_tree_level(mesh_dev mesh, uint32_t level, float4* __restrict__ node,
                                                       float4* __restrict__ sum)
{
    for (uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); i < mesh.level_count[level];
         i += gridDim.x * (kBlock / 64))
        tree_node(mesh, level, i, node, sum);
}

}  // namespace

// A triangle mesh on the device: its non-degenerate triangles and, where there are more than a scan takes, the
// tree over them, made there; then the normals that give the distance its sign, made on the host (FP64, no FMA contraction) while the device walks
// the tree. (The tree made on the host, and everything before the walk: 3.57 ms for the 20,480-triangle ball and
// 24^3 cells, 1.53 ms so, 0.93 of it the walk.)
struct mesh_upload {
    dev_buf<uint32_t> tri, orig, face_off, faces, key, ws;
    dev_buf<double> position, corners, vnormal, fnormal;
    dev_buf<float4> node, corners32, sum;
    mesh_dev view{};
    std::vector<uint32_t> t;  // vertices of the non-degenerate triangles

    static void cross(const double a[3], const double b[3], double o[3])
    {
#pragma clang fp contract(off)
        o[0] = a[1] * b[2] - a[2] * b[1];
        o[1] = a[2] * b[0] - a[0] * b[2];
        o[2] = a[0] * b[1] - a[1] * b[0];
    }
    static double dot(const double a[3], const double b[3])
    {
#pragma clang fp contract(off)
        return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
    }

    mesh_upload(hipStream_t s, const double* pos, uint32_t nv, const uint32_t* tris, uint32_t nt)
    {
#pragma clang fp contract(off)
        auto at = [&](uint32_t v, int d) { return pos[3 * std::size_t(v) + d]; };
        double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
        t.reserve(3 * std::size_t(nt));
        for (uint32_t f = 0; f < nt; ++f) {
            double e1[3], e2[3], n[3];
            for (int d = 0; d < 3; ++d) {
                e1[d] = at(tris[3 * f + 1], d) - at(tris[3 * f], d);
                e2[d] = at(tris[3 * f + 2], d) - at(tris[3 * f], d);
            }
            cross(e1, e2, n);
            if (dot(n, n) > 0.0)
                for (int k = 0; k < 3; ++k) {
                    t.push_back(tris[3 * f + k]);
                    for (int d = 0; d < 3; ++d) {
                        lo[d] = std::min(lo[d], at(tris[3 * f + k], d));
                        hi[d] = std::max(hi[d], at(tris[3 * f + k], d));
                    }
                }
        }
        uint32_t const m = uint32_t(t.size() / 3);
        require(m < kMaxTriangles, "too many triangles");
        view.m = m;
        tri.upload(t.data(), t.size(), s);
        view.tri = tri.p;
        if (!m) return;
        if (m <= kScanTriangles) {
            upload_corners(s, pos, lo, hi);
            return;
        }
        morton_box box;
        for (int d = 0; d < 3; ++d) {
            box.lo[d] = lo[d];
            box.scale[d] = hi[d] > lo[d] ? 1024.0 / (hi[d] - lo[d]) : 0.0;
        }
        center(lo, hi);
        uint32_t nodes = 0;
        for (uint32_t n = m; view.levels < kTreeLevels;) {
            n = (n + kTreeArity - 1) / kTreeArity;
            view.level_off[view.levels] = nodes;
            view.level_count[view.levels++] = n;
            nodes += n;
            if (n <= kTreeArity) break;
        }
        position.upload(pos, 3 * std::size_t(nv), s);
        key.alloc(m);
        orig.alloc(m);
        ws.alloc(sort_workspace(m));
        corners.alloc(9 * std::size_t(m));
        corners32.alloc(3 * std::size_t(m));
        node.alloc(3 * std::size_t(nodes));
        sum.alloc(nodes);
        view.orig = orig.p, view.corners = corners.p, view.corners32 = corners32.p, view.node = node.p;
        k_tree_keys<<<(m + 255) / 256, 256, 0, s>>>(position.p, tri.p, m, box, key.p, orig.p);
        radix_sort_pairs(s, key.p, orig.p, m, 30, ws.p);
        k_tree_corners<<<(3 * m + 255) / 256, 256, 0, s>>>(view, position.p, corners.p, corners32.p);
        for (uint32_t l = 0; l < view.levels; ++l)
            k_tree_level<<<level_blocks(view.level_count[l]), kBlock, 0, s>>>(view, l, node.p, sum.p);
        hip_check(hipGetLastError(), "mesh tree");
    }

    // The corners alone, in the triangles' own order, for k_grid_scan: FP64 and then relative to the center in FP32.
    void upload_corners(hipStream_t s, const double* pos, const double lo[3], const double hi[3])
    {
        center(lo, hi);
        std::size_t const n = 3 * std::size_t(view.m), first32 = (3 * n + 1) & ~std::size_t(1);
        host_corners.resize(first32 + 2 * n);
        auto* const c32 = reinterpret_cast<float4*>(host_corners.data() + first32);
        for (std::size_t i = 0; i < n; ++i) {
            const double* x = pos + 3 * std::size_t(t[i]);
            std::copy(x, x + 3, host_corners.data() + 3 * i);
            c32[i] = make_float4(float(x[0] - view.center[0]), float(x[1] - view.center[1]), float(x[2] - view.center[2]),
                                 0.0f);
        }
        corners.upload(host_corners.data(), host_corners.size(), s);
        view.corners = corners.p, view.corners32 = reinterpret_cast<const float4*>(corners.p + first32);
    }

    void center(const double lo[3], const double hi[3])
    {
        for (int d = 0; d < 3; ++d) {
            view.center[d] = 0.5 * (lo[d] + hi[d]);
            view.reach = std::max(view.reach, float(0.5 * (hi[d] - lo[d])) * (1.0f + 1e-6f));
        }
    }

    // The host arrays stay until the stream has taken them.
    std::vector<double> host_corners;
    std::vector<double> vn, fn;
    std::vector<uint32_t> off, inc;

    mesh_normals normals(hipStream_t s, const double* pos, uint32_t nv)
    {
#pragma clang fp contract(off)
        auto at = [&](uint32_t v, int d) { return pos[3 * std::size_t(v) + d]; };
        uint32_t const m = view.m;
        vn.assign(3 * std::size_t(nv), 0.0);
        fn.resize(3 * std::size_t(m));
        for (uint32_t f = 0; f < m; ++f) {
            double p[3][3];
            for (int k = 0; k < 3; ++k)
                for (int d = 0; d < 3; ++d) p[k][d] = at(t[3 * f + k], d);
            double e1[3], e2[3], n[3];
            for (int d = 0; d < 3; ++d) {
                e1[d] = p[1][d] - p[0][d];
                e2[d] = p[2][d] - p[0][d];
            }
            cross(e1, e2, n);
            double const ln = std::sqrt(dot(n, n));
            for (int d = 0; d < 3; ++d) {
                n[d] = n[d] / ln;
                fn[3 * std::size_t(f) + d] = n[d];
            }
            for (int k = 0; k < 3; ++k) {
                double a1[3], a2[3];
                for (int d = 0; d < 3; ++d) {
                    a1[d] = p[(k + 1) % 3][d] - p[k][d];
                    a2[d] = p[(k + 2) % 3][d] - p[k][d];
                }
                double const cs = dot(a1, a2) / (std::sqrt(dot(a1, a1)) * std::sqrt(dot(a2, a2)));
                double const alpha = std::acos(std::max(-1.0, std::min(1.0, cs)));
                uint32_t const v = t[3 * f + k];
                for (int d = 0; d < 3; ++d) vn[3 * std::size_t(v) + d] = vn[3 * std::size_t(v) + d] + alpha * n[d];
            }
        }
        // each vertex's triangles in increasing order
        off.assign(std::size_t(nv) + 1, 0);
        inc.resize(t.size());
        for (uint32_t v : t) ++off[v + 1];
        for (std::size_t v = 0; v < nv; ++v) off[v + 1] += off[v];
        std::vector<uint32_t> fill(off.begin(), off.end() - 1);
        for (std::size_t i = 0; i < t.size(); ++i) inc[fill[t[i]]++] = uint32_t(i / 3);
        vnormal.upload(vn.data(), vn.size(), s);
        fnormal.upload(fn.data(), fn.size(), s);
        face_off.upload(off.data(), off.size(), s);
        faces.upload(inc.data(), inc.size(), s);
        return {vnormal.p, fnormal.p, face_off.p, faces.p};
    }
};

void grid_cell_size(const double dmin[3], const double dmax[3], const uint32_t res[3], double cell[3],
                    double inv_cell[3])
{
    for (int d = 0; d < 3; ++d) {
        cell[d] = (dmax[d] - dmin[d]) / double(res[d]);
        inv_cell[d] = 1.0 / cell[d];
    }
}

void check_grid(const double dmin[3], const double dmax[3], const uint32_t res[3])
{
    require(dmin && dmax && res, "null grid argument");
    for (int d = 0; d < 3; ++d) {
        require(res[d] >= 1, "grid resolution must be at least 1 cell per axis");
        require(std::isfinite(dmin[d]) && std::isfinite(dmax[d]) && dmax[d] > dmin[d],
                "grid domain must be a finite box with max > min");
    }
    require(grid_dims(res).nodes() < (uint64_t(1) << 32), "grid has too many nodes");
}

void build_mesh_grid(hipStream_t s, const double* pos, uint32_t nv, const uint32_t* tris, uint32_t nt,
                     const double dmin[3], const double dmax[3], const uint32_t res[3], double* dev_nodes)
{
    require((pos || nv == 0) && (tris || nt == 0), "null mesh argument");
    for (std::size_t i = 0; i < 3 * std::size_t(nt); ++i) require(tris[i] < nv, "triangle vertex index out of range");
    check_grid(dmin, dmax, res);
    grid_params gp{};
    double inv_cell[3];
    grid_cell_size(dmin, dmax, res, gp.cell, inv_cell);
    for (int d = 0; d < 3; ++d) {
        gp.res[d] = res[d];
        gp.dmin[d] = dmin[d];
    }
    uint64_t const n = grid_dims(res).nodes(), per_block = uint64_t(kRun) * (kBlock / 64);
    dev_buf<uint32_t> nearest_of;
    if (nt > kScanTriangles) nearest_of.alloc(n);
    mesh_upload mesh(s, pos, nv, tris, nt);
    if (mesh.view.m <= kScanTriangles) {
        mesh_normals const nm = mesh.normals(s, pos, nv);
        uint32_t const split = n <= kSplitNodes ? 8u : 1u;
        auto const scan = split > 1 ? k_grid_scan<8> : k_grid_scan<1>;
        scan<<<unsigned((n * split + kBlock - 1) / kBlock), kBlock, 0, s>>>(mesh.view, nm, gp, n, dev_nodes);
        hip_check(hipGetLastError(), "grid node kernel");
        hip_check(hipStreamSynchronize(s), "grid node kernel");
        return;
    }
    k_grid_nodes<<<unsigned((n + per_block - 1) / per_block), kBlock, 0, s>>>(mesh.view, gp, n, nearest_of.p);
    hip_check(hipGetLastError(), "grid node kernel");
    mesh_normals const nm = mesh.normals(s, pos, nv);
    k_grid_signs<<<unsigned((n + kBlock - 1) / kBlock), kBlock, 0, s>>>(mesh.view, nm, gp, n, nearest_of.p, dev_nodes);
    hip_check(hipGetLastError(), "grid node kernel");
    hip_check(hipStreamSynchronize(s), "grid node kernel");
}

void environment_domain(const double* pos, uint32_t nv, const double lo_in[3], const double hi_in[3], double lo[3],
                        double hi[3])
{
#pragma clang fp contract(off)
    for (int d = 0; d < 3; ++d) {
        lo[d] = lo_in[d];
        hi[d] = hi_in[d];
    }
    for (uint32_t i = 0; i < nv; ++i)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], pos[3 * std::size_t(i) + d]);
            hi[d] = std::max(hi[d], pos[3 * std::size_t(i) + d]);
        }
    // environment_body.cpp:54-64: once per vertex, max grows by 1e-3 |diagonal|, then min by
    // 1e-3 |diagonal| of the grown box (re-extending by the vertices inside the loop changes nothing
    // after the first pass)
    auto diag_norm = [&] {
        double const a = hi[0] - lo[0], b = hi[1] - lo[1], c = hi[2] - lo[2];
        return std::sqrt(a * a + b * b + c * c);
    };
    for (uint32_t v = 0; v < nv; ++v) {
        double const g1 = 1.0e-3 * diag_norm();
        for (int d = 0; d < 3; ++d) hi[d] += g1 * 1.0;
        double const g2 = 1.0e-3 * diag_norm();
        for (int d = 0; d < 3; ++d) lo[d] -= g2 * 1.0;
    }
}

namespace {

__global__ void k_eval_sdf(sdf_dev f, const double* __restrict__ pts, uint32_t n, double* __restrict__ sd,
                           double* __restrict__ grad)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    pos4 const p = make_double4(pts[3 * std::size_t(i)], pts[3 * std::size_t(i) + 1], pts[3 * std::size_t(i) + 2], 0.0);
    double v, g[3];
    sdf_eval(f, p, v, g);
    sd[i] = v;
    grad[3 * std::size_t(i)] = g[0];
    grad[3 * std::size_t(i) + 1] = g[1];
    grad[3 * std::size_t(i) + 2] = g[2];
}

}  // namespace

void evaluate_sdf(hipStream_t s, sdf_dev const& f, const double* pts, uint32_t n, double* sd, double* grad)
{
    if (n == 0) return;
    dev_buf<double> dp, dsd, dg;
    dp.upload(pts, 3 * std::size_t(n), s);
    dsd.alloc(n);
    dg.alloc(3 * std::size_t(n));
    k_eval_sdf<<<(n + 255) / 256, 256, 0, s>>>(f, dp.p, n, dsd.p, dg.p);
    hip_check(hipGetLastError(), "sdf evaluation");
    hip_check(hipMemcpyAsync(sd, dsd.p, n * sizeof(double), hipMemcpyDeviceToHost, s), "read sdf values");
    hip_check(hipMemcpyAsync(grad, dg.p, 3 * std::size_t(n) * sizeof(double), hipMemcpyDeviceToHost, s),
              "read sdf gradients");
    hip_check(hipStreamSynchronize(s), "sdf evaluation");
}

}  // namespace sbs

using namespace sbs;

extern "C" int sbs_sdf_grid_node_count(const uint32_t resolution[3], uint64_t* count)
{
    return guarded([&] {
        require(resolution && count, "null argument");
        *count = grid_dims(resolution).nodes();
    });
}

extern "C" int sbs_sdf_grid_node_positions(const double domain_min[3], const double domain_max[3],
                                           const uint32_t resolution[3], double* positions)
{
    return guarded([&] {
        check_grid(domain_min, domain_max, resolution);
        require(positions != nullptr, "positions is null");
        double cell[3], inv_cell[3];
        grid_cell_size(domain_min, domain_max, resolution, cell, inv_cell);
        grid_dims const g(resolution);
        for (uint64_t l = 0; l < g.nodes(); ++l) grid_node_position(g, domain_min, cell, l, positions + 3 * l);
    });
}

extern "C" int sbs_sdf_environment_domain(const double* positions, uint32_t num_vertices, const double domain_min[3],
                                          const double domain_max[3], double out_min[3], double out_max[3])
{
    return guarded([&] {
        require((positions || num_vertices == 0) && domain_min && domain_max && out_min && out_max, "null argument");
        environment_domain(positions, num_vertices, domain_min, domain_max, out_min, out_max);
    });
}

extern "C" int sbs_sdf_grid_from_mesh(int device, const double* positions, uint32_t num_vertices,
                                      const uint32_t* triangles, uint32_t num_triangles, const double domain_min[3],
                                      const double domain_max[3], const uint32_t resolution[3], double* nodes)
{
    return guarded([&] {
        require(nodes != nullptr, "nodes is null");
        check_grid(domain_min, domain_max, resolution);
        hip_check(hipSetDevice(device), "hipSetDevice");
        hipStream_t s;
        hip_check(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "hipStreamCreate");
        try {
            uint64_t const n = grid_dims(resolution).nodes();
            dev_buf<double> dn;
            dn.alloc(n);
            build_mesh_grid(s, positions, num_vertices, triangles, num_triangles, domain_min, domain_max, resolution,
                            dn.p);
            hip_check(hipMemcpyAsync(nodes, dn.p, n * sizeof(double), hipMemcpyDeviceToHost, s), "read grid nodes");
            hip_check(hipStreamSynchronize(s), "read grid nodes");
        } catch (...) {
            (void)hipStreamDestroy(s);
            throw;
        }
        hip_check(hipStreamDestroy(s), "hipStreamDestroy");
    });
}
