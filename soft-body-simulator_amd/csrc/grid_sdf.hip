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
// A wave per grid node walks a tree of bounds over the triangles in Morton order (k_grid_nodes). What bounds
// it: the FP32 tests of a few hundred tree nodes and triangles a grid node and the round trips to L2 between
// the batches. On the 20,480-triangle ball and 24^3 cells (104,625 nodes) 963 us, where the scan of
// 128-triangle tiles through LDS that it replaces took 12.4 ms.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <utility>
#include <vector>

#include "abi_util.h"
#include "grid_sdf.h"
#include "sdf.h"

namespace sbs {

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kRun = 16;  // grid nodes a wave takes (6,500 waves for 24^3 cells: six a SIMD)
// Each of at most 16 levels leaves at most 48 children of one batch waiting while the walk goes deeper.
constexpr uint32_t kStack = 1024, kList = 256;

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
// coordinates, which is several times what their roundings add up to.
struct seeker {
    float x, y, z, margin, limit;
    __device__ __forceinline__ void set(mesh_dev const& mesh, const double p[3])
    {
        x = float(p[0] - mesh.center[0]);
        y = float(p[1] - mesh.center[1]);
        z = float(p[2] - mesh.center[2]);
        margin = 4e-6f * (mesh.reach + fabsf(x) + fabsf(y) + fabsf(z));
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
    // its centroid (about ten triangles a node are left for the FP64 closest point).
    __device__ __forceinline__ bool may_be(float4 a, float4 b, float4 c) const
    {
        float const ax = a.x - x, ay = a.y - y, az = a.z - z, bx = b.x - x, by = b.y - y, bz = b.z - z,
                    cx = c.x - x, cy = c.y - y, cz = c.z - z;
        float const wx = ax + bx + cx, wy = ay + by + cy, wz = az + bz + cz;
        float const r = __builtin_amdgcn_rsqf(fmaf(wx, wx, fmaf(wy, wy, wz * wz)));
        float const m = fminf(fminf(fmaf(ax, wx, fmaf(ay, wy, az * wz)), fmaf(bx, wx, fmaf(by, wy, bz * wz))),
                              fmaf(cx, wx, fmaf(cy, wy, cz * wz)));
        return !(m * r > limit);
    }
};

// Triangle t's exact closest point against the best so far.
__device__ __forceinline__ void visit(mesh_dev const& mesh, uint32_t t, const double p[3], nearest& best)
{
#pragma clang fp contract(off)
    double c[9], q[3];
    for (int k = 0; k < 9; ++k) c[k] = mesh.corners[9 * std::size_t(t) + k];
    int feat;
    tri_closest_point(p, c, q, &feat);
    double const e0 = p[0] - q[0], e1 = p[1] - q[1], e2 = p[2] - q[2];
    double const d2 = e0 * e0 + e1 * e1 + e2 * e2;
    uint32_t const o = mesh.orig[t];
    if (d2 < best.d2 || (d2 == best.d2 && o < best.o)) best = nearest{d2, t, o};
}

// Every lane gets the nearest of the wave's.
__device__ __forceinline__ void wave_nearest(nearest& best)
{
    for (int o = 32; o > 0; o >>= 1) {
        nearest const b{__shfl_xor(best.d2, o, 64), uint32_t(__shfl_xor(best.t, o, 64)), uint32_t(__shfl_xor(best.o, o, 64))};
        if (b.d2 < best.d2 || (b.d2 == best.d2 && b.o < best.o)) best = b;
    }
}

// The signed distance from the nearest triangle: its closest point again, the pseudo-normal of the
// feature that holds it (an edge's is the sum of its triangles' unit normals in original order).
__device__ __forceinline__ double signed_distance(mesh_dev const& mesh, const double p[3], nearest const& best)
{
#pragma clang fp contract(off)
    if (best.t == 0xffffffffu) return DBL_MAX;
    double c[9], q[3], nrm[3] = {0.0, 0.0, 0.0};
    for (int k = 0; k < 9; ++k) c[k] = mesh.corners[9 * std::size_t(best.t) + k];
    int feat;
    tri_closest_point(p, c, q, &feat);
    const uint32_t* tv = mesh.tri + 3 * std::size_t(best.o);
    if (feat < 3) {
        for (int d = 0; d < 3; ++d) nrm[d] = mesh.vnormal[3 * std::size_t(tv[feat]) + d];
    } else if (feat < 6) {
        uint32_t const v = tv[feat - 3], w = tv[feat == 5 ? 0 : feat - 2];
        for (uint32_t i = mesh.face_off[v], e = mesh.face_off[v + 1]; i < e; ++i) {
            uint32_t const f = mesh.faces[i];
            const uint32_t* fv = mesh.tri + 3 * std::size_t(f);
            if (fv[0] != w && fv[1] != w && fv[2] != w) continue;
            for (int d = 0; d < 3; ++d) nrm[d] = nrm[d] + mesh.fnormal[3 * std::size_t(f) + d];
        }
    } else {
        for (int d = 0; d < 3; ++d) nrm[d] = mesh.fnormal[3 * std::size_t(best.o) + d];
    }
    double const s = (p[0] - q[0]) * nrm[0] + (p[1] - q[1]) * nrm[1] + (p[2] - q[2]) * nrm[2];
    double const d = sqrt(best.d2);
    return s < 0.0 ? -d : d;
}

// One wave walks the tree for one grid node, kRun consecutive nodes one after the other. The walk takes up
// to 16 tree nodes off a stack in LDS and tests their 64 children at once, one a lane, each with FP32
// bounds; children that may hold something go back on the stack, triangles that may be the nearest to a
// list whose exact FP64 closest points the lanes then share. (A lane per grid node walked 64 different
// paths: 4.3 ms on the 20,480-triangle ball and 24^3 cells, 0.96 ms so.) The first bound is exact distances
// to 64 triangles that are neighbours in Morton order: those of the last node's nearest one, for a run's
// first node those of the nearest box.
__global__ void __launch_bounds__(kBlock) k_grid_nodes(mesh_dev mesh, grid_params gp, uint64_t n,
                                                       double* __restrict__ out)
{
    constexpr uint32_t kWaves = kBlock / 64;
    __shared__ uint32_t stack_lds[kWaves][kStack], list_lds[kWaves][kList];
    uint32_t const wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint64_t const l0 = (uint64_t(blockIdx.x) * kWaves + wave) * kRun;
    if (l0 >= n) return;
    uint32_t const cnt = uint32_t(n - l0 < kRun ? n - l0 : kRun);
    if (mesh.m == 0) {
        if (lane < cnt) out[l0 + lane] = DBL_MAX;
        return;
    }
    uint32_t* const stack = stack_lds[wave];
    uint32_t* const list = list_lds[wave];
    uint64_t const below = (uint64_t(1) << lane) - 1;
    grid_dims const dims(gp.res);
    uint32_t const top = mesh.levels - 1, start = top < 2 ? top : 2;
    nearest mine;  // lane r: the nearest of node l0 + r
    uint32_t block = 0;  // of 64 triangles
    for (uint32_t r = 0; r < cnt; ++r) {
        double p[3];
        grid_node_position(dims, gp.dmin, gp.cell, l0 + r, p);
        seeker at;
        at.set(mesh, p);
        if (r == 0 && top >= 2) {  // a node two levels up is one block of 64 triangles
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
        if (64 * block + lane < mesh.m) visit(mesh, 64 * block + lane, p, best);
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
            for (uint32_t i = lane; i < candidates; i += 64) visit(mesh, list[i], p, best);
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
        if (lane == r) mine = best;
    }
    if (lane < cnt) {
        double p[3];
        grid_node_position(dims, gp.dmin, gp.cell, l0 + lane, p);
        out[l0 + lane] = signed_distance(mesh, p, mine);
    }
}

}  // namespace

void launch_grid_nodes(hipStream_t s, mesh_dev const& mesh, const uint32_t res[3], const double dmin[3],
                       const double cell[3], double* nodes)
{
    grid_params gp{};
    for (int d = 0; d < 3; ++d) {
        gp.res[d] = res[d];
        gp.dmin[d] = dmin[d];
        gp.cell[d] = cell[d];
    }
    uint64_t const n = grid_dims(res).nodes(), per_block = uint64_t(kRun) * (kBlock / 64);
    k_grid_nodes<<<unsigned((n + per_block - 1) / per_block), kBlock, 0, s>>>(mesh, gp, n, nodes);
}

// Host side of the mesh: non-degenerate triangles, corners and pseudonormals (FP64, no FMA
// contraction), uploaded to the device.
struct mesh_upload {
    dev_buf<uint32_t> tri, orig, face_off, faces;
    dev_buf<double> corners, vnormal, fnormal;
    dev_buf<float4> node, corners32;
    mesh_dev view{};

    mesh_upload(hipStream_t s, const double* pos, uint32_t nv, const uint32_t* tris, uint32_t nt)
    {
#pragma clang fp contract(off)
        auto at = [&](uint32_t v, int d) { return pos[3 * std::size_t(v) + d]; };
        auto cross = [](const double a[3], const double b[3], double o[3]) {
            o[0] = a[1] * b[2] - a[2] * b[1];
            o[1] = a[2] * b[0] - a[0] * b[2];
            o[2] = a[0] * b[1] - a[1] * b[0];
        };
        auto dot = [](const double a[3], const double b[3]) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; };
        std::vector<uint32_t> t;
        for (uint32_t f = 0; f < nt; ++f) {
            double e1[3], e2[3], n[3];
            for (int d = 0; d < 3; ++d) {
                e1[d] = at(tris[3 * f + 1], d) - at(tris[3 * f], d);
                e2[d] = at(tris[3 * f + 2], d) - at(tris[3 * f], d);
            }
            cross(e1, e2, n);
            if (dot(n, n) > 0.0)
                for (int k = 0; k < 3; ++k) t.push_back(tris[3 * f + k]);
        }
        uint32_t const m = uint32_t(t.size() / 3);
        std::vector<double> c(9 * std::size_t(m)), vn(3 * std::size_t(nv), 0.0), fn(3 * std::size_t(m));
        for (uint32_t f = 0; f < m; ++f) {
            double p[3][3];
            for (int k = 0; k < 3; ++k)
                for (int d = 0; d < 3; ++d) {
                    p[k][d] = at(t[3 * f + k], d);
                    c[9 * std::size_t(f) + 3 * k + d] = p[k][d];
                }
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
        std::vector<uint32_t> off(std::size_t(nv) + 1, 0), inc(t.size());
        for (uint32_t v : t) ++off[v + 1];
        for (std::size_t v = 0; v < nv; ++v) off[v + 1] += off[v];
        {
            std::vector<uint32_t> fill(off.begin(), off.end() - 1);
            for (std::size_t i = 0; i < t.size(); ++i) inc[fill[t[i]]++] = uint32_t(i / 3);
        }
        // triangles in Morton order of their centroids (10 bits per axis over the mesh's box),
        // corners in that order, each with its original index; boxes of every kTreeArity of them, of
        // every kTreeArity of those, and so on up to at most kTreeArity
        std::vector<uint32_t> ord(m);
        {
            double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
            for (std::size_t i = 0; i < 9 * std::size_t(m); ++i) {
                lo[i % 3] = std::min(lo[i % 3], c[i]);
                hi[i % 3] = std::max(hi[i % 3], c[i]);
            }
            auto spread = [](uint32_t v) {
                uint64_t x = v & 0x3ffu;
                x = (x | (x << 16)) & 0x30000ffull;
                x = (x | (x << 8)) & 0x300f00full;
                x = (x | (x << 4)) & 0x30c30c3ull;
                x = (x | (x << 2)) & 0x9249249ull;
                return x;
            };
            std::vector<std::pair<uint64_t, uint32_t>> key(m);
            for (uint32_t f = 0; f < m; ++f) {
                uint64_t code = 0;
                for (int d = 0; d < 3; ++d) {
                    double const cen = (c[9 * std::size_t(f) + d] + c[9 * std::size_t(f) + 3 + d] +
                                        c[9 * std::size_t(f) + 6 + d]) / 3.0;
                    double const ext = hi[d] - lo[d];
                    double const u = ext > 0.0 ? (cen - lo[d]) / ext : 0.0;
                    uint32_t const q = uint32_t(std::min(1023.0, std::max(0.0, u * 1024.0)));
                    code |= spread(q) << d;
                }
                key[f] = {code, f};
            }
            std::sort(key.begin(), key.end());
            for (uint32_t i = 0; i < m; ++i) ord[i] = key[i].second;
        }
        std::vector<double> cs(9 * std::size_t(m));
        for (uint32_t i = 0; i < m; ++i)
            std::copy(c.begin() + 9 * std::size_t(ord[i]), c.begin() + 9 * std::size_t(ord[i]) + 9,
                      cs.begin() + 9 * std::size_t(i));
        // relative to the middle of the mesh's box, in FP32 (the walk's margin covers the rounding)
        double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
        for (std::size_t i = 0; i < cs.size(); ++i) {
            lo[i % 3] = std::min(lo[i % 3], cs[i]);
            hi[i % 3] = std::max(hi[i % 3], cs[i]);
        }
        for (int d = 0; d < 3 && m; ++d) {
            view.center[d] = 0.5 * (lo[d] + hi[d]);
            view.reach = std::max(view.reach, float(0.5 * (hi[d] - lo[d])) * (1.0f + 1e-6f));
        }
        std::vector<float4> c32(3 * std::size_t(m));
        for (std::size_t i = 0; i < c32.size(); ++i)
            c32[i] = make_float4(float(cs[3 * i] - view.center[0]), float(cs[3 * i + 1] - view.center[1]),
                                 float(cs[3 * i + 2] - view.center[2]), 0.0f);
        std::vector<float4> nd;
        std::vector<std::array<float, 3>> below(m), sums;  // normals of the triangles, then of the level below
        for (uint32_t i = 0; i < m; ++i)
            for (int d = 0; d < 3; ++d) below[i][d] = float(fn[3 * std::size_t(ord[i]) + d]);
        std::size_t per = 1;  // triangles under a node of the level
        for (uint32_t n = m, child = 0; n > 0 && view.levels < kTreeLevels; ++view.levels) {
            uint32_t const cnt = uint32_t((uint64_t(n) + kTreeArity - 1) / kTreeArity), first = uint32_t(nd.size() / 3);
            nd.resize(nd.size() + 3 * std::size_t(cnt));
            sums.assign(cnt, {0.0f, 0.0f, 0.0f});
            per *= kTreeArity;
            for (uint32_t i = 0; i < cnt; ++i) {
                float4 l = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
                float4 h = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
                auto cover = [&](float4 const& a, float4 const& b) {
                    l = make_float4(std::min(l.x, a.x), std::min(l.y, a.y), std::min(l.z, a.z), 0.0f);
                    h = make_float4(std::max(h.x, b.x), std::max(h.y, b.y), std::max(h.z, b.z), 0.0f);
                };
                std::size_t const j0 = std::size_t(i) * kTreeArity, j1 = std::min<std::size_t>(n, j0 + kTreeArity);
                std::array<float, 3>& u = sums[i];
                for (std::size_t j = j0; j < j1; ++j) {
                    if (view.levels == 0)
                        for (int k = 0; k < 3; ++k) cover(c32[3 * j + k], c32[3 * j + k]);
                    else
                        cover(nd[3 * (child + j)], nd[3 * (child + j) + 1]);
                    for (int d = 0; d < 3; ++d) u[d] += below[j][d];
                }
                float const ln = std::sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
                // slabs for patches of up to 256 triangles; larger ones bend too far for one
                bool const slab = ln > 1e-3f && std::isfinite(ln) && view.levels < 4;
                float const g[3] = {slab ? u[0] / ln : 0.0f, slab ? u[1] / ln : 0.0f, slab ? u[2] / ln : 0.0f};
                float s0 = slab ? INFINITY : -INFINITY, s1 = slab ? -INFINITY : INFINITY;
                for (std::size_t j = 3 * i * per; slab && j < std::min<std::size_t>(c32.size(), 3 * (i + 1) * per); ++j) {
                    float const e = c32[j].x * g[0] + c32[j].y * g[1] + c32[j].z * g[2];
                    s0 = std::min(s0, e);
                    s1 = std::max(s1, e);
                }
                l.w = g[0];
                h.w = g[1];
                float4* o = nd.data() + 3 * (std::size_t(first) + i);
                o[0] = l;
                o[1] = h;
                // where its children are: bit 31 a leaf, bits 29-30 their count less one, the rest the leaf's
                // index or the first child's place in the node array
                uint32_t const info = (view.levels == 0 ? 0x80000000u | i : child + uint32_t(j0)) |
                                      (uint32_t(j1 - j0 - 1) << 29);
                float word;
                std::memcpy(&word, &info, sizeof word);
                o[2] = make_float4(g[2], s0, s1, word);
            }
            view.level_off[view.levels] = child = first;
            view.level_count[view.levels] = n = cnt;
            below.swap(sums);
            if (cnt <= kTreeArity) {
                ++view.levels;
                break;
            }
        }
        tri.upload(t.data(), t.size(), s);
        corners.upload(cs.data(), cs.size(), s);
        orig.upload(ord.data(), ord.size(), s);
        face_off.upload(off.data(), off.size(), s);
        faces.upload(inc.data(), inc.size(), s);
        node.upload(nd.data(), nd.size(), s);
        corners32.upload(c32.data(), c32.size(), s);
        vnormal.upload(vn.data(), vn.size(), s);
        fnormal.upload(fn.data(), fn.size(), s);
        hip_check(hipStreamSynchronize(s), "mesh upload");
        view.tri = tri.p, view.corners = corners.p, view.vnormal = vnormal.p, view.fnormal = fnormal.p;
        view.orig = orig.p, view.face_off = face_off.p, view.faces = faces.p;
        view.node = node.p, view.corners32 = corners32.p;
        view.m = m;
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
    mesh_upload const mesh(s, pos, nv, tris, nt);
    double cell[3], inv_cell[3];
    grid_cell_size(dmin, dmax, res, cell, inv_cell);
    require(mesh.view.m < (1u << 30), "too many triangles");
    launch_grid_nodes(s, mesh.view, res, dmin, cell, dev_nodes);
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
