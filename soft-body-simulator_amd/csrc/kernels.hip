// gfx950 kernels of the XPBD time step: prediction, per-color constraint projection (green strain,
// stable neo-Hookean, distance), clustered Gauss-Seidel, SDF contact detection and projection,
// velocity update, FP64 residual / energy reductions and Jones-Plassmann graph coloring.
//
// Particle state lives in HBM as SoA streams: xi (working positions, w = inverse mass) and xn
// (substep start = committed positions, w = inverse mass) as double4, velocities as float4.
// Positions are stored in FP64 so that a tet's edge vectors keep FP32 relative precision wherever
// the body is: every constraint forms its edge differences in FP64, does all of its arithmetic in
// FP32 on those differences, and adds its FP32 correction back in FP64. Constraint data of a group
// is stored in execution (color) order so that one color is one contiguous, coalesced range.
#include <algorithm>

#include "device_math.h"
#include "kernels.h"
#include "mlp_device.h"
#include "sdf.h"
#include "solver_device.h"

namespace sbs {

namespace {

inline unsigned grid_for(uint32_t n, int block) { return (n + uint32_t(block) - 1) / uint32_t(block); }

// ---------------------------------------------------------------- prediction / commit

__global__ void k_predict(pos4* __restrict__ xi, const pos4* __restrict__ xn, float4* __restrict__ v, uint32_t n,
                          float gx, float gy, float gz, int force, float dt)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    pos4 const x = xn[i];
    float4 vel = v[i];
    pos4 p;
    predict_one(p, x, vel, gx, gy, gz, force, dt);
    v[i] = vel;
    xi[i] = p;
}

__global__ void k_commit(const pos4* __restrict__ xi, pos4* __restrict__ xn, float4* __restrict__ v, uint32_t n,
                         float dt)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    pos4 const p = xi[i], q = xn[i];
    v[i] = velocity(p, q, dt);
    xn[i] = p;
}

// Commit of one substep fused with the prediction of the next (same per-particle order). With prow,
// thread r handles particle prow[r] (rows [0, n); padding rows hold 0xffffffff), else particle r.
__global__ void k_commit_predict(pos4* __restrict__ xi, pos4* __restrict__ xn, float4* __restrict__ v, uint32_t n,
                                 float gx, float gy, float gz, int force, float dt, const uint32_t* __restrict__ prow)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (prow) {
        i = prow[i];
        if (i == 0xffffffffu) return;
    }
    pos4 const p = xi[i], q = xn[i];
    float4 vel = velocity(p, q, dt);
    pos4 np;
    predict_one(np, p, vel, gx, gy, gz, force, dt);
    xn[i] = p;
    v[i] = vel;
    xi[i] = np;
}

// ---------------------------------------------------------------- green strain constraint
__global__ void __launch_bounds__(256) k_green(tet_group_dev g, pos4* xi, const pos4* __restrict__ xn, uint32_t begin,
                                               uint32_t count, float alpha_tilde, float gamma, int first)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    uint32_t const t = begin + i;
    int4 const id = g.idx[t];
    float4 const a = g.m0[t], b = g.m1[t], c = g.m2[t];
    float lm = first ? 0.0f : g.lambda[t];
    pos4 P[4] = {xi[id.x], xi[id.y], xi[id.z], xi[id.w]};
    auto xn_of = [&](int k) { return xn[k == 0 ? id.x : (k == 1 ? id.y : (k == 2 ? id.z : id.w))]; };
    if (!green_project(P, xn_of, a, b, c, alpha_tilde, gamma, lm)) {
        if (first) g.lambda[t] = 0.0f;
        return;
    }
    g.lambda[t] = lm;
    xi[id.x] = P[0];
    xi[id.y] = P[1];
    xi[id.z] = P[2];
    xi[id.w] = P[3];
}

// x += d in FP64 (read, add, write) for the x, y, z of one particle.
__device__ __forceinline__ void add_displacement(pos4* x, v3 d)
{
    double* q = reinterpret_cast<double*>(x);
    q[0] += double(d.x);
    q[1] += double(d.y);
    q[2] += double(d.z);
}

template <bool DAMPED>
__global__ void __launch_bounds__(256) k_neohookean(tet_group_dev g, pos4* xi, const pos4* __restrict__ xn,
                                                    uint32_t begin, uint32_t count, float inv_dt2, float beta_dt,
                                                    int mode, float hyd_scale)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    uint32_t const t = begin + i;
    int4 const id = g.idx[t];
    float4 const a = g.m0[t], b = g.m1[t];
    float2 const c = nh_m2(g, t);
    float2 lm = mode == kSolveFirst ? make_float2(0.0f, 0.0f) : reinterpret_cast<const float2*>(g.lambda)[t];
    if (mode >= kApplyWarmStart) {  // gradients at the predicted positions (xn holds a copy of them)
        pos4 const P[4] = {xn[id.x], xn[id.y], xn[id.z], xn[id.w]};
        v3 d[4];
        // in the warm-start modes beta_dt carries the deviatoric multiplier's scale (no damping term
        // applies), hyd_scale the hydrostatic one's
        neohookean_displacement(P, a, b, c, inv_dt2, mode == kApplyExplicit, make_float2(beta_dt, hyd_scale), lm, d);
        reinterpret_cast<float2*>(g.lambda)[t] = lm;
        add_displacement(&xi[id.x], d[0]);
        add_displacement(&xi[id.y], d[1]);
        add_displacement(&xi[id.z], d[2]);
        add_displacement(&xi[id.w], d[3]);
        return;
    }
    pos4 P[4] = {xi[id.x], xi[id.y], xi[id.z], xi[id.w]};
    auto xn_of = [&](int k) { return xn[k == 0 ? id.x : (k == 1 ? id.y : (k == 2 ? id.z : id.w))]; };
    neohookean_project<DAMPED>(P, xn_of, a, b, c, inv_dt2, beta_dt, lm);
    reinterpret_cast<float2*>(g.lambda)[t] = lm;
    xi[id.x] = P[0];
    xi[id.y] = P[1];
    xi[id.z] = P[2];
    xi[id.w] = P[3];
}

// ---------------------------------------------------------------- multiplier warm start

__global__ void k_copy_pos(const pos4* __restrict__ a, pos4* __restrict__ b, uint32_t n)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = a[i];
}

// One component a thread, so that a wave's stores to host memory are one run of 512 (256) bytes; bounded
// by the link to the host.
__global__ void __launch_bounds__(256) k_pack_state(const pos4* __restrict__ x, const float4* __restrict__ v,
                                                    uint32_t n, double* __restrict__ xo, float* __restrict__ vo)
{
    std::size_t const i = std::size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= 3 * std::size_t(n)) return;
    std::size_t const p = i / 3, c = i % 3;
    if (xo) xo[i] = reinterpret_cast<const double*>(x)[4 * p + c];
    if (vo) vo[i] = reinterpret_cast<const float*>(v)[4 * p + c];
}

// ---------------------------------------------------------------- clustered Gauss-Seidel

// One thread per cluster: the cluster's particles are staged in LDS (slot-major, so that the
// threads of a wave hit consecutive words), its constraints run in order against the staged
// copies, and the particles are written back once. Clusters of one color share no particle, so
// this equals the sequential sweep over the color's clusters.
template <int BLOCK>
struct cluster_stage {
    pos4 p[kClusterSlots][BLOCK];
};

__device__ __forceinline__ int slot_id(int4 va, int4 vb, uint32_t s)
{
    int const lo = s == 0 ? va.x : (s == 1 ? va.y : (s == 2 ? va.z : va.w));
    int const hi = s == 4 ? vb.x : (s == 5 ? vb.y : (s == 6 ? vb.z : vb.w));
    return s < 4 ? lo : hi;
}

template <int BLOCK, class Project>
__device__ __forceinline__ void run_cluster(cluster_dev const& cl, pos4* xi, const pos4* __restrict__ xn,
                                            uint32_t begin, uint32_t count, Project&& project)
{
    __shared__ cluster_stage<BLOCK> st;
    uint32_t const i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= count) return;
    uint32_t const c = begin + i;
    int4 const va = cl.v0[c], vb = cl.v1[c];
    int const ids[kClusterSlots] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
    pos4 (*P)[BLOCK] = st.p;
#pragma unroll
    for (int k = 0; k < kClusterSlots; ++k)
        if (ids[k] >= 0) P[k][threadIdx.x] = xi[ids[k]];
    uint32_t const t0 = cl.off[c], t1 = cl.off[c + 1];
    for (uint32_t t = t0; t < t1; ++t) {
        uint32_t const loc = cl.loc[t];
        uint32_t const s0 = loc & 0xffu, s1 = (loc >> 8) & 0xffu, s2 = (loc >> 16) & 0xffu, s3 = loc >> 24;
        pos4 Q[4] = {P[s0][threadIdx.x], P[s1][threadIdx.x], P[s2][threadIdx.x], P[s3][threadIdx.x]};
        int const id[4] = {slot_id(va, vb, s0), slot_id(va, vb, s1), slot_id(va, vb, s2), slot_id(va, vb, s3)};
        auto xn_of = [&](int k) { return xn[id[k]]; };
        project(t, Q, xn_of);
        P[s0][threadIdx.x] = Q[0];
        P[s1][threadIdx.x] = Q[1];
        P[s2][threadIdx.x] = Q[2];
        P[s3][threadIdx.x] = Q[3];
    }
#pragma unroll
    for (int k = 0; k < kClusterSlots; ++k)
        if (ids[k] >= 0) xi[ids[k]] = P[k][threadIdx.x];
}

template <int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_green_clusters(tet_group_dev g, cluster_dev cl, pos4* xi,
                                                          const pos4* __restrict__ xn, uint32_t begin, uint32_t count,
                                                          float alpha_tilde, float gamma, int first)
{
    run_cluster<BLOCK>(cl, xi, xn, begin, count, [&](uint32_t t, pos4 P[4], auto&& xn_of) {
        float lm = first ? 0.0f : g.lambda[t];
        if (green_project(P, xn_of, g.m0[t], g.m1[t], g.m2[t], alpha_tilde, gamma, lm) || first) g.lambda[t] = lm;
    });
}

template <int BLOCK, bool DAMPED>
__global__ void __launch_bounds__(BLOCK) k_neohookean_clusters(tet_group_dev g, cluster_dev cl, pos4* xi,
                                                               const pos4* __restrict__ xn, uint32_t begin,
                                                               uint32_t count, float inv_dt2, float beta_dt, int mode)
{
    run_cluster<BLOCK>(cl, xi, xn, begin, count, [&](uint32_t t, pos4 P[4], auto&& xn_of) {
        float2 lm = mode == kSolveFirst ? make_float2(0.0f, 0.0f) : reinterpret_cast<const float2*>(g.lambda)[t];
        neohookean_project<DAMPED>(P, xn_of, g.m0[t], g.m1[t], nh_m2(g, t), inv_dt2, beta_dt, lm);
        reinterpret_cast<float2*>(g.lambda)[t] = lm;
    });
}

// Warm-start displacement of the clusters of one color: every tet's gradients at the predicted
// positions xt, its displacement added to xi at once (clusters of a color share no particle, and
// one thread runs a cluster's tets in order, so the additions do not race).
__global__ void __launch_bounds__(128) k_neohookean_clusters_apply(tet_group_dev g, cluster_dev cl, pos4* xi,
                                                                   const pos4* __restrict__ xt, uint32_t begin,
                                                                   uint32_t count, float inv_dt2, int expl,
                                                                   float2 scale)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    uint32_t const c = begin + i;
    int4 const va = cl.v0[c], vb = cl.v1[c];
    for (uint32_t t = cl.off[c]; t < cl.off[c + 1]; ++t) {
        uint32_t const loc = cl.loc[t];
        int const id[4] = {slot_id(va, vb, loc & 0xffu), slot_id(va, vb, (loc >> 8) & 0xffu),
                           slot_id(va, vb, (loc >> 16) & 0xffu), slot_id(va, vb, loc >> 24)};
        pos4 const P[4] = {xt[id[0]], xt[id[1]], xt[id[2]], xt[id[3]]};
        float2 lm = reinterpret_cast<const float2*>(g.lambda)[t];
        v3 d[4];
        neohookean_displacement(P, g.m0[t], g.m1[t], nh_m2(g, t), inv_dt2, expl != 0, scale, lm, d);
        reinterpret_cast<float2*>(g.lambda)[t] = lm;
#pragma unroll
        for (int k = 0; k < 4; ++k) add_displacement(&xi[id[k]], d[k]);
    }
}

// ---------------------------------------------------------------- hex-cell clusters

// PREFETCH: every tet's material and multipliers are loaded before the first projection (one
// memory round trip, ~240 VGPRs, 2 waves per SIMD: for launches too small to fill the chip, where
// latency rules); otherwise each tet's are loaded just before it is projected (fewer registers,
// more waves in flight: for launches that fill the chip, where bandwidth rules).
// FIRST: the first iteration of a substep (multipliers start at zero). A compile-time switch: a
// multiplier load under a run-time condition sat in a branch, after which the compiler drained the
// memory queue, serializing the prefetch of the six tets' data into several round trips.
template <int BLOCK, bool PREFETCH, int MIN_WAVES, bool DAMPED, bool FIRST>
__global__ void __launch_bounds__(BLOCK, MIN_WAVES) k_neohookean_hex(tet_group_dev g, cluster_dev cl, pos4* xi,
                                                                     const pos4* __restrict__ xn, uint32_t begin,
                                                                     uint32_t count, uint32_t tbase, xcd_split sp,
                                                                     float inv_dt2, float beta_dt)
{
    uint32_t const x = blockIdx.x % kXcds, local = (blockIdx.x / kXcds) * BLOCK + threadIdx.x;
    if (local >= sp.off[x + 1] - sp.off[x]) return;
    uint32_t const i = sp.off[x] + local;
    int4 const va = lane_load(cl.v0 + begin, i), vb = lane_load(cl.v1 + begin, i);
    int const ids[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
    constexpr int NP = PREFETCH ? kHexTets : 1;
    float4 A[NP], B[NP];
    float2 Cm[NP];
    float2 L[NP];
    // tet k of the color's clusters is one contiguous run: its start is uniform (scalar registers),
    // the lane's offset in it a 32-bit byte offset 
    auto load = [&](int k, int slot) {
        std::size_t const t = std::size_t(tbase) + std::size_t(uint32_t(k)) * count;
        A[slot] = lane_load(g.m0 + t, i);
        B[slot] = lane_load(g.m1 + t, i);
        Cm[slot] = lane_load(reinterpret_cast<const float2*>(g.m2) + t, i);
        L[slot] = FIRST ? make_float2(0.0f, 0.0f) : lane_load(reinterpret_cast<const float2*>(g.lambda) + t, i);
    };
    auto store = [&](int k, int slot) {
        lane_store(reinterpret_cast<float2*>(g.lambda) + (std::size_t(tbase) + std::size_t(uint32_t(k)) * count), i, L[slot]);
    };
    if (PREFETCH) {
#pragma unroll
        for (int k = 0; k < kHexTets; ++k) load(k, k);
    }
    pos4 P[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) P[k] = xi[ids[k]];
    if (PREFETCH) loads_issued();
#pragma unroll
    for (int k = 0; k < kHexTets; ++k) {
        int const m = PREFETCH ? k : 0;
        if (!PREFETCH) load(k, 0);
        int const s0 = kHexSlots[k][0], s1 = kHexSlots[k][1], s2 = kHexSlots[k][2], s3 = kHexSlots[k][3];
        pos4 Q[4] = {P[s0], P[s1], P[s2], P[s3]};
        int const id[4] = {ids[s0], ids[s1], ids[s2], ids[s3]};
        auto xn_of = [&](int q) { return xn[id[q]]; };
        neohookean_project<DAMPED>(Q, xn_of, A[m], B[m], Cm[m], inv_dt2, beta_dt, L[m]);
        P[s0] = Q[0];
        P[s1] = Q[1];
        P[s2] = Q[2];
        P[s3] = Q[3];
        if (!PREFETCH) store(k, 0);
    }
    if (PREFETCH) {
#pragma unroll
        for (int k = 0; k < kHexTets; ++k) store(k, k);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) xi[ids[k]] = P[k];
}

// Warm-start displacement of the hex clusters of one color (gradients at the predicted positions
// xt, the 6 tets' displacements summed per particle, then added to xi).
template <int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_neohookean_hex_apply(tet_group_dev g, cluster_dev cl, pos4* xi,
                                                                const pos4* __restrict__ xt, uint32_t begin,
                                                                uint32_t count, uint32_t tbase, float inv_dt2, int expl,
                                                                float2 scale)
{
    uint32_t const i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= count) return;
    uint32_t const c = begin + i;
    int4 const va = cl.v0[c], vb = cl.v1[c];
    int const ids[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
    pos4 P[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) P[k] = xt[ids[k]];
    v3 D[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) D[k] = mk(0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < kHexTets; ++k) {
        uint32_t const t = tbase + uint32_t(k) * count + i;
        int const s0 = kHexSlots[k][0], s1 = kHexSlots[k][1], s2 = kHexSlots[k][2], s3 = kHexSlots[k][3];
        pos4 const Q[4] = {P[s0], P[s1], P[s2], P[s3]};
        float2 lm = reinterpret_cast<const float2*>(g.lambda)[t];
        v3 d[4];
        neohookean_displacement(Q, g.m0[t], g.m1[t], nh_m2(g, t), inv_dt2, expl != 0, scale, lm, d);
        reinterpret_cast<float2*>(g.lambda)[t] = lm;
        D[s0] = D[s0] + d[0];
        D[s1] = D[s1] + d[1];
        D[s2] = D[s2] + d[2];
        D[s3] = D[s3] + d[3];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) add_displacement(&xi[ids[k]], D[k]);
}

// Constraint values of a neo-Hookean tet at edges e (the quantities nh_deviatoric and
// nh_hydrostatic return, without their gradients).
__device__ __forceinline__ float2 nh_values(v3 const e[3], nh_rest const& q, float gamma0)
{
    float const g00 = fdot(e[0], e[0]), g11 = fdot(e[1], e[1]), g22 = fdot(e[2], e[2]);
    float const g01 = fdot(e[0], e[1]), g02 = fdot(e[0], e[2]), g12 = fdot(e[1], e[2]);
    float const off = fmaf(q.q01, g01, fmaf(q.q02, g02, q.q12 * g12));
    float const c2 = fmaf(q.q00, g00, fmaf(q.q11, g11, fmaf(q.q22, g22, 2.0f * off)));
    return make_float2(hw_sqrt(fmaxf(c2, 0.0f)), fmaf(q.detr, fdot(e[0], fcross(e[1], e[2])), -gamma0));
}

// Warm-start displacements of every hex cluster of a group in one launch (all colors): nothing
// moves during the launch, so every gradient is taken at the predicted positions xi (a copy of
// them, or the working positions themselves before any displacement is added). Workgroup b (64
// rows) runs the clusters cinfo[2b].w + t, t < cinfo[2b + 1].x, of one color (cinfo[2b]: the first
// one's index in its color, the color's cluster count and first constraint); the summed
// displacement of the cluster's slot k goes to disp[k * nrows + 64 b + t] (one coalesced store per
// slot).
// MODE kWarmFeatures (capture) and kWarmLearned also form the cluster's network features (see
// launch_hex_warm_start) and store the multipliers they start from as the history; kWarmFeatures
// writes the features to raw[row], kWarmLearned runs the network on the workgroup's 64 rows (two
// 32-row matrix-core tiles, rows staged through LDS) and adds its predicted change to the
// multipliers before the displacement.
constexpr int kWarmPlain = kWarmNetNone, kWarmFeatures = kWarmNetFeatures, kWarmLearned = kWarmNetLearned;
constexpr int kFeatures = 39;  // used network inputs of a hex cluster

template <int MODE>
__device__ __forceinline__ void hex_warm_disp(tet_group_dev const& g, cluster_dev const& cl, const pos4* xi,
                                              const uint4* __restrict__ cinfo, uint32_t nrows, float inv_dt2,
                                              int expl, float2 scale, float4* __restrict__ disp,
                                              warm_net_dev const& net)
{
    uint4 const info = cinfo[2 * blockIdx.x];
    uint32_t const used = cinfo[2 * blockIdx.x + 1].x;
    if (MODE != kWarmLearned && threadIdx.x >= used) return;
    if (used == 0) return;  // a padding workgroup (uniform)
    bool const active = threadIdx.x < used;
    uint32_t const r = blockIdx.x * 64u + threadIdx.x;
    // inactive lanes (learned mode only) run the network on zero rows and touch no memory of theirs
    uint32_t const i = info.x + (active ? threadIdx.x : 0u), count = info.y, tbase = info.z;
    uint32_t const ci = info.w + (active ? threadIdx.x : 0u);
    int4 const va = cl.v0[ci], vb = cl.v1[ci];
    int const ids[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
    // every tet's material and multipliers are loaded before the first multiplier is stored back
    float4 A[kHexTets], B[kHexTets];
    float2 C[kHexTets], L[kHexTets], H[kHexTets];
#pragma unroll
    for (int k = 0; k < kHexTets; ++k) {
        uint32_t const t = tbase + uint32_t(k) * count + i;
        A[k] = g.m0[t];
        B[k] = g.m1[t];
        C[k] = nh_m2(g, t);
        L[k] = reinterpret_cast<const float2*>(g.lambda)[t];
        if (MODE != kWarmPlain) H[k] = net.hist[t];
    }
    pos4 P[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) P[k] = xi[ids[k]];
    if (MODE != kWarmPlain) {
        // features: alpha~ lambda_prev (12), alpha~ lambda_prev2 (12), C at the predicted positions
        // (12), log alpha~ of tet 0 (deviatoric, hydrostatic), the body-size feature
        float f[kFeatures];
#pragma unroll
        for (int k = 0; k < kHexTets; ++k) {
            int const s0 = kHexSlots[k][0], s1 = kHexSlots[k][1], s2 = kHexSlots[k][2], s3 = kHexSlots[k][3];
            v3 const e[3] = {sub(P[s0], P[s3]), sub(P[s1], P[s3]), sub(P[s2], P[s3])};
            float2 const cv = nh_values(e, load_nh(A[k], B[k]), C[k].y);
            float const atd = B[k].w * inv_dt2, ath = C[k].x * inv_dt2;
            f[2 * k] = atd * L[k].x;
            f[2 * k + 1] = ath * L[k].y;
            f[12 + 2 * k] = atd * H[k].x;
            f[13 + 2 * k] = ath * H[k].y;
            f[24 + 2 * k] = cv.x;
            f[25 + 2 * k] = cv.y;
        }
        f[36] = logf(B[0].w * inv_dt2);
        f[37] = logf(C[0].x * inv_dt2);
        f[38] = net.body_size[tbase + i];
        if (active) {
#pragma unroll
            for (int k = 0; k < kHexTets; ++k) net.hist[tbase + uint32_t(k) * count + i] = L[k];
        }
        if (MODE == kWarmFeatures) {
            float* o = net.raw + std::size_t(r) * mlp::kMaxInputs;
#pragma unroll
            for (int m = 0; m < mlp::kMaxInputs; ++m) o[m] = m < kFeatures ? f[m] : 0.0f;
        } else {
            // the network corrects carried-over multipliers: a cluster whose multipliers or their
            // history are all zero (the first two substeps after a reset) keeps the previous start
            bool carried = false, history = false;
#pragma unroll
            for (int m = 0; m < 2 * kHexTets; ++m) {
                carried = carried || f[m] != 0.0f;
                history = history || f[2 * kHexTets + m] != 0.0f;
            }
            using mlp::bf16x8;
            __shared__ bf16x8 rows_lds[64 * mlp::kIn / 8];  // [row][48] BF16 inputs, then [row][12] FP32 outputs
            __shared__ float bias_lds[mlp::kBiasTotal];
            for (int m = threadIdx.x; m < int(mlp::kBiasTotal); m += 64) bias_lds[m] = net.bias[m];
            {
                bf16x8 v[mlp::kIn / 8];
#pragma unroll
                for (int m = 0; m < mlp::kIn; ++m)
                    v[m / 8][m % 8] = static_cast<mlp::bf16>(
                        active && m < kFeatures ? (f[m] - net.norm->mean[m]) * net.norm->inv_std[m] : 0.0f);
#pragma unroll
                for (int m = 0; m < mlp::kIn / 8; ++m) rows_lds[threadIdx.x * (mlp::kIn / 8) + m] = v[m];
            }
            __syncthreads();
            int const lane = threadIdx.x, h = lane >> 5, c = lane & 31;
            // the two 32-row tiles one after the other, not unrolled (each pass reads the weights
            // again, from L2): half the accumulators and activations live at a time. A tile's
            // outputs ([row][12] FP32) overwrite only inputs of rows already read (the workgroup is
            // one wave: tile t's 32 rows of inputs are in registers before its outputs are written;
            // its outputs occupy bytes [1536 t, 1536 t + 1536), tile 1's inputs start at 3072).
            float* out = reinterpret_cast<float*>(rows_lds);
#pragma unroll 1
            for (int t2 = 0; t2 < 2; ++t2) {
                bf16x8 xin[1][mlp::kQ1];
#pragma unroll
                for (int q = 0; q < mlp::kQ1; ++q) xin[0][q] = rows_lds[(32 * t2 + c) * (mlp::kIn / 8) + 2 * q + h];
                mlp::f32x16 yt[1];
                mlp::forward_tiles<1>(reinterpret_cast<const bf16x8*>(net.pack), bias_lds, xin, lane, yt);
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    int const o = mlp::acc_unit(j, h);
                    if (o < 2 * kHexTets) out[(32 * t2 + c) * (2 * kHexTets) + o] = yt[0][j];
                }
            }
            __syncthreads();
            if (!active) return;
            // the material and the positions again (the same values): read back after the network
            // instead of held across it, so that the network runs with the registers it needs
#pragma unroll
            for (int k = 0; k < kHexTets; ++k) {
                uint32_t const t = tbase + uint32_t(k) * count + i;
                A[k] = g.m0[t];
                B[k] = g.m1[t];
                C[k] = nh_m2(g, t);
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) P[k] = xi[ids[k]];
            // the predicted change of alpha~ lambda over the substep, back to multipliers
            if (carried && history) {
#pragma unroll
                for (int k = 0; k < kHexTets; ++k) {
                    float const yd = out[threadIdx.x * (2 * kHexTets) + 2 * k] * net.norm->out_scale[2 * k];
                    float const yh = out[threadIdx.x * (2 * kHexTets) + 2 * k + 1] * net.norm->out_scale[2 * k + 1];
                    L[k].x += yd / (B[k].w * inv_dt2);
                    L[k].y += yh / (C[k].x * inv_dt2);
                }
            }
        }
    }
    v3 D[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) D[k] = mk(0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < kHexTets; ++k) {
        int const s0 = kHexSlots[k][0], s1 = kHexSlots[k][1], s2 = kHexSlots[k][2], s3 = kHexSlots[k][3];
        pos4 const Q[4] = {P[s0], P[s1], P[s2], P[s3]};
        v3 d[4];
        neohookean_displacement(Q, A[k], B[k], C[k], inv_dt2, expl != 0, scale, L[k], d);
        D[s0] = D[s0] + d[0];
        D[s1] = D[s1] + d[1];
        D[s2] = D[s2] + d[2];
        D[s3] = D[s3] + d[3];
    }
#pragma unroll
    for (int k = 0; k < kHexTets; ++k) reinterpret_cast<float2*>(g.lambda)[tbase + uint32_t(k) * count + i] = L[k];
#pragma unroll
    for (int k = 0; k < 8; ++k) disp[std::size_t(k) * nrows + r] = make_float4(D[k].x, D[k].y, D[k].z, 0.0f);
}

template <int MODE>
__global__ void __launch_bounds__(64) k_hex_warm_disp(tet_group_dev g, cluster_dev cl, const pos4* __restrict__ xi,
                                                      const uint4* __restrict__ cinfo, uint32_t nrows, float inv_dt2,
                                                      int expl, float2 scale, float4* __restrict__ disp,
                                                      warm_net_dev net)
{
    hex_warm_disp<MODE>(g, cl, xi, cinfo, nrows, inv_dt2, expl, scale, disp, net);
}

// The learned variant, held to at most 256 registers a lane (2 waves per SIMD); its positions are
// read through a pointer without restrict so that the reads after the network are real loads.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
k_hex_warm_learned(tet_group_dev g, cluster_dev cl, const pos4* xi, const uint4* __restrict__ cinfo, uint32_t nrows,
                   float inv_dt2, int expl, float2 scale, float4* __restrict__ disp, warm_net_dev net)
{
    hex_warm_disp<kWarmLearned>(g, cl, xi, cinfo, nrows, inv_dt2, expl, scale, disp, net);
}

// Training rows of a hex group's captured substep: for j < rows, cluster ci = offset + j * stride,
// its row rowof[ci] of raw (the features at the substep start) and, as targets, the change of
// alpha~ lambda of its 12 multipliers over the substep (the final multipliers against feature
// values 0..11); a row holding a non-finite value is stored as zeros.
__global__ void k_hex_capture(tet_group_dev g, const uint4* __restrict__ cinfo, const uint32_t* __restrict__ rowof,
                              const float* __restrict__ raw, uint32_t stride, uint32_t offset, float inv_dt2,
                              float* __restrict__ ds_x, float* __restrict__ ds_t, uint64_t base, uint32_t rows)
{
    uint32_t const j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= rows) return;
    uint32_t const row = rowof[offset + j * stride];
    uint4 const info = cinfo[2 * (row / 64)];
    uint32_t const i = info.x + row % 64, count = info.y, tbase = info.z;
    const float* f = raw + std::size_t(row) * mlp::kMaxInputs;
    float t[2 * kHexTets];
    bool ok = true;
#pragma unroll
    for (int k = 0; k < kHexTets; ++k) {
        uint32_t const tk = tbase + uint32_t(k) * count + i;
        float2 const lf = reinterpret_cast<const float2*>(g.lambda)[tk];
        t[2 * k] = g.m1[tk].w * inv_dt2 * lf.x - f[2 * k];
        t[2 * k + 1] = nh_m2(g, tk).x * inv_dt2 * lf.y - f[2 * k + 1];
        ok = ok && isfinite(t[2 * k]) && isfinite(t[2 * k + 1]);
    }
#pragma unroll
    for (int m = 0; m < kFeatures; ++m) ok = ok && isfinite(f[m]);
    std::size_t const o = base + j;
#pragma unroll
    for (int m = 0; m < mlp::kMaxInputs; ++m) ds_x[o * mlp::kMaxInputs + m] = ok ? f[m] : 0.0f;
#pragma unroll
    for (int m = 0; m < mlp::kMaxOutputs; ++m) ds_t[o * mlp::kMaxOutputs + m] = ok && m < 2 * kHexTets ? t[m] : 0.0f;
}

// x_p += the displacements of p's cluster slots, in FP64, in the order of the list (execution
// order of the clusters: the order of the colored pass).
__global__ void k_gather_disp(const uint32_t* __restrict__ off, const uint32_t* __restrict__ ent,
                              const float4* __restrict__ disp, pos4* __restrict__ xi, uint32_t n)
{
    uint32_t const p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    uint32_t const b = off[p], e = off[p + 1];
    if (b == e) return;
    pos4 x = xi[p];
    for (uint32_t j = b; j < e; ++j) {
        float4 const d = disp[ent[j]];
        x.x += double(d.x);
        x.y += double(d.y);
        x.z += double(d.z);
    }
    xi[p] = x;
}

// The same with the list as a dense row of 8 slot indices per particle (unused: 0xffffffff), when
// no particle is in more than 8 clusters (hex lattices): the 8 loads of a row go out together and
// the unused ones add an exact 0.
// With surface_of (particle -> surface vertex or -1), the first iteration's contact projections of
// the surface vertices follow in the same thread, as k_contact(first) would run them next.
// With prow, thread r handles particle prow[r] (rows [0, n); padding rows hold 0xffffffff).
__global__ void k_gather_disp8(const uint4* __restrict__ ent, const float4* __restrict__ disp, pos4* __restrict__ xi,
                               uint32_t n, const int* __restrict__ surface_of, contact_dev c, float c_at,
                               const uint32_t* __restrict__ prow)
{
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    if (prow) {
        p = prow[p];
        if (p == 0xffffffffu) return;
    }
    uint4 const a = ent[2 * std::size_t(p)], b = ent[2 * std::size_t(p) + 1];
    uint32_t const e[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    int const sv = surface_of ? surface_of[p] : -1;
    if (e[0] == 0xffffffffu && sv < 0) return;
    float4 d[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) d[m] = disp[e[m] != 0xffffffffu ? e[m] : 0u];
    pos4 x = xi[p];
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        bool const ok = e[m] != 0xffffffffu;
        x.x += ok ? double(d[m].x) : 0.0;
        x.y += ok ? double(d[m].y) : 0.0;
        x.z += ok ? double(d[m].z) : 0.0;
    }
    if (sv >= 0) contact_vertex_at(c, x, uint32_t(sv), c_at, true);
    xi[p] = x;
}

// FIRST: the first iteration of a substep, a compile-time switch for the reason given at
// k_neohookean_hex.
template <int BLOCK, bool FIRST>
__global__ void __launch_bounds__(BLOCK) k_green_hex(tet_group_dev g, cluster_dev cl, pos4* xi,
                                                     const pos4* __restrict__ xn, uint32_t begin, uint32_t count,
                                                     uint32_t tbase, xcd_split sp, float alpha_tilde, float gamma)
{
    uint32_t const x = blockIdx.x % kXcds, local = (blockIdx.x / kXcds) * BLOCK + threadIdx.x;
    if (local >= sp.off[x + 1] - sp.off[x]) return;
    uint32_t const i = sp.off[x] + local;
    uint32_t const c = begin + i;
    int4 const va = cl.v0[c], vb = cl.v1[c];
    int const ids[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
    float4 A[kHexTets], B[kHexTets], Cm[kHexTets];
    float L[kHexTets];
#pragma unroll
    for (int k = 0; k < kHexTets; ++k) {
        uint32_t const t = tbase + uint32_t(k) * count + i;
        A[k] = g.m0[t];
        B[k] = g.m1[t];
        Cm[k] = g.m2[t];
        L[k] = FIRST ? 0.0f : g.lambda[t];
    }
    pos4 P[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) P[k] = xi[ids[k]];
#pragma unroll
    for (int k = 0; k < kHexTets; ++k) {
        int const s0 = kHexSlots[k][0], s1 = kHexSlots[k][1], s2 = kHexSlots[k][2], s3 = kHexSlots[k][3];
        pos4 Q[4] = {P[s0], P[s1], P[s2], P[s3]};
        int const id[4] = {ids[s0], ids[s1], ids[s2], ids[s3]};
        auto xn_of = [&](int q) { return xn[id[q]]; };
        // on the early-out the multiplier stays as loaded (0 on the first iteration)
        green_project(Q, xn_of, A[k], B[k], Cm[k], alpha_tilde, gamma, L[k]);
        P[s0] = Q[0];
        P[s1] = Q[1];
        P[s2] = Q[2];
        P[s3] = Q[3];
    }
#pragma unroll
    for (int k = 0; k < kHexTets; ++k) g.lambda[tbase + uint32_t(k) * count + i] = L[k];
#pragma unroll
    for (int k = 0; k < 8; ++k) xi[ids[k]] = P[k];
}

// ---------------------------------------------------------------- distance constraint

// distance_constraint.cpp:24-53 (no guard against zero length, as there).
__global__ void __launch_bounds__(256) k_distance(distance_group_dev g, pos4* xi, const pos4* __restrict__ xn,
                                                  uint32_t begin, uint32_t count, float alpha_tilde, float gamma,
                                                  int first)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    uint32_t const t = begin + i;
    uint2 const id = g.idx[t];
    float const d = g.rest[t];
    float const lm = first ? 0.0f : g.lambda[t];
    pos4 P1 = xi[id.x], P2 = xi[id.y];
    v3 const diff = sub(P1, P2);
    float const length = sqrtf(dot(diff, diff));
    v3 const n = (1.0f / length) * diff;
    float const C = length - d;
    float gdd = 0.0f;
    if (gamma != 0.0f) gdd = dot(n, sub(P1, xn[id.x])) - dot(n, sub(P2, xn[id.y]));
    float const w1 = wof(P1), w2 = wof(P2);
    float const dl = (-(C + alpha_tilde * lm) + gamma * gdd) / ((1.0f + gamma) * (w1 + w2) + alpha_tilde);
    g.lambda[t] = lm + dl;
    add_to(P1, (w1 * dl) * n);
    add_to(P2, -(w2 * dl) * n);
    xi[id.x] = P1;
    xi[id.y] = P2;
}

// ---------------------------------------------------------------- contacts

// One thread per surface vertex: contacts against every SDF, in SDF order, from the positions at
// the start of the frame (bvh_model.cpp:72-95, contact_handler.cpp:39-52). A vertex keeps at most
// c.slots contacts; more are counted in c.overflow.
__global__ void k_detect(contact_dev c, const pos4* __restrict__ x, const sdf_dev* __restrict__ sdfs, uint32_t nsdf)
{
    uint32_t const s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= c.S) return;
    pos4 const p = x[c.surf[s]];
    uint32_t cnt = 0;
    for (uint32_t k = 0; k < nsdf; ++k) {
        double q[3], n[3];
        if (!sdf_contact(sdfs[k], p, q, n)) continue;
        if (cnt == c.slots) {
            atomicAdd(c.overflow, 1u);
            continue;
        }
        store_contact(c, s, cnt++, k, q, n);
    }
    c.count[s] = cnt;
}

// collision_constraint.cpp:21-41, all contacts of one particle in SDF order by one thread.
__global__ void k_snapshot_surface(const uint32_t* __restrict__ surf, const pos4* __restrict__ xi,
                                   pos4* __restrict__ snap, uint32_t S)
{
    uint32_t const s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < S) snap[s] = xi[surf[s]];
}

__global__ void k_contact(contact_dev c, pos4* xi, float alpha_tilde, int first)
{
    uint32_t const s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= c.S) return;
    if (c.count[s] == 0) return;
    uint32_t const vi = c.surf[s];
    pos4 P = xi[vi];
    contact_vertex_at(c, P, s, alpha_tilde, first != 0);
    xi[vi] = P;
}

// ---------------------------------------------------------------- reductions (FP64)

template <int BLOCK>
__device__ __forceinline__ double block_sum(double v)
{
    static_assert(BLOCK % 64 == 0, "wave64 blocks");
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    __shared__ double part[BLOCK / 64];
    int const lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) part[wave] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < BLOCK / 64; ++i) r += part[i];
    __syncthreads();
    return r;
}

constexpr int kRedBlock = 256;

__global__ void __launch_bounds__(kRedBlock) k_green_residual(tet_group_dev g, const pos4* __restrict__ x,
                                                              uint32_t begin, uint32_t count, float alpha_tilde,
                                                              double* partial)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    double h2 = 0.0;
    if (i < count) {
        uint32_t const t = begin + i;
        int4 const id = g.idx[t];
        float4 const c = g.m2[t];
        pos4 const p3 = x[id.w];
        v3 f[4];
        float const C = green_core(sub(x[id.x], p3), sub(x[id.y], p3), sub(x[id.z], p3), load_rows(g.m0[t], g.m1[t], c),
                                   c.y, c.z, c.w, f);
        double const h = double(C) + double(alpha_tilde) * double(g.lambda[t]);
        h2 = h * h;
    }
    double const s = block_sum<kRedBlock>(h2);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// ||F||_F^2 and det F - gamma0 of neo-Hookean tet id at positions x, in FP64 from the FP64 edge
// vectors and the FP32 rest data (the forms at nh_rest).
__device__ __forceinline__ void nh_constraints_f64(pos4 p0, pos4 p1, pos4 p2, pos4 p3, nh_rest const& q, float gamma0,
                                                   double& f2, double& det_minus)
{
    double const e[3][3] = {{p0.x - p3.x, p0.y - p3.y, p0.z - p3.z},
                            {p1.x - p3.x, p1.y - p3.y, p1.z - p3.z},
                            {p2.x - p3.x, p2.y - p3.y, p2.z - p3.z}};
    auto d = [&](int m, int n) { return e[m][0] * e[n][0] + e[m][1] * e[n][1] + e[m][2] * e[n][2]; };
    f2 = double(q.q00) * d(0, 0) + double(q.q11) * d(1, 1) + double(q.q22) * d(2, 2) +
         2.0 * (double(q.q01) * d(0, 1) + double(q.q02) * d(0, 2) + double(q.q12) * d(1, 2));
    f2 = f2 > 0.0 ? f2 : 0.0;
    double const vol = e[0][0] * (e[1][1] * e[2][2] - e[1][2] * e[2][1]) +
                       e[0][1] * (e[1][2] * e[2][0] - e[1][0] * e[2][2]) +
                       e[0][2] * (e[1][0] * e[2][1] - e[1][1] * e[2][0]);
    det_minus = double(q.detr) * vol - double(gamma0);
}

__device__ __forceinline__ void nh_constraints_f64(const pos4* __restrict__ x, int4 id, nh_rest const& q, float gamma0,
                                                   double& f2, double& det_minus)
{
    nh_constraints_f64(x[id.x], x[id.y], x[id.z], x[id.w], q, gamma0, f2, det_minus);
}

// h^2 of both constraints of neo-Hookean tet t at positions P0..P3 (FP64).
__device__ __forceinline__ double nh_residual2(tet_group_dev const& g, uint32_t t, pos4 p0, pos4 p1, pos4 p2, pos4 p3,
                                               float inv_dt2)
{
    float4 const b = g.m1[t];
    float2 const c = nh_m2(g, t);
    double cd, ch;
    nh_constraints_f64(p0, p1, p2, p3, load_nh(g.m0[t], b), c.y, cd, ch);
    float2 const lm = reinterpret_cast<const float2*>(g.lambda)[t];
    cd = sqrt(cd);
    double const hd = cd + double(b.w) * double(inv_dt2) * double(lm.x);
    double const hh = ch + double(c.x) * double(inv_dt2) * double(lm.y);
    return hd * hd + hh * hh;
}

// The same over a hex-cluster group, one thread per row of the all-color rows (a cluster of any
// color, or padding): the cluster's eight particles are read once for its six tets. One 64-row
// workgroup per record pair, so that workgroup b runs on the XCD of its rows' region (b mod 8).
constexpr int kHexRedBlock = 64;
__global__ void __launch_bounds__(kHexRedBlock) k_neohookean_hex_residual(tet_group_dev g, cluster_dev cl,
                                                                       const pos4* __restrict__ x,
                                                                       const uint4* __restrict__ cinfo,
                                                                       uint32_t nrows, float inv_dt2,
                                                                       double* partial)
{
    // the workgroup's run of clusters, as at k_hex_warm_disp
    uint4 const info = cinfo[2 * blockIdx.x];
    uint32_t const used = cinfo[2 * blockIdx.x + 1].x;
    double h2 = 0.0;
    if (threadIdx.x < used) {
        uint32_t const ci = info.w + threadIdx.x, i = info.x + threadIdx.x;
        int4 const va = cl.v0[ci], vb = cl.v1[ci];
        pos4 const P[8] = {x[va.x], x[va.y], x[va.z], x[va.w], x[vb.x], x[vb.y], x[vb.z], x[vb.w]};
#pragma unroll
        for (int k = 0; k < kHexTets; ++k)
            h2 += nh_residual2(g, info.z + uint32_t(k) * info.y + i, P[kHexSlots[k][0]], P[kHexSlots[k][1]],
                               P[kHexSlots[k][2]], P[kHexSlots[k][3]], inv_dt2);
    }
    double const s = block_sum<kHexRedBlock>(h2);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void __launch_bounds__(kRedBlock) k_neohookean_residual(tet_group_dev g, const pos4* __restrict__ x,
                                                                   uint32_t begin, uint32_t count, float inv_dt2,
                                                                   double* partial)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    double h2 = 0.0;
    if (i < count) {
        uint32_t const t = begin + i;
        int4 const id = g.idx[t];
        h2 = nh_residual2(g, t, x[id.x], x[id.y], x[id.z], x[id.w], inv_dt2);
    }
    double const s = block_sum<kRedBlock>(h2);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void __launch_bounds__(kRedBlock) k_distance_residual(distance_group_dev g, const pos4* __restrict__ x,
                                                                 uint32_t begin, uint32_t count, float alpha_tilde,
                                                                 double* partial)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    double h2 = 0.0;
    if (i < count) {
        uint32_t const t = begin + i;
        uint2 const id = g.idx[t];
        pos4 const a = x[id.x], b = x[id.y];
        double const dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
        double const h =
            (sqrt(dx * dx + dy * dy + dz * dz) - double(g.rest[t])) + double(alpha_tilde) * double(g.lambda[t]);
        h2 = h * h;
    }
    double const s = block_sum<kRedBlock>(h2);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void __launch_bounds__(kRedBlock) k_particle_energy(const pos4* __restrict__ x, const float4* __restrict__ v,
                                                               const float* __restrict__ mass, uint32_t n, float gx,
                                                               float gy, float gz, int force, double* partial)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    double ke = 0, pe = 0, px = 0, py = 0, pz = 0;
    if (i < n) {
        double const m = mass[i];
        pos4 const p = x[i];
        float4 const u = v[i];
        ke = 0.5 * m * (double(u.x) * u.x + double(u.y) * u.y + double(u.z) * u.z);
        pe = -(force ? 1.0 : m) * (double(gx) * p.x + double(gy) * p.y + double(gz) * p.z);
        px = m * u.x;
        py = m * u.y;
        pz = m * u.z;
    }
    double r[5] = {block_sum<kRedBlock>(ke), block_sum<kRedBlock>(pe), block_sum<kRedBlock>(px),
                   block_sum<kRedBlock>(py), block_sum<kRedBlock>(pz)};
    if (threadIdx.x == 0) {
        double* o = partial + 6 * blockIdx.x;
        o[0] = r[0];
        o[1] = r[1];
        o[2] = 0.0;
        o[3] = r[2];
        o[4] = r[3];
        o[5] = r[4];
    }
}

__global__ void __launch_bounds__(kRedBlock) k_green_energy(tet_group_dev g, const pos4* __restrict__ x, uint32_t count,
                                                            double* partial)
{
    uint32_t const t = blockIdx.x * blockDim.x + threadIdx.x;
    double e = 0.0;
    if (t < count) {
        int4 const id = g.idx[t];
        float4 const c = g.m2[t];
        pos4 const p3 = x[id.w];
        v3 f[4];
        e = green_core(sub(x[id.x], p3), sub(x[id.y], p3), sub(x[id.z], p3), load_rows(g.m0[t], g.m1[t], c), c.y, c.z,
                       c.w, f);
    }
    double const s = block_sum<kRedBlock>(e);
    if (threadIdx.x == 0) {
        double* o = partial + 6 * blockIdx.x;
        o[0] = o[1] = o[3] = o[4] = o[5] = 0.0;
        o[2] = s;
    }
}

__global__ void __launch_bounds__(kRedBlock) k_neohookean_energy(tet_group_dev g, const pos4* __restrict__ x,
                                                                 uint32_t count, double* partial)
{
    uint32_t const t = blockIdx.x * blockDim.x + threadIdx.x;
    double e = 0.0;
    if (t < count) {
        int4 const id = g.idx[t];
        float4 const b = g.m1[t];
        float2 const c = nh_m2(g, t);
        double ic, j;
        nh_constraints_f64(x, id, load_nh(g.m0[t], b), c.y, ic, j);
        // mu |V0| = 1 / m1.w, lambda |V0| = 1 / m2.x
        e = 0.5 / double(b.w) * (ic - 3.0) + 0.5 / double(c.x) * j * j;
    }
    double const s = block_sum<kRedBlock>(e);
    if (threadIdx.x == 0) {
        double* o = partial + 6 * blockIdx.x;
        o[0] = o[1] = o[3] = o[4] = o[5] = 0.0;
        o[2] = s;
    }
}

// ---------------------------------------------------------------- Jones-Plassmann coloring

__device__ __forceinline__ uint32_t hash32(uint32_t x)
{
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

// Priority of element t: (previous color, hash32(t)) -- higher first; ties are impossible because
// hash32 is a bijection on 32-bit indices.
__global__ void k_jp_keys(uint32_t n, const uint32_t* __restrict__ prev, uint64_t* __restrict__ key)
{
    uint32_t const t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    key[t] = (uint64_t(prev ? prev[t] : 0u) << 32) | hash32(t);
}

// An element whose key exceeds the keys of all its uncolored neighbours takes the smallest color
// unused by its colored neighbours. Over all rounds this equals sequential greedy coloring in
// descending key order: when an element is colored, exactly its higher-key neighbours are.
__global__ void k_jp_round(uint32_t n, uint32_t arity, const uint32_t* __restrict__ elem_off,
                           const uint32_t* __restrict__ verts, const uint32_t* __restrict__ inc_off,
                           const uint32_t* __restrict__ inc, const uint64_t* __restrict__ key,
                           const uint32_t* __restrict__ color_in, uint32_t* __restrict__ color_out, uint32_t* remaining,
                           uint32_t* overflow)
{
    uint32_t const t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    uint32_t const mine = color_in[t];
    if (mine != kUncolored) {
        color_out[t] = mine;
        return;
    }
    uint64_t const kt = key[t];
    uint64_t used[kMaxColors / 64] = {0, 0, 0, 0};
    size_t const a0 = elem_off ? elem_off[t] : size_t(t) * arity;
    size_t const a1 = elem_off ? elem_off[t + 1] : a0 + arity;
    for (size_t a = a0; a < a1; ++a) {
        uint32_t const v = verts[a];
        uint32_t const e1 = inc_off[v + 1];
        for (uint32_t e = inc_off[v]; e < e1; ++e) {
            uint32_t const u = inc[e];
            if (u == t) continue;
            uint32_t const cu = color_in[u];
            if (cu == kUncolored) {
                if (key[u] > kt) {
                    color_out[t] = kUncolored;
                    atomicAdd(remaining, 1u);
                    return;
                }
            } else if (cu < kMaxColors) {
                used[cu >> 6] |= (uint64_t(1) << (cu & 63));
            }
        }
    }
    uint32_t c = kMaxColors;
#pragma unroll
    for (int w = 0; w < int(kMaxColors / 64); ++w) {
        if (c == kMaxColors && ~used[w] != 0) c = uint32_t(w) * 64 + uint32_t(__builtin_ctzll(~used[w]));
    }
    if (c >= kMaxColors) {
        atomicAdd(overflow, 1u);
        c = kMaxColors - 1;
    }
    color_out[t] = c;
}

__global__ void k_fill_u32(uint32_t* p, uint32_t value, uint32_t n)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

}  // namespace

// ---------------------------------------------------------------- launchers

void launch_predict(hipStream_t s, pos4* xi, const pos4* xn, float4* v, uint32_t n, float gx, float gy, float gz,
                    int force, float dt, int block)
{
    if (n) k_predict<<<grid_for(n, block), block, 0, s>>>(xi, xn, v, n, gx, gy, gz, force, dt);
}

void launch_commit(hipStream_t s, const pos4* xi, pos4* xn, float4* v, uint32_t n, float dt, int block)
{
    if (n) k_commit<<<grid_for(n, block), block, 0, s>>>(xi, xn, v, n, dt);
}

void launch_commit_predict(hipStream_t s, pos4* xi, pos4* xn, float4* v, uint32_t n, float gx, float gy, float gz,
                           int force, float dt, int block, const uint32_t* prow, uint32_t nprows)
{
    if (prow && nprows)
        k_commit_predict<<<grid_for(nprows, kParticleRowBlock), kParticleRowBlock, 0, s>>>(xi, xn, v, nprows, gx, gy,
                                                                                          gz, force, dt, prow);
    else if (n)
        k_commit_predict<<<grid_for(n, block), block, 0, s>>>(xi, xn, v, n, gx, gy, gz, force, dt, nullptr);
}

void launch_green(hipStream_t s, tet_group_dev g, pos4* xi, const pos4* xn, uint32_t begin, uint32_t count,
                  float alpha_tilde, float gamma, int first, int block)
{
    if (count) k_green<<<grid_for(count, block), block, 0, s>>>(g, xi, xn, begin, count, alpha_tilde, gamma, first);
}

void launch_neohookean(hipStream_t s, tet_group_dev g, pos4* xi, const pos4* xn, uint32_t begin, uint32_t count,
                       float inv_dt2, float beta_dt, int mode, int block, float hyd_scale)
{
    if (!count) return;
    // the warm-start modes carry a scale in beta_dt and take no damping
    auto const kernel = mode < kApplyWarmStart && beta_dt != 0.0f ? k_neohookean<true> : k_neohookean<false>;
    kernel<<<grid_for(count, block), block, 0, s>>>(g, xi, xn, begin, count, inv_dt2, beta_dt, mode, hyd_scale);
}

void launch_distance(hipStream_t s, distance_group_dev g, pos4* xi, const pos4* xn, uint32_t begin, uint32_t count,
                     float alpha_tilde, float gamma, int first, int block)
{
    if (count)
        k_distance<<<grid_for(count, block), block, 0, s>>>(g, xi, xn, begin, count, alpha_tilde, gamma, first);
}

void launch_green_clusters(hipStream_t s, tet_group_dev g, cluster_dev cl, pos4* xi, const pos4* xn, uint32_t begin,
                           uint32_t count, float alpha_tilde, float gamma, int first, int block)
{
    if (!count) return;
    if (block <= 64)
        k_green_clusters<64><<<grid_for(count, 64), 64, 0, s>>>(g, cl, xi, xn, begin, count, alpha_tilde, gamma, first);
    else
        k_green_clusters<128><<<grid_for(count, 128), 128, 0, s>>>(g, cl, xi, xn, begin, count, alpha_tilde, gamma, first);
}

void launch_neohookean_clusters(hipStream_t s, tet_group_dev g, cluster_dev cl, pos4* xi, const pos4* xn,
                                uint32_t begin, uint32_t count, float inv_dt2, float beta_dt, int mode, int block,
                                float hyd_scale)
{
    if (!count) return;
    if (mode >= kApplyWarmStart) {
        k_neohookean_clusters_apply<<<grid_for(count, 128), 128, 0, s>>>(g, cl, xi, xn, begin, count, inv_dt2,
                                                                         mode == kApplyExplicit,
                                                                         make_float2(beta_dt, hyd_scale));
        return;
    }
    bool const damped = beta_dt != 0.0f;
    auto go = [&](auto kernel, int b) {
        kernel<<<grid_for(count, b), b, 0, s>>>(g, cl, xi, xn, begin, count, inv_dt2, beta_dt, mode);
    };
    if (block <= 64)
        damped ? go(k_neohookean_clusters<64, true>, 64) : go(k_neohookean_clusters<64, false>, 64);
    else
        damped ? go(k_neohookean_clusters<128, true>, 128) : go(k_neohookean_clusters<128, false>, 128);
}

void launch_neohookean_hex(hipStream_t s, tet_group_dev g, cluster_dev cl, pos4* xi, const pos4* xn, uint32_t begin,
                           uint32_t count, uint32_t tbase, xcd_split const& sp, float inv_dt2, float beta_dt, int mode,
                           int block, float hyd_scale)
{
    if (!count) return;
    if (mode >= kApplyWarmStart) {
        k_neohookean_hex_apply<64><<<grid_for(count, 64), 64, 0, s>>>(g, cl, xi, xn, begin, count, tbase, inv_dt2,
                                                                       mode == kApplyExplicit,
                                                                       make_float2(beta_dt, hyd_scale));
        return;
    }
    // block 64 / 128: material prefetched; kHexStreamed: 64 threads, material loaded per tet, at
    // least 3 waves per SIMD (2 with damping, which would spill at 3). Damping (beta != 0) takes the
    // variants that carry the xn differences.
    bool const damped = beta_dt != 0.0f, first = mode == kSolveFirst;
    auto go = [&](auto kernel, int b) {
        uint32_t most = 0;  // workgroups per XCD
        for (int x = 0; x < kXcds; ++x) most = std::max(most, uint32_t(grid_for(sp.off[x + 1] - sp.off[x], b)));
        if (most) kernel<<<most * kXcds, b, 0, s>>>(g, cl, xi, xn, begin, count, tbase, sp, inv_dt2, beta_dt);
    };
    if (block == kHexStreamed) {
        if (damped)
            first ? go(k_neohookean_hex<64, false, 2, true, true>, 64) : go(k_neohookean_hex<64, false, 2, true, false>, 64);
        else
            first ? go(k_neohookean_hex<64, false, 3, false, true>, 64)
                  : go(k_neohookean_hex<64, false, 3, false, false>, 64);
    } else if (block <= 64) {
        if (damped)
            first ? go(k_neohookean_hex<64, true, 1, true, true>, 64) : go(k_neohookean_hex<64, true, 1, true, false>, 64);
        else
            first ? go(k_neohookean_hex<64, true, 1, false, true>, 64) : go(k_neohookean_hex<64, true, 1, false, false>, 64);
    } else {
        if (damped)
            first ? go(k_neohookean_hex<128, true, 1, true, true>, 128)
                  : go(k_neohookean_hex<128, true, 1, true, false>, 128);
        else
            first ? go(k_neohookean_hex<128, true, 1, false, true>, 128)
                  : go(k_neohookean_hex<128, true, 1, false, false>, 128);
    }
}

void launch_green_hex(hipStream_t s, tet_group_dev g, cluster_dev cl, pos4* xi, const pos4* xn, uint32_t begin,
                      uint32_t count, uint32_t tbase, xcd_split const& sp, float alpha_tilde, float gamma, int first,
                      int block)
{
    if (!count) return;
    int const b = block <= 64 ? 64 : 128;
    uint32_t most = 0;  // workgroups per XCD
    for (int x = 0; x < kXcds; ++x) most = std::max(most, uint32_t(grid_for(sp.off[x + 1] - sp.off[x], b)));
    if (!most) return;
    auto go = [&](auto kernel) { kernel<<<most * kXcds, b, 0, s>>>(g, cl, xi, xn, begin, count, tbase, sp, alpha_tilde, gamma); };
    if (b == 64)
        first ? go(k_green_hex<64, true>) : go(k_green_hex<64, false>);
    else
        first ? go(k_green_hex<128, true>) : go(k_green_hex<128, false>);
}

void launch_detect(hipStream_t s, contact_dev c, const pos4* x, const sdf_dev* sdfs, uint32_t nsdf, int block)
{
    if (c.S) k_detect<<<grid_for(c.S, block), block, 0, s>>>(c, x, sdfs, nsdf);
}

void launch_snapshot_surface(hipStream_t s, const uint32_t* surf, const pos4* xi, pos4* snap, uint32_t S)
{
    if (S) k_snapshot_surface<<<grid_for(S, 256), 256, 0, s>>>(surf, xi, snap, S);
}

void launch_contact(hipStream_t s, contact_dev c, pos4* xi, float alpha_tilde, int first, int block)
{
    if (c.S) k_contact<<<grid_for(c.S, block), block, 0, s>>>(c, xi, alpha_tilde, first);
}

void launch_green_residual(hipStream_t s, tet_group_dev g, const pos4* x, uint32_t begin, uint32_t count,
                           float alpha_tilde, double* partial, int)
{
    if (count) k_green_residual<<<grid_for(count, kRedBlock), kRedBlock, 0, s>>>(g, x, begin, count, alpha_tilde, partial);
}

void launch_neohookean_residual(hipStream_t s, tet_group_dev g, const pos4* x, uint32_t begin, uint32_t count,
                                float inv_dt2, double* partial, int)
{
    if (count)
        k_neohookean_residual<<<grid_for(count, kRedBlock), kRedBlock, 0, s>>>(g, x, begin, count, inv_dt2, partial);
}

__global__ void __launch_bounds__(256) k_copy_spans(copy_spans sp)
{
    uint64_t const tid = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x, stride = uint64_t(gridDim.x) * blockDim.x;
    for (int k = 0; k < sp.n; ++k) {
        uint64_t const words = sp.bytes[k] / 16;
        uint4* d = static_cast<uint4*>(sp.dst[k]);
        const uint4* s = static_cast<const uint4*>(sp.src[k]);
        for (uint64_t i = tid; i < words; i += stride) d[i] = s[i];
        uint64_t const tail = (sp.bytes[k] - words * 16) / 4;  // the last < 16 bytes, 4 at a time
        if (tid < tail)
            static_cast<uint32_t*>(sp.dst[k])[words * 4 + tid] = static_cast<const uint32_t*>(sp.src[k])[words * 4 + tid];
    }
}

void launch_neohookean_hex_residual(hipStream_t s, tet_group_dev g, cluster_dev cl, const pos4* x,
                                    const uint4* cinfo, uint32_t nrows, float inv_dt2, double* partial)
{
    if (nrows)
        k_neohookean_hex_residual<<<grid_for(nrows, kHexRedBlock), kHexRedBlock, 0, s>>>(g, cl, x, cinfo, nrows,
                                                                                           inv_dt2, partial);
}

void launch_copy_spans(hipStream_t s, copy_spans const& spans)
{
    if (spans.n > 0) k_copy_spans<<<1024, 256, 0, s>>>(spans);
}

__global__ void __launch_bounds__(256) k_sum_partials(const double* __restrict__ partial, uint32_t n, double* out)
{
    double v = 0.0;
    for (uint32_t i = threadIdx.x; i < n; i += 256) v += partial[i];
    double const t = block_sum<256>(v);
    if (threadIdx.x == 0) out[0] = t;
}

void launch_sum_partials(hipStream_t s, const double* partial, uint32_t n, double* out)
{
    k_sum_partials<<<1, 256, 0, s>>>(partial, n, out);
}

__global__ void k_publish_u32(const uint32_t* __restrict__ src, uint32_t* dst)
{
    if (threadIdx.x == 0) *reinterpret_cast<volatile uint32_t*>(dst) = *src;
}

void launch_publish_u32(hipStream_t s, const uint32_t* src, uint32_t* dst)
{
    k_publish_u32<<<1, 64, 0, s>>>(src, dst);
}

void launch_distance_residual(hipStream_t s, distance_group_dev g, const pos4* x, uint32_t begin, uint32_t count,
                              float alpha_tilde, double* partial, int)
{
    if (count)
        k_distance_residual<<<grid_for(count, kRedBlock), kRedBlock, 0, s>>>(g, x, begin, count, alpha_tilde, partial);
}

void launch_particle_energy(hipStream_t s, const pos4* x, const float4* v, const float* mass, uint32_t n, float gx,
                            float gy, float gz, int force, double* partial, int)
{
    if (n) k_particle_energy<<<grid_for(n, kRedBlock), kRedBlock, 0, s>>>(x, v, mass, n, gx, gy, gz, force, partial);
}

void launch_green_energy(hipStream_t s, tet_group_dev g, const pos4* x, uint32_t count, double* partial, int)
{
    if (count) k_green_energy<<<grid_for(count, kRedBlock), kRedBlock, 0, s>>>(g, x, count, partial);
}

void launch_neohookean_energy(hipStream_t s, tet_group_dev g, const pos4* x, uint32_t count, double* partial, int)
{
    if (count) k_neohookean_energy<<<grid_for(count, kRedBlock), kRedBlock, 0, s>>>(g, x, count, partial);
}

void launch_jp_round(hipStream_t s, uint32_t n, uint32_t arity, const uint32_t* elem_off, const uint32_t* verts,
                     const uint32_t* inc_off, const uint32_t* inc, const uint64_t* key, const uint32_t* color_in,
                     uint32_t* color_out, uint32_t* remaining, uint32_t* overflow, int block)
{
    if (n)
        k_jp_round<<<grid_for(n, block), block, 0, s>>>(n, arity, elem_off, verts, inc_off, inc, key, color_in,
                                                        color_out, remaining, overflow);
}

void launch_jp_keys(hipStream_t s, uint32_t n, const uint32_t* prev, uint64_t* key, int block)
{
    if (n) k_jp_keys<<<grid_for(n, block), block, 0, s>>>(n, prev, key);
}

void launch_fill_u32(hipStream_t s, uint32_t* p, uint32_t value, uint32_t n)
{
    if (n) k_fill_u32<<<grid_for(n, 256), 256, 0, s>>>(p, value, n);
}

void launch_hex_warm_start(hipStream_t s, tet_group_dev g, cluster_dev cl, const pos4* xt, pos4* xi,
                           const uint4* cinfo, uint32_t nrows, float inv_dt2, int expl, float2 scale,
                           float4* disp, const uint32_t* csr_off, const uint32_t* csr, uint32_t n,
                           const int* surface_of, contact_dev const& c, float c_at, const uint32_t* prow,
                           uint32_t nprows, int net_mode, warm_net_dev const& net)
{
    if (!nrows) return;
    if (net_mode == kWarmLearned)
        k_hex_warm_learned<<<grid_for(nrows, 64), 64, 0, s>>>(g, cl, xt, cinfo, nrows, inv_dt2, expl, scale,
                                                                         disp, net);
    else if (net_mode == kWarmFeatures)
        k_hex_warm_disp<kWarmFeatures><<<grid_for(nrows, 64), 64, 0, s>>>(g, cl, xt, cinfo, nrows, inv_dt2, expl,
                                                                          scale, disp, net);
    else
        k_hex_warm_disp<kWarmPlain><<<grid_for(nrows, 64), 64, 0, s>>>(g, cl, xt, cinfo, nrows, inv_dt2, expl, scale,
                                                                       disp, net);
    if (csr_off)
        k_gather_disp<<<grid_for(n, 256), 256, 0, s>>>(csr_off, csr, disp, xi, n);
    else if (prow && nprows)
        k_gather_disp8<<<grid_for(nprows, kParticleRowBlock), kParticleRowBlock, 0, s>>>(
            reinterpret_cast<const uint4*>(csr), disp, xi, nprows, surface_of, c, c_at, prow);
    else
        k_gather_disp8<<<grid_for(n, 256), 256, 0, s>>>(reinterpret_cast<const uint4*>(csr), disp, xi, n, surface_of,
                                                        c, c_at, nullptr);
}

void launch_hex_capture(hipStream_t s, tet_group_dev g, const uint4* cinfo, const uint32_t* rowof, const float* raw,
                        uint32_t stride, uint32_t offset, float inv_dt2, float* ds_x, float* ds_t, uint64_t base,
                        uint32_t rows)
{
    if (!rows) return;
    k_hex_capture<<<grid_for(rows, 256), 256, 0, s>>>(g, cinfo, rowof, raw, stride, offset, inv_dt2, ds_x, ds_t, base,
                                                      rows);
}

void launch_pack_state(hipStream_t s, const pos4* x, const float4* v, uint32_t n, double* xo, float* vo)
{
    if (n) k_pack_state<<<grid_for(3 * n, 256), 256, 0, s>>>(x, v, n, xo, vo);
}

void launch_copy_pos(hipStream_t s, const pos4* a, pos4* b, uint32_t n)
{
    if (n) k_copy_pos<<<grid_for(n, 256), 256, 0, s>>>(a, b, n);
}

}  // namespace sbs
