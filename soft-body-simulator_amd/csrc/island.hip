// A whole frame of small bodies in one launch: one workgroup per island (a body that no constraint joins to
// another) keeps the island's working positions in LDS and runs prediction, every iteration's
// contacts and colors, and the velocity update with a workgroup barrier between stages, instead of
// one launch per stage.
//
// What bounds it: the chain of stages. A stage is one color's constraints of the island, at most a
// few waves, so its time is one wave's dependent arithmetic (about 2.8 us for the six neo-Hookean
// tets of a hex cell, 0.45 us for one tet) plus the exchange with the next stage: through LDS and a
// barrier here, through a kernel boundary and two memory round trips when every stage is a launch
// (5.4-6.5 us a stage whatever its size). The next stage's particle ids, material and multipliers
// are loaded into the registers that the running stage has just used, and nothing waits for them before
// their use: the records of the chunks lie in LDS, the barrier orders LDS only, the sweep has no branch
// that some waves take. (With records from memory, __syncthreads and a skip for waves without an element,
// the compiler waited for all loads in flight three times a stage: a frame of the demo bar 361 us now and
// 405 then, 864 hex cells 902 and 960.)
//
// The stages and their order are those of the per-launch path, each element is projected by the same
// device functions, and elements of one color share no particle: positions, velocities and
// multipliers are the same bits.
#include "abi_util.h"
#include "island.h"
#include "solver_device.h"

namespace sbs {

namespace {

using lds_double = __attribute__((address_space(3))) double;
using lds_float = __attribute__((address_space(3))) float;
using lds_uint = __attribute__((address_space(3))) uint32_t;

// The island's working positions: one LDS array per coordinate and one of the FP32 inverse masses. 32-byte
// rows (two 16-byte accesses) had fewer addresses but more bank conflicts: the corners of one color's
// cells lie two particles apart (soft block of 864 cells 1,117 us a frame against 1,086).
struct island_pos {
    lds_double *x, *y, *z;
    lds_float* w;
    lds_uint* chunk;  // 4 words a chunk
    __device__ __forceinline__ uint4 record(uint32_t k) const
    {
        return uniform(make_uint4(chunk[4 * k], chunk[4 * k + 1], chunk[4 * k + 2], chunk[4 * k + 3]));
    }
    __device__ __forceinline__ pos4 get(uint32_t l) const { return make_double4(x[l], y[l], z[l], double(w[l])); }
    __device__ __forceinline__ void put(uint32_t l, pos4 p) const
    {
        x[l] = p.x;
        y[l] = p.y;
        z[l] = p.z;
    }
};

__device__ __forceinline__ island_pos island_lds(uint32_t cap)
{
    extern __shared__ double lds[];
    lds_double* const x = (lds_double*)lds;
    lds_float* const w = (lds_float*)(x + 3 * cap);
    return {x, x + cap, x + 2 * cap, w, (lds_uint*)(w + cap)};
}

// A chunk's lane: its element, or the last one for lanes past the end.
__device__ __forceinline__ uint32_t chunk_size(uint4 rec) { return rec.w & 0x7fffffffu; }
__device__ __forceinline__ uint32_t chunk_lane(uint4 rec) { return min(threadIdx.x, chunk_size(rec) - 1u); }

// The frame (or the part of it that p names) around the sweep: per-particle passes, contacts, and
// `item(chunk now, chunk next, now starts from zero multipliers)` for every chunk of every stage, with a
// barrier after the last chunk of a stage. ids(chunk), data(chunk): load the first item's.
template <int BLOCK, class Data, class Item>
__device__ __forceinline__ void run_island(island_dev const& d, pos4* xi, pos4* xn, float4* v, contact_dev const& c,
                                           solve_params const& p, island_pos const& P, uint4 isl, Data&& data,
                                           Item&& item)
{
    __shared__ uint32_t nlist;  // surface vertices of the island that hold contacts
    uint32_t const tid = threadIdx.x;
    uint4 const where = uniform(d.islands[2 * blockIdx.x + 1]);
    const uint32_t* __restrict__ recs = reinterpret_cast<const uint32_t*>(d.chunks + where.x);
    uint32_t const n = where.y;
    bool const work = n && p.iterations > 0;
    for (uint32_t k = tid; k < 4 * n; k += BLOCK) P.chunk[k] = recs[k];
    if (tid == 0) nlist = 0;
    __syncthreads();
    uint4 now = work ? P.record(0) : uint4{};
    if (work) data(now);
    if (c.S && c.slots)
        for (uint32_t s = isl.z + tid; s < isl.z + isl.w; s += BLOCK)
            if (c.count[s]) d.clist[isl.z + atomicAdd(&nlist, 1u)] = s;
    __syncthreads();
    // the thread's first vertex of the list keeps its first contact in registers for the frame: read from
    // memory in every iteration they were three dependent round trips between two barriers (at 512 threads
    // and more the registers would spill)
    constexpr bool kKeep = BLOCK <= 256;
    uint32_t const nl = nlist;
    bool const mine = kKeep && tid < nl;
    uint32_t const s0 = mine ? d.clist[isl.z + tid] : 0u, l0 = mine ? c.surf[s0] - isl.x : 0u;
    uint32_t const cnt0 = mine ? c.count[s0] : 0u;
    pos4 const q0 = mine ? c.q[s0] : pos4{};
    v3 const n0 = mine ? xyz(c.n[s0]) : mk(0.0f, 0.0f, 0.0f);
    float lam0 = mine && p.skip_first_contacts ? c.lambda[s0] : 0.0f;
    for (uint32_t sub = 0; sub < p.substeps; ++sub) {
        for (uint32_t i = tid; i < isl.y; i += BLOCK) {
            uint32_t const gi = isl.x + i;
            if (sub == 0) {
                pos4 x = p.predict ? xn[gi] : xi[gi];
                if (p.predict) {
                    float4 vel = v[gi];
                    pos4 np;
                    predict_one(np, x, vel, p.g[0], p.g[1], p.g[2], p.force, p.dt);
                    x = np;
                }
                P.put(i, x);
                P.w[i] = wof(x);
            } else {  // commit of the last substep, prediction of this one
                pos4 const q = xn[gi];
                pos4 x = P.get(i);
                x.w = q.w;
                float4 vel = velocity(x, q, p.dt);
                pos4 np;
                predict_one(np, x, vel, p.g[0], p.g[1], p.g[2], p.force, p.dt);
                xn[gi] = x;
                P.put(i, np);
            }
        }
        __syncthreads();
        for (uint32_t it = 0; it < p.iterations; ++it) {
            if (nl && !(it == 0 && p.skip_first_contacts)) {
                if (mine) {
                    pos4 x = P.get(l0);
                    lam0 = contact_slot(x, q0, n0, wof(x), 0.0f, p.contact_at, it == 0 ? 0.0f : lam0);
                    c.lambda[s0] = lam0;
                    contact_slots(c, x, s0, 1, cnt0, p.contact_at, it == 0);
                    P.put(l0, x);
                }
                for (uint32_t k = tid + (kKeep ? BLOCK : 0); k < nl; k += BLOCK) {
                    uint32_t const s = d.clist[isl.z + k], l = c.surf[s] - isl.x;
                    pos4 x = P.get(l);
                    contact_vertex_at(c, x, s, p.contact_at, it == 0);
                    P.put(l, x);
                }
                lds_barrier();
            }
            bool const zero = p.zero_first && it == 0;
            for (uint32_t k = 0; work && k < n; ++k) {
                uint4 const next = P.record(k + 1 < n ? k + 1 : 0);
                item(now, next, zero);
                if (now.w >> 31) lds_barrier();
                now = next;
            }
        }
    }
    for (uint32_t i = tid; i < isl.y; i += BLOCK) {
        uint32_t const gi = isl.x + i;
        pos4 const q = xn[gi];
        pos4 x = P.get(i);
        x.w = q.w;
        if (p.commit) {
            v[gi] = velocity(x, q, p.dt);
            xn[gi] = x;
        }
        xi[gi] = x;
    }
}

// Hex-cell clusters: a lane runs one cluster's six tets, particles in registers (as k_neohookean_hex
// and k_green_hex). A tet's material and multipliers of the next chunk are loaded as soon as the
// running chunk has used its own, by every lane (lanes past the end repeat the last element, so no
// load sits in a branch) and only lanes with an element write.
// One wave per SIMD at 256 threads (and room for a second workgroup beside it: at most 256 registers a
// lane); 512 threads where a stage of an island has more than 256 clusters.
template <int KIND, bool DAMPED, int BLOCK>
__global__ void __launch_bounds__(BLOCK, 2) k_island_hex(island_dev d, tet_group_dev g, cluster_dev cl, pos4* xi, pos4* xn,
                                                      float4* v, contact_dev c, solve_params p)
{
    uint4 const isl = uniform(d.islands[2 * blockIdx.x]);
    island_pos const P = island_lds(d.cap);
    float4 A[kHexTets], B[kHexTets];
    float4 G[KIND == 0 ? kHexTets : 1];
    float2 C[KIND == 0 ? 1 : kHexTets], L[kHexTets];
    int4 va, vb;
    // t: the constraint's index, its 16-byte offset in a 32-bit register (a scene of islands has fewer
    // than 2^28 constraints): one vector addition a tet, where a scalar 64-bit base per tet and array took
    // 230 scalar instructions a stage, each an issue slot of a wave that has its SIMD to itself
    auto load = [&](uint32_t t, int m) {
        A[m] = lane_load(g.m0, t);
        B[m] = lane_load(g.m1, t);
        if (KIND == 0) {
            G[m] = lane_load(g.m2, t);
            L[m].x = lane_load(g.lambda, t);
        } else {
            C[m] = lane_load(reinterpret_cast<const float2*>(g.m2), t);
            L[m] = lane_load(reinterpret_cast<const float2*>(g.lambda), t);
        }
    };
    auto load_ids = [&](uint4 rec) {
        va = lane_load(cl.v0, rec.x + chunk_lane(rec));
        vb = lane_load(cl.v1, rec.x + chunk_lane(rec));
    };
    auto data = [&](uint4 rec) {
        load_ids(rec);
#pragma unroll
        for (int m = 0; m < kHexTets; ++m) load(rec.y + uint32_t(m) * rec.z + chunk_lane(rec), m);
    };
    auto item = [&](uint4 now, uint4 next, bool zero) {
        bool const active = threadIdx.x < chunk_size(now);
        uint32_t const l[8] = {va.x - isl.x, va.y - isl.x, va.z - isl.x, va.w - isl.x,
                               vb.x - isl.x, vb.y - isl.x, vb.z - isl.x, vb.w - isl.x};
        pos4 X[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) X[k] = P.get(l[k]);
        loads_issued();
        load_ids(next);
        loads_issued();
        uint32_t const t0 = now.y + chunk_lane(now), n0 = next.y + chunk_lane(next);
#pragma unroll
        for (int m = 0; m < kHexTets; ++m) {
            int const s0 = kHexSlots[m][0], s1 = kHexSlots[m][1], s2 = kHexSlots[m][2], s3 = kHexSlots[m][3];
            pos4 Q[4] = {X[s0], X[s1], X[s2], X[s3]};
            uint32_t const id[4] = {l[s0], l[s1], l[s2], l[s3]};
            auto xn_of = [&](int k) { return xn[isl.x + id[k]]; };
            uint32_t const t = t0 + uint32_t(m) * now.z;
            float2 lm = zero ? make_float2(0.0f, 0.0f) : L[m];
            if (KIND == 0) {
                green_project(Q, xn_of, A[m], B[m], G[m], p.alpha_tilde, DAMPED ? p.gamma : 0.0f, lm.x);
                if (active) lane_store(g.lambda, t, lm.x);
            } else {
                neohookean_project<DAMPED>(Q, xn_of, A[m], B[m], C[m], p.inv_dt2, p.beta_dt, lm);
                if (active) lane_store(reinterpret_cast<float2*>(g.lambda), t, lm);
            }
            X[s0] = Q[0];
            X[s1] = Q[1];
            X[s2] = Q[2];
            X[s3] = Q[3];
            if (m == kHexTets - 1 && active) {
#pragma unroll
                for (int k = 0; k < 8; ++k) P.put(l[k], X[k]);
            }
            __builtin_amdgcn_sched_barrier(0);  // the registers are free: no use of them sinks past the loads
            load(n0 + uint32_t(m) * next.z, m);
            loads_issued();
        }
    };
    run_island<BLOCK>(d, xi, xn, v, c, p, P, isl, data, item);
}

// One constraint per lane (tets without clusters).
template <int KIND, bool DAMPED, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_island_tets(island_dev d, tet_group_dev g, pos4* xi, pos4* xn, float4* v,
                                                       contact_dev c, solve_params p)
{
    uint4 const isl = uniform(d.islands[2 * blockIdx.x]);
    island_pos const P = island_lds(d.cap);
    int4 id;
    float4 A, B, G;
    float2 C, L;
    auto data = [&](uint4 rec) {
        uint32_t const t = rec.y + chunk_lane(rec);
        id = lane_load(g.idx, t);
        A = lane_load(g.m0, t);
        B = lane_load(g.m1, t);
        if (KIND == 0) {
            G = lane_load(g.m2, t);
            L.x = lane_load(g.lambda, t);
        } else {
            C = lane_load(reinterpret_cast<const float2*>(g.m2), t);
            L = lane_load(reinterpret_cast<const float2*>(g.lambda), t);
        }
    };
    auto item = [&](uint4 now, uint4 next, bool zero) {
        bool const active = threadIdx.x < chunk_size(now);
        uint32_t const t = now.y + chunk_lane(now);
        uint32_t const l[4] = {id.x - isl.x, id.y - isl.x, id.z - isl.x, id.w - isl.x};
        pos4 Q[4] = {P.get(l[0]), P.get(l[1]), P.get(l[2]), P.get(l[3])};
        auto xn_of = [&](int k) { return xn[isl.x + l[k]]; };
        bool moved = true;
        float2 lm = zero ? make_float2(0.0f, 0.0f) : L;
        if (KIND == 0) {
            moved = green_project(Q, xn_of, A, B, G, p.alpha_tilde, DAMPED ? p.gamma : 0.0f, lm.x);
            if (active) lane_store(g.lambda, t, lm.x);
        } else {
            neohookean_project<DAMPED>(Q, xn_of, A, B, C, p.inv_dt2, p.beta_dt, lm);
            if (active) lane_store(reinterpret_cast<float2*>(g.lambda), t, lm);
        }
        if (active && moved) {
#pragma unroll
            for (int k = 0; k < 4; ++k) P.put(l[k], Q[k]);
        }
        __builtin_amdgcn_sched_barrier(0);
        data(next);
        loads_issued();
    };
    run_island<BLOCK>(d, xi, xn, v, c, p, P, isl, data, item);
}

template <class K, class... Args>
void launch_island(hipStream_t s, K kernel, uint32_t blocks, int block, std::size_t lds, Args... args)
{
    kernel<<<blocks, block, lds, s>>>(args...);
    hip_check(hipGetLastError(), "island launch");
}

template <int KIND, bool DAMPED>
void allow_island_kernels()
{
    allow_lds(kIslandDynamicLds, k_island_hex<KIND, DAMPED, 256>, k_island_hex<KIND, DAMPED, 512>,
              k_island_tets<KIND, DAMPED, 256>, k_island_tets<KIND, DAMPED, 1024>);
}

}  // namespace

void allow_island_lds()
{
    allow_island_kernels<0, false>();
    allow_island_kernels<0, true>();
    allow_island_kernels<1, false>();
    allow_island_kernels<1, true>();
}

void launch_island_frame(hipStream_t s, island_dev const& d, int kind, bool hex, tet_group_dev const& g,
                         cluster_dev const& cl, pos4* xi, pos4* xn, float4* v, contact_dev const& c,
                         solve_params const& p)
{
    if (!d.count) return;
    std::size_t const lds = island_lds_bytes(d.cap, d.chunks_cap);
    bool const wide = d.block > 256, damped = kind == 0 ? p.gamma != 0.0f : p.beta_dt != 0.0f;
    auto hexes = [&](auto kernel, int block) { launch_island(s, kernel, d.count, block, lds, d, g, cl, xi, xn, v, c, p); };
    auto tets = [&](auto kernel, int block) { launch_island(s, kernel, d.count, block, lds, d, g, xi, xn, v, c, p); };
    if (hex) {
        if (kind == 0)
            damped ? (wide ? hexes(k_island_hex<0, true, 512>, 512) : hexes(k_island_hex<0, true, 256>, 256))
                   : (wide ? hexes(k_island_hex<0, false, 512>, 512) : hexes(k_island_hex<0, false, 256>, 256));
        else
            damped ? (wide ? hexes(k_island_hex<1, true, 512>, 512) : hexes(k_island_hex<1, true, 256>, 256))
                   : (wide ? hexes(k_island_hex<1, false, 512>, 512) : hexes(k_island_hex<1, false, 256>, 256));
        return;
    }
    if (kind == 0)
        damped ? (wide ? tets(k_island_tets<0, true, 1024>, 1024) : tets(k_island_tets<0, true, 256>, 256))
               : (wide ? tets(k_island_tets<0, false, 1024>, 1024) : tets(k_island_tets<0, false, 256>, 256));
    else
        damped ? (wide ? tets(k_island_tets<1, true, 1024>, 1024) : tets(k_island_tets<1, true, 256>, 256))
               : (wide ? tets(k_island_tets<1, false, 1024>, 1024) : tets(k_island_tets<1, false, 256>, 256));
}

}  // namespace sbs
