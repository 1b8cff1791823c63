// Several colors of a large body in one launch. The particles are divided into tiles, one workgroup each; a
// workgroup loads its tile's particles and those around it that its elements reach into LDS, runs the
// elements of one color after the other with a barrier between, and writes its own particles to the other of
// two position arrays. Elements at a tile's rim are run by every tile whose particles depend on them: with
// the same inputs and the same device functions they give the same bits everywhere, so no workgroup waits
// for another.
//
// What bounds it: the chain of stages (one color of a tile), each one wave's dependent arithmetic, 3.3-3.7 us
// for hex cells of neo-Hookean tets up to 256 of them (2.8 us of it vector instructions of a wave that has its
// SIMD to itself), 0.9 us for single tets. A launch of its own took 5.4 us a stage at 2,700 cells a color and
// 8.2 at 20,800 (a kernel boundary, two dependent round trips, and particles of the stage before read from
// beyond the L2); a launch here takes 3-6 us beside its stages. Per iteration, contacts included, launched
// color by color and here: 129k tets 43.5 and 32.8 us, 1M 68 and 49, 2M 93 and 75, 4M 140 and 130; 40k single
// tets 140 and 48, 1M 236 and 112; 129k tets of Green cells 125 and 119.
//
// Waiting for the neighbours' progress instead of running the rims twice was no faster than the launches: a
// hand-over between XCDs costs a store drained to memory, a flag and a poll, about 2 us.
#include "solver_device.h"
#include "tile.h"

namespace sbs {

namespace {

constexpr uint32_t kTopBit = 0x80000000u, kNone = 0xffffffffu;

using lds_double = __attribute__((address_space(3))) double;
using lds_float = __attribute__((address_space(3))) float;
using lds_uint = __attribute__((address_space(3))) uint32_t;

struct tile_dev {
    const uint4* blocks;
    const uint4* chunks;
    const uint2* particles;
    const uint32_t* elems;
    const uint4* corners8;
    const uint2* corners4;
    float* lambda;
    uint32_t tiles, per, cap, instances;
};

struct tile_lds {
    lds_double *x, *y, *z, *w;
    lds_float* f;     // the inverse masses again, in FP32
    lds_uint* id;
    lds_uint* chunk;  // 4 words a chunk
    __device__ __forceinline__ explicit tile_lds(uint32_t cap)
    {
        extern __shared__ double lds[];
        x = (lds_double*)lds;
        y = x + cap;
        z = y + cap;
        w = z + cap;
        f = (lds_float*)(w + cap);
        id = (lds_uint*)(f + cap);
        chunk = id + cap;
    }
    __device__ __forceinline__ pos4 get(uint32_t l) const { return make_double4(x[l], y[l], z[l], double(f[l])); }
    __device__ __forceinline__ void put(uint32_t l, pos4 p) const
    {
        x[l] = p.x;
        y[l] = p.y;
        z[l] = p.z;
    }
    __device__ __forceinline__ uint4 record(uint32_t k) const
    {
        return uniform(make_uint4(chunk[4 * k], chunk[4 * k + 1], chunk[4 * k + 2], chunk[4 * k + 3]));
    }
};

// Where the tile's k-th particle lies in LDS: of every 64 the even ones first. The corners of a color's cells
// are two particles apart along a lattice line, every second bank.
__device__ __forceinline__ uint32_t slot_of(uint32_t k) { return (k & ~63u) | (k & 1u) << 5 | (k >> 1 & 31u); }

__device__ __forceinline__ uint32_t instance(uint4 rec) { return rec.x + min(threadIdx.x, max(rec.y, 1u) - 1u); }

// The tile's particles into LDS (contacts projected on the way), the chunks, its own particles out again.
// ids(first chunk, second), data(first chunk): load the elements and then the constraints of the first item;
// item(chunk, next, the one after): runs a chunk and loads the next one's data (past the end the last chunk
// is repeated). Before the first item there are three dependent memory round trips: the tile's record with its
// first two chunks; its particles' entries and the elements; the rows and the constraints.
template <class Ids, class Data, class Item>
__device__ __forceinline__ void run_tile(tile_dev const& d, const pos4* __restrict__ in, pos4* __restrict__ out,
                                         contact_dev const& c, tile_params const& p, tile_lds const& P, Ids&& ids,
                                         Data&& data, Item&& item)
{
    // neighbouring tiles on one XCD, the same ones in every launch: its L2 holds their shared constraints
    uint32_t const tile = (blockIdx.x % kXcds) * d.per + blockIdx.x / kXcds, tid = threadIdx.x;
    if (tile >= d.tiles) return;
    uint4 const blk = uniform(d.blocks[3 * tile]), first = uniform(d.blocks[3 * tile + 1]);
    uint4 const second = uniform(d.blocks[3 * tile + 2]);
    const uint32_t* __restrict__ recs = reinterpret_cast<const uint32_t*>(d.chunks + blk.z);
    uint32_t const n = blk.w;
    constexpr uint32_t kBatch = 8;  // particles of a thread in flight together
    uint2 e[kBatch];
    pos4 x[kBatch];
    uint32_t cnt[kBatch];
    auto load_entries = [&](uint32_t base) {
        uint32_t const l0 = base + tid;
#pragma unroll
        for (uint32_t k = 0; k < kBatch; ++k)
            if (base + k * kTileThreads < blk.y) e[k] = lane_load(d.particles + blk.x, min(l0 + k * kTileThreads, blk.y - 1));
    };
    // (without contacts, or for an inner particle, some word: a load under a condition would be waited for)
    const uint32_t* const counts = p.contacts ? c.count : d.elems;
    auto load_rows = [&](uint32_t base) {
#pragma unroll
        for (uint32_t k = 0; k < kBatch; ++k) {
            if (base + k * kTileThreads >= blk.y) continue;
            x[k] = in[e[k].x & ~kTopBit];
            cnt[k] = counts[p.contacts && e[k].y != kNone ? e[k].y : 0u];
        }
    };
    uint32_t touched = 0;  // which of the thread's particles hold contacts
    auto put_rows = [&](uint32_t base) {
        uint32_t const l0 = base + tid;
#pragma unroll
        for (uint32_t k = 0; k < kBatch; ++k) {
            if (base + k * kTileThreads >= blk.y) continue;
            bool const real = l0 + k * kTileThreads < blk.y;
            uint32_t const l = slot_of(l0 + k * kTileThreads);
            if (real && p.contacts && e[k].y != kNone && cnt[k]) touched |= 1u << (l0 / kTileThreads + k);
            if (real) {
                P.put(l, x[k]);
                P.w[l] = x[k].w;
                P.f[l] = wof(x[k]);
                P.id[l] = e[k].x;
            }
        }
    };
    bool const runs = __builtin_amdgcn_readfirstlane(int(tid)) < kTileBlock;
    load_entries(0);
    if (runs) ids(first, second);
    uint32_t const rec = recs[min(tid, 4 * n - 1)];
    loads_issued();
    load_rows(0);
    if (runs) data(first);
    loads_issued();
    // (a tile holds at most one batch of particles and kTileThreads words of chunks: the loops below never turn.
    // Without them the compiler schedules the loads above otherwise, and four frames of 1M tets take 6,664 us
    // instead of 6,533, two of 129k 2,250 instead of 2,228)
    if (tid < 4 * n) P.chunk[tid] = rec;
    for (uint32_t k = tid + kTileThreads; k < 4 * n; k += kTileThreads) P.chunk[k] = recs[k];
    put_rows(0);
    for (uint32_t base = kBatch * kTileThreads; base < blk.y; base += kBatch * kTileThreads) {
        load_entries(base);
        load_rows(base);
        put_rows(base);
    }
    static_assert(kTileParticles <= 32 * kTileThreads, "a bit per particle of a thread");
    for (; touched; touched &= touched - 1) {
        uint32_t const k = tid + (uint32_t(__ffs(int(touched))) - 1u) * kTileThreads, l = slot_of(k);
        uint2 const q = d.particles[blk.x + k];
        pos4 y = make_double4(P.x[l], P.y[l], P.z[l], P.w[l]);
        contact_slots(c, y, q.y, 0, c.count[q.y], p.contact_at, p.first_contacts != 0,
                      [&](uint32_t r) { return in[c.surf[r]]; },
                      [&](uint32_t slot, float lm) { if (q.x & kTopBit) p.lambda_out[slot] = lm; });
        P.put(l, y);
    }
    __syncthreads();
    if (runs) {
        uint4 now = P.record(0), next = P.record(min(1u, n - 1));
        for (uint32_t k = 0; k < n; ++k) {
            uint4 const after = P.record(min(k + 2, n - 1));
            item(now, next, after);
            if (now.w) lds_barrier();
            now = next;
            next = after;
        }
    } else {  // the waves that only carry particles
        for (uint32_t k = 0; k < n; ++k)
            if (P.record(k).w) lds_barrier();
    }
    for (uint32_t l0 = tid; l0 < blk.y; l0 += 4 * kTileThreads) {
        uint32_t id[4];
        pos4 o[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            uint32_t const l = slot_of(min(l0 + k * kTileThreads, blk.y - 1));
            id[k] = l0 + k * kTileThreads < blk.y ? P.id[l] : 0u;
            o[k] = make_double4(P.x[l], P.y[l], P.z[l], P.w[l]);
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (id[k] & kTopBit) out[id[k] & ~kTopBit] = o[k];
    }
}

// Hex-cell clusters, a lane each. No branch in the sweep but the masks of its stores: where one skipped the
// arithmetic of waves without a cluster, the compiler waited for every load in flight at its join.
template <int KIND, bool DAMPED>
__global__ void __launch_bounds__(kTileThreads, 2) k_tile_hex(tile_dev d, tet_group_dev g, const pos4* __restrict__ in,
                                                            pos4* __restrict__ out, const pos4* __restrict__ xn,
                                                            contact_dev c, tile_params p)
{
    tile_lds const P(d.cap);
    using mult = std::conditional_t<KIND == 0, float, float2>;
    float4 A[kHexTets], B[kHexTets];
    float4 G[KIND == 0 ? kHexTets : 1];
    float2 C[KIND == 0 ? 1 : kHexTets];
    mult L[kHexTets];
    uint4 corners{};
    uint32_t word = 0, word_next = 0;  // the running and the next chunk's element
    mult* const lambda_in = reinterpret_cast<mult*>(p.from_group ? g.lambda : d.lambda);
    mult* const lambda_out = reinterpret_cast<mult*>(p.to_group ? g.lambda : d.lambda);
    // t, u: the constraint and where its multipliers come from
    auto load = [&](uint32_t t, uint32_t u, int m) {
        A[m] = lane_load(g.m0, t);
        B[m] = lane_load(g.m1, t);
        if (KIND == 0)
            G[m] = lane_load(g.m2, t);
        else
            C[m] = lane_load(reinterpret_cast<const float2*>(g.m2), t);
        L[m] = lane_load(lambda_in, u);
    };
    auto ids = [&](uint4 now, uint4 next) {
        word = lane_load(d.elems, instance(now));
        word_next = lane_load(d.elems, instance(next));
        corners = lane_load(d.corners8, instance(now));
    };
    auto data = [&](uint4 now) {
        uint32_t const t = word & ~kTopBit, i = instance(now);
#pragma unroll
        for (uint32_t m = 0; m < kHexTets; ++m)
            load(t + m * now.z, p.from_group ? t + m * now.z : i + m * d.instances, int(m));
    };
    auto item = [&](uint4 now, uint4 next, uint4 after) {
        uint32_t const l[8] = {corners.x & 0xffffu, corners.x >> 16, corners.y & 0xffffu, corners.y >> 16,
                               corners.z & 0xffffu, corners.z >> 16, corners.w & 0xffffu, corners.w >> 16};
        pos4 X[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) X[k] = P.get(l[k]);
        bool const active = threadIdx.x < now.y, store = active && (!p.to_group || (word & kTopBit));
        uint32_t const o = p.to_group ? word & ~kTopBit : instance(now), os = p.to_group ? now.z : d.instances;
        uint32_t const t = word_next & ~kTopBit, n = instance(next);
        uint32_t const u = p.from_group ? t : n, us = p.from_group ? next.z : d.instances;
        loads_issued();
        word = word_next;
        word_next = lane_load(d.elems, instance(after));
        corners = lane_load(d.corners8, n);
        loads_issued();
#pragma unroll
        for (int m = 0; m < kHexTets; ++m) {
            int const s0 = kHexSlots[m][0], s1 = kHexSlots[m][1], s2 = kHexSlots[m][2], s3 = kHexSlots[m][3];
            pos4 Q[4] = {X[s0], X[s1], X[s2], X[s3]};
            uint32_t const id[4] = {l[s0], l[s1], l[s2], l[s3]};
            auto xn_of = [&](int k) { return xn[P.id[id[k]] & ~kTopBit]; };
            mult lm = p.zero ? mult{} : L[m];
            if constexpr (KIND == 0)
                green_project(Q, xn_of, A[m], B[m], G[m], p.alpha_tilde, DAMPED ? p.gamma : 0.0f, lm);
            else
                neohookean_project<DAMPED>(Q, xn_of, A[m], B[m], C[m], p.inv_dt2, p.beta_dt, lm);
            if (store) lane_store(lambda_out, o + uint32_t(m) * os, lm);
            X[s0] = Q[0];
            X[s1] = Q[1];
            X[s2] = Q[2];
            X[s3] = Q[3];
            if (m == kHexTets - 1 && active) {
#pragma unroll
                for (int k = 0; k < 8; ++k) P.put(l[k], X[k]);
            }
            __builtin_amdgcn_sched_barrier(0);  // the registers are free: no use of them sinks past the loads
            load(t + uint32_t(m) * next.z, u + uint32_t(m) * us, m);
            loads_issued();
        }
    };
    run_tile(d, in, out, c, p, P, ids, data, item);
}

// One constraint per lane (tets without clusters).
template <int KIND, bool DAMPED>
__global__ void __launch_bounds__(kTileThreads, 2) k_tile_tets(tile_dev d, tet_group_dev g, const pos4* __restrict__ in,
                                                          pos4* __restrict__ out, const pos4* __restrict__ xn,
                                                          contact_dev c, tile_params p)
{
    tile_lds const P(d.cap);
    using mult = std::conditional_t<KIND == 0, float, float2>;
    float4 A, B, G;
    float2 C;
    mult L;
    uint2 corners{};
    uint32_t word = 0, word_next = 0;
    mult* const lambda_in = reinterpret_cast<mult*>(p.from_group ? g.lambda : d.lambda);
    mult* const lambda_out = reinterpret_cast<mult*>(p.to_group ? g.lambda : d.lambda);
    auto load = [&](uint32_t w, uint32_t inst) {
        uint32_t const t = w & ~kTopBit;
        A = lane_load(g.m0, t);
        B = lane_load(g.m1, t);
        if (KIND == 0)
            G = lane_load(g.m2, t);
        else
            C = lane_load(reinterpret_cast<const float2*>(g.m2), t);
        L = lane_load(lambda_in, p.from_group ? t : inst);
        corners = lane_load(d.corners4, inst);
    };
    auto ids = [&](uint4 now, uint4 next) {
        word = lane_load(d.elems, instance(now));
        word_next = lane_load(d.elems, instance(next));
    };
    auto data = [&](uint4 now) { load(word, instance(now)); };
    auto item = [&](uint4 now, uint4 next, uint4 after) {
        uint32_t const i = instance(now), w = word, t = w & ~kTopBit;
        word = word_next;
        word_next = lane_load(d.elems, instance(after));
        bool const active = threadIdx.x < now.y, store = active && (!p.to_group || (w & kTopBit));
        uint32_t const l[4] = {corners.x & 0xffffu, corners.x >> 16, corners.y & 0xffffu, corners.y >> 16};
        pos4 Q[4] = {P.get(l[0]), P.get(l[1]), P.get(l[2]), P.get(l[3])};
        auto xn_of = [&](int k) { return xn[P.id[l[k]] & ~kTopBit]; };
        bool moved = true;
        mult lm = p.zero ? mult{} : L;
        if constexpr (KIND == 0)
            moved = green_project(Q, xn_of, A, B, G, p.alpha_tilde, DAMPED ? p.gamma : 0.0f, lm);
        else
            neohookean_project<DAMPED>(Q, xn_of, A, B, C, p.inv_dt2, p.beta_dt, lm);
        if (store) lane_store(lambda_out, p.to_group ? t : i, lm);
        if (active && moved) {
#pragma unroll
            for (int k = 0; k < 4; ++k) P.put(l[k], Q[k]);
        }
        __builtin_amdgcn_sched_barrier(0);
        load(word, instance(next));
        loads_issued();
    };
    run_tile(d, in, out, c, p, P, ids, data, item);
}

// ---------------------------------------------------------------- the plan

struct plan_dev {
    uint32_t V, elements, ncolors, tiles;
    const int4 *v0, *v1;
    const uint32_t *cfirst, *tfirst;  // elements and constraints before each color
    const uint32_t *own_first, *own, *tile_of;
    const uint32_t* table;   // [color][particle]: the color's element at the particle, or ~0
    const uint32_t* bounds;  // first color of each segment, then ncolors
    uint32_t* bits;          // per (segment, tile): particles, then elements
    uint32_t vwords, ewords;
};

template <bool HEX>
__device__ __forceinline__ uint32_t corner(plan_dev const& d, uint32_t e, int k)
{
    int4 const v = k < 4 ? d.v0[e] : d.v1[e];
    int const j = k & 3;
    return uint32_t(j == 0 ? v.x : (j == 1 ? v.y : (j == 2 ? v.z : v.w)));
}

template <bool HEX>
__global__ void k_tile_table(plan_dev d, uint32_t* __restrict__ table)
{
    uint32_t const e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= d.elements) return;
    uint32_t c = 0;
    while (e >= d.cfirst[c + 1]) ++c;
    for (int k = 0; k < (HEX ? 8 : 4); ++k) table[std::size_t(c) * d.V + corner<HEX>(d, e, k)] = e;
}

// Marks what tile blockIdx.x needs for segment blockIdx.y: from the last color back, the color's elements at
// a marked particle, then those elements' other corners. counts: instances per color of [tile], then
// particles per [segment][tile].
template <bool HEX>
__global__ void __launch_bounds__(kTileBlock) k_tile_cone(plan_dev d, uint32_t* __restrict__ instances,
                                                          uint32_t* __restrict__ particles)
{
    extern __shared__ uint32_t marked[];  // particles, then the color's elements
    __shared__ uint32_t np, ne;
    uint32_t* const found = marked + kTileParticles;
    uint32_t const tile = blockIdx.x, seg = blockIdx.y, tid = threadIdx.x;
    uint32_t* const vb = d.bits + (std::size_t(seg) * d.tiles + tile) * (d.vwords + d.ewords);
    uint32_t* const eb = vb + d.vwords;
    uint32_t const o0 = d.own_first[tile], own = d.own_first[tile + 1] - o0;
    bool fits = own <= kTileParticles;
    if (fits)
        for (uint32_t i = tid; i < own; i += kTileBlock) {
            uint32_t const v = d.own[o0 + i];
            marked[i] = v;
            atomicOr(&vb[v >> 5], 1u << (v & 31u));
        }
    if (tid == 0) np = own, ne = 0;
    __syncthreads();
    for (uint32_t c = d.bounds[seg + 1]; fits && c-- > d.bounds[seg];) {
        uint32_t const n = np;
        for (uint32_t i = tid; i < n; i += kTileBlock) {
            uint32_t const e = d.table[std::size_t(c) * d.V + marked[i]];
            if (e == kNone) continue;
            uint32_t const bit = 1u << (e & 31u);
            if (!(atomicOr(&eb[e >> 5], bit) & bit)) found[atomicAdd(&ne, 1u)] = e;
        }
        __syncthreads();
        uint32_t const m = ne;
        for (uint32_t i = tid; i < m; i += kTileBlock)
            for (int k = 0; k < (HEX ? 8 : 4); ++k) {
                uint32_t const v = corner<HEX>(d, found[i], k), bit = 1u << (v & 31u);
                if (atomicOr(&vb[v >> 5], bit) & bit) continue;
                uint32_t const at = atomicAdd(&np, 1u);
                if (at < kTileParticles) marked[at] = v;
            }
        if (tid == 0) instances[std::size_t(tile) * d.ncolors + c] = m;
        __syncthreads();
        fits = np <= kTileParticles;
        if (tid == 0) ne = 0;
        __syncthreads();
    }
    if (tid == 0) particles[std::size_t(seg) * d.tiles + tile] = fits ? np : kNone;
}

// Exclusive prefix of v over the workgroup; total: its sum.
__device__ __forceinline__ uint32_t prefix(uint32_t v, uint32_t& total)
{
    __shared__ uint32_t sums[kTileBlock / 64];
    uint32_t const lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (uint32_t s = 1; s < 64; s <<= 1) {
        uint32_t const u = __shfl_up(inc, s, 64);
        if (lane >= s) inc += u;
    }
    if (lane == 63) sums[wave] = inc;
    __syncthreads();
    uint32_t base = 0;
    total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kTileBlock / 64; ++w) {
        if (w < wave) base += sums[w];
        total += sums[w];
    }
    __syncthreads();
    return base + inc - v;
}

// Calls item(i, place) for every set bit i of [lo, hi), places in ascending order.
template <class Item>
__device__ __forceinline__ void for_bits(const uint32_t* __restrict__ words, uint32_t lo, uint32_t hi, Item&& item,
                                         uint32_t* count = nullptr)
{
    uint32_t at = 0;
    if (lo >= hi) return;
    for (uint32_t w0 = lo >> 5; w0 <= (hi - 1) >> 5; w0 += kTileBlock) {
        uint32_t const w = w0 + threadIdx.x;
        uint32_t b = w <= (hi - 1) >> 5 ? words[w] : 0u;
        if (w == lo >> 5) b &= ~0u << (lo & 31u);
        if (w == (hi - 1) >> 5) b &= ~0u >> (31u - ((hi - 1) & 31u));
        uint32_t total, place = at + prefix(uint32_t(__popc(b)), total);
        for (; b; b &= b - 1) item(w * 32u + uint32_t(__ffs(int(b))) - 1u, place++);
        at += total;
    }
    if (count) *count = at;
}

// Writes the tile's particle entries and instances from its marks.
template <bool HEX>
__global__ void __launch_bounds__(kTileBlock) k_tile_emit(plan_dev d, const uint4* __restrict__ blocks,
                                                          const uint32_t* __restrict__ firsts,
                                                          const int* __restrict__ surface_of, uint2* __restrict__ parts,
                                                          uint32_t* __restrict__ elems, uint4* __restrict__ corners8,
                                                          uint2* __restrict__ corners4)
{
    extern __shared__ uint32_t marked[];
    uint32_t const tile = blockIdx.x, seg = blockIdx.y;
    std::size_t const at = std::size_t(seg) * d.tiles + tile;
    const uint32_t* const vb = d.bits + at * (d.vwords + d.ewords);
    uint4 const blk = blocks[3 * at];
    // the marks in order first, then an even share of them for every thread (the marks cluster in few words)
    for_bits(vb, 0, d.V, [&](uint32_t v, uint32_t place) { marked[place] = v; });
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < blk.y; i += kTileBlock) {
        uint32_t const v = marked[i];
        int const s = surface_of[v];
        parts[blk.x + i] = make_uint2(v | (d.tile_of[v] == tile ? kTopBit : 0u), s >= 0 ? uint32_t(s) : kNone);
    }
    auto place_of = [&](uint32_t v) {
        uint32_t lo = 0, n = blk.y;
        while (n > 1) {
            uint32_t const h = n >> 1;
            bool const up = marked[lo + h] <= v;
            lo = up ? lo + h : lo;
            n = up ? n - h : h;
        }
        return slot_of(lo);
    };
    for (uint32_t c = d.bounds[seg]; c < d.bounds[seg + 1]; ++c) {
        uint32_t const first = firsts[std::size_t(tile) * d.ncolors + c];
        uint32_t total = 0;
        for_bits(vb + d.vwords, d.cfirst[c], d.cfirst[c + 1],
                 [&](uint32_t e, uint32_t place) { elems[first + place] = e; }, &total);
        __syncthreads();
        for (uint32_t i = first + threadIdx.x; i < first + total; i += kTileBlock) {
            uint32_t const e = elems[i];
            elems[i] = (d.tfirst[c] + (e - d.cfirst[c])) | (d.tile_of[corner<HEX>(d, e, 0)] == tile ? kTopBit : 0u);
            uint32_t pair[HEX ? 4 : 2];
#pragma unroll
            for (int k = 0; k < (HEX ? 4 : 2); ++k)
                pair[k] = place_of(corner<HEX>(d, e, 2 * k)) | place_of(corner<HEX>(d, e, 2 * k + 1)) << 16;
            if (HEX)
                corners8[i] = make_uint4(pair[0], pair[1], pair[HEX ? 2 : 0], pair[HEX ? 3 : 0]);
            else
                corners4[i] = make_uint2(pair[0], pair[1]);
        }
    }
}

plan_dev view(tile_source const& src, dev_buf<uint32_t> const& cfirst, dev_buf<uint32_t> const& tfirst,
              dev_buf<uint32_t> const& own_first, dev_buf<uint32_t> const& own, dev_buf<uint32_t> const& tile_of,
              dev_buf<uint32_t> const& table, dev_buf<uint32_t> const& bounds, dev_buf<uint32_t> const& bits,
              std::size_t vwords, std::size_t ewords)
{
    return {src.V,       src.elements, src.ncolors, src.tiles, src.v0,   src.v1, cfirst.p,         tfirst.p,
            own_first.p, own.p,        tile_of.p,   table.p,   bounds.p, bits.p, uint32_t(vwords), uint32_t(ewords)};
}

}  // namespace

tile_scratch::tile_scratch(hipStream_t stream, tile_source const& source)
    : s(stream), src(source), vwords((std::size_t(source.V) + 31) / 32), ewords((std::size_t(source.elements) + 31) / 32)
{
    std::vector<uint32_t> first(src.tiles + 1, 0), list(src.V);
    for (uint32_t v = 0; v < src.V; ++v) ++first[src.tile_of[v] + 1];
    for (uint32_t t = 0; t < src.tiles; ++t) first[t + 1] += first[t];
    std::vector<uint32_t> fill(first.begin(), first.end() - 1);
    for (uint32_t v = 0; v < src.V; ++v) list[fill[src.tile_of[v]]++] = v;
    own_first.upload(first.data(), first.size(), s);
    own.upload(list.data(), list.size(), s);
    tile_of.upload(src.tile_of, src.V, s);
    cfirst.upload(src.color_elements, src.ncolors + 1, s);
    tfirst.upload(src.color_constraints, src.ncolors + 1, s);
    table.alloc(std::size_t(src.ncolors) * src.V);
    launch_fill_u32(s, table.p, kNone, uint32_t(table.n));
    plan_dev const d = view(src, cfirst, tfirst, own_first, own, tile_of, table, bounds_dev, bits, vwords, ewords);
    unsigned const grid = (src.elements + 255) / 256;
    src.hex ? k_tile_table<true><<<grid, 256, 0, s>>>(d, table.p) : k_tile_table<false><<<grid, 256, 0, s>>>(d, table.p);
    hip_check(hipGetLastError(), "tile table");
    hip_check(hipStreamSynchronize(s), "tile table");  // the host lists end here
}

tile_counts tile_scratch::count(std::vector<uint32_t> const& bounds)
{
    uint32_t const nseg = uint32_t(bounds.size()) - 1;
    tile_counts n;
    n.instances.assign(std::size_t(src.tiles) * src.ncolors, 0);
    n.particles.assign(std::size_t(nseg) * src.tiles, kNone);
    std::size_t const words = std::size_t(nseg) * src.tiles * (vwords + ewords);
    if (words * 4 > kTileScratch || words >= (std::size_t(1) << 32)) return n;
    if (bits.n < words) bits.alloc(words);
    bounds_dev.upload(bounds.data(), bounds.size(), s);
    counts.alloc(n.instances.size() + n.particles.size());
    launch_fill_u32(s, bits.p, 0u, uint32_t(words));
    launch_fill_u32(s, counts.p, 0u, uint32_t(counts.n));
    plan_dev const d = view(src, cfirst, tfirst, own_first, own, tile_of, table, bounds_dev, bits, vwords, ewords);
    std::size_t const lds = 2 * std::size_t(kTileParticles) * 4;
    auto const kernel = src.hex ? k_tile_cone<true> : k_tile_cone<false>;
    kernel<<<dim3(src.tiles, nseg), kTileBlock, lds, s>>>(d, counts.p, counts.p + n.instances.size());
    hip_check(hipGetLastError(), "tile counts");
    hip_check(hipMemcpyAsync(n.instances.data(), counts.p, n.instances.size() * 4, hipMemcpyDeviceToHost, s), "tile counts");
    hip_check(hipMemcpyAsync(n.particles.data(), counts.p + n.instances.size(), n.particles.size() * 4,
                             hipMemcpyDeviceToHost, s),
              "tile counts");
    hip_check(hipStreamSynchronize(s), "tile counts");
    return n;
}

void tile_scratch::build(std::vector<uint32_t> const& bounds, tile_counts const& n, tile_plan& plan)
{
    uint32_t const nseg = uint32_t(bounds.size()) - 1;
    std::vector<uint4> blocks, chunks;
    std::vector<uint32_t> firsts(n.instances.size());  // [tile][color]: its first instance
    // Instance 0 stands where a tile has no element of the segment's colors: the group's first constraints at the
    // tile's first place, read but never run. (Any other instance's places need hold no particle in this tile,
    // and the damping term follows a place's particle into the substep start positions.)
    std::size_t parts = 0, insts = 1;
    plan.segments.clear();
    for (uint32_t sg = 0; sg < nseg; ++sg) {
        tile_segment seg{bounds[sg], bounds[sg + 1], 0, 0, blocks.size()};
        for (uint32_t t = 0; t < src.tiles; ++t) {
            uint32_t const np = n.particles[std::size_t(sg) * src.tiles + t];
            std::size_t const chunk0 = chunks.size();
            uint32_t const part0 = uint32_t(parts);
            parts += np;
            for (uint32_t c = bounds[sg]; c < bounds[sg + 1]; ++c) {
                uint32_t const m = n.instances[std::size_t(t) * src.ncolors + c];
                firsts[std::size_t(t) * src.ncolors + c] = uint32_t(insts);
                for (uint32_t q = 0; q < m; q += kTileBlock)
                    chunks.push_back(make_uint4(uint32_t(insts) + q, std::min<uint32_t>(m - q, kTileBlock),
                                                src.color_elements[c + 1] - src.color_elements[c], q + kTileBlock >= m));
                insts += m;
            }
            seg.cap = std::max(seg.cap, (np + 63) & ~63u);
            if (chunks.size() == chunk0) chunks.push_back(make_uint4(0, 0, 1, 1));  // a tile without elements
            seg.chunks = std::max(seg.chunks, uint32_t(chunks.size() - chunk0));
            blocks.push_back(make_uint4(part0, np, uint32_t(chunk0), uint32_t(chunks.size() - chunk0)));
            blocks.push_back(chunks[chunk0]);
            blocks.push_back(chunks[std::min(chunk0 + 1, chunks.size() - 1)]);
        }
        plan.segments.push_back(seg);
    }
    int const per = src.hex ? kHexTets : 1;
    // offsets of 32 bits; as with a plan that memory has no room for, the caller does without
    require(parts < (std::size_t(1) << 31) && insts * per < (std::size_t(1) << 29), "tile plan too large",
            SBS_ERR_OUT_OF_MEMORY);
    plan.blocks.upload(blocks.data(), blocks.size(), s);
    plan.chunks.upload(chunks.data(), chunks.size(), s);
    counts.upload(firsts.data(), firsts.size(), s);
    plan.particles.alloc(parts);
    plan.elems.alloc(insts);
    if (src.hex)
        plan.corners8.alloc(insts);
    else
        plan.corners4.alloc(insts);
    launch_fill_u32(s, plan.elems.p, 0u, 1);
    launch_fill_u32(s, src.hex ? reinterpret_cast<uint32_t*>(plan.corners8.p) : reinterpret_cast<uint32_t*>(plan.corners4.p),
                    0u, src.hex ? 4 : 2);
    plan.lambda.alloc(2 * insts * per);
    plan.instances = uint32_t(insts);
    bounds_dev.upload(bounds.data(), bounds.size(), s);
    plan_dev const d = view(src, cfirst, tfirst, own_first, own, tile_of, table, bounds_dev, bits, vwords, ewords);
    std::size_t const lds = std::size_t(kTileParticles) * 4;
    auto const kernel = src.hex ? k_tile_emit<true> : k_tile_emit<false>;
    kernel<<<dim3(src.tiles, nseg), kTileBlock, lds, s>>>(d, plan.blocks.p, counts.p, src.surface_of, plan.particles.p,
                                                          plan.elems.p, plan.corners8.p, plan.corners4.p);
    hip_check(hipGetLastError(), "tile plan");
    // the largest tile's LDS, whatever this plan's: the limit belongs to the kernels and is shared by all
    // simulations of the process, so it is always set to the same size
    allow_lds(kTileLds, k_tile_hex<0, false>, k_tile_hex<0, true>, k_tile_hex<1, false>, k_tile_hex<1, true>,
              k_tile_tets<0, false>, k_tile_tets<0, true>, k_tile_tets<1, false>, k_tile_tets<1, true>);
    hip_check(hipStreamSynchronize(s), "tile plan");
    plan.tiles = src.tiles;
}

void launch_tile_segment(hipStream_t s, tile_plan const& plan, std::size_t segment, int kind, bool hex,
                         tet_group_dev const& g, const pos4* in, pos4* out, const pos4* xn, contact_dev const& c,
                         tile_params const& p)
{
    tile_segment const& seg = plan.segments[segment];
    uint32_t const per = (plan.tiles + kXcds - 1) / kXcds;
    tile_dev const d{plan.blocks.p + seg.blocks, plan.chunks.p,   plan.particles.p, plan.elems.p,
                     plan.corners8.p,            plan.corners4.p, plan.lambda.p,    plan.tiles,
                     per,                        seg.cap,         plan.instances};
    std::size_t const lds = std::size_t(seg.cap) * kTileBytes + std::size_t(seg.chunks) * 16;
    auto run = [&](auto kernel) { kernel<<<per * kXcds, kTileThreads, lds, s>>>(d, g, in, out, xn, c, p); };
    bool const damped = kind == 0 ? p.gamma != 0.0f : p.beta_dt != 0.0f;
    if (hex && kind == 0)
        damped ? run(k_tile_hex<0, true>) : run(k_tile_hex<0, false>);
    else if (hex)
        damped ? run(k_tile_hex<1, true>) : run(k_tile_hex<1, false>);
    else if (kind == 0)
        damped ? run(k_tile_tets<0, true>) : run(k_tile_tets<0, false>);
    else
        damped ? run(k_tile_tets<1, true>) : run(k_tile_tets<1, false>);
    hip_check(hipGetLastError(), "tile launch");
}

}  // namespace sbs
