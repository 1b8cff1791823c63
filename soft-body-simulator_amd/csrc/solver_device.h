// Device functions of the time step shared by the kernels that run one stage per launch (kernels.hip), several
// colors of a large body (tile.hip), or a whole frame of a small body (island.hip): position arithmetic,
// prediction and velocity update, the Green, stable neo-Hookean and contact projections.
#pragma once
#include <type_traits>

#include "device_math.h"
#include "kernels.h"

namespace sbs {

namespace {

// base[i] with base uniform over the wave: one 32-bit byte offset per lane beside the scalar base (a
// 64-bit address per lane and array costs two more instructions each). i * sizeof(T) must stay below
// 2^32. For the index of a cluster in its color it does at 16 bytes: 2^28 clusters of one color, which
// share no particle, would hold 2^31 particles, 172 GB of positions beside 100 GB of constraints.
template <class T>
__device__ __forceinline__ auto lane_address(T* base, uint32_t i)
{
    // the base in scalar registers: folded into the lane's part it would make that 64 bits again
    auto b = (__attribute__((address_space(1))) char*)(const_cast<std::remove_const_t<T>*>(base));
    asm("" : "+s"(b));
    using bits = __attribute__((ext_vector_type(sizeof(T) / 4))) float;
    return (__attribute__((address_space(1))) bits*)(b + uint32_t(i * uint32_t(sizeof(T))));
}

template <class T>
__device__ __forceinline__ std::remove_const_t<T> lane_load(T* base, uint32_t i)
{
    return __builtin_bit_cast(std::remove_const_t<T>, *lane_address(base, i));
}

template <class T>
__device__ __forceinline__ void lane_store(T* base, uint32_t i, T v)
{
    auto o = lane_address(base, i);
    *o = __builtin_bit_cast(std::remove_reference_t<decltype(*lane_address(base, i))>, v);
}

// The loads before this point are issued before it, and nothing moves across: without a branch between
// a prefetch and its uses the compiler sinks the loads down to them (the empty asm orders the memory
// instructions, the scheduling barrier keeps the asm where it stands).
__device__ __forceinline__ void loads_issued()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// A record that every lane holds, in scalar registers.
__device__ __forceinline__ uint4 uniform(uint4 r)
{
    auto word = [](uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); };
    return make_uint4(word(r.x), word(r.y), word(r.z), word(r.w));
}

// A workgroup barrier that orders LDS only. __syncthreads also waits for every global load and store in
// flight, the next stage's prefetched data among them.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// a - b of two positions, rounded to FP32
__device__ __forceinline__ v3 sub(pos4 a, pos4 b)
{
    return {float(a.x - b.x), float(a.y - b.y), float(a.z - b.z)};
}
// p += d (an FP32 correction) in FP64
__device__ __forceinline__ void add_to(pos4& p, v3 d)
{
    p.x += double(d.x);
    p.y += double(d.y);
    p.z += double(d.z);
}
__device__ __forceinline__ float wof(pos4 p) { return float(p.w); }

// timestep.cpp:35-43: v += a dt, xi = x + v dt. With gravity_is_force the acceleration is
// g * w (the reference's f = g, a = f w); otherwise g for every particle with w > 0.
__device__ __forceinline__ void predict_one(pos4& xi, pos4 const& x, float4& v, float gx, float gy, float gz,
                                            int force, float dt)
{
    float const w = wof(x);
    float ax, ay, az;
    if (force) {
        ax = gx * w;
        ay = gy * w;
        az = gz * w;
    } else if (w > 0.0f) {
        ax = gx;
        ay = gy;
        az = gz;
    } else {
        ax = ay = az = 0.0f;
    }
    v.x = v.x + ax * dt;
    v.y = v.y + ay * dt;
    v.z = v.z + az * dt;
    double const d = dt;
    xi = make_double4(x.x + double(v.x) * d, x.y + double(v.y) * d, x.z + double(v.z) * d, x.w);
}

// timestep.cpp:48-57: x = xi, v = (x - xn)/dt, xn = x.
__device__ __forceinline__ float4 velocity(pos4 p, pos4 q, float dt)
{
    double const d = dt;
    return make_float4(float((p.x - q.x) / d), float((p.y - q.y) / d), float((p.z - q.z) / d), 0.0f);
}

struct tet_rows {
    v3 r0, r1, r2;
};

__device__ __forceinline__ tet_rows load_rows(float4 a, float4 b, float4 c)
{
    return {mk(a.x, a.y, a.z), mk(a.w, b.x, b.y), mk(b.z, b.w, c.x)};
}

// green_constraint.cpp:61-133 on the edge vectors e_k = p_k - p_4. Computes C = |V0| psi and
// f1..f4 = -grad C, with the reference's inversion flip of the smallest singular value (:92-96),
// the 0.577 clamp (:99-102), the StVK first Piola stress of the clamped F^ mapped back with U, V
// (:104-112), and psi from E = U E^ V^T: |E|_F^2 = sum e_i^2, tr(E) = sum e_i (u_i . v_i) (:108-110).
__device__ __forceinline__ float green_core(v3 e0, v3 e1, v3 e2, tet_rows const& R, float V0, float mu, float la,
                                            v3 f[4])
{
    float const det = dot(e0, cross(e1, e2));
    bool const inverted = (det >= 0.0f) != (V0 >= 0.0f);
    m3 const F = deformation_gradient(e0, e1, e2, R.r0, R.r1, R.r2);
    m3 U, V;
    float s[3];
    svd3(F, U, s, V);
    // reference convention: non-negative singular values, the smallest negated iff inverted
    float s2 = inverted ? -fabsf(s[2]) : fabsf(s[2]);
    if ((s2 < 0.0f) != (s[2] < 0.0f)) U.c2 = -U.c2;
    float const f0 = fmaxf(s[0], 0.577f), f1 = fmaxf(s[1], 0.577f), f2 = fmaxf(s2, 0.577f);
    float const h0 = 0.5f * (f0 * f0 - 1.0f), h1 = 0.5f * (f1 * f1 - 1.0f), h2 = 0.5f * (f2 * f2 - 1.0f);
    float const tr = h0 + h1 + h2;
    float const ph0 = f0 * (2.0f * mu * h0 + la * tr);
    float const ph1 = f1 * (2.0f * mu * h1 + la * tr);
    float const ph2 = f2 * (2.0f * mu * h2 + la * tr);
    float const trE = h0 * dot(U.c0, V.c0) + h1 * dot(U.c1, V.c1) + h2 * dot(U.c2, V.c2);
    float const psi = mu * (h0 * h0 + h1 * h1 + h2 * h2) + 0.5f * la * trE * trE;
    float const aV0 = fabsf(V0);
    // f_k = -|V0| P r_k, P = sum_i ph_i u_i v_i^T
    float const a0 = -aV0 * ph0, a1 = -aV0 * ph1, a2 = -aV0 * ph2;
    auto force = [&](v3 r) { return (a0 * dot(V.c0, r)) * U.c0 + (a1 * dot(V.c1, r)) * U.c1 + (a2 * dot(V.c2, r)) * U.c2; };
    f[0] = force(R.r0);
    f[1] = force(R.r1);
    f[2] = force(R.r2);
    f[3] = -(f[0] + f[1] + f[2]);
    return aV0 * psi;
}

// One green projection of the tet (P0..P3) with material (a, b, c) and multiplier lm; xn_of(k) is
// the substep start position of vertex k in P's frame, read only for the damping term. Returns
// false on the epsilon early-out.
template <class Pos, class XnOf>
__device__ __forceinline__ bool green_project(Pos P[4], XnOf&& xn_of, float4 a, float4 b, float4 c, float alpha_tilde,
                                              float gamma, float& lm)
{
    v3 f[4];
    float const C = green_core(sub(P[0], P[3]), sub(P[1], P[3]), sub(P[2], P[3]), load_rows(a, b, c), c.y, c.z, c.w, f);
    float const wsum = wof(P[0]) * dot(f[0], f[0]) + wof(P[1]) * dot(f[1], f[1]) + wof(P[2]) * dot(f[2], f[2]) +
                       wof(P[3]) * dot(f[3], f[3]);
    if (wsum < 1e-20f) return false;  // green_constraint.cpp:130-131
    float gdd = 0.0f;
    if (gamma != 0.0f) {  // damping term (:140-144)
        gdd = dot(f[0], sub(P[0], xn_of(0))) + dot(f[1], sub(P[1], xn_of(1))) + dot(f[2], sub(P[2], xn_of(2))) +
              dot(f[3], sub(P[3], xn_of(3)));
    }
    float const dl = hw_div(-(C + alpha_tilde * lm) + gamma * gdd, (1.0f + gamma) * wsum + alpha_tilde);
    lm += dl;
    // xi += w (-f) dl (:154-157)
#pragma unroll
    for (int k = 0; k < 4; ++k) add_to(P[k], -(wof(P[k]) * dl) * f[k]);
    return true;
}

// ---------------------------------------------------------------- stable neo-Hookean constraint

// A tet in FP32 relative form for a sequence of constraint updates: edges e_k = p_k - p_3, the
// displacements dx_k = p_k - xn_k since the substep start (only with damping), the inverse masses
// and the corrections d_k accumulated so far. The FP64 differences are taken once; each update
// then moves the FP32 quantities, and the positions receive the sum of the corrections once.
struct tet_frame {
    v3 e[3], dx[4], d[4];
    float w[4];
};

template <class Pos, class XnOf>
__device__ __forceinline__ tet_frame make_frame(Pos const P[4], XnOf&& xn_of, bool damped)
{
    tet_frame f;
#pragma unroll
    for (int k = 0; k < 3; ++k) f.e[k] = sub(P[k], P[3]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f.w[k] = wof(P[k]);
        f.d[k] = mk(0.0f, 0.0f, 0.0f);
        f.dx[k] = damped ? sub(P[k], xn_of(k)) : mk(0.0f, 0.0f, 0.0f);
    }
    return f;
}

// Rest data of a neo-Hookean tet: with R = DmInv (rows r_k), Ds = [e0 e1 e2] and F = Ds R,
//   ||F||_F^2 = sum_mn (e_m . e_n) Q_mn and F r_k = sum_m Q_mk e_m, Q = R R^T (symmetric);
//   cof(F) r_k = cof(Ds) cof(R) r_k = det(R) (e_{k+1} x e_{k+2}), det F = det(R) e0 . (e1 x e2)
// (cof(R) = det(R) R^-T and R^-T r_k = Dm^T r_k is the unit vector k). So the deviatoric gradient
// dC/dx_k = F r_k / ||F|| and the hydrostatic one cof(F) r_k need no F and no cofactor matrix.
// Material layout (40 B per tet): m0 = (Q00, Q11, Q22, Q01), m1 = (Q02, Q12, det R, 1/(mu|V0|)),
// and m2 read as float2 per tet = (1/(lambda|V0|), 1 + mu/lambda).
struct nh_rest {
    float q00, q11, q22, q01, q02, q12, detr;
};

__device__ __forceinline__ nh_rest load_nh(float4 a, float4 b) { return {a.x, a.y, a.z, a.w, b.x, b.y, b.z}; }

__device__ __forceinline__ float2 nh_m2(tet_group_dev const& g, uint32_t t)
{
    return reinterpret_cast<const float2*>(g.m2)[t];
}

// The neo-Hookean updates below spell out every fused multiply-add and contract nothing else, so
// their rounding is fixed by the source and not by the kernel they are inlined into: the hex
// kernel's launch variants (material prefetched or streamed) give bit-identical positions.
#pragma clang fp contract(on)

__device__ __forceinline__ float fdot(v3 a, v3 b) { return fmaf(a.z, b.z, fmaf(a.y, b.y, a.x * b.x)); }

__device__ __forceinline__ v3 fcross(v3 a, v3 b)
{
    return {fmaf(a.y, b.z, -(a.z * b.y)), fmaf(a.z, b.x, -(a.x * b.z)), fmaf(a.x, b.y, -(a.y * b.x))};
}

// a e0 + b e1 + c e2
__device__ __forceinline__ v3 fcomb(float a, v3 e0, float b, v3 e1, float c, v3 e2)
{
    return {fmaf(c, e2.x, fmaf(b, e1.x, a * e0.x)), fmaf(c, e2.y, fmaf(b, e1.y, a * e0.y)),
            fmaf(c, e2.z, fmaf(b, e1.z, a * e0.z))};
}

// x + s a
__device__ __forceinline__ v3 faxpy(float s, v3 a, v3 x) { return {fmaf(s, a.x, x.x), fmaf(s, a.y, x.y), fmaf(s, a.z, x.z)}; }

// -(a + b + c)
__device__ __forceinline__ v3 fnegsum(v3 a, v3 b, v3 c)
{
    return {-((a.x + b.x) + c.x), -((a.y + b.y) + c.y), -((a.z + b.z) + c.z)};
}

// Deviatoric constraint C = ||F||_F at edges e; gradients s h_k with s = 1/C (0 when C = 0).
__device__ __forceinline__ float nh_deviatoric(v3 const e[3], nh_rest const& q, v3 h[4], float& s)
{
    float const g00 = fdot(e[0], e[0]), g11 = fdot(e[1], e[1]), g22 = fdot(e[2], e[2]);
    float const g01 = fdot(e[0], e[1]), g02 = fdot(e[0], e[2]), g12 = fdot(e[1], e[2]);
    float const off = fmaf(q.q01, g01, fmaf(q.q02, g02, q.q12 * g12));
    float const c2 = fmaf(q.q00, g00, fmaf(q.q11, g11, fmaf(q.q22, g22, 2.0f * off)));
    float const C = hw_sqrt(fmaxf(c2, 0.0f));
    s = C > 0.0f ? hw_rcp(C) : 0.0f;
    h[0] = fcomb(q.q00, e[0], q.q01, e[1], q.q02, e[2]);
    h[1] = fcomb(q.q01, e[0], q.q11, e[1], q.q12, e[2]);
    h[2] = fcomb(q.q02, e[0], q.q12, e[1], q.q22, e[2]);
    h[3] = fnegsum(h[0], h[1], h[2]);
    return C;
}

// Hydrostatic constraint C = det F - gamma0 at edges e; gradients s h_k with s = det R.
__device__ __forceinline__ float nh_hydrostatic(v3 const e[3], nh_rest const& q, float gamma0, v3 h[4], float& s)
{
    h[0] = fcross(e[1], e[2]);
    h[1] = fcross(e[2], e[0]);
    h[2] = fcross(e[0], e[1]);
    h[3] = fnegsum(h[0], h[1], h[2]);
    s = q.detr;
    return fmaf(q.detr, fdot(e[0], h[0]), -gamma0);
}

// Sum over the tet's vertices of w_k |s h_k|^2.
__device__ __forceinline__ float grad_norm2(float const w[4], v3 const h[4], float s)
{
    float const n = fmaf(w[3], fdot(h[3], h[3]), fmaf(w[2], fdot(h[2], h[2]), fmaf(w[1], fdot(h[1], h[1]), w[0] * fdot(h[0], h[0]))));
    return (s * s) * n;
}

// One XPBD update of a tet constraint with gradients g_k = s h_k: dl from the multiplier and the
// damping term, then d_k += w_k s dl h_k (and dx_k), e_k += (corr_k - corr_3). FIRST: the tet's first
// update (d_k starts at zero). A constraint whose sum w|g|^2 is below the epsilon gets dl = 0, which
// leaves every value as it is: a select, where an early return cost a branch and the registers' zeroing
// at its join. Undamped the damping terms are compiled out (x + 0 * y keeps x's bits); as a run-time
// zero they stayed, with a second branch: 19 VALU and 10 scalar instructions a tet of 266 in all
// (k_neohookean_hex 8.93 -> 8.17 us per launch on the 1M beam, 6.42 -> 5.87 on a 129k beam, kernel trace).
template <bool DAMPED, bool FIRST>
__device__ __forceinline__ void tet_update(tet_frame& f, v3 const h[4], float s, float C, float alpha_tilde,
                                           float gamma, float& lm)
{
    float const wsum = grad_norm2(f.w, h, s);
    float dl;
    if (DAMPED) {
        float const gdd =
            s * (((fdot(h[0], f.dx[0]) + fdot(h[1], f.dx[1])) + fdot(h[2], f.dx[2])) + fdot(h[3], f.dx[3]));
        dl = hw_div(fmaf(gamma, gamma != 0.0f ? gdd : 0.0f, -fmaf(alpha_tilde, lm, C)),
                    fmaf(1.0f + gamma, wsum, alpha_tilde));
    } else {
        dl = hw_div(-fmaf(alpha_tilde, lm, C), wsum + alpha_tilde);
    }
    dl = wsum < 1e-20f ? 0.0f : dl;
    lm += dl;
    float const sd = s * dl;
    float ws[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        ws[k] = f.w[k] * sd;
        f.d[k] = FIRST ? mk(ws[k] * h[k].x, ws[k] * h[k].y, ws[k] * h[k].z) : faxpy(ws[k], h[k], f.d[k]);
        if (DAMPED) f.dx[k] = faxpy(ws[k], h[k], f.dx[k]);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) f.e[k] = faxpy(ws[k], h[k], faxpy(-ws[3], h[3], f.e[k]));
}

// Deviatoric then hydrostatic projection of one tet (P0..P3), multipliers lm = (deviatoric,
// hydrostatic), material (a, b, c) as laid out at nh_rest. xn_of(k) is the substep start position
// of vertex k, read only with damping.
template <bool DAMPED, class Pos, class XnOf>
__device__ __forceinline__ void neohookean_project(Pos P[4], XnOf&& xn_of, float4 a, float4 b, float2 c, float inv_dt2,
                                                   float beta_dt, float2& lm)
{
    nh_rest const q = load_nh(a, b);
    tet_frame f = make_frame(P, xn_of, DAMPED);
    {  // deviatoric: C = ||F||_F, compliance 1/(mu |V0|)
        v3 h[4];
        float s;
        float const C = nh_deviatoric(f.e, q, h, s);
        float const at = b.w * inv_dt2;
        tet_update<DAMPED, true>(f, h, s, C, at, DAMPED ? at * beta_dt : 0.0f, lm.x);
    }
    {  // hydrostatic: C = det F - (1 + mu/lambda), compliance 1/(lambda |V0|)
        v3 h[4];
        float s;
        float const C = nh_hydrostatic(f.e, q, c.y, h, s);
        float const at = c.x * inv_dt2;
        tet_update<DAMPED, false>(f, h, s, C, at, DAMPED ? at * beta_dt : 0.0f, lm.y);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) add_to(P[k], f.d[k]);
}

// Warm-start displacement of one tet at positions P (the predicted positions): both gradients at
// P, d_k = w_k (grad_k C_dev lm.x + grad_k C_hyd lm.y). With explicit the multipliers are first
// set to -C(P) / alpha~, the pair that zeroes the XPBD residual at P; then they are multiplied by
// scale (x: deviatoric, y: hydrostatic; the caller stores them back). A constraint whose
// sum w|grad C|^2 is below the projection's epsilon contributes nothing, as it would not project.
template <class Pos>
__device__ __forceinline__ void neohookean_displacement(Pos const P[4], float4 a, float4 b, float2 c, float inv_dt2,
                                                        bool expl, float2 scale, float2& lm, v3 d[4])
{
    nh_rest const q = load_nh(a, b);
    tet_frame const f = make_frame(P, [](int) { return pos4{}; }, false);
    v3 hd[4], hh[4];
    float sd, sh;
    float const Cd = nh_deviatoric(f.e, q, hd, sd);
    float const Ch = nh_hydrostatic(f.e, q, c.y, hh, sh);
    if (expl) lm = make_float2(-Cd / (b.w * inv_dt2), -Ch / (c.x * inv_dt2));
    lm = make_float2(scale.x * lm.x, scale.y * lm.y);
    float const wd = grad_norm2(f.w, hd, sd), wh = grad_norm2(f.w, hh, sh);
    float const ld = wd < 1e-20f ? 0.0f : lm.x * sd, lh = wh < 1e-20f ? 0.0f : lm.y * sh;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float const a = f.w[k] * ld, b = f.w[k] * lh;
        d[k] = faxpy(b, hh[k], mk(a * hd[k].x, a * hd[k].y, a * hd[k].z));
    }
}

// The contacts of surface vertex s (all its slots in SDF order) projected onto P, the vertex's
// position (collision_constraint.cpp:21-41): C = (p - q).n; when C < 0, dl = -(C + alpha~ lm) /
// (w + alpha~), lm += dl, p += w n dl. first: the first iteration (multipliers start at zero, and
// are stored as zero for slots without penetration). For a contact with a surface triangle, q is the
// triangle's point of the stored barycentric weights b at the copied surface positions, plus h n, and
// the denominator adds that point's inverse mass sum_k b_k^2 w_k: the vertex moves by its share of
// the two-sided projection (the triangle's corners take theirs through their own contacts).
// One slot: q and n the plane, wt the plane point's inverse mass, lm the multiplier; returns it updated.
__device__ __forceinline__ float contact_slot(pos4& P, pos4 q, v3 n, float w, float wt, float alpha_tilde, float lm)
{
    float const C = fdot(sub(P, q), n);
    if (C >= 0.0f) return lm;
    float const dl = -fmaf(alpha_tilde, lm, C) / (w + wt + alpha_tilde);
    float const sd = w * dl;
    P.x += double(sd * n.x);
    P.y += double(sd * n.y);
    P.z += double(sd * n.z);
    return lm + dl;
}

// Slots [k0, cnt) of vertex s. snap(r): the position of surface vertex r that triangle contacts refer to;
// set(slot, lm) takes the updated multiplier, which is read from c.lambda.
template <class Snap, class Set>
__device__ __forceinline__ void contact_slots(contact_dev const& c, pos4& P, uint32_t s, uint32_t k0, uint32_t cnt,
                                              float alpha_tilde, bool first, Snap&& snap, Set&& set)
{
    float const w = wof(P);
    for (uint32_t k = k0; k < cnt; ++k) {
        uint32_t const slot = k * c.S + s;
        pos4 q = c.q[slot];
        v3 const n = xyz(c.n[slot]);
        float wt = 0.0f;
        if (c.snap && q.w >= double(c.nsdf)) {  // a surface triangle: its closest point as it is now
            uint4 const tr = c.btris[uint32_t(q.w) - c.nsdf];
            pos4 const a = snap(tr.x), b = snap(tr.y), d = snap(tr.z);
            wt = float(q.x * q.x * a.w + q.y * q.y * b.w + q.z * q.z * d.w);
            double const hx = c.body_h * double(n.x), hy = c.body_h * double(n.y), hz = c.body_h * double(n.z);
            q = make_double4(q.x * a.x + q.y * b.x + q.z * d.x + hx, q.x * a.y + q.y * b.y + q.z * d.y + hy,
                             q.x * a.z + q.y * b.z + q.z * d.z + hz, q.w);
        }
        set(slot, contact_slot(P, q, n, w, wt, alpha_tilde, first ? 0.0f : c.lambda[slot]));
    }
}

__device__ __forceinline__ void contact_slots(contact_dev const& c, pos4& P, uint32_t s, uint32_t k0, uint32_t cnt,
                                              float alpha_tilde, bool first)
{
    contact_slots(c, P, s, k0, cnt, alpha_tilde, first, [&](uint32_t r) { return c.snap[r]; },
                  [&](uint32_t slot, float lm) { c.lambda[slot] = lm; });
}

__device__ __forceinline__ void contact_vertex_at(contact_dev const& c, pos4& P, uint32_t s, float alpha_tilde,
                                                  bool first)
{
    contact_slots(c, P, s, 0, c.count[s], alpha_tilde, first);
}

#pragma clang fp contract(fast)

// Slot pattern shared by every cluster made of the 6 tets of one hex cell of the box split (slots
// numbered by first appearance). With the pattern known at compile time the 8 particles live in
// registers, and every constraint's material and multipliers are loaded before the first one
// runs. Inside a color the constraints are slot-major: tet k of the color's i-th cluster sits at
// tbase + k * count + i, so the loads of a wave coalesce.
constexpr int kHexTets = 6;

constexpr int kHexSlots[kHexTets][4] = {{0, 1, 2, 3}, {0, 4, 1, 3}, {0, 2, 5, 3}, {0, 5, 6, 3}, {0, 7, 4, 3}, {0, 6, 7, 3}};

}  // namespace

}  // namespace sbs
