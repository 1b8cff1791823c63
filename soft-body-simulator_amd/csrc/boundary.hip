// Boundary surface extraction on the device (tetrahedral_mesh_boundary_t::extract_boundary_surface,
// src/physics/tetrahedral_mesh_boundary.cpp:65-120, with the face numbering of
// tetrahedron_set_t::add_tetrahedron, src/physics/topology.cpp:904-956).
//
// Face q = 4 t + f of tet t has the vertex order of tetrahedron_t::faces_copy
// {v1v2v4, v2v3v4, v3v1v4, v1v3v2} (topology.cpp:335-342). Equal faces (the same three vertices) are one
// triangle of the mesh, created by its first face. A face finds the others in a hash table of face indices: the
// one that takes the slot stands for all, and the others count themselves there and leave the smallest index.
// Triangles of other than two faces are the boundary, in the order of their first faces and with those faces'
// vertex orders; surface vertices are numbered by first appearance along the boundary triangles. Both orders
// are bits set at indices and the bits' prefix sums, so nothing is sorted.
//
// What bounds it: at 1M tets (4M faces, 1.65 ms a call) the upload of 16 MB from the caller's memory, 0.9 ms;
// then the insertion's random accesses, an atomic on the table and a look at another tet for each face, 279 us
// of 430 on the device. Sorting the faces by their keys moved them through seven radix passes, 149 launches
// and 860 us; its 18 buffers took 2.6 ms of a call of 4.5 to allocate and free, the two here 0.4.
#include "abi_util.h"
#include "kernels.h"
#include "scan_sort.h"
#include "sbs_gpu.h"

namespace sbs {

namespace {

unsigned grid_for(std::size_t n) { return unsigned((n + 255) / 256); }

__device__ __forceinline__ void face_vertices(const uint32_t* tets, uint32_t q, uint32_t v[3])
{
    uint32_t const t = q >> 2, f = q & 3u;
    int const a = f == 0 ? 0 : (f == 1 ? 1 : (f == 2 ? 2 : 0));
    int const b = f == 0 ? 1 : (f == 1 ? 2 : (f == 2 ? 0 : 2));
    int const c = f == 3 ? 1 : 3;
    v[0] = tets[4 * std::size_t(t) + a];
    v[1] = tets[4 * std::size_t(t) + b];
    v[2] = tets[4 * std::size_t(t) + c];
}

// the vertices ascending
struct face_key {
    uint32_t a, b, c;
    __device__ __forceinline__ face_key(const uint32_t* tets, uint32_t q)
    {
        uint32_t v[3];
        face_vertices(tets, q, v);
        a = min(v[0], min(v[1], v[2]));
        c = max(v[0], max(v[1], v[2]));
        b = v[0] + v[1] + v[2] - a - c;
    }
    __device__ __forceinline__ bool operator==(face_key const& o) const { return a == o.a && b == o.b && c == o.c; }
    __device__ __forceinline__ uint32_t hash() const
    {
        uint32_t h = a * 0x9e3779b1u;
        h = (h ^ (h >> 15)) + b;
        h *= 0x85ebca77u;
        h = (h ^ (h >> 13)) + c;
        h *= 0xc2b2ae3du;
        h ^= h >> 16;
        h *= 0x27d4eb2fu;
        return h ^ (h >> 15);
    }
};

constexpr uint32_t kEmpty = 0xffffffffu, kNotFirst = 0x80000000u;

__global__ void k_check_indices(const uint4* __restrict__ tets, uint32_t n, uint32_t nv, uint32_t* __restrict__ bad)
{
    uint32_t const t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    uint4 const v = tets[t];
    if (max(max(v.x, v.y), max(v.z, v.w)) >= nv) *bad = 1;
}

// table (slots words, more than there are faces): a face of each triangle; others[q]: how many more faces the
// triangle of such a face q has, kNotFirst for the rest; least[q]: the smallest of those
__global__ void k_insert_faces(const uint32_t* __restrict__ tets, uint32_t nf, uint32_t slots,
                               uint32_t* __restrict__ table, uint32_t* __restrict__ others, uint32_t* __restrict__ least)
{
    uint32_t const q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nf) return;
    face_key const key(tets, q);
    uint32_t at = uint32_t((uint64_t(key.hash()) * slots) >> 32);
    for (;;) {
        uint32_t const r = atomicCAS(&table[at], kEmpty, q);
        if (r == kEmpty) return;
        if (face_key(tets, r) == key) {
            others[q] = kNotFirst;
            atomicAdd(&others[r], 1u);
            atomicMin(&least[r], q);
            return;
        }
        if (++at == slots) at = 0;
    }
}

// a bit for the first face of every boundary triangle
__global__ void k_boundary_bits(const uint32_t* __restrict__ others, const uint32_t* __restrict__ least, uint32_t nf,
                                uint32_t* __restrict__ bits)
{
    uint32_t const q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nf) return;
    uint32_t const n = others[q];
    if (n == kNotFirst || n == 1) return;
    uint32_t const f = min(q, least[q]);
    atomicOr(&bits[f >> 5], 1u << (f & 31u));
}

__global__ void k_count_bits(const uint32_t* __restrict__ bits, uint32_t words, uint32_t* __restrict__ count)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < words) count[i] = uint32_t(__popc(bits[i]));
}

// the indices of the set bits, in order
__global__ void k_list_bits(const uint32_t* __restrict__ bits, const uint32_t* __restrict__ before, uint32_t words,
                            uint32_t* __restrict__ out)
{
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= words) return;
    uint32_t at = before[i];
    for (uint32_t b = bits[i]; b; b &= b - 1) out[at++] = 32u * i + uint32_t(__ffs(int(b))) - 1u;
}

// each vertex's first corner along the boundary triangles
__global__ void k_first_corners(const uint32_t* __restrict__ tets, const uint32_t* __restrict__ faces, uint32_t nt,
                                uint32_t* __restrict__ first)
{
    uint32_t const j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nt) return;
    uint32_t v[3];
    face_vertices(tets, faces[j], v);
    for (uint32_t c = 0; c < 3; ++c) atomicMin(&first[v[c]], 3 * j + c);
}

__global__ void k_corner_bits(const uint32_t* __restrict__ first, uint32_t nv, uint32_t* __restrict__ bits)
{
    uint32_t const v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv || first[v] == kEmpty) return;
    atomicOr(&bits[first[v] >> 5], 1u << (first[v] & 31u));
}

// the vertices by their first corners
__global__ void k_number_vertices(const uint32_t* __restrict__ first, uint32_t nv, const uint32_t* __restrict__ bits,
                                  const uint32_t* __restrict__ before, uint32_t* __restrict__ s_of,
                                  uint32_t* __restrict__ verts)
{
    uint32_t const v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv || first[v] == kEmpty) return;
    uint32_t const c = first[v], w = c >> 5;
    uint32_t const s = before[w] + uint32_t(__popc(bits[w] & ((1u << (c & 31u)) - 1u)));
    s_of[v] = s;
    verts[s] = v;
}

__global__ void k_triangles(const uint32_t* __restrict__ tets, const uint32_t* __restrict__ faces, uint32_t nt,
                            const uint32_t* __restrict__ s_of, uint32_t* __restrict__ tri)
{
    uint32_t const j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nt) return;
    uint32_t v[3];
    face_vertices(tets, faces[j], v);
    for (int c = 0; c < 3; ++c) tri[3 * j + c] = s_of[v[c]];
}

uint32_t read_word(hipStream_t s, const uint32_t* p)
{
    uint32_t h = 0;
    hip_check(hipMemcpyAsync(&h, p, sizeof(uint32_t), hipMemcpyDeviceToHost, s), "read count");
    hip_check(hipStreamSynchronize(s), "read count");
    return h;
}

// Parts of one device allocation, each at a multiple of 256 bytes: reserve() first, then alloc(), then at().
struct device_arena {
    dev_buf<uint32_t> mem;
    std::size_t words = 0;
    std::size_t reserve(std::size_t n)
    {
        std::size_t const o = words;
        words += (n + 63) & ~std::size_t(63);
        return o;
    }
    void alloc() { mem.alloc(words); }
    uint32_t* at(std::size_t offset) const { return mem.p + offset; }
};

}  // namespace

}  // namespace sbs

using namespace sbs;

extern "C" int sbs_gpu_extract_boundary(int device, uint32_t num_vertices, const uint32_t* tets, uint32_t num_tets,
                                        uint32_t* surface_to_tet, uint32_t* triangles, uint32_t* num_surface_vertices,
                                        uint32_t* num_triangles)
{
    return guarded([&] {
        require(tets != nullptr || num_tets == 0, "tets is null");
        require(num_surface_vertices && num_triangles, "size outputs are null");
        require(num_vertices <= (1u << 21), "at most 2^21 vertices");
        require(num_tets <= (1u << 28), "at most 2^28 tets");
        // Bad indices are the caller's error whatever fails beside them, and leave the outputs alone. The device
        // looks for them; where it cannot, the host does.
        auto check_here = [&] {
            for (std::size_t i = 0; i < 4 * std::size_t(num_tets); ++i)
                require(tets[i] < num_vertices, "tet vertex index out of range");
            *num_surface_vertices = *num_triangles = 0;
        };
        if (num_tets == 0) return check_here();
        hipStream_t s = nullptr;
        hipError_t e = hipSetDevice(device);
        if (e == hipSuccess) e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
        if (e != hipSuccess) {
            check_here();
            hip_check(e, "boundary extraction");
        }
        bool checked = false;
        try {
            uint32_t const nf = 4 * num_tets, nv = num_vertices, fwords = (nf + 31) / 32;
            uint32_t const slots = uint32_t(nf + nf / 2 + 1);
            device_arena mem;
            std::size_t const o_tets = mem.reserve(nf), o_table = mem.reserve(slots), o_least = mem.reserve(nf);
            std::size_t const o_first = mem.reserve(nv);
            std::size_t const o_zero = mem.words;
            std::size_t const o_others = mem.reserve(nf), o_bits = mem.reserve(fwords), o_bad = mem.reserve(1);
            std::size_t const zeros = mem.words - o_zero;
            std::size_t const o_count = mem.reserve(fwords), o_before = mem.reserve(std::size_t(fwords) + 1);
            std::size_t const o_ws = mem.reserve(scan_workspace(fwords));
            mem.alloc();
            uint32_t* const dt = mem.at(o_tets);
            hip_check(hipMemcpyAsync(dt, tets, nf * sizeof(uint32_t), hipMemcpyHostToDevice, s), "upload tets");
            // the table, least and first start as ~0, one after the other
            launch_fill_u32(s, mem.at(o_table), kEmpty, uint32_t(o_zero - o_table));
            launch_fill_u32(s, mem.at(o_zero), 0u, uint32_t(zeros));
            k_check_indices<<<grid_for(num_tets), 256, 0, s>>>(reinterpret_cast<const uint4*>(dt), num_tets, nv, mem.at(o_bad));
            hip_check(hipGetLastError(), "boundary face kernels");
            bool const bad = read_word(s, mem.at(o_bad)) != 0;
            checked = true;
            require(!bad, "tet vertex index out of range");
            *num_surface_vertices = *num_triangles = 0;
            uint32_t *const bits = mem.at(o_bits), *const count = mem.at(o_count), *const before = mem.at(o_before);
            k_insert_faces<<<grid_for(nf), 256, 0, s>>>(dt, nf, slots, mem.at(o_table), mem.at(o_others), mem.at(o_least));
            k_boundary_bits<<<grid_for(nf), 256, 0, s>>>(mem.at(o_others), mem.at(o_least), nf, bits);
            k_count_bits<<<grid_for(fwords), 256, 0, s>>>(bits, fwords, count);
            exclusive_scan(s, count, before, fwords, mem.at(o_ws));
            hip_check(hipGetLastError(), "boundary face kernels");
            uint32_t const nt = read_word(s, before + fwords);
            if (nt > 0) {
                uint32_t const nc = 3 * nt, cwords = (nc + 31) / 32;  // nt <= nf
                device_arena out;
                std::size_t const p_faces = out.reserve(nt), p_tri = out.reserve(nc), p_verts = out.reserve(nv);
                std::size_t const p_sof = out.reserve(nv), p_bits = out.reserve(cwords), p_count = out.reserve(cwords);
                std::size_t const p_before = out.reserve(std::size_t(cwords) + 1), p_ws = out.reserve(scan_workspace(cwords));
                out.alloc();
                uint32_t *const faces = out.at(p_faces), *const first = mem.at(o_first), *const cbits = out.at(p_bits);
                launch_fill_u32(s, cbits, 0u, cwords);
                k_list_bits<<<grid_for(fwords), 256, 0, s>>>(bits, before, fwords, faces);
                k_first_corners<<<grid_for(nt), 256, 0, s>>>(dt, faces, nt, first);
                k_corner_bits<<<grid_for(nv), 256, 0, s>>>(first, nv, cbits);
                k_count_bits<<<grid_for(cwords), 256, 0, s>>>(cbits, cwords, out.at(p_count));
                exclusive_scan(s, out.at(p_count), out.at(p_before), cwords, out.at(p_ws));
                k_number_vertices<<<grid_for(nv), 256, 0, s>>>(first, nv, cbits, out.at(p_before), out.at(p_sof),
                                                               out.at(p_verts));
                k_triangles<<<grid_for(nt), 256, 0, s>>>(dt, faces, nt, out.at(p_sof), out.at(p_tri));
                hip_check(hipGetLastError(), "boundary kernels");
                uint32_t const ns = read_word(s, out.at(p_before) + cwords);
                if (surface_to_tet)
                    hip_check(hipMemcpyAsync(surface_to_tet, out.at(p_verts), ns * sizeof(uint32_t),
                                             hipMemcpyDeviceToHost, s),
                              "read surface vertices");
                if (triangles)
                    hip_check(hipMemcpyAsync(triangles, out.at(p_tri), nc * sizeof(uint32_t), hipMemcpyDeviceToHost, s),
                              "read triangles");
                hip_check(hipStreamSynchronize(s), "boundary extraction");
                *num_surface_vertices = ns;
                *num_triangles = nt;
            }
        } catch (...) {
            (void)hipStreamDestroy(s);
            if (!checked) check_here();
            throw;
        }
        hip_check(hipStreamDestroy(s), "hipStreamDestroy");
    });
}
