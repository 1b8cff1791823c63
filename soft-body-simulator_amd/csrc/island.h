// Whole-frame kernels of small bodies (island.hip): one workgroup per island (body).
#pragma once
#include "kernels.h"

namespace sbs {

// LDS of a compute unit a workgroup may use for positions, and the bytes a particle takes there (three
// FP64 coordinates and its FP32 inverse mass); the rest holds the chunks, 16 bytes each, and the kernels' own
// words.
constexpr std::size_t kIslandLds = 160 * 1024, kIslandBytes = 28;
constexpr uint32_t kIslandChunks = 320;
constexpr std::size_t kIslandDynamicLds = kIslandLds - 512;
constexpr uint32_t kIslandParticles = uint32_t((kIslandDynamicLds - 16 * kIslandChunks) / kIslandBytes);
constexpr std::size_t island_lds_bytes(uint32_t particles, uint32_t chunks) { return particles * kIslandBytes + chunks * 16; }
static_assert(island_lds_bytes(kIslandParticles, kIslandChunks) <= kIslandDynamicLds, "the largest island fits");
// Constraints of a scene of islands: 16-byte offsets into its arrays fit 32 bits.
constexpr uint32_t kIslandConstraints = 1u << 28;

// The islands of a scene whose single constraint group is laid out island by island inside each color.
struct island_dev {
    const uint4* islands;  // 2 a piece: first particle, particles, first surface vertex, surface vertices;
                           // first chunk, chunks, 0, 0
    const uint4* chunks;   // up to a workgroup's elements of one color: first element, first constraint,
                           // constraint stride of a cluster's tets, elements (top bit: the color ends here)
    uint32_t* clist;       // scratch, one word per surface vertex
    uint32_t count;
    uint32_t cap;         // particles of the largest island (the stride of its LDS arrays)
    uint32_t chunks_cap;  // chunks of the island with the most
    uint32_t block;       // elements of a chunk, threads of a workgroup: island_block()
};

// 256 threads keep a wave to a SIMD; more where a stage of an island (largest: its elements) has more.
constexpr uint32_t island_block(bool hex, uint32_t largest) { return largest <= 256 ? 256 : (hex ? 512 : 1024); }

struct solve_params {
    uint32_t substeps, iterations;
    int predict, commit;          // start with the prediction, end with the velocity update
    int zero_first;               // multipliers start at zero in the first iteration of a substep
    int skip_first_contacts;      // the first iteration's contacts have been projected already
    float dt, g[3];
    int force;
    float contact_at;
    float alpha_tilde, gamma;     // Green
    float inv_dt2, beta_dt;       // neo-Hookean
};

// Lets the kernels take the largest island's LDS. To be called on a device before a launch of more than
// kDefaultLds: the limit belongs to the kernel, not to the launch, and is shared by all simulations of the
// process, so it is always set to the same size.
void allow_island_lds();

// One launch: p.substeps substeps of every island. kind: 0 Green, 1 neo-Hookean; hex: the group's
// elements are hex-cell clusters, else single tets.
void launch_island_frame(hipStream_t s, island_dev const& d, int kind, bool hex, tet_group_dev const& g,
                         cluster_dev const& cl, pos4* xi, pos4* xn, float4* v, contact_dev const& c,
                         solve_params const& p);

}  // namespace sbs
