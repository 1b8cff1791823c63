// Whole-frame kernels of small bodies (island.hip): one workgroup per island.
#pragma once
#include "kernels.h"

namespace sbs {

// LDS of a compute unit a workgroup may use for positions, and the bytes a particle takes there (three
// FP64 coordinates and its FP32 inverse mass); some hundred bytes are left for the kernels' own.
constexpr std::size_t kIslandLds = 160 * 1024, kIslandBytes = 28;
constexpr uint32_t kIslandParticles = uint32_t((kIslandLds - 512) / kIslandBytes);
// Constraints of a scene of islands: 16-byte offsets into its arrays fit 32 bits.
constexpr uint32_t kIslandConstraints = 1u << 28;

// The islands of a scene whose single constraint group is laid out island by island inside each color.
struct island_dev {
    const uint4* islands;  // first particle, particles, first surface vertex, surface vertices
    const uint4* stages;   // [island][color]: first element, first constraint, constraint stride of a
                           // cluster's tets, elements
    uint32_t* clist;       // scratch, one word per surface vertex
    uint32_t count, ncolors;
    uint32_t cap;            // particles of the largest island (the stride of its LDS arrays)
    uint32_t largest_stage;  // elements of the largest stage of any island
};

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

// One launch: p.substeps substeps of every island. kind: 0 Green, 1 neo-Hookean; hex: the group's
// elements are hex-cell clusters, else single tets.
void launch_island_frame(hipStream_t s, island_dev const& d, int kind, bool hex, tet_group_dev const& g,
                         cluster_dev const& cl, pos4* xi, pos4* xn, float4* v, contact_dev const& c,
                         solve_params const& p);

}  // namespace sbs
