// Time steps of large bodies, several colors per launch (tile.hip): each workgroup carries one part of the
// particles through them in LDS.
#pragma once
#include <vector>

#include "abi_util.h"
#include "kernels.h"

namespace sbs {

// LDS bytes of a particle: its row (three coordinates and the inverse mass, FP64), the inverse mass as the
// projections take it (FP32), its index.
constexpr std::size_t kTileBytes = 40;
// LDS of a compute unit, and the particles of a tile, a multiple of 64: what it holds beside the chunks.
constexpr std::size_t kTileLds = 160 * 1024;
constexpr uint32_t kTileParticles = 3968;
// Instances of a chunk, one a lane: a wave to a SIMD. Particles are loaded and stored by twice as many threads
// (1M tets 6,554 us for four frames, 6,728 with 256 threads).
constexpr int kTileBlock = 256, kTileThreads = 512;
// Colors of a launch, and chunks of a tile in one: elements of a color share no particle.
constexpr uint32_t kTileColors = 8, kTileChunks = kTileColors * ((kTileParticles + kTileBlock - 1) / kTileBlock);
static_assert(kTileParticles * kTileBytes + kTileChunks * 16 <= kTileLds, "the largest tile fits");
// Constraints of a scene of tiles: 16-byte offsets into its arrays fit 32 bits.
constexpr uint32_t kTileConstraints = 1u << 28;
// Largest scratch memory of the plan.
constexpr std::size_t kTileScratch = std::size_t(1) << 30;

// One segment (a run of colors) of a planned sweep.
struct tile_segment {
    uint32_t first_color, last_color;  // [first, last)
    uint32_t cap;                      // particles of its largest tile
    uint32_t chunks;                   // chunks of the tile with the most
    std::size_t blocks;                // its records in tile_plan::blocks
};

// Tiles are parts of the particles; a tile's workgroup needs, for the colors of a segment, every element
// that moves one of its own particles, and for each of those the elements of the segment's earlier colors
// that move its corners: the elements a tile runs beside its own are run by the neighbouring tile too.
struct tile_plan {
    uint32_t tiles = 0;
    std::vector<tile_segment> segments;
    // [segment][tile], 3 records: (first particle entry, particles, first chunk, chunks), its first two chunks
    dev_buf<uint4> blocks;
    // up to kTileBlock instances of one color: first instance, instances, constraint stride of a cluster's
    // tets, whether the color ends here
    dev_buf<uint4> chunks;
    dev_buf<uint2> particles;  // particle (top bit: the tile's own), surface vertex or ~0
    dev_buf<uint32_t> elems;   // instance: first constraint (top bit: the tile keeps its multipliers)
    dev_buf<uint4> corners8;   // hex cells: 8 16-bit places in the tile
    dev_buf<uint2> corners4;   // single tets: 4
    dev_buf<float> lambda;     // instances' multipliers, [tet of the cluster][instance]
    uint32_t instances = 0;
    bool ready() const { return tiles != 0; }
};

struct tile_source {
    uint32_t V, elements, ncolors;
    bool hex;
    const int4 *v0, *v1;             // hex: corners of an element; else v0: a constraint's particles
    const uint32_t* color_elements;  // host: elements before each color, ncolors + 1
    const uint32_t* color_constraints;
    const int* surface_of;           // device: surface vertex of a particle, or -1
    const uint32_t* tile_of;         // host: tile of each particle
    uint32_t tiles;
};

// What a plan over given segments would hold: instances per [tile][color], particles per [segment][tile]
// (~0u: more than a tile can hold).
struct tile_counts {
    std::vector<uint32_t> instances, particles;
};

// Plans in two steps: tile_scratch::count() for candidate segmentations, build() for the chosen one.
struct tile_scratch {  // (build() throws SBS_ERR_OUT_OF_MEMORY for a plan that is too large as well)
    tile_scratch(hipStream_t s, tile_source const& src);
    // (all particles ~0u: the plan would take more scratch memory than kTileScratch)
    tile_counts count(std::vector<uint32_t> const& bounds);  // bounds: first color of each segment, then ncolors
    void build(std::vector<uint32_t> const& bounds, tile_counts const& n, tile_plan& plan);

private:
    hipStream_t s;
    tile_source src;
    std::size_t vwords, ewords;
    dev_buf<uint32_t> table, own_first, own, tile_of, cfirst, tfirst, bits, bounds_dev, counts;
};

struct tile_params {
    int zero;         // multipliers start at zero
    int from_group;   // multipliers come from the group's array (a warm-started first iteration)
    int to_group;     // the last iteration: they go back there
    int contacts;     // project the contacts first
    int first_contacts;
    float* lambda_out;  // contact multipliers' output (input: contact_dev::lambda)
    float contact_at;
    float alpha_tilde, gamma;  // Green
    float inv_dt2, beta_dt;    // neo-Hookean
};

// One segment of the sweep: positions from `in` to `out`. kind: 0 Green, 1 neo-Hookean.
void launch_tile_segment(hipStream_t s, tile_plan const& plan, std::size_t segment, int kind, bool hex,
                         tet_group_dev const& g, const pos4* in, pos4* out, const pos4* xn, contact_dev const& c,
                         tile_params const& p);

}  // namespace sbs
