// The tile plan of an XPBD substep: which consecutive stencil groups run in one launch, and what each workgroup of
// that launch loads, projects and writes.
//
// Stencils of one group share no particle, but consecutive groups depend on each other, so one launch per group costs
// a dependent launch (about 4.4 us) for work that takes a microsecond. Here the particles are split into compact tiles,
// one per workgroup, and a launch (a batch) runs several groups: a tile loads the particles that its own particles'
// results depend on through those groups, runs the groups in order in LDS with a workgroup barrier between two, and
// writes its own particles to another buffer. What a tile needs of its neighbours it computes itself (the stencils of
// the halo are projected by several tiles), so workgroups never wait for each other, and every particle goes through
// the same projections in the same order as with one launch per group: the result is the same bit for bit.
#pragma once

#include <cstdint>
#include <functional>
#include <vector>

namespace spgvbd {

// The energy types a tile kernel holds: springs, membranes, hinges and anchors; with tetrahedra; with the further ones.
constexpr int kTileSurface = 0, kTileFive = 1, kTileFurther = 2;
constexpr int tileSet(int type) { return type >= 6 ? kTileFurther : type == 4 ? kTileFive : kTileSurface; }
// Threads of a tile's workgroup. A group takes a round per this many of the tile's stencils; 1024 threads leave 128
// registers each, too few for a tetrahedron with its FP64 solve, whose path few projections take but whose registers all
// hold (170; 512x512 cloth: 30 us a substep with 1024 threads, 36 with 512, 44 with 256; 17^3-cell cube: 153, 59 and 78).
constexpr int tileThreads(int set) { return set == kTileSurface ? 1024 : 512; }
constexpr int kTileMaxParticles = 3968;  // particles a tile loads at most: 62 KB of LDS
constexpr int kTileMaxGroups = 64;       // groups of a batch at most

// One stencil group, in launch order.
struct TileGroup {
    int32_t type;          // energy type
    int32_t size;          // particles per stencil
    int32_t count;         // stencils
    int32_t record;        // the group's first record in its type's table
    const int32_t *stencils = nullptr;  // particles, no particle twice in the group (set by the plan)
};

struct TileHeader {
    int32_t particleBegin, particleEnd, owned;  // range of the particle list; its first `owned` are written
    int32_t segBegin;                           // one segment per group of the batch
};
struct TileSegment {
    int32_t type, count;
    int32_t base;  // first float4 of the segment's records
};
// A stencil projected by a tile: its particles' places in the tile's list, and its record in its type's table.
// kTileCounts is set in the first place where the tile owns the stencil's first particle: of all tiles that project
// the stencil, that one counts it in the statistics.
constexpr uint16_t kTileCounts = 0x8000;
struct TileEntry {
    uint16_t place[4];
    int32_t record;
};
struct TileBatch {
    int32_t firstGroup, groups;
    int32_t headerBase, tiles;  // tiles 0: the groups run one launch each
    int32_t maxParticles;
};

struct TilePlan {
    std::vector<TileBatch> batches;     // in order; empty: no plan
    std::vector<TileHeader> headers;
    std::vector<int32_t> particles;
    std::vector<TileSegment> segments;
    std::vector<int64_t> segmentEntry;  // first entry of each segment, and the end
    std::vector<TileEntry> entries;
    int64_t recordSize = 0;             // float4 of all records
};

// float4 planes of a tile record of an energy type
constexpr int tilePlanes(int type) { return type == 1 || type == 3 ? 1 : type == 5 ? 2 : type == 2 ? 3 : 4; }

// The plan, or one without batches where one launch per group is estimated to be as fast. xyz: 3 floats every `stride`,
// the particles' positions; objects: their particle ranges (n + 1 offsets); stencils(g, out): writes group g's particles,
// size per stencil (called from several threads); threads: of a tile's workgroup.
TilePlan buildTilePlan(const float *xyz, int stride, const std::vector<int64_t> &objects, std::vector<TileGroup> groups,
                       const std::function<void(int32_t, int32_t *)> &stencils, int threads);

}  // namespace spgvbd
