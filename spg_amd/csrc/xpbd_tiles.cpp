#include "xpbd_tiles.h"

#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <limits>
#include <numeric>

#include "host_threads.h"

namespace spgvbd {

namespace {

// The times the plan is chosen by, in microseconds, measured on MI355X. A compute unit holds one workgroup of a tile
// kernel at a time (its registers), so a launch of more tiles than compute units takes its time per tile several times
// over; and each tile gathers its particles, a cache line each where they are scattered. Without these two a solid of
// 64^3 cells took 538 tiles, whose five launches take 221 us, where its 34 groups take 152 us by themselves, and 10^6
// particles with springs anywhere 230 us for 214. A 512x512 cloth (256 tiles): 37 us by this estimate, 33 measured;
// 700x700 (479): 68 and 62; 1024x1024 (1024): 133 and 123.
constexpr double kGroupLaunchUs = 4.4;    // one launch of one group, a small one
constexpr double kGroupBytesPerUs = 4e6;  // of the records and particles of a large one
constexpr double kTileLaunchUs = 5.0;     // a tile launch without its groups
constexpr double kBytesPerUs = 5e6;       // record streaming and particle gathers of a tile launch
constexpr double kParticleBytes = 64;     // of a particle that a tile loads
constexpr int kComputeUnits = 256;

// Host threads that build the plan. Starting them takes 0.5 ms, more than the whole plan of a small mesh: 0.07 ms for a cloth
// of 16x16 particles in 20 groups.
constexpr int kPlanThreads = 8;
constexpr int64_t kThreadedFrom = 16384;  // particles times groups

// A round of one group in a tile: steps of one launch of one round a group (a 100x100 cloth of each kind, solids of 12^3
// and 17^3 cells) less the launch, by group.
double groupUs(int32_t type)
{
    switch (type) {
    case 4: return 1.2;
    case 8: return 3.0;
    case 9: return 4.5;
    case 10: return 3.0;
    case 11: return 1.5;
    case 12: return 1.7;
    case 13: return 1.5;
    default: return 1.0;
    }
}
// One group by itself. The kernels of types 8 to 10 keep an array in scratch memory: 5.5 us at 2,800 stencils, 9 at
// 19,000, 15 at 45,000, 18 at 140,000.
double aloneUs(const TileGroup &g)
{
    const double bytes = g.count * (16.0 * tilePlanes(g.type) + 32.0 * g.size);
    const double least = g.type >= 8 && g.type <= 10 ? 5.0 + 10.0 * std::min(1.0, g.count / 40000.0) : kGroupLaunchUs;
    return std::max(least, bytes / kGroupBytesPerUs);
}
// how often a compute unit takes a tile
double waves(int64_t tiles) { return static_cast<double>((tiles + kComputeUnits - 1) / kComputeUnits); }

// Bisects particles [b, e) of `order` along the longer side of their box, again and again, into `parts` ranges of equal
// size; writes the ranges' ends to ends[0 .. parts).
void bisect(const float *xyz, int stride, int32_t *order, int64_t b, int64_t e, int64_t parts, int64_t *ends)
{
    if (parts <= 1) {
        ends[0] = e;
        return;
    }
    std::array<float, 3> lo, hi;
    lo.fill(std::numeric_limits<float>::max());
    hi.fill(std::numeric_limits<float>::lowest());
    for (int64_t i = b; i < e; ++i)
        for (int d = 0; d < 3; ++d) {
            const float v = xyz[static_cast<int64_t>(order[i]) * stride + d];
            lo[d] = std::min(lo[d], v);
            hi[d] = std::max(hi[d], v);
        }
    int axis = 0;
    for (int d = 1; d < 3; ++d)
        if (hi[d] - lo[d] > hi[axis] - lo[axis]) axis = d;
    const int64_t left = parts / 2, mid = b + (e - b) * left / parts;
    std::nth_element(order + b, order + mid, order + e, [&](int32_t p, int32_t q) {
        const float u = xyz[static_cast<int64_t>(p) * stride + axis], v = xyz[static_cast<int64_t>(q) * stride + axis];
        return u != v ? u < v : p < q;
    });
    if (e - b > 65536) {
        forAll(2, kPlanThreads, [&](int64_t k) {
            if (k == 0)
                bisect(xyz, stride, order, b, mid, left, ends);
            else
                bisect(xyz, stride, order, mid, e, parts - left, ends + left);
        });
        return;
    }
    bisect(xyz, stride, order, b, mid, left, ends);
    bisect(xyz, stride, order, mid, e, parts - left, ends + left);
}

// Compact tiles of particles, none across objects.
struct Tiles {
    std::vector<int32_t> order;
    std::vector<int64_t> ends;  // tile t: order[ends[t - 1] .. ends[t])

    int64_t count() const { return static_cast<int64_t>(ends.size()); }
    const int32_t *begin(int64_t t) const { return order.data() + (t ? ends[t - 1] : 0); }
    int64_t size(int64_t t) const { return ends[t] - (t ? ends[t - 1] : 0); }
};

// Tiles of at most 256 particles, and from them tiles of up to twice and four times as many: the halves and quarters
// of a tile are consecutive.
constexpr int64_t kLargeTile = 1024;
std::array<Tiles, 3> makeTiles(const float *xyz, int stride, const std::vector<int64_t> &objects)
{
    std::array<Tiles, 3> out;
    auto &order = out[0].order;
    order.resize(objects.back());
    std::iota(order.begin(), order.end(), 0);
    for (size_t o = 0; o + 1 < objects.size(); ++o) {
        const int64_t n = objects[o + 1] - objects[o];
        if (n == 0) continue;
        const int64_t large = (n + kLargeTile - 1) / kLargeTile;
        std::vector<int64_t> ends(large);
        bisect(xyz, stride, order.data(), objects[o], objects[o + 1], large, ends.data());
        int64_t b = objects[o];
        for (int64_t e : ends) {
            out[2].ends.push_back(e);
            // an object of one tile may be much smaller than 1024 particles
            const int64_t halves = e - b > kLargeTile / 2 ? 2 : 1;
            std::vector<int64_t> half(halves);
            bisect(xyz, stride, order.data(), b, e, halves, half.data());
            int64_t c = b;
            for (int64_t f : half) {
                out[1].ends.push_back(f);
                const int64_t quarters = f - c > kLargeTile / 4 ? 2 : 1;
                std::vector<int64_t> quarter(quarters);
                bisect(xyz, stride, order.data(), c, f, quarters, quarter.data());
                out[0].ends.insert(out[0].ends.end(), quarter.begin(), quarter.end());
                c = f;
            }
            b = e;
        }
    }
    out[1].order = out[2].order = order;
    return out;
}

// The stencil of a group that holds a particle: at most one does.
class Holders {
  public:
    Holders(int64_t nv, const std::vector<TileGroup> &groups, int hostThreads) : m_nv(nv), m_of(nv * groups.size())
    {
        forAll(groups.size(), hostThreads, [&](int64_t g) {
            int32_t *of = m_of.data() + g * nv;
            std::fill(of, of + nv, -1);
            for (int32_t s = 0; s < groups[g].count; ++s)
                for (int d = 0; d < groups[g].size; ++d) of[groups[g].stencils[int64_t(s) * groups[g].size + d]] = s;
        });
    }
    // its number in group g; -1: none
    int32_t of(int32_t p, int32_t g) const { return m_of[g * m_nv + p]; }

  private:
    int64_t m_nv;
    std::vector<int32_t> m_of;
};
constexpr int64_t kHoldersMax = int64_t(1) << 28;  // entries of that table at most (1 GB)

// What a tile loads and projects, grown backwards over the groups: `particles` starts as the tile's own. The places of
// the particles are kept in an open-addressing table of a size that does not depend on the mesh.
class Grower {
  public:
    Grower(const Holders &h, const std::vector<TileGroup> &g) : m_holders(h), m_groups(g), m_key(kSlots, -1), m_place(kSlots)
    {
        int32_t most = 0;
        for (const auto &group : g) most = std::max(most, group.count);
        m_found.resize(most);
    }
    std::vector<int32_t> particles;

    void start(const int32_t *own, int64_t n)
    {
        std::fill(m_key.begin(), m_key.end(), -1);
        particles.clear();
        for (int64_t k = 0; k < n; ++k) place(own[k]);
    }
    // the stencils of group g that the particles depend on, and their particles; false: more particles than a tile may
    // load
    bool grow(int32_t g, std::vector<int32_t> &out)
    {
        out.clear();
        const TileGroup &G = m_groups[g];
        for (const int32_t p : particles) {
            const int32_t s = m_holders.of(p, g);
            if (s < 0 || m_found[s]) continue;
            m_found[s] = 1;
            out.push_back(s);
        }
        for (const int32_t s : out) {
            m_found[s] = 0;
            for (int d = 0; d < G.size; ++d) place(G.stencils[static_cast<int64_t>(s) * G.size + d]);
        }
        return static_cast<int64_t>(particles.size()) <= kTileMaxParticles;
    }
    // the place of particle p, appended to the list if it is new
    int32_t place(int32_t p)
    {
        uint32_t h = (static_cast<uint32_t>(p) * 2654435761u) >> (32 - kBits);
        while (m_key[h] != p) {
            if (m_key[h] < 0) {
                // past the limit the list only tells that it is exceeded (grow): the table keeps free slots
                if (static_cast<int64_t>(particles.size()) > kTileMaxParticles) return 0;
                m_key[h] = p;
                m_place[h] = static_cast<int32_t>(particles.size());
                particles.push_back(p);
                break;
            }
            h = (h + 1) & (kSlots - 1);
        }
        return m_place[h];
    }

  private:
    static constexpr int kBits = 14, kSlots = 1 << kBits;
    static_assert(kSlots > 2 * kTileMaxParticles, "the table never fills");
    const Holders &m_holders;
    const std::vector<TileGroup> &m_groups;
    std::vector<int32_t> m_key, m_place;
    std::vector<uint8_t> m_found;  // per stencil of the group being grown
};

// Cuts the groups into batches from the last one backwards: a batch takes one more group as long as what its halo adds
// costs less than another launch. Decided on up to kSamples tiles; `margin`: how many times a sampled tile's particles
// have to fit, for the tiles that are not. Returns the batches (ascending) and their time.
std::vector<TileBatch> cut(const Tiles &tiles, const Holders &holders, const std::vector<TileGroup> &groups,
                           int threads, double margin, double &us)
{
    constexpr int kSamples = 5;
    const int64_t nt = tiles.count(), ns = std::min<int64_t>(nt, kSamples);
    std::vector<Grower> grower(ns, Grower(holders, groups));
    auto groupCost = [&](int32_t g, double stencils) {  // of a tile's stencils of the group
        return waves(nt) * groupUs(groups[g].type) * std::max(1.0, std::ceil(stencils / threads));
    };
    std::vector<TileBatch> out;
    std::vector<int32_t> list;
    us = 0.0;
    for (int32_t last = static_cast<int32_t>(groups.size()) - 1; last >= 0;) {
        for (int64_t k = 0; k < ns; ++k) {
            const int64_t t = (2 * k + 1) * nt / (2 * ns);
            grower[k].start(tiles.begin(t), tiles.size(t));
        }
        int32_t first = last + 1;
        double compute = 0.0, bytes = 0.0, loads = 0.0;
        while (first > 0 && last - first + 1 < kTileMaxGroups) {
            const int32_t g = first - 1;
            double largest = 0.0, total = 0.0;
            bool fits = true;
            for (int64_t k = 0; k < ns && fits; ++k) {
                fits = grower[k].grow(g, list) && grower[k].particles.size() * margin <= kTileMaxParticles;
                largest = std::max<double>(largest, list.size());
                total += static_cast<double>(list.size()) * nt / ns;
            }
            const double with = groupCost(g, largest), without = groupCost(g, static_cast<double>(groups[g].count) / nt);
            if (!fits || (first <= last && with - without > kTileLaunchUs)) break;
            compute += with;
            bytes += total * 16.0 * tilePlanes(groups[g].type);
            loads = 0.0;
            for (int64_t k = 0; k < ns; ++k) loads += static_cast<double>(grower[k].particles.size()) * nt / ns;
            first = g;
        }
        const int32_t count = std::max(1, last - first + 1);
        first = last - count + 1;
        const double tile = kTileLaunchUs + std::max(compute, bytes / kBytesPerUs) + loads * kParticleBytes / kBytesPerUs;
        double separate = 0.0;
        for (int32_t g = first; g <= last; ++g) separate += aloneUs(groups[g]);
        const bool use = count > 1 && tile < separate;
        us += use ? tile : separate;
        out.push_back({first, count, 0, use ? static_cast<int32_t>(nt) : 0, 0});
        last = first - 1;
    }
    std::reverse(out.begin(), out.end());
    return out;
}

// Fills the plan's lists for its batches. Returns false where a tile that was not sampled needs more particles than a
// tile may load, or the lists outgrow their indices.
bool fill(TilePlan &plan, const Tiles &tiles, const Holders &holders, const std::vector<TileGroup> &groups, int hostThreads)
{
    struct Built {
        std::vector<int32_t> particles;
        std::vector<int32_t> count;      // stencils per group of the batch
        std::vector<TileEntry> entries;  // in group order
    };
    const int64_t nt = tiles.count();
    int64_t records = 0;
    for (auto &batch : plan.batches) {
        if (!batch.tiles) continue;
        std::vector<Built> built(nt);
        std::atomic<bool> ok{true};
        const int64_t chunk = std::max<int64_t>(1, nt / (8 * kPlanThreads));
        forAll((nt + chunk - 1) / chunk, hostThreads, [&](int64_t c) {
            Grower grower(holders, groups);
            std::vector<std::vector<int32_t>> stencils(batch.groups);
            for (int64_t t = c * chunk; t < std::min(nt, (c + 1) * chunk) && ok; ++t) {
                Built &b = built[t];
                grower.start(tiles.begin(t), tiles.size(t));
                size_t total = 0;
                for (int32_t k = batch.groups - 1; k >= 0; --k) {
                    if (!grower.grow(batch.firstGroup + k, stencils[k])) {
                        ok = false;
                        return;
                    }
                    std::sort(stencils[k].begin(), stencils[k].end());  // records that were neighbours stay so
                    total += stencils[k].size();
                }
                b.entries.reserve(total);
                for (int32_t k = 0; k < batch.groups; ++k) {
                    const TileGroup &G = groups[batch.firstGroup + k];
                    b.count.push_back(static_cast<int32_t>(stencils[k].size()));
                    for (const int32_t s : stencils[k]) {
                        TileEntry e{{0, 0, 0, 0}, G.record + s};
                        for (int d = 0; d < G.size; ++d)
                            e.place[d] = static_cast<uint16_t>(grower.place(G.stencils[int64_t(s) * G.size + d]));
                        if (e.place[0] < tiles.size(t)) e.place[0] |= kTileCounts;
                        b.entries.push_back(e);
                    }
                }
                b.particles = grower.particles;
            }
        });
        if (!ok) return false;
        batch.headerBase = static_cast<int32_t>(plan.headers.size());
        std::vector<int64_t> particleAt(nt + 1, plan.particles.size()), entryAt(nt + 1, plan.entries.size());
        for (int64_t t = 0; t < nt; ++t) {
            const Built &b = built[t];
            particleAt[t + 1] = particleAt[t] + static_cast<int64_t>(b.particles.size());
            entryAt[t + 1] = entryAt[t] + static_cast<int64_t>(b.entries.size());
            if (particleAt[t + 1] > std::numeric_limits<int32_t>::max()) return false;
            batch.maxParticles = std::max(batch.maxParticles, static_cast<int32_t>(b.particles.size()));
            plan.headers.push_back({static_cast<int32_t>(particleAt[t]), static_cast<int32_t>(particleAt[t + 1]),
                                    static_cast<int32_t>(tiles.size(t)), static_cast<int32_t>(plan.segments.size())});
            int64_t at = entryAt[t];
            for (int32_t k = 0; k < batch.groups; ++k) {
                const int32_t type = groups[batch.firstGroup + k].type;
                plan.segments.push_back({type, b.count[k], static_cast<int32_t>(records)});
                plan.segmentEntry.push_back(at);
                at += b.count[k];
                records += static_cast<int64_t>(b.count[k]) * tilePlanes(type);
                if (records > std::numeric_limits<int32_t>::max()) return false;
            }
        }
        plan.particles.resize(particleAt[nt]);
        plan.entries.resize(entryAt[nt]);
        forAll(nt, hostThreads, [&](int64_t t) {
            std::copy(built[t].particles.begin(), built[t].particles.end(), plan.particles.begin() + particleAt[t]);
            std::copy(built[t].entries.begin(), built[t].entries.end(), plan.entries.begin() + entryAt[t]);
        });
    }
    plan.segmentEntry.push_back(static_cast<int64_t>(plan.entries.size()));
    plan.recordSize = records;
    return true;
}

}  // namespace

TilePlan buildTilePlan(const float *xyz, int stride, const std::vector<int64_t> &objects, std::vector<TileGroup> groups,
                       const std::function<void(int32_t, int32_t *)> &stencils, int threads)
{
    const int64_t nv = objects.back();
    if (nv == 0 || groups.size() < 2) return {};
    if (nv * static_cast<int64_t>(groups.size()) > kHoldersMax) return {};
    // with so many tiles, the largest there are, that no group is faster in a tile than by itself there is nothing to plan
    int64_t fewest = 0;
    for (size_t o = 0; o + 1 < objects.size(); ++o) fewest += (objects[o + 1] - objects[o] + kLargeTile - 1) / kLargeTile;
    double alone = 0.0;
    bool any = false;
    for (const auto &g : groups) {
        alone += aloneUs(g);
        any |= waves(fewest) * groupUs(g.type) < aloneUs(g);
    }
    if (!any) return {};
    const int hostThreads = nv * static_cast<int64_t>(groups.size()) < kThreadedFrom ? 1 : kPlanThreads;
    std::vector<std::vector<int32_t>> stencilsOf(groups.size());
    forAll(groups.size(), hostThreads, [&](int64_t g) {
        stencilsOf[g].resize(static_cast<size_t>(groups[g].count) * groups[g].size);
        stencils(static_cast<int32_t>(g), stencilsOf[g].data());
        groups[g].stencils = stencilsOf[g].data();
    });
    const Holders holders(nv, groups, hostThreads);
    auto tiles = makeTiles(xyz, stride, objects);
    for (double margin : {1.125, 1.5, 2.0}) {
        std::array<std::vector<TileBatch>, 3> batches;
        std::array<double, 3> us;
        forAll(3, hostThreads, [&](int64_t k) {
            if (k > 0 && tiles[k].count() == tiles[k - 1].count()) {  // small objects: the same tiles
                us[k] = std::numeric_limits<double>::max();
                return;
            }
            batches[k] = cut(tiles[k], holders, groups, threads, margin, us[k]);
        });
        // larger tiles where they are 2% faster: the smaller ones use more of the chip (17^3-cell solid: 24 tiles 60 us, 12
        // tiles 62, by the estimate 63.4 and 62.7)
        size_t best = 0;
        for (size_t k = 1; k < us.size(); ++k)
            if (us[k] < 0.98 * us[best]) best = k;
        const bool tiled = std::any_of(batches[best].begin(), batches[best].end(), [](const TileBatch &b) { return b.tiles > 0; });
        if (!tiled || us[best] >= alone) return {};
        Tiles &t = tiles[best];
        int64_t b = 0;
        for (int64_t e : t.ends) {  // ascending within a tile: its particles are then mostly consecutive in memory
            std::sort(t.order.begin() + b, t.order.begin() + e);
            b = e;
        }
        TilePlan plan;
        plan.batches = std::move(batches[best]);
        if (fill(plan, t, holders, groups, hostThreads)) return plan;
    }
    return {};
}

}  // namespace spgvbd
