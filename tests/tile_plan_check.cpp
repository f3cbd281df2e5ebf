// Runs stencil groups in tile-plan order on 64-bit hashes and compares with running them one group after the other: a
// particle's hash depends on every projection it went through, on what the stencil's other particles held then, and on
// their order. Also checks the plan's lists. Arguments: kind (cloth, cube, net), size, serial (0 / 1), threads. Prints
// "batches B tiled T"; exits with 1 on a difference.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "coloring.h"
#include "xpbd_tiles.h"

using namespace spgvbd;

static uint64_t mix(uint64_t a)
{
    a = (a ^ (a >> 33)) * 0xff51afd7ed558ccdULL;
    a = (a ^ (a >> 33)) * 0xc4ceb9fe1a85ec53ULL;
    return a ^ (a >> 33);
}

static void project(uint64_t *p, const int *id, int n, uint64_t key)
{
    uint64_t h = key;
    for (int d = 0; d < n; ++d) h = mix(h + p[id[d]] * (d + 1));
    for (int d = 0; d < n; ++d) p[id[d]] = mix(h + d + p[id[d]]);
}

int main(int argc, char **argv)
{
    if (argc != 5) return 2;
    const char *kind = argv[1];
    const int n = atoi(argv[2]), serial = atoi(argv[3]), threads = atoi(argv[4]);
    std::vector<float> x;
    std::vector<int64_t> objects{0};
    struct Set {
        int type, size;
        std::vector<int32_t> st;
    };
    std::vector<Set> sets;
    if (!strcmp(kind, "cloth")) {  // hinges, triangles, one anchored row; then a particle of its own
        Set hinge{3, 4, {}}, tri{2, 3, {}}, anchor{5, 1, {}};
        auto id = [&](int i, int j) { return i * n + j; };
        for (int i = 0; i < n; ++i)
            for (int j = 0; j < n; ++j) x.insert(x.end(), {float(j), float(i), 0.f});
        for (int i = 0; i + 1 < n; ++i)
            for (int j = 0; j + 1 < n; ++j) {
                tri.st.insert(tri.st.end(), {id(i, j), id(i, j + 1), id(i + 1, j + 1), id(i, j), id(i + 1, j + 1), id(i + 1, j)});
                hinge.st.insert(hinge.st.end(), {id(i, j), id(i + 1, j + 1), id(i, j + 1), id(i + 1, j)});
                if (i) hinge.st.insert(hinge.st.end(), {id(i, j), id(i, j + 1), id(i + 1, j + 1), id(i - 1, j)});
                if (j) hinge.st.insert(hinge.st.end(), {id(i, j), id(i + 1, j), id(i + 1, j + 1), id(i, j - 1)});
            }
        for (int j = 0; j < n; ++j) anchor.st.push_back(id(n - 1, j));
        sets = {hinge, tri, anchor};
        objects.push_back(n * n);
        x.insert(x.end(), {0.f, 0.f, 0.f});
        objects.push_back(n * n + 1);
    } else if (!strcmp(kind, "cube")) {
        Set tet{4, 4, {}};
        const int m = n + 1, step[3] = {m * m, m, 1}, perm[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
        for (int i = 0; i < m * m * m; ++i) x.insert(x.end(), {float(i / (m * m)), float(i / m % m), float(i % m)});
        for (int c = 0; c < n * n * n; ++c) {
            const int a = (c / (n * n) * m + c / n % n) * m + c % n;
            for (auto &p : perm)
                tet.st.insert(tet.st.end(), {a, a + step[p[0]], a + step[p[0]] + step[p[1]], a + step[0] + step[1] + step[2]});
        }
        sets = {tet};
        objects.push_back(m * m * m);
    } else {  // springs between arbitrary particles: halves of the tiles' particles lie far away
        Set spring{1, 2, {}};
        uint64_t s = 7;
        auto draw = [&](int k) { return static_cast<int>((s = mix(s + 1)) % k); };
        for (int i = 0; i < 3 * n; ++i) x.push_back(float(draw(1000)));
        for (int i = 0; i < 3 * n; ++i) {
            const int a = draw(n), b = draw(n);
            if (a != b) spring.st.insert(spring.st.end(), {a, b});
        }
        sets = {spring};
        objects.push_back(n);
    }
    const int64_t nv = objects.back();
    std::vector<std::vector<int32_t>> lists;
    std::vector<TileGroup> groups;
    for (const Set &s : sets) {
        const int64_t ns = s.st.size() / s.size;
        const auto col = serial ? serialLevels(s.st.data(), ns, s.size) : colorStencils(s.st.data(), ns, s.size);
        std::vector<std::vector<int32_t>> by;
        for (int64_t i = 0; i < ns; ++i) {
            if (static_cast<int64_t>(by.size()) <= col[i]) by.resize(col[i] + 1);
            by[col[i]].insert(by[col[i]].end(), s.st.begin() + i * s.size, s.st.begin() + (i + 1) * s.size);
        }
        int record = 0;
        for (auto &g : by) {
            lists.push_back(g);
            groups.push_back({s.type, s.size, static_cast<int32_t>(g.size() / s.size), record});
            record += groups.back().count;
        }
    }
    const TilePlan plan = buildTilePlan(
        x.data(), 3, objects, groups, [&](int32_t g, int32_t *out) { std::copy(lists[g].begin(), lists[g].end(), out); }, threads);
    auto key = [](int type, int record) { return mix(type * 1000003ull + record); };
    std::vector<uint64_t> one(nv), tiled(nv), out(nv);
    for (int64_t i = 0; i < nv; ++i) one[i] = tiled[i] = mix(i + 1);
    for (size_t k = 0; k < groups.size(); ++k) groups[k].stencils = lists[k].data();
    auto alone = [&](std::vector<uint64_t> &p, const TileGroup &g) {
        for (int s = 0; s < g.count; ++s) project(p.data(), g.stencils + int64_t(s) * g.size, g.size, key(g.type, g.record + s));
        return static_cast<int64_t>(g.count);
    };
    int64_t total = 0, counted = 0, wrong = 0, tiles = 0;
    for (const auto &g : groups) total += alone(one, g);
    std::vector<char> record(plan.recordSize, 0);
    int32_t nextGroup = 0;
    for (const auto &b : plan.batches) {
        wrong += b.firstGroup != nextGroup;
        nextGroup += b.groups;
        if (!b.tiles) {
            for (int k = 0; k < b.groups; ++k) counted += alone(tiled, groups[b.firstGroup + k]);
            continue;
        }
        ++tiles;
        std::vector<char> owned(nv, 0);
        wrong += b.groups > kTileMaxGroups || b.maxParticles > kTileMaxParticles;
        for (int t = 0; t < b.tiles; ++t) {
            const TileHeader &h = plan.headers.at(b.headerBase + t);
            const int m = h.particleEnd - h.particleBegin;
            wrong += m > b.maxParticles || h.owned > m;
            std::vector<uint64_t> local(m);
            for (int i = 0; i < m; ++i) local[i] = tiled.at(plan.particles.at(h.particleBegin + i));
            for (int k = 0; k < b.groups; ++k) {
                const TileGroup &g = groups[b.firstGroup + k];
                const TileSegment &s = plan.segments.at(h.segBegin + k);
                const int64_t first = plan.segmentEntry.at(h.segBegin + k);
                wrong += s.type != g.type || plan.segmentEntry.at(h.segBegin + k + 1) != first + s.count;
                for (int i = 0; i < s.count; ++i) {
                    const TileEntry &e = plan.entries.at(first + i);
                    int id[4];
                    for (int d = 0; d < g.size; ++d) wrong += (id[d] = e.place[d] & ~kTileCounts) >= m;
                    if (wrong) return printf("a place outside its tile\n"), 1;
                    counted += (e.place[0] & kTileCounts) != 0;
                    project(local.data(), id, g.size, key(s.type, e.record));
                    for (int q = 0; q < tilePlanes(s.type); ++q) wrong += record.at(s.base + int64_t(q) * s.count + i)++ != 0;
                }
            }
            for (int i = 0; i < h.owned; ++i) {
                const int p = plan.particles[h.particleBegin + i];
                wrong += owned.at(p)++ != 0;
                out[p] = local[i];
            }
        }
        for (char o : owned) wrong += o == 0;
        tiled = out;
    }
    for (char r : record) wrong += r == 0;
    if (!plan.batches.empty()) wrong += one != tiled || counted != total || nextGroup != static_cast<int32_t>(groups.size());
    printf("batches %zu tiled %lld\n", plan.batches.size(), static_cast<long long>(tiles));
    return wrong ? 1 : 0;
}
