// The tile plan when memory runs out: allocation K of buildTilePlan, counted over all its threads, and all after it fail,
// for K = 0, 1, 2, ... spread over the plan; then a callback that throws. Every time std::bad_alloc has to arrive here. Prints the
// number of allocations of a whole plan.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>

#include "coloring.h"
#include "xpbd_tiles.h"

using namespace spgvbd;

static std::atomic<int64_t> made{0}, allowed{INT64_MAX};

void *operator new(size_t n)
{
    if (made.fetch_add(1) >= allowed.load()) throw std::bad_alloc();
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

int main()
{
    const int n = 150;  // quads of a square grid: several colours, some ninety tiles of 256 particles
    std::vector<float> x;
    std::vector<int32_t> quads;
    for (int i = 0; i < n; ++i)
        for (int j = 0; j < n; ++j) x.insert(x.end(), {float(j), float(i), 0.f});
    for (int i = 0; i + 1 < n; ++i)
        for (int j = 0; j + 1 < n; ++j) quads.insert(quads.end(), {i * n + j, (i + 1) * n + j + 1, i * n + j + 1, (i + 1) * n + j});
    const int64_t count = quads.size() / 4;
    const auto color = colorStencils(quads.data(), count, 4);
    std::vector<std::vector<int32_t>> lists;
    for (int64_t s = 0; s < count; ++s) {
        if (static_cast<int64_t>(lists.size()) <= color[s]) lists.resize(color[s] + 1);
        lists[color[s]].insert(lists[color[s]].end(), quads.begin() + 4 * s, quads.begin() + 4 * s + 4);
    }
    const std::vector<int64_t> objects{0, int64_t(n) * n};
    auto plan = [&](bool throwing) {
        std::vector<TileGroup> groups;
        int32_t record = 0;
        for (const auto &l : lists) {
            groups.push_back({3, 4, static_cast<int32_t>(l.size() / 4), record});
            record += groups.back().count;
        }
        return buildTilePlan(x.data(), 3, objects, groups, [&](int32_t g, int32_t *out) {
            if (throwing && g > 0) throw std::bad_alloc();
            std::copy(lists[g].begin(), lists[g].end(), out);
        }, 1024).batches.size();
    };
    made = 0;
    if (plan(false) == 0) return printf("no plan\n"), 1;
    const int64_t whole = made.load();
    printf("%lld allocations\n", static_cast<long long>(whole));
    auto fails = [&](bool throwing, int64_t k) {
        made = 0;
        allowed = k;
        bool caught = false;
        try {
            plan(throwing);
        } catch (const std::bad_alloc &) {
            caught = true;
        }
        allowed = INT64_MAX;
        return caught;
    };
    // how many allocations the threads make varies with their number: the last ones may not come
    for (int64_t k = 0; k < whole * 9 / 10; k += k < 40 ? 1 : whole / 50)
        if (!fails(false, k)) return printf("allocation %lld failed unnoticed\n", static_cast<long long>(k)), 1;
    if (!fails(true, INT64_MAX)) return printf("the callback's exception was lost\n"), 1;
    return 0;
}
