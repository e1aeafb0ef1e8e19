// Host-side check of the work plans that the device makes for ensembles
// (plan_cluster and exact_wide in h4_kernels.hpp).  Built and run by
// tests/test_plan_rules.py; exit status 0 means every case held.
#include "h4_kernels.hpp"

#include <algorithm>
#include <cstdio>
#include <vector>

using namespace h4;

static int failures = 0;

#define CHECK(cond, ...)                                  \
    do {                                                  \
        if (!(cond) && failures++ < 10) {                 \
            std::printf("FAIL %s: ", #cond);              \
            std::printf(__VA_ARGS__);                     \
            std::printf("\n");                            \
        }                                                 \
    } while (0)

// The tables of an ensemble that a plan reads.
struct Clusters {
    std::vector<uint32_t> n;
    Ens e{};
    explicit Clusters(std::vector<uint32_t> sizes) : n(std::move(sizes)) {
        e.K = (uint32_t)n.size();
        e.cnt = n.data();
        e.grid = 2048;
        e.max_split = 1024;
        e.iw_fill = DEFAULT_IW_FILL;
    }
    ExactLoad load(const std::vector<uint32_t> &nact) const {
        ExactLoad l{};
        for (size_t c = 0; c < n.size(); ++c) {
            const double lanes = (nact[c] + BS - 1) / BS * BS;
            l.pairs += (double)nact[c] * n[c];
            l.act += nact[c];
            l.lanes += lanes;
            l.lane_pairs += lanes * n[c];
            if (nact[c]) l.nmax = std::max(l.nmax, (double)n[c]);
        }
        return l;
    }
};

// Exact precision: ensembles whose particles fill the chip get a lane each
// although no cluster does by itself, smaller ones do not.
static void check_exact() {
    const struct {
        uint32_t K, n;
        bool wide;
    } all[] = {{64, 10000, true}, {16, 16384, true}, {64, 1000, true}, {256, 700, true},
               {6, 9000, true},   {200, 1025, true}, {512, 300, true}, {1024, 100, true},
               {4, 3000, false},  {8, 300, false},   {32, 300, false}, {64, 200, false},
               {2, 20000, false}};
    for (const auto &a : all) {
        const Clusters c(std::vector<uint32_t>(a.K, a.n));
        const ExactLoad l = c.load(c.n);
        CHECK(exact_wide(l) == a.wide, "%u clusters of %u", a.K, a.n);
        const ClPlan pl = plan_cluster(c.e, 0, a.n, l.pairs, true, false, exact_wide(l));
        CHECK((pl.iw == (uint32_t)BS) == a.wide && (uint64_t)pl.n_it * pl.iw >= a.n && pl.S == 1,
              "%u clusters of %u: %u slots, %u items", a.K, a.n, pl.iw, pl.n_it);
        // a few active particles each are left to workgroups of their own
        const std::vector<uint32_t> few(a.K, 3);
        CHECK(!exact_wide(c.load(few)), "%u clusters of %u, 3 active", a.K, a.n);
    }
    // one system: by its active count alone
    const Clusters one({100000});
    for (uint32_t nact : {1u, 768u, 769u, 45055u, 45056u, 100000u}) {
        const ClPlan pl = plan_cluster(one.e, 0, nact, (double)nact * 100000.0, true, false,
                                       nact >= EXACT_WIDE);
        CHECK(pl.iw == (nact <= 768 ? 1u : nact < 45056 ? 3u : 256u), "%u active: %u slots", nact,
              pl.iw);
    }
}

// A block step's finish: one pass up to 2048 blocks, two for larger ensembles.
static void check_finish() {
    CHECK(finish_by_blocks(1, 1) && finish_by_blocks(1, 100000), "one system");
    CHECK(finish_by_blocks(2, 2048) && !finish_by_blocks(2, 2049), "two clusters");
    CHECK(!finish_by_blocks(512, 4096), "512 clusters of 2048");
}

// Chunks of one tile in ensembles: only where chunks of four make few items.
static void check_chunks() {
    const struct {
        uint32_t K, n, nact;
        bool mixed;
        uint32_t S;
    } all[] = {{2, 10000, 78, false, 40}, {2, 10000, 78, true, 40},   {8, 4096, 32, false, 16},
               {512, 1100, 9, false, 2},  {512, 1100, 9, true, 2},    {256, 2048, 16, false, 2},
               {8, 1000, 8, false, 1},    {2, 70000, 40, false, 69}, {64, 4096, 32, false, 4}};
    for (const auto &a : all) {
        const Clusters c(std::vector<uint32_t>(a.K, a.n));
        const ClPlan pl =
            plan_cluster(c.e, 0, a.nact, (double)a.K * a.nact * a.n, false, a.mixed, false);
        CHECK(pl.S == a.S, "%u clusters of %u, %u active: %u chunks of %u, %u slots", a.K, a.n, a.nact,
              pl.S, pl.tpc, pl.iw);
    }
}

int main() {
    check_exact();
    check_chunks();
    check_finish();
    if (failures) {
        std::printf("%d failures\n", failures);
        return 1;
    }
    std::printf("plan rules ok\n");
    return 0;
}
