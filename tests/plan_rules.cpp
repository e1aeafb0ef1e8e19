// Host-side check of the work plans that the device makes for ensembles
// (plan_cluster and exact_wide in h4_kernels.hpp).  Built and run by
// tests/test_plan_rules.py; exit status 0 means every case held.
#include "h4_kernels.hpp"

#include <algorithm>
#include <cstdio>
#include <random>
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

// The plans of random ensembles, as the device makes them, cover their tiles and
// fit the buffer that their partial sums share (ensemble_partial_bound, or the
// clusters' own bounds).
static void check_partials(uint32_t trials, uint32_t grid, uint32_t max_split, bool mixed) {
    const uint32_t target = grid * QUEUE_FACTOR;
    std::mt19937_64 rng(20261205 + grid + mixed);
    for (uint32_t t = 0; t < trials; ++t) {
        const uint32_t K = 2 + rng() % 80, spread = 1 + rng() % 40000;
        std::vector<uint32_t> n(K), nact(K);
        unsigned long long n_total = 0, per_cluster = 0;
        double W = 0.0;
        for (uint32_t c = 0; c < K; ++c) {
            n[c] = 1 + rng() % spread;
            nact[c] = rng() % 4 == 0 ? 0 : 1 + rng() % (rng() % 2 ? n[c] : std::min(n[c], 600u));
            n_total += n[c];
            per_cluster += partial_bound(n[c], target);
            W += (double)nact[c] * (double)n[c];
        }
        Clusters cl(n);
        cl.e.grid = grid;
        cl.e.max_split = max_split;
        unsigned long long used = 0;
        for (uint32_t c = 0; c < K; ++c) {
            if (!nact[c]) continue;
            const ClPlan pl = plan_cluster(cl.e, c, nact[c], W, false, mixed, false);
            const uint32_t nt = ntiles(cl.e, c);
            CHECK((unsigned long long)pl.n_it * pl.iw >= nact[c] && pl.rows == pl.n_it * pl.iw &&
                      (unsigned long long)pl.S * pl.tpc >= nt && (pl.S - 1) * pl.tpc < nt &&
                      pl.S <= max_split,
                  "n %u, %u active: %u x %u slots, %u chunks of %u tiles", n[c], nact[c], pl.n_it,
                  pl.iw, pl.S, pl.tpc);
            CHECK(!pl.jrun || (mixed && pl.iw == 64), "jrun with %u slots", pl.iw);
            if (pl.S > 1) used += 6ull * pl.S * pl.rows;
        }
        const unsigned long long sum = ensemble_partial_bound(K, n_total, target);
        CHECK(used <= std::min(per_cluster, sum), "trial %u, K %u: %llu doubles", t, K, used);
    }
}

int main() {
    check_exact();
    for (int mixed = 0; mixed < 2; ++mixed) {
        check_partials(4000, 4096, 1024, mixed);
        check_partials(4000, 2048, 1024, mixed);
        check_partials(2000, 256, 16, mixed);
        check_partials(2000, 1, 1u << 30, mixed);
    }
    check_chunks();
    check_finish();
    if (failures) {
        std::printf("%d failures\n", failures);
        return 1;
    }
    std::printf("plan rules ok\n");
    return 0;
}
