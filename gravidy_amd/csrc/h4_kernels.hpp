// h4_kernels.hpp -- gfx950 device code of the Hermite-4 block-timestep path.
//
// State lives in HBM as structure-of-arrays (one double array per
// component) so every kernel's per-particle loads are coalesced 8-byte
// lanes; the predictor is kept as two double4 arrays in the layout of an
// LDS j tile.  The pairwise kernels stage j particles through LDS in tiles
// of JT and read them back as wave-uniform (broadcast) LDS loads.
//
// Rounding rules.  Predictor, corrector, timestep and init_dt are compiled
// with FP contraction off and use IEEE division and sqrt, so each
// operation rounds exactly as the reference's x86-64 build does
// (Hermite4CPU.cpp:340-411, NbodyUtils.cpp:337-424, Hermite4.cpp:108-140);
// the energy sum keeps the reference's terms and rounds within 1e-13.
// The FP64_EXACT pair kernel does the same for the pair terms and keeps the
// ascending-j order of Hermite4CPU::update_acc_jrk.  The FP64 pair kernel
// contracts to FMA, uses a refined v_rsq_f64 and may split the j range.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace h4 {

constexpr int BS = 256;           // threads per workgroup: 4 wave64
constexpr int JT = 256;           // j particles per LDS tile (== BS)
constexpr double PAD_POS = 1.0e18;  // position of zero-mass padding particles

// Pointer table of the SoA state (all arrays n_pad long).
struct Soa {
    double *r[3];    // corrected position
    double *m;       // mass as uploaded (double; energy uses it)
    double *v[3];    // corrected velocity
    double *f[6];    // acceleration a[3], jerk a1[3]
    double *old[6];  // forces at the start of the step
    double *a2[3];   // 2nd derivative from the Hermite interpolant
    double *a3[3];   // 3rd derivative
    double *t;       // particle time
    double *dt;      // particle block timestep
    // Predictor (Predictor, common.hpp:213-221) as two double4 arrays, the
    // layout of an LDS j tile: pp = (x, y, z, m) with m the float-rounded
    // mass as a double, pv = (vx, vy, vz, bits) with the float mass's bit
    // pattern in the low 32 bits of w (read by the mixed kernel).
    double4 *pp;
    double4 *pv;
};

// Float mass bit pattern stored in pv[i].w.
__host__ __device__ inline double mass_bits(float m) {
    unsigned long long u = __builtin_bit_cast(uint32_t, m);
    return __builtin_bit_cast(double, u);
}

// Device-side scalars of the block-step loop of one cluster (one
// independent N-body system; a plain context is one cluster).  Every step
// kernel reads the block time and the active count from here, so a step
// (or a captured chain of steps) needs no host round trip.
struct ClState {
    double itime;                     // ITIME: block time of the last step
    double atime;                     // ATIME: next block time
    uint32_t nact;                    // active count (compaction target)
    uint32_t done;                    // 1: this cluster's loop has stopped
    unsigned long long tmin_key;      // order-preserving key of min(t+dt)
    unsigned long long steps;         // block steps since the last setup
    unsigned long long interactions;  // sum of nact * n
    unsigned long long nsteps;        // sum of nact
    unsigned long long small_steps;   // block steps made by the one-workgroup kernel
    // Loop tail of the cluster's last block step, left by the step's last
    // launch for the next launch that needs the next block time to make:
    double tail_t;                    // the step's block time
    unsigned long long tail_steps;    // steps done before it
    uint32_t tail_nact;               // its active count
    uint32_t tail_pend;               // 1: that tail is still to be made
};

// Work plan of one step for one cluster (computed on the device after the
// active sets are known).
struct ClPlan {
    uint32_t iw;        // i slots per workgroup (lane-group width)
    uint32_t S;         // j chunks
    uint32_t tpc;       // JT tiles per chunk
    uint32_t n_it;      // i tiles
    uint32_t rows;      // n_it * iw
    uint32_t lanes;     // finish lanes per particle (finish_lanes(S, nact))
    uint32_t grid;      // workgroup share given to decompose()
    uint32_t cmaj;      // 1: partials chunk-major (partial_at)
    uint32_t jrun;      // 1: a j sub-group takes consecutive j (lane_group)
};

// Place of the j-chunk partial sum of component q, chunk sc, active
// particle k in a plan's partial buffer (6 S rows doubles).  Component and
// chunk major, particle minor (a work item writes its particles' sums of
// one chunk as contiguous runs), unless the finish pass gives each
// particle 16 or more lanes and the plan has at least 64 i slots: then
// chunk minor, so that those lanes read whole 128-byte lines of one
// particle's chunks rather than one double of each of 16 or more lines
// (the items' scattered writes then cost less than the finish saves; with
// fewer i slots they cost more).  Either way the finish adds the chunks in
// the same order, so the sums do not depend on the layout.
__host__ __device__ inline size_t partial_at(const ClPlan &pl, uint32_t q, uint32_t sc,
                                             uint32_t k) {
    return pl.cmaj ? ((size_t)q * pl.rows + k) * pl.S + sc
                   : ((size_t)q * pl.S + sc) * pl.rows + k;
}

// Loop control shared by all clusters.
struct RunCtl {
    double t_end;                  // steps run while itime < t_end
    double t_stop;                 // stop after a step with itime >= t_stop
    unsigned long long max_steps;  // stop after this many steps
    uint32_t ndirty[2];            // blocks with active particles, by step parity
    uint32_t ndone;                // clusters that have stopped
    uint32_t qdone;                // update workgroups done with the work queue
    unsigned long long items;      // update work items this step
    unsigned long long fin_units;  // finish workgroup units this step
    unsigned long long team_retry; // k_team_run leaves the steps before this one alone
    unsigned long long team_steps; // block steps made by k_team_run
    uint32_t team_err;             // 1: a wait inside k_team_run ran out
    uint32_t team_fails;           // teams in a row that did not form
    unsigned long long qnext;      // update work queue: items claimed beyond the
                                   // first gridDim.x (zero between launches)
};

// The stop test of the reference's loop after a block step made at time T,
// the next block time being mn (Hermite4CPU_integration.cpp:81,102): an
// output time reached (t_stop), the step budget spent, ITIME >= t_end, or
// no particle left ahead of T.
__host__ __device__ inline bool loop_stops(const RunCtl &ctl, double T, unsigned long long steps,
                                           double mn) {
    return T >= ctl.t_stop || steps >= ctl.max_steps || !(T < ctl.t_end) || !(mn > T);
}

// Cluster tables and per-step scratch, by pointer (device memory).
struct Ens {
    uint32_t K;              // clusters
    uint32_t nblk;           // JT blocks of the padded state
    const uint32_t *off;     // [K] first device index (multiple of JT)
    const uint32_t *cnt;     // [K] particles
    const uint32_t *hoff;    // [K] first host index (clusters back to back)
    const uint32_t *bcl;     // [nblk] cluster of each block
    ClState *cs;             // [K]
    ClPlan *plan;            // [K]
    unsigned long long *items_pre;  // [K+1] exclusive prefix of work items
    unsigned long long *fin_pre;    // [K+1] exclusive prefix of finish units
    unsigned long long *part_pre;   // [K+1] exclusive prefix of partial doubles
    RunCtl *ctl;
    uint32_t *dirty;         // [2][nblk][3] blocks with active particles (block, first
                             // place in the cluster's active list, count), by step
                             // parity (the step's slot in its captured chunk, mod 2)
    double *bmin;            // [nblk] min(t + dt) per block
    uint32_t *bcnt;          // [nblk] particles that have it (BCNT_MANY or more:
                             // not known)
    double4 *arec;           // [4][nblk * JT] the step's active particles in the order
                             // of the active list (index off[c] + k): predictor
                             // (pp, pv), then old forces and step ((a, dt), (jerk, 0));
                             // written by the selection of a device-loop step
    double *hist_t;          // per-step history of cluster 0 (ring, pinned host memory)
    uint32_t *hist_n;
    uint32_t hist_cap;
    uint32_t grid;           // persistent workgroups of the update kernel
    uint32_t max_split;
    uint32_t iw_fill;        // pick_iw fill rule, sixteenths
    uint32_t tuned;          // 1: tune[] holds a table for single-cluster plans
    const uint32_t *tune;    // [64]: workgroup share [0..31], lane-group width
                             // [32..63], by floor(log2(nact)); 0 = default
};

// Order-preserving map double -> uint64 for atomicMin.
__host__ __device__ inline unsigned long long dkey(double x) {
    unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__host__ __device__ inline double dkey_inv(unsigned long long k) {
    unsigned long long u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __builtin_bit_cast(double, u);
}

// Work split of the pairwise update.  A workgroup handles IW active
// particles ("i slots") at a time; its BS lanes are IW slots x BS/IW j
// sub-groups.  The nact active particles form n_it = ceil(nact/IW) i tiles
// and the j range (n_jt tiles of JT) is cut into S chunks, giving n_it * S
// work items.  S is large enough that every one of `grid` workgroups gets
// an item when nact is small, and beyond that up to QUEUE_FACTOR items per
// workgroup (taken from the update kernel's work queue, which evens out
// faster and slower CUs and XCDs) as long as a chunk keeps CHUNK_TILES
// tiles (more chunks would mostly add partial sums to write and read).  A
// chunk of a narrow group (IW 4 or 16) holds at least 4 tiles, 4K or 16K
// pairs: shorter items cost more in partial sums than they gain (IW 16),
// longer ones leave small steps waiting on one item's tile copies (IW 4).
// (Fewer in single systems of up to TEAM_TILES tiles and small ensembles of
// them: one_tile_chunks.)
// Large active sets of large systems (nact >= 8192 over more than 256
// tiles) keep chunks of CHUNK_TILES_LARGE tiles: 8 to 32 items per resident
// workgroup even out the end of the launch, and their finish pass reads
// whole lines of partials (finish_lanes: 4 lanes per particle); measured at
// N = 262144, nact 8192 to 32768: 2-5 % less update time.
constexpr uint32_t TEAM_TILES = 256;  // largest system of k_team_run, in j tiles
constexpr uint32_t NARROW_ACT = 128;  // largest nact that lane_group does not narrow
constexpr uint32_t QUEUE_FACTOR = 16;
constexpr uint32_t CHUNK_TILES = 16;
constexpr uint32_t CHUNK_TILES_LARGE = 4;

struct Decomp {
    uint32_t n_it;             // i tiles
    uint32_t S;                // j chunks
    uint32_t tiles_per_chunk;  // JT tiles per chunk
    uint32_t n_items;          // n_it * S
    uint32_t rows;             // n_it * IW: stride of one chunk in partials
};

// Whether a chunk of a narrow group may be one tile.  In single systems of 5 to
// TEAM_TILES tiles at any width: their small steps are made by one workgroup
// per tile, k_team_run, with these chunks' sums, and the launches gain as well
// (n = 10007 with a tuning table, so without a team: 22.8 -> 21.4 us a step).  In
// those of up to 4 for the larger steps, nact > NARROW_ACT.  Of an ensemble (share: the cluster's
// part of its pairs) in clusters of 5 to TEAM_TILES tiles as long as chunks of 4
// would give all clusters fewer than 256 items, one per CU; more items than
// that cost in partial sums what they gain.  Block steps, us, chunks of 4 | 1 |
// by this rule, FP64:
//   2 clusters of 10000  32.0 | 29.6 | 29.8     64 of 128 to 4096  48.8 |  52.2 |  49.2
//   8 of 4096            34.5 | 32.7 | 32.2    512 of 1100        129.8 | 139.4 | 130.2
constexpr uint32_t ITEMS_ONE = 256;
__host__ __device__ inline bool one_tile_chunks(uint32_t nact, uint32_t iw, uint32_t n_jt,
                                                bool ensemble, double share) {
    if (n_jt > TEAM_TILES) return false;
    if (!ensemble) return n_jt > 4 || nact > NARROW_ACT;
    return n_jt > 4 && (double)((nact + iw - 1) / iw) * ((n_jt + 3) / 4) < share * ITEMS_ONE;
}

__host__ __device__ inline Decomp decompose(uint32_t nact, uint32_t iw,
                                            uint32_t n_jt, uint32_t grid,
                                            uint32_t max_split, bool ensemble = false,
                                            double share = 1.0) {
    Decomp d;
    d.n_it = (nact + iw - 1) / iw;
    uint32_t min_tiles = iw >= 64 || one_tile_chunks(nact, iw, n_jt, ensemble, share) ? 1u : 4u;
    uint32_t S = 1;
    const uint32_t target = grid * QUEUE_FACTOR;
    if (d.n_it > 0 && d.n_it < target) {
        const uint32_t s_fill = d.n_it < grid ? (grid + d.n_it - 1) / d.n_it : 1u;
        const uint32_t s_queue = (target + d.n_it - 1) / d.n_it;
        const uint32_t ct = (nact >= 8192 && n_jt > 256) ? CHUNK_TILES_LARGE : CHUNK_TILES;
        const uint32_t s_tiles = n_jt / ct;
        const uint32_t s_most = s_fill > s_tiles ? s_fill : s_tiles;
        S = s_queue < s_most ? s_queue : s_most;
    }
    if (S > max_split) S = max_split;
    uint32_t s_cap = (n_jt + min_tiles - 1) / min_tiles;
    if (S > s_cap) S = s_cap;
    if (S < 1) S = 1;
    d.tiles_per_chunk = (n_jt + S - 1) / S;
    d.S = d.tiles_per_chunk ? (n_jt + d.tiles_per_chunk - 1) / d.tiles_per_chunk : 1;
    d.n_items = d.n_it * d.S;
    d.rows = d.n_it * iw;
    return d;
}

// Upper bound of the j-split partials (doubles) of one cluster of n
// particles over every plan decompose() can make for a workgroup share of
// at most g / QUEUE_FACTOR: any active count, any lane-group width
// iw <= BS, any split cap.  With S > 1 chunks, S <= ceil(g / n_it) (the
// queue target), so S n_it <= g + n_it - 1
// and 6 S rows = 6 S n_it iw <= 6 (g iw + n + iw); also S <= n_jt and
// rows <= n + iw, so 6 S rows <= 6 n_jt (n + iw).
__host__ __device__ inline unsigned long long partial_bound(uint32_t n, uint32_t g) {
    const unsigned long long iw = BS, n_jt = (n + JT - 1) / JT;
    const unsigned long long a = (unsigned long long)g * iw + n + iw;
    const unsigned long long b = n_jt * ((unsigned long long)n + iw);
    return 6ull * (a < b ? a : b);
}

// The same for K clusters of total size n_total whose workgroup shares
// w_c = max(1, floor(share_c * w)) (shares summing to at most 1) give
// queue targets g_c = QUEUE_FACTOR w_c adding up to at most g + QUEUE_FACTOR K,
// g = QUEUE_FACTOR w: 6 sum_c (g_c BS + n_c + BS) <= 6 (BS (g + (QUEUE_FACTOR + 1) K) + n_total).
__host__ __device__ inline unsigned long long ensemble_partial_bound(uint32_t K,
                                                                     unsigned long long n_total,
                                                                     uint32_t g) {
    return 6ull * ((unsigned long long)BS * ((unsigned long long)g + (QUEUE_FACTOR + 1ull) * K) +
                   n_total);
}

// Lanes of the finish pass that share one particle's S chunk sums: each
// lane adds at most 8 of them (1, 4, 16 or 64 lanes), except that many
// active particles (nact >= 8192, enough to fill the part) take at most 4
// lanes each: a wave then reads whole 128-byte lines of consecutive
// particles' partials rather than one double per line.
__host__ __device__ inline uint32_t finish_lanes(uint32_t S, uint32_t nact) {
    if (S <= 8) return 1u;
    if (S <= 32 || nact >= 8192) return 4u;
    return S <= 128 ? 16u : 64u;
}

// Whether the finish of a block step is one pass over the blocks with active
// particles (k_finish_blocks), or, for ensembles of many blocks, one over the
// active particles and one over the blocks (k_finish_correct,
// k_blockmin_dirty).  The former saves a launch, but has a workgroup's barriers
// for each block, most of which have one or two active particles: beyond what
// is resident at once, that is the longer.  Block steps, us, one pass | two, FP64:
//   1024 blocks (64 clusters of 4096)     79.0 |  81.5
//   2048 (256 of 2048; 32 of 16384)      120.6 | 119.4, 206.2 | 207.2
//   2526 (64 of 1024 to 32768)           252.2 | 246.6
//   4096 (512 of 2048; 64 of 16384)      218.7 | 212.1, 381.7 | 380.6
constexpr uint32_t FINISH_BLOCKS = 2048;
__host__ __device__ inline bool finish_by_blocks(uint32_t K, uint32_t nblk) {
    return K == 1 || nblk <= FINISH_BLOCKS;
}

// Lane-group width for nact active particles: the widest of 256/64/16/4
// that keeps at least fill16/16 of the i slots busy (default 12/16), else
// the least padded.
constexpr uint32_t DEFAULT_IW_FILL = 12;
__host__ __device__ inline uint32_t pick_iw(uint32_t nact, uint32_t fill16 = DEFAULT_IW_FILL) {
    const uint32_t opts[4] = {256, 64, 16, 4};
    uint32_t best = 256, best_pad = 0xffffffffu;
    for (int k = 0; k < 4; ++k) {
        uint32_t iw = opts[k];
        uint32_t slots = (nact + iw - 1) / iw * iw;
        if (16ull * nact >= (unsigned long long)fill16 * slots) return iw;
        if (slots < best_pad) {
            best_pad = slots;
            best = iw;
        }
    }
    return best;
}

// Lane-group width of an FP64 or mixed plan: pick_iw's, but narrower where a
// j range of n_jt chunks at most gives too few work items that wide.  An
// item of 256 slots keeps its workgroup for 256 pairs per lane and tile (some
// 30 us with one wave per SIMD) while, say, 500 of 10007 particles make 80 of
// them.  64 slots make 320 items of a quarter of the work, 16 slots 1280 of a
// sixteenth.  Update times, FP64, 256 | 64 | 16 slots, us:
//   n =  1024, nact  400: 33 | 15 | 10     n = 10007, nact  500: 34 | 21 | 19
//   n =  4096, nact 1000: 33 | 17 | 16     n = 10007, nact 1000: 34 | 25 | 24
//   n =  4096, nact 2000: 35 | 21 | 21     n = 10007, nact 2000: 49 | 35 | 36
//   n =  4096, nact 4096: 37 | 30 | 31     n = 10007, nact 4300: 69 | 66 | 94
//   n = 65536, nact  500: 56 | 53 | 54     n = 10007, nact 6000: 85 | 83 | 117
//   n = 65536, nact 1500: 127 | 164 | 147  n = 20000, nact 4000: 105 | 108 | 111
// The lines: 1024 items of 256 slots (4 per CU), 512 of 64 slots.
// nact <= NARROW_ACT keeps pick_iw's width: those steps are k_small_run's and
// k_team_run's (which takes larger ones too, at the width they have here), whose
// workgroups keep their j and gain nothing.
// Mixed precision narrows to 64 only (n = 4096, nact 1000: 33 -> 13 us), with
// jrun = 1: each j sub-group then takes 64 consecutive j, so that the FP32
// runs are the 32 consecutive pairs that 256 slots sum; with 16 slots they
// would be others.
// share: of the part, in an ensemble.  Its clusters of up to 4 tiles keep
// pick_iw's width, and with it the order of their sums over the thousands of
// steps that k_small_run leaves to the launches a few of (256 clusters of 128 to
// 1024: 50.5 us a step with it, 50.0 narrowed).  Beside a larger cluster, where
// all their steps are launches, narrower groups would gain: with one of 4096
// 65.2 us a step, 49.6 narrowed.
constexpr uint32_t ITEMS_256 = 1024, ITEMS_64 = 512;
struct LaneGroup {
    uint32_t iw, jrun;
};
__host__ __device__ inline LaneGroup lane_group(uint32_t nact, uint32_t fill16, uint32_t n_jt,
                                                bool mixed, double share = 1.0) {
    LaneGroup g{pick_iw(nact ? nact : 1, fill16), 0u};
    if (nact <= NARROW_ACT) return g;
    if (g.iw == 256 && (double)((nact + 255) / 256) * n_jt < share * ITEMS_256) {
        g.iw = 64;
        g.jrun = mixed ? 1u : 0u;
    }
    if (!mixed && g.iw == 64 && (double)((nact + 63) / 64) * n_jt < share * ITEMS_64) g.iw = 16;
    return g;
}

// Whether the exact kernel gives every active particle of a launch a lane of
// its own, or a few of them a workgroup (exact_iw).  Of one system: from
// EXACT_WIDE active ones on, which fill the CUs (n = 65536: 16.0 ms at any nact
// up to 65536, against 0.356 us times nact).
constexpr uint32_t EXACT_WIDE = 45056;
// Of an ensemble's clusters, summed up; all of them the same way, as a lane's
// chain takes twice as long beside the other kind's workgroups (24 clusters of
// 500 to 20000: 6.4 ms mixed, 5.4 and 5.7 unmixed).
struct ExactLoad {
    double pairs;       // nact n
    double act;         // nact
    double lanes;       // nact rounded up to whole workgroups
    double lane_pairs;  // of those with n
    double nmax;        // largest n with an active particle
};
// Times in us.  A few per workgroup: 1.8e11 pairs/s, 250 more of them per
// particle for filling and emptying its pipeline.  A lane each: 4.0e11 pairs/s
// with full CUs, and no less than the chain of the largest cluster, 0.25 us per
// j with one workgroup on a CU and 0.5 with more of them.  Initial forces, wide
// and not, us: 64 clusters of 10000 16050 and 35100, of 1000 290 and 475, of
// 700 205 and 250; 6 of 9000 2270 and 2970; 4 of 3000 760 and 250.
__host__ __device__ inline bool exact_wide(const ExactLoad &l) {
    const double few = 5.6e-6 * (l.pairs + 250.0 * l.act);
    const double per_cu = l.lanes / (256.0 * BS);
    const double chain = 0.25 * l.nmax * (per_cu < 1.0 ? 1.0 : per_cu > 2.0 ? 2.0 : per_cu);
    return chain < few && 2.5e-6 * l.lane_pairs < few;
}

// Active particles per work item of the exact kernel for nact active ones of
// a cluster; load: the nact of a single system of its size with the pairs of
// all clusters (sum of nact n over n), so nact itself for one system.  Few get a
// workgroup each: the ordered add chain bounds it (n = 16385: nact 256 88 us,
// 117 us with 3 per workgroup; both 170 us at 1024).  More share one, 3 chains
// on one wave and its term waves busier (nact 4096: 391 against 631 us; initial
// forces of 64 clusters of 200: 49 against 76 us).
__host__ __device__ inline uint32_t exact_iw(uint32_t nact, double load, bool wide) {
    return wide ? (uint32_t)BS : load <= 768.0 || nact <= 1 ? 1u : 3u;
}

// Work items of the energy of n particles: i blocks of ENERGY_I particles
// against the j chunks of jc particles from the block's first one on, in
// wgs contiguous runs.  The chunk is the largest of 256 ... 16 that gives
// 2048 items, so that a small system's pairs are spread over the CUs too
// (n = 1024: 96 items of 16, not 6 of 256); small items go two to a
// workgroup (fewer workgroup sums to add on the host; n = 4096: 52 us with
// 1024 workgroups), and 2048 workgroups, 8 per CU, take 16 items or more
// each (n = 131072: 3783 -> 3714 us, but n = 65536: 1125 -> 1134 us).
constexpr uint32_t ENERGY_GRID = 2048;  // most workgroups of one cluster
constexpr uint32_t ENERGY_I = 512;
struct EnergyItems {
    uint32_t jc;      // particles per j chunk
    uint32_t chunks;  // j chunks
    uint32_t wgs;     // workgroups
    uint64_t items;
};
__host__ __device__ inline EnergyItems energy_items(uint32_t n) {
    EnergyItems e;
    const uint64_t nb = ((uint64_t)n + ENERGY_I - 1) / ENERGY_I;
    for (e.jc = JT;; e.jc /= 2) {
        e.chunks = (uint32_t)(((uint64_t)n + e.jc - 1) / e.jc);
        e.items = nb * e.chunks - (ENERGY_I / e.jc) * (nb * (nb - 1) / 2);
        if (e.items >= 2048 || e.jc == 16) break;
    }
    e.wgs = e.items >= 16 * ENERGY_GRID ? ENERGY_GRID
            : e.items >= 2048           ? 1024u
            : e.items >= 512            ? (uint32_t)(e.items / 2)
                                        : (uint32_t)(e.items < 256 ? e.items : 256);
    return e;
}

// j tiles of cluster c.
__host__ __device__ __forceinline__ uint32_t ntiles(const Ens &e, uint32_t c) {
    return (e.cnt[c] + JT - 1) / JT;
}

// Work plan of cluster c for nact active particles; W = sum over the
// clusters of nact * n (the update workgroups are shared in proportion);
// wide: of an exact plan, exact_wide.
__host__ __device__ __forceinline__ ClPlan plan_cluster(const Ens &e, uint32_t c, uint32_t nact,
                                                        double W, bool exact, bool mixed,
                                                        bool wide) {
    ClPlan pl;
    pl.cmaj = pl.jrun = 0;
    if (exact) {
        pl.iw = exact_iw(nact, e.K == 1 ? (double)nact : W / (double)e.cnt[c], wide);
        pl.S = 1;
        pl.tpc = ntiles(e, c);
        pl.n_it = (nact + pl.iw - 1) / pl.iw;
        pl.rows = pl.n_it * pl.iw;
        pl.lanes = 1;
        pl.grid = e.grid;
    } else {
        double share = W > 0.0 ? (double)nact * (double)e.cnt[c] / W : 0.0;
        uint32_t g = (uint32_t)(share * e.grid);
        pl.grid = g < 1 ? 1 : g;
        pl.iw = pick_iw(nact ? nact : 1, e.iw_fill);
        const uint32_t nt = ntiles(e, c);
        if (e.K == 1 || nt > 4) {
            const LaneGroup lg = lane_group(nact, e.iw_fill, nt < e.max_split ? nt : e.max_split,
                                            mixed, e.K == 1 ? 1.0 : share);
            pl.iw = lg.iw;
            pl.jrun = lg.jrun;
        }
        if (e.tuned && e.K == 1 && nact) {
            uint32_t bucket = 31u - (uint32_t)__builtin_clz(nact);
            if (e.tune[bucket]) pl.grid = e.tune[bucket] < e.grid ? e.tune[bucket] : e.grid;
            if (e.tune[32 + bucket]) {
                pl.iw = e.tune[32 + bucket];
                pl.jrun = 0;
            }
        }
        Decomp d = decompose(nact, pl.iw, nt, pl.grid, e.max_split, e.K > 1, share);
        pl.S = d.S;
        pl.tpc = d.tiles_per_chunk;
        pl.n_it = d.n_it;
        pl.rows = d.rows;
        pl.lanes = finish_lanes(d.S, nact);
        pl.cmaj = (d.S > 1 && pl.lanes >= 16 && d.rows >= 64) ? 1u : 0u;
    }
    return pl;
}

// ---------------------------------------------------------------------------
// Pair terms
// ---------------------------------------------------------------------------

// The six terms one pair adds in Hermite4CPU::force_calculation
// (Hermite4CPU.cpp:55-82), operation for operation: no contraction, IEEE
// sqrt and division, same association.
__device__ __forceinline__ void terms_exact(const double pi[6], double xj,
                                            double yj, double zj, double vxj,
                                            double vyj, double vzj, double mj,
                                            double e2, double tm[6]) {
#pragma clang fp contract(off)
    double rx = xj - pi[0];
    double ry = yj - pi[1];
    double rz = zj - pi[2];
    double vx = vxj - pi[3];
    double vy = vyj - pi[4];
    double vz = vzj - pi[5];

    double r2 = rx * rx + ry * ry + rz * rz + e2;
    double rinv = 1.0 / sqrt(r2);
    double r2inv = rinv * rinv;
    double r3inv = r2inv * rinv;
    double r5inv = r2inv * r3inv;
    double mr3inv = r3inv * mj;
    double mr5inv = r5inv * mj;

    double rv = rx * vx + ry * vy + rz * vz;

    tm[0] = (rx * mr3inv);
    tm[1] = (ry * mr3inv);
    tm[2] = (rz * mr3inv);
    tm[3] = (vx * mr3inv - (3 * rv) * rx * mr5inv);
    tm[4] = (vy * mr3inv - (3 * rv) * ry * mr5inv);
    tm[5] = (vz * mr3inv - (3 * rv) * rz * mr5inv);
}

// The FP64 pair loop works with s = sqrt(3) / r and q = s^2 = 3 / r^2:
// the jerk coefficient 3 (r.v) / r^2 is then (r.v) q, with no multiply by
// 3, and m s q = 3 sqrt(3) m / r^3, so every pair term it sums is
// 3 sqrt(3) times the true one.  The sums are multiplied by
// PAIR_SCALE = 1 / (3 sqrt 3) once, when the update writes them out.
constexpr double PAIR_SCALE = 0.19245008972987526;

// sqrt(3) / sqrt(x) for x > 0: hardware estimate y = (1 + d) / sqrt(x)
// (v_rsq_f64; |d| < 2^-24 over the FP64 range, measured on the part over 4M inputs),
// then one Newton step sqrt(3) y (1 + e/2), e = 1 - x y^2, which leaves a
// relative error of about -1.5 d^2, below 2^-47.
__device__ __forceinline__ double rsqrt3_fp64(double x) {
    double y = __builtin_amdgcn_rsq(x);
    double e = fma(-x, y * y, 1.0);
    return y * fma(e, 0.8660254037844386, 1.7320508075688772);  // sqrt3 / 2, sqrt3
}

// Same pair as terms_exact with FMA contraction and rsqrt3_fp64, scaled by
// 3 sqrt(3) (see PAIR_SCALE):
//   a  += m r / |r|^3
//   j  += m/|r|^3 (v - 3 (r.v)/|r|^2 r)
__device__ __forceinline__ void pair_fp64(const double pi[6], double xj,
                                          double yj, double zj, double vxj,
                                          double vyj, double vzj, double mj,
                                          double e2, double fo[6]) {
    double rx = xj - pi[0];
    double ry = yj - pi[1];
    double rz = zj - pi[2];
    double vx = vxj - pi[3];
    double vy = vyj - pi[4];
    double vz = vzj - pi[5];
    double r2 = fma(rx, rx, fma(ry, ry, fma(rz, rz, e2)));
    double s = rsqrt3_fp64(r2);  // sqrt(3) / r
    double q = s * s;            // 3 / r^2
    double mr3 = (mj * s) * q;   // 3 sqrt(3) m / r^3
    double rv = fma(rx, vx, fma(ry, vy, rz * vz));
    double c = rv * q;           // 3 (r.v) / r^2
    fo[0] = fma(rx, mr3, fo[0]);
    fo[1] = fma(ry, mr3, fo[1]);
    fo[2] = fma(rz, mr3, fo[2]);
    fo[3] = fma(mr3, fma(-c, rx, vx), fo[3]);
    fo[4] = fma(mr3, fma(-c, ry, vy), fo[4]);
    fo[5] = fma(mr3, fma(-c, rz, vz), fo[5]);
}

// FP32 pair terms from FP32 differences r = x_j - x_i, v = v_j - v_i:
// r^2, 1/r, the force and jerk terms, added into the FP32 partial sums
// t[6].  The caller folds t into FP64 accumulators every few pairs.
// 1/r is v_rsq_f32 itself (within 1 ulp): a Newton step on it (4 more
// instructions per pair) changed the N = 262144 Plummer forces' RMS
// relative error from 2.7e-8 to 1.5e-8 (acceleration) and 2.5e-7 to
// 2.4e-7 (jerk), both inside the mixed contract, the largest errors not at
// all (they come from FP32 cancellation in v - c r), and cost 8 % of the
// kernel's time.  (No sqrt(3) scaling either: the FP32 value of sqrt(3) is
// 1.8e-8 off, a bias every pair term would share.)
__device__ __forceinline__ void pair_terms_f32(float rx, float ry, float rz, float vx,
                                               float vy, float vz, float mj, float e2,
                                               float t[6]) {
    float r2 = fmaf(rx, rx, fmaf(ry, ry, fmaf(rz, rz, e2)));
    float rinv = __builtin_amdgcn_rsqf(r2);
    float rinv2 = rinv * rinv;
    float mr3 = (mj * rinv) * rinv2;
    float rv = fmaf(rx, vx, fmaf(ry, vy, rz * vz));
    float c = (3.0f * rv) * rinv2;
    t[0] = fmaf(rx, mr3, t[0]);
    t[1] = fmaf(ry, mr3, t[1]);
    t[2] = fmaf(rz, mr3, t[2]);
    t[3] = fmaf(mr3, fmaf(-c, rx, vx), t[3]);
    t[4] = fmaf(mr3, fmaf(-c, ry, vy), t[4]);
    t[5] = fmaf(mr3, fmaf(-c, rz, vz), t[5]);
}

// Mixed-precision pair: position and velocity differences in FP64 (they
// cancel for close pairs), rounded once to FP32, then pair_terms_f32.
__device__ __forceinline__ void pair_mixed(const double pi[6], double xj,
                                           double yj, double zj, double vxj,
                                           double vyj, double vzj, float mj,
                                           float e2, float t[6]) {
    pair_terms_f32((float)(xj - pi[0]), (float)(yj - pi[1]), (float)(zj - pi[2]),
                   (float)(vxj - pi[3]), (float)(vyj - pi[4]), (float)(vzj - pi[5]), mj, e2, t);
}

}  // namespace h4
