// h4hip.hip -- libh4hip.so: HIP kernels and C ABI of the MI355X Hermite-4
// block-timestep backend (declarations and contracts in include/h4hip.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "h4hip.h"
#include "h4_kernels.hpp"

using namespace h4;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg) {
    g_err = msg;
    return code;
}

#define H4H_HIP(call)                                                        \
    do {                                                                     \
        hipError_t e_ = (call);                                              \
        if (e_ != hipSuccess)                                                \
            return fail(H4H_EHIP, std::string(#call) + ": " +                \
                                      hipGetErrorString(e_));                \
    } while (0)

#define H4H_LAUNCHED()                                                       \
    do {                                                                     \
        hipError_t e_ = hipGetLastError();                                   \
        if (e_ != hipSuccess)                                                \
            return fail(H4H_EHIP, std::string("kernel launch: ") +           \
                                      hipGetErrorString(e_));                \
    } while (0)

// FP32 partial sums of the mixed kernel are folded into FP64 every
// H4_MIXED_FOLD pairs per lane.
#ifndef H4_MIXED_FOLD
#define H4_MIXED_FOLD 32
#endif
// Unroll of the mixed inner loop: 2 keeps the kernel at 108 VGPRs (4 waves
// per SIMD); 4 needs 132 (3 waves) and measured 1-8 % slower.
#ifndef H4_MIXED_UNROLL
#define H4_MIXED_UNROLL 2
#endif

// Columns of a context's state from r[0] on (create_impl lays them out).
constexpr uint32_t COL_R = 0, COL_M = 3, COL_V = 4, COL_F = 7, COL_OLD = 13, COL_A2 = 19,
                   COL_A3 = 22, COL_T = 25, COL_DT = 26;

constexpr uint32_t DEFAULT_GRID = 2048;       // persistent workgroups
constexpr uint32_t DEFAULT_MAX_SPLIT = 1024;  // largest j split
constexpr uint32_t ENERGY_OUT = 8 * ENERGY_GRID;  // workgroup sums of one energy launch

// ---------------------------------------------------------------------------
// Cluster geometry helpers
// ---------------------------------------------------------------------------
//
// A context holds K independent clusters (K = 1 for a single system).
// Cluster c occupies device indices off[c] .. off[c] + cnt[c] - 1, padded
// to a multiple of JT with zero-mass particles, so every JT block belongs
// to exactly one cluster (bcl[block]) and j tiles never straddle clusters.
// Host arrays hold the clusters back to back (hoff[c]).

__device__ __forceinline__ uint32_t cluster_of_block(const Ens &e, uint32_t b) { return e.bcl[b]; }


// Index of the cluster whose [pre[c], pre[c+1]) range holds x (pre has
// K+1 entries, non-decreasing, pre[0] = 0, x < pre[K]).
__device__ __forceinline__ uint32_t find_cluster(const unsigned long long *pre, uint32_t K,
                                                 unsigned long long x) {
    uint32_t lo = 0, hi = K;  // answer in [lo, hi)
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (pre[mid] <= x)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// Layout kernels (one thread per padded device index)
// ---------------------------------------------------------------------------

struct Cols {
    double *c[8];
    uint32_t stride[8];  // doubles between consecutive particles (0 means 1)
};

__device__ __forceinline__ size_t col_at(const Cols &c, uint32_t k, uint32_t i) {
    return (size_t)i * (c.stride[k] ? c.stride[k] : 1u);
}

// dst.c[k][i] = src[h*ncols + k] for the host index h of device index i.
__global__ __launch_bounds__(BS) void k_aos_to_soa(const double *src, uint32_t ncols, Cols dst,
                                                  Ens e) {
    uint32_t i = blockIdx.x * BS + threadIdx.x;
    if (i >= e.nblk * JT) return;
    uint32_t c = cluster_of_block(e, i / JT);
    uint32_t local = i - e.off[c];
    if (local >= e.cnt[c]) return;
    size_t h = (size_t)e.hoff[c] + local;
    for (uint32_t k = 0; k < ncols; ++k)
        if (dst.c[k]) dst.c[k][col_at(dst, k, i)] = src[h * ncols + k];
}

// dst[h*ncols + k] = src.c[k][i] (NULL columns write 0).
__global__ __launch_bounds__(BS) void k_soa_to_aos(Cols src, uint32_t ncols, double *dst, Ens e) {
    uint32_t i = blockIdx.x * BS + threadIdx.x;
    if (i >= e.nblk * JT) return;
    uint32_t c = cluster_of_block(e, i / JT);
    uint32_t local = i - e.off[c];
    if (local >= e.cnt[c]) return;
    size_t h = (size_t)e.hoff[c] + local;
    for (uint32_t k = 0; k < ncols; ++k)
        dst[h * ncols + k] = src.c[k] ? src.c[k][col_at(src, k, i)] : 0.0;
}

// Same for one array of scalars (t, dt) and for the u32 active list of a
// single cluster context.
__global__ __launch_bounds__(BS) void k_scalar_to_soa(const double *src, double *dst, Ens e) {
    uint32_t i = blockIdx.x * BS + threadIdx.x;
    if (i >= e.nblk * JT) return;
    uint32_t c = cluster_of_block(e, i / JT);
    uint32_t local = i - e.off[c];
    if (local < e.cnt[c]) dst[i] = src[e.hoff[c] + local];
}

__global__ __launch_bounds__(BS) void k_soa_to_scalar(const double *src, double *dst, Ens e) {
    uint32_t i = blockIdx.x * BS + threadIdx.x;
    if (i >= e.nblk * JT) return;
    uint32_t c = cluster_of_block(e, i / JT);
    uint32_t local = i - e.off[c];
    if (local < e.cnt[c]) dst[e.hoff[c] + local] = src[i];
}

// Host arrays of rows (host index h, nc doubles each), numbered one after the
// other: array a's first double is number at[a].  Row element k is state
// column col[a] + k, except element 3 of four: column fourth[a] (NO_COL: 0).
constexpr uint32_t NO_COL = 0xffffffffu;
struct RowArrays {
    uint32_t n;
    unsigned long long at[9];
    uint32_t nc[8], col[8], fourth[8];
};

// Doubles [b, b + len) of the arrays to out, consecutive threads to
// consecutive doubles: out is host memory, and only whole lines cross the bus
// at its rate.
__global__ __launch_bounds__(BS) void k_rows_out(const double *state, RowArrays t, Ens e,
                                                 unsigned long long b, uint32_t len, double *out) {
    const uint32_t x = blockIdx.x * BS + threadIdx.x;
    if (x >= len) return;
    uint32_t a = 0;
    while (a + 1 < t.n && t.at[a + 1] <= b + x) ++a;
    const unsigned long long el = b + x - t.at[a];
    const uint32_t nc = t.nc[a];
    const unsigned long long h = nc == 1 ? el : nc == 3 ? el / 3 : nc == 4 ? el / 4 : el / 6;
    const uint32_t k = (uint32_t)(el - h * nc);
    const uint32_t col = nc == 4 && k == 3 ? t.fourth[a] : t.col[a] + k;
    uint32_t lo = 0, hi = e.K;  // the cluster of host index h
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (e.hoff[mid] <= h)
            lo = mid;
        else
            hi = mid;
    }
    const size_t i = e.off[lo] + (size_t)(h - e.hoff[lo]);
    out[x] = col == NO_COL ? 0.0 : state[(size_t)col * e.nblk * JT + i];
}

// Predictor at t_i (Hermite4::init_data, Hermite4.cpp:194-240): position
// and velocity as corrected, mass rounded to float.  Padding slots get zero
// mass far away and never become active (t = 0, dt = +inf).
__global__ __launch_bounds__(BS) void k_init_predictor(Soa s, Ens e) {
    uint32_t i = blockIdx.x * BS + threadIdx.x;
    if (i >= e.nblk * JT) return;
    uint32_t c = cluster_of_block(e, i / JT);
    if (i - e.off[c] < e.cnt[c]) {
        const float mf = (float)s.m[i];
        s.pp[i] = make_double4(s.r[0][i], s.r[1][i], s.r[2][i], (double)mf);
        s.pv[i] = make_double4(s.v[0][i], s.v[1][i], s.v[2][i], mass_bits(mf));
    } else {
        s.pp[i] = make_double4(PAD_POS, PAD_POS, PAD_POS, 0.0);
        s.pv[i] = make_double4(0.0, 0.0, 0.0, mass_bits(0.0f));
        s.dt[i] = INFINITY;
    }
}

// Active list of every cluster = all its particles (init_acc_jrk).
__global__ __launch_bounds__(BS) void k_identity_active(uint32_t *move, Ens e) {
    uint32_t i = blockIdx.x * BS + threadIdx.x;
    if (i >= e.nblk * JT) return;
    uint32_t c = cluster_of_block(e, i / JT);
    uint32_t local = i - e.off[c];
    if (local < e.cnt[c]) move[i] = i;
    if (local == 0) e.cs[c].nact = e.cnt[c];
}

// ---------------------------------------------------------------------------
// Exchanges inside a wave
// ---------------------------------------------------------------------------

// Lane exchanges by DPP (a few cycles; a ds_bpermute shuffle takes ~100):
// CTRL is the DPP control, BANK the banks of four lanes that take it (the
// others keep `old`).
template <int CTRL, int BANK = 0xf>
__device__ __forceinline__ double dpp(double old, double x) {
    const unsigned long long o = __builtin_bit_cast(unsigned long long, old);
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)o, (int)(uint32_t)u,
                                                              CTRL, 0xf, BANK, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(
        (int)(uint32_t)(o >> 32), (int)(uint32_t)(u >> 32), CTRL, 0xf, BANK, false);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E;     // quad_perm 1,0,3,2 and 2,3,0,1
constexpr int DPP_QUADS = 0x141, DPP_EIGHTS = 0x140;  // row_half_mirror, row_mirror
template <int K>
__device__ __forceinline__ double quad_lane(double x) {  // lane K of each quad
    return dpp<K * 0x55>(x, x);
}
// The value of lane ^ 4: row_shl:4 into banks 0 and 2, row_shr:4 into 1 and 3.
__device__ __forceinline__ double xor4(double x) {
    return dpp<0x114, 0xa>(dpp<0x104, 0x5>(x, x), x);
}
// Swaps the odd rows of 16 lanes (ROWS = 1; the upper half of 32: ROWS = 2)
// of x with the even ones of y: an even row has then x of itself (a) and of
// its odd neighbour (b), an odd row y of its even neighbour (a) and of
// itself (b).
template <int ROWS>
__device__ __forceinline__ void swap_rows(double x, double y, double &a, double &b) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    const unsigned long long t = __builtin_bit_cast(unsigned long long, y);
    uint32_t l0, l1, h0, h1;
    if constexpr (ROWS == 1) {
        const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)u, (uint32_t)t, false, false);
        const auto hi =
            __builtin_amdgcn_permlane16_swap((uint32_t)(u >> 32), (uint32_t)(t >> 32), false, false);
        l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
    } else {
        const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)t, false, false);
        const auto hi =
            __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), (uint32_t)(t >> 32), false, false);
        l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
    }
    a = __builtin_bit_cast(double, ((unsigned long long)h0 << 32) | l0);
    b = __builtin_bit_cast(double, ((unsigned long long)h1 << 32) | l1);
}
// v_min_f64 as it is (fmin also quiets both operands: two more instructions
// each time; a NaN loses either way).
__device__ __forceinline__ double vmin(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Sum over the lane's group of L = 1, 4, 16 or 64 consecutive lanes (all
// lanes of the wave active; every lane of the group gets it): lane ^ 1 first.
__device__ __forceinline__ double lanes_sum(double x, uint32_t L) {
    double a, b;
    if (L >= 4) {
        x += dpp<DPP_XOR1>(x, x);
        x += dpp<DPP_XOR2>(x, x);
    }
    if (L >= 16) {
        x += dpp<DPP_QUADS>(x, x);   // (the quads are uniform by now,
        x += dpp<DPP_EIGHTS>(x, x);  // and the eights)
    }
    if (L >= 64) {
        swap_rows<1>(x, x, a, b);
        x = a + b;
        swap_rows<2>(x, x, a, b);
        x = a + b;
    }
    return x;
}

// Minimum over the wave (all lanes active; every lane gets it).
__device__ __forceinline__ double wave_min(double x) {
    double a, b;
    x = vmin(x, dpp<DPP_XOR1>(x, x));
    x = vmin(x, dpp<DPP_XOR2>(x, x));
    x = vmin(x, dpp<DPP_QUADS>(x, x));   // (the quads are uniform by now,
    x = vmin(x, dpp<DPP_EIGHTS>(x, x));  // and the eights)
    swap_rows<1>(x, x, a, b);
    x = vmin(a, b);
    swap_rows<2>(x, x, a, b);
    return vmin(a, b);
}

// Sums fo over the wave's lanes with the same slot (lane mod P, P < 64 a
// power of two) and stores each slot's six sums at its row.  Swapping halves
// and rows of 16 between two components leaves each half its own three and
// each row one or two, so the later levels move 2 values instead of 6 (41
// instructions at P = 1; 156 with all six carried through six levels).
__device__ __forceinline__ void slot_sums(const double fo[6], uint32_t P, double *row) {
    const uint32_t lane = __lane_id();
    double a, b, u[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {  // lower half: components 0..2, upper: 3..5
        swap_rows<2>(fo[k], fo[3 + k], a, b);
        u[k] = a + b;
    }
    const uint32_t q = lane >= 32 ? 3u : 0u;
    if (P == 32) {
        for (int k = 0; k < 3; ++k) row[q + k] = u[k];
        return;
    }
    swap_rows<1>(u[0], u[1], a, b);  // even rows: component q, odd: q + 1
    double x = a + b;
    swap_rows<1>(u[2], u[2], a, b);  // both: q + 2
    double y = a + b;
    // rotations by 8, 4, 2, 1 inside the rows: lane ^ 8, and so on (uniform
    // under the larger ones by then)
    if (P <= 8) {
        x += dpp<0x128>(x, x);
        y += dpp<0x128>(y, y);
    }
    if (P <= 4) {
        x += dpp<0x124>(x, x);
        y += dpp<0x124>(y, y);
    }
    if (P <= 2) {
        x += dpp<0x122>(x, x);
        y += dpp<0x122>(y, y);
    }
    if (P == 1) {
        x += dpp<0x121>(x, x);
        y += dpp<0x121>(y, y);
    }
    if ((lane & 15u) < P) {
        const bool odd = (lane & 16u) != 0;
        row[q + (odd ? 1u : 0u)] = x;
        if (!odd) row[q + 2] = y;
    }
}

// ---------------------------------------------------------------------------
// Work plan of a step (one workgroup)
// ---------------------------------------------------------------------------

// Per cluster: lane-group width, j split and work items from its active
// count; the update workgroups are shared in proportion to nact * n.
// Exclusive prefix sums over clusters go to items_pre / fin_pre /
// part_pre, totals to ctl.

// Plan of a single-cluster context, made by every workgroup of the update
// kernel from the active count (so the device step needs no k_plan
// launch); workgroup 0 publishes it for the finish pass.
__device__ __forceinline__ ClPlan plan_single(const Ens &e, int prec,
                                              unsigned long long &items) {
    const uint32_t nact = e.cs[0].nact;
    const ClPlan pl = plan_cluster(e, 0, nact, (double)nact * (double)e.cnt[0],
                                   prec == H4H_FP64_EXACT, prec == H4H_MIXED,
                                   nact >= EXACT_WIDE);
    items = nact ? (unsigned long long)pl.n_it * pl.S : 0ull;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const uint32_t per = BS / pl.lanes;
        const unsigned long long units = (nact + per - 1) / per;
        e.plan[0] = pl;
        e.items_pre[0] = e.fin_pre[0] = e.part_pre[0] = 0ull;
        e.items_pre[1] = items;
        e.fin_pre[1] = units;
        e.part_pre[1] = (nact && pl.S > 1) ? 6ull * pl.S * pl.rows : 0ull;
        e.ctl->items = items;
        e.ctl->fin_units = units;
    }
    return pl;
}

__device__ void plan_all(const Ens &e, int prec) {
    __shared__ double wsum[5][BS / 64];
    // nact n of all clusters; the others of ExactLoad for an exact plan
    const bool exact = prec == H4H_FP64_EXACT;
    double w[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (uint32_t c = threadIdx.x; c < e.K; c += BS) {
        const uint32_t nact = e.cs[c].nact;
        const double n = (double)e.cnt[c], lanes = (double)((nact + BS - 1) / BS * BS);
        w[0] += (double)nact * n;
        w[1] += (double)nact;
        w[2] += lanes;
        w[3] += lanes * n;
        w[4] = nact ? fmax(w[4], n) : w[4];
    }
    const uint32_t wave = threadIdx.x >> 6, lane = __lane_id();
    w[0] = lanes_sum(w[0], 64);
    if (lane == 0) wsum[0][wave] = w[0];
    if (exact && e.K > 1) {
        for (int q = 1; q < 4; ++q) w[q] = lanes_sum(w[q], 64);
        w[4] = -wave_min(-w[4]);
        if (lane == 0)
            for (int q = 1; q < 5; ++q) wsum[q][wave] = w[q];
    }
    __syncthreads();
    double W = 0.0;
    for (uint32_t k = 0; k < BS / 64; ++k) W += wsum[0][k];
    bool wide = W >= (double)EXACT_WIDE * (double)e.cnt[0];  // (one system: nact)
    if (exact && e.K > 1) {
        ExactLoad l{W, 0.0, 0.0, 0.0, 0.0};
        for (uint32_t k = 0; k < BS / 64; ++k) {
            l.act += wsum[1][k];
            l.lanes += wsum[2][k];
            l.lane_pairs += wsum[3][k];
            l.nmax = fmax(l.nmax, wsum[4][k]);
        }
        wide = exact_wide(l);
    }
    // The plans, and exclusive prefix sums of work items, finish units and
    // partial doubles over the clusters, BS clusters at a time.
    __shared__ unsigned long long wtot[3][BS / 64];
    unsigned long long carry[3] = {0ull, 0ull, 0ull};
    for (uint32_t base = 0; base < e.K; base += BS) {
        const uint32_t c = base + threadIdx.x;
        unsigned long long v[3] = {0ull, 0ull, 0ull};
        const uint32_t nact = c < e.K ? e.cs[c].nact : 0u;
        if (nact) {
            const ClPlan pl = plan_cluster(e, c, nact, W, exact, prec == H4H_MIXED, wide);
            e.plan[c] = pl;
            const uint32_t per = BS / pl.lanes;
            v[0] = (unsigned long long)pl.n_it * pl.S;
            v[1] = (nact + per - 1) / per;
            v[2] = pl.S > 1 ? 6ull * pl.S * pl.rows : 0ull;
        }
        unsigned long long inc[3] = {v[0], v[1], v[2]};
        for (uint32_t o = 1; o < 64; o <<= 1)
            for (int q = 0; q < 3; ++q) {
                unsigned long long y = __shfl_up(inc[q], o);
                if (__lane_id() >= o) inc[q] += y;
            }
        const uint32_t w = threadIdx.x >> 6;
        if (__lane_id() == 63)
            for (int q = 0; q < 3; ++q) wtot[q][w] = inc[q];
        __syncthreads();
        unsigned long long tot[3];
        for (int q = 0; q < 3; ++q) {
            unsigned long long before = 0ull, all = 0ull;
            for (uint32_t k = 0; k < BS / 64; ++k) {
                if (k < w) before += wtot[q][k];
                all += wtot[q][k];
            }
            inc[q] += before + carry[q];  // inclusive, with earlier chunks
            tot[q] = all;
        }
        if (c < e.K) {
            e.items_pre[c] = inc[0] - v[0];
            e.fin_pre[c] = inc[1] - v[1];
            e.part_pre[c] = inc[2] - v[2];
        }
        for (int q = 0; q < 3; ++q) carry[q] += tot[q];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        e.items_pre[e.K] = carry[0];
        e.fin_pre[e.K] = carry[1];
        e.part_pre[e.K] = carry[2];
        e.ctl->items = carry[0];
        e.ctl->fin_units = carry[1];
    }
}

__global__ __launch_bounds__(BS) void k_plan(Ens e, int prec) { plan_all(e, prec); }

// ---------------------------------------------------------------------------
// Predictor / active selection / save old (one workgroup per JT block)
// ---------------------------------------------------------------------------

enum : uint32_t {
    PS_PREDICT = 1,   // Hermite4CPU::predicted_pos_vel (Hermite4CPU.cpp:340-365)
    PS_SELECT = 2,    // Hermite4::find_particles_to_move (Hermite4.cpp:63-84)
    PS_SAVE_OLD = 4,  // Hermite4::save_old_acc_jrk (Hermite4.cpp:145-153)
    PS_DEVTIME = 8,   // block time = the cluster's ATIME (device step loop)
    PS_DIRTY = 16,    // record blocks holding active particles
    PS_TAIL = 32,     // make the loop tail the previous step left (device loop)
    PS_COMPACT = 64,  // the active particles' records in Ens::arec (with
                      // PS_PREDICT | PS_SELECT | PS_SAVE_OLD)
};

// The loop tail of cluster c's block step number `steps` (1-based in this
// loop) made at block time T with nact active particles, the next block
// time being mn (Hermite4CPU_integration.cpp:81-124): ITIME and ATIME, the
// step and interaction counters, the step history of cluster 0, and the
// stop.  One thread.
__device__ __forceinline__ void record_tail(const Ens &e, uint32_t c, double T, uint32_t nact,
                                            unsigned long long steps, double mn, bool stop) {
    ClState *cs = &e.cs[c];
    if (c == 0) {
        e.hist_t[(steps - 1) % e.hist_cap] = T;
        e.hist_n[(steps - 1) % e.hist_cap] = nact;
    }
    cs->itime = T;
    cs->atime = mn;
    cs->steps = steps;
    cs->interactions += (unsigned long long)nact * e.cnt[c];
    cs->nsteps += nact;
    if (stop) {
        cs->done = 1;
        atomicAdd(&e.ctl->ndone, 1u);
    }
}

// The active set of a cluster is appended to its segment of move[] with one
// atomic per workgroup that has active particles (ballot per wave, prefix
// over the waves in LDS).  Clusters whose loop has stopped are skipped.
// The work plan is made by k_plan afterwards: a last-workgroup pattern
// here would need a device-scope fence per workgroup, i.e. an L2
// write-back on every workgroup of this multi-XCD part.
// Hermite4CPU::predicted_pos_vel (Hermite4CPU.cpp:340-365) of one particle
// (position r, velocity v, forces f, float mass mf) over dt = itime - t,
// as the two predictor records.
__device__ __forceinline__ void predict_vals(const double r[3], const double v[3],
                                             const double f[6], double dt, float mf,
                                             double4 &a, double4 &b) {
#pragma clang fp contract(off)
    double dt2 = (dt * dt);
    double dt3 = (dt2 * dt);
    double dt2c = dt2 / 2.0;
    double dt3c = dt3 / 6.0;
    double pr[3], pvel[3];
    for (int k = 0; k < 3; ++k) {
        pr[k] = (dt3c * f[3 + k]) + (dt2c * f[k]) + (dt * v[k]) + r[k];
        pvel[k] = (dt2c * f[3 + k]) + (dt * f[k]) + v[k];
    }
    a = make_double4(pr[0], pr[1], pr[2], (double)mf);
    b = make_double4(pvel[0], pvel[1], pvel[2], mass_bits(mf));
}

// PS_TAIL (device loop): each cluster's last block step left its loop tail
// in its ClState (tail_*); every workgroup of the cluster takes the next
// block time as the minimum of the cluster's block minima and makes the
// stop decision itself, the cluster's first workgroup records the tail, and
// the step proceeds at that time unless the cluster's loop stops.  This
// launch reads the tail records and the block minima and writes only fields
// no workgroup of it reads (the stop flag aside: a workgroup that sees it
// set would have stopped anyway).  Blocks with active particles go to the
// dirty list `par` (the step's slot in its captured chunk, mod 2).
__global__ __launch_bounds__(BS) void k_select(Soa s, Ens e, uint32_t flags, double itime_arg,
                                              uint32_t par, uint32_t *move) {
#pragma clang fp contract(off)
    __shared__ uint32_t wave_off[BS / 64 + 1];
    __shared__ double wmin[BS / 64];
    __shared__ double s_time;
    __shared__ uint32_t s_go;
    const uint32_t b = blockIdx.x;
    const uint32_t i = b * JT + threadIdx.x;  // inside the padded arrays
    const bool single = e.K == 1;
    const uint32_t c = single ? 0u : cluster_of_block(e, b);
    ClState *cs = &e.cs[c];
    const bool devloop = (flags & (PS_TAIL | PS_DEVTIME)) != 0;
    // The particle's state does not depend on the block time, so its loads
    // go out before the loop tail's minimum is known and their latency
    // overlaps that of the cluster record and the block minima.  A single
    // system loads it at once (the step slots of a captured chunk that find
    // the loop stopped load it for nothing); an ensemble, whose stopped
    // clusters can be most of it, first reads whether the cluster stopped.
    const bool load = single || !devloop || cs->done == 0;
    const bool need_f = (flags & (PS_PREDICT | PS_SAVE_OLD)) != 0;
    double ti = 0.0, dti = 0.0, f[6], r[3], v[3];
    float mf = 0.f;
    for (int k = 0; k < 6; ++k) f[k] = 0.0;
    for (int k = 0; k < 3; ++k) r[k] = v[k] = 0.0;
    if (load) {
        if (flags & (PS_PREDICT | PS_SELECT)) ti = s.t[i];
        if (flags & PS_SELECT) dti = s.dt[i];
        if (need_f)
            for (int k = 0; k < 6; ++k) f[k] = s.f[k][i];
        if (flags & PS_PREDICT) {
            for (int k = 0; k < 3; ++k) {
                r[k] = s.r[k][i];
                v[k] = s.v[k][i];
            }
            mf = (float)s.m[i];
        }
    }
    bool live;
    double itime;
    if (flags & PS_TAIL) {
        // the cluster record, read ahead of the barrier (this launch writes
        // none of these fields that another workgroup reads)
        const uint32_t done = cs->done, pend = cs->tail_pend;
        const double tail_t = cs->tail_t, atime = cs->atime;
        const unsigned long long tail_steps = cs->tail_steps;
        const uint32_t tail_nact = cs->tail_nact;
        const uint32_t b0 = single ? 0u : e.off[c] / JT, nb = single ? e.nblk : ntiles(e, c);
        double mn = INFINITY;
        for (uint32_t k = threadIdx.x; k < nb; k += BS) mn = fmin(mn, e.bmin[b0 + k]);
        mn = wave_min(mn);
        if (__lane_id() == 0) wmin[threadIdx.x >> 6] = mn;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (uint32_t k = 1; k < BS / 64; ++k) mn = fmin(mn, wmin[k]);
            uint32_t go = 0;
            double T = 0.0;
            if (done) {
            } else if (pend) {
                const unsigned long long steps = tail_steps + 1;
                const bool stop = loop_stops(*e.ctl, tail_t, steps, mn);
                if (b == b0) record_tail(e, c, tail_t, tail_nact, steps, mn, stop);
                go = !stop;
                T = mn;
            } else {
                go = 1;
                T = atime;
            }
            s_go = go;
            s_time = T;
        }
        __syncthreads();
        live = s_go != 0;
        itime = s_time;
    } else {
        live = (flags & PS_DEVTIME) ? cs->done == 0 : true;
        itime = (flags & PS_DEVTIME) ? cs->atime : itime_arg;
    }
    const bool in = live && (i - e.off[c]) < e.cnt[c];
    bool act = false;
    double4 pa = {}, pb = {};
    if (in) {
        if (flags & PS_PREDICT) {
            predict_vals(r, v, f, itime - ti, mf, pa, pb);
            s.pp[i] = pa;
            s.pv[i] = pb;
        }
        if (flags & PS_SELECT) {
            double tmp_time = ti + dti;
            act = fabs(itime - tmp_time) < 2 * DBL_EPSILON;
        }
    }
    if (flags & PS_SELECT) {
        unsigned long long mask = __ballot(act);
        uint32_t lane = __lane_id();
        uint32_t w = threadIdx.x >> 6;
        if (lane == 0) wave_off[w] = (uint32_t)__popcll(mask);
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t total = 0;
            for (uint32_t k = 0; k < BS / 64; ++k) {
                uint32_t n = wave_off[k];
                wave_off[k] = total;
                total += n;
            }
            wave_off[BS / 64] = total ? atomicAdd(&cs->nact, total) : 0;
            if (total && (flags & PS_DIRTY)) {
                const uint32_t d = atomicAdd(&e.ctl->ndirty[par], 1u);
                uint32_t *dl = e.dirty + (size_t)par * 3 * e.nblk;
                dl[3 * d] = b;
                dl[3 * d + 1] = wave_off[BS / 64];
                dl[3 * d + 2] = total;
            }
        }
        __syncthreads();
        if (act) {
            unsigned long long below = mask & ((1ull << lane) - 1ull);
            const uint32_t slot =
                e.off[c] + wave_off[BS / 64] + wave_off[w] + (uint32_t)__popcll(below);
            move[slot] = i;
            if (flags & PS_SAVE_OLD)
                for (int k = 0; k < 6; ++k) s.old[k][i] = f[k];
            if (flags & PS_COMPACT) {
                const size_t np = (size_t)e.nblk * JT;
                e.arec[slot] = pa;
                e.arec[np + slot] = pb;
                e.arec[2 * np + slot] = make_double4(f[0], f[1], f[2], dti);
                e.arec[3 * np + slot] = make_double4(f[3], f[4], f[5], 0.0);
            }
        }
    }
}

__global__ __launch_bounds__(BS) void k_save_old(Soa s, Ens e, const uint32_t *move) {
    for (uint32_t c = 0; c < e.K; ++c) {
        uint32_t nact = e.cs[c].nact;
        for (uint32_t k = blockIdx.x * BS + threadIdx.x; k < nact; k += gridDim.x * BS) {
            uint32_t i = move[e.off[c] + k];
            for (int q = 0; q < 6; ++q) s.old[q][i] = s.f[q][i];
        }
    }
}

// ---------------------------------------------------------------------------
// Pairwise acceleration + jerk
// ---------------------------------------------------------------------------

// Loads JT consecutive predictor records starting at j0 into an LDS tile;
// each of the BS (= JT) threads moves one record (two coalesced double4
// loads).  ES = 1: pp records at [0, JT), pv records at [JT, 2 JT);
// ES = 2: record t at [2t] (pp) and [2t + 1] (pv).  Thread t's record goes to place at.
template <uint32_t ES = 1>
__device__ __forceinline__ void load_jtile(const Soa &s, uint32_t j0, double4 *tile,
                                           uint32_t at) {
    tile[ES * at] = s.pp[j0 + threadIdx.x];
    tile[ES == 2 ? 2 * at + 1 : JT + at] = s.pv[j0 + threadIdx.x];
}

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void global_void_t;

// Copies predictor records j0 .. j0 + JT - 1 into an LDS tile (pp records
// at [0, JT), pv records at [JT, 2 JT)) with global_load_lds_dwordx4: the
// data goes from memory to LDS without registers, so the copy of the next
// tile runs while the workgroup computes on the current one; the barrier
// after the computation waits for it (vmcnt).  Each wave moves 64
// consecutive 16-byte units per instruction to consecutive LDS units.
__device__ __forceinline__ void dma_jtile(const Soa &s, uint32_t j0, double4 *dst) {
    const double2 *gp = reinterpret_cast<const double2 *>(s.pp + j0);
    const double2 *gv = reinterpret_cast<const double2 *>(s.pv + j0);
    double2 *lp = reinterpret_cast<double2 *>(dst);
    double2 *lv = reinterpret_cast<double2 *>(dst + JT);
    const uint32_t w = threadIdx.x & ~63u;  // first unit of this wave
    static_assert(2 * JT == 2 * BS, "a tile is 2 x BS 16-byte units per array");
    __builtin_amdgcn_global_load_lds((global_void_t *)(gp + threadIdx.x), (lds_void_t *)(lp + w), 16,
                                     0, 0);
    __builtin_amdgcn_global_load_lds((global_void_t *)(gp + BS + threadIdx.x),
                                     (lds_void_t *)(lp + BS + w), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((global_void_t *)(gv + threadIdx.x), (lds_void_t *)(lv + w), 16,
                                     0, 0);
    __builtin_amdgcn_global_load_lds((global_void_t *)(gv + BS + threadIdx.x),
                                     (lds_void_t *)(lv + BS + w), 16, 0, 0);
}

// Predicted position and velocity of particle i.
__device__ __forceinline__ void load_predictor(const Soa &s, uint32_t i, double pi[6]) {
    const double4 a = s.pp[i], b = s.pv[i];
    pi[0] = a.x;
    pi[1] = a.y;
    pi[2] = a.z;
    pi[3] = b.x;
    pi[4] = b.y;
    pi[5] = b.z;
}

__device__ __forceinline__ float mass_f32(const double4 &b) {
    return __builtin_bit_cast(float, (uint32_t)__builtin_bit_cast(unsigned long long, b.w));
}

// Inner loop of one lane over one LDS tile: the lane's j sub-group js
// takes tile entries js, js + G, ..., G = BS/IW (all JT entries when
// IW = BS).  Entry jj is sp[ES jj] (position, mass) and sv[ES jj]
// (velocity): ES = 1 for a tile stored as two arrays, 2 for one stored as
// interleaved record pairs.  SELF: the tile may hold the lane's own i, whose term is
// skipped (mass 0, and r2 kept finite when e2 == 0).  MIXED: FP32 pair
// terms summed in FP32 over runs of at most 32 pairs, each run then added
// to the FP64 accumulators.
template <int IW, bool SELF, bool MIXED, uint32_t ES>
__device__ __forceinline__ void tile_pairs(const double pi[6], uint32_t i,
                                           uint32_t j0, uint32_t js,
                                           const double4 *sp, const double4 *sv,
                                           double e2, double fo[6]) {
    constexpr uint32_t G = BS / IW;
    constexpr uint32_t NQ = JT / G;
    if constexpr (!MIXED) {
#pragma unroll 4
        for (uint32_t q = 0; q < NQ; ++q) {
            uint32_t jj = js + q * G;
            double4 a = sp[ES * jj];
            double4 b = sv[ES * jj];
            if (SELF) {
                bool me = (j0 + jj) == i;
                double mj = me ? 0.0 : a.w;
                double x = me ? pi[0] + 1.0 : a.x;
                pair_fp64(pi, x, a.y, a.z, b.x, b.y, b.z, mj, e2, fo);
            } else {
                pair_fp64(pi, a.x, a.y, a.z, b.x, b.y, b.z, a.w, e2, fo);
            }
        }
    } else {
        constexpr uint32_t FOLD = NQ < H4_MIXED_FOLD ? NQ : H4_MIXED_FOLD;
        const float e2f = (float)e2;
        for (uint32_t q0 = 0; q0 < NQ; q0 += FOLD) {
            float t[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll H4_MIXED_UNROLL
            for (uint32_t q = q0; q < q0 + FOLD; ++q) {
                uint32_t jj = js + q * G;
                double4 a = sp[ES * jj];
                double4 b = sv[ES * jj];
                if (SELF) {
                    bool me = (j0 + jj) == i;
                    float mj = me ? 0.f : mass_f32(b);
                    double x = me ? pi[0] + 1.0 : a.x;
                    pair_mixed(pi, x, a.y, a.z, b.x, b.y, b.z, mj, e2f, t);
                } else {
                    pair_mixed(pi, a.x, a.y, a.z, b.x, b.y, b.z, mass_f32(b), e2f, t);
                }
            }
            for (int c = 0; c < 6; ++c) fo[c] += (double)t[c];
        }
    }
}

// j sub-group of thread t of an IW-slot group: with IW < 64 slots a wave
// holds 64 / IW sub-groups, numbered by their lane bits reversed so that
// slot_sums adds neighbouring ones first.
template <int IW>
__device__ __forceinline__ uint32_t subgroup(uint32_t t) {
    if constexpr (IW < 64) {
        constexpr uint32_t bits = IW == 4 ? 4 : 2;
        static_assert((IW << bits) == 64, "IW is 4 or 16");
        return (t >> 6) * (64 / IW) + (__brev((t & 63u) / IW) >> (32 - bits));
    } else {
        return t / IW;
    }
}

// Sums fo over the BS/IW j sub-groups of each i slot (thread t of BS): in
// the wave (slot_sums), then over the waves in order through red.  The fixed
// tree makes it deterministic.  IW < BS: leaves, after a barrier, sum q of
// slot k of wave g at red[(g IW + k) 6 + q]; IW = BS: fo already is the slot's.
template <int IW>
__device__ __forceinline__ void reduce_subgroups(const double fo[6], double *red, uint32_t t) {
    if constexpr (IW < BS) {
        const uint32_t w = t >> 6;
        __syncthreads();
        if constexpr (IW < 64) {
            slot_sums(fo, IW, red + (w * IW + t % IW) * 6);
        } else {
            static_assert(IW == 64, "one slot per lane");
            for (int c = 0; c < 6; ++c) red[t * 6 + c] = fo[c];
        }
        __syncthreads();
    }
}

// FP64_EXACT: the pair terms of Hermite4CPU::update_acc_jrk
// (Hermite4CPU.cpp:309-336) added in its order, j ascending, j == i skipped.
// The order makes every component of a particle's sum a chain of n - 1
// dependent FP64 adds (5.5 ns each on the part), but the terms (some 80
// instructions, with an IEEE square root and division) do not depend on each
// other.  One lane per active particle that computes and adds takes 161-235
// ns per j whatever nact is, until its waves fill the SIMDs; with the terms
// spread over waves and one wave adding them, an update takes (n = 1024)
// nact 32: 247 -> 12.6 us, 1024: 250 -> 16 us; (n = 16385) 256: 3870 -> 88
// us, 4096: 3930 -> 390 us, 16385: 3960 -> 1476 us.
constexpr uint32_t XW = BS / 64 - 1;  // waves that compute terms; the last one adds them

// Doubles of LDS of an item of IX particles over j tiles of TJ: two buffers
// of 6 IX rows.  A row's stride of 4 dwords mod 64 lets the adding lanes,
// one row each, read 16 bytes at a time without bank conflicts, and a wave's
// term stores are 64 consecutive doubles.
template <uint32_t IX, uint32_t TJ>
constexpr uint32_t exact_lds() {
    return 2 * 6 * IX * (TJ + 2);
}

// IX active particles against the whole cluster in j tiles of TJ: XW waves
// compute tile t's terms into one LDS buffer (one pair per lane and unit of
// one particle x 64 j) while lane 6 x + q of the remaining wave adds
// component q of particle x of tile t - 1 from the other, in j order.  The
// adding wave is another one of the four from one workgroup of a CU to the
// next, so that they do not share a SIMD.  The skipped
// term (j == i) is stored as +0.0, which leaves every sum as it is (a sum
// that starts at +0.0 is never -0.0).
template <uint32_t IX, uint32_t TJ>
__device__ __forceinline__ void exact_item(const Soa &s, const uint32_t *mv, uint32_t nact,
                                           uint32_t it, uint32_t j_begin, uint32_t n, double e2,
                                           double *lds) {
    constexpr uint32_t TS = TJ + 2, NJ = TJ / 64, UPW = IX * NJ / XW;
    static_assert(IX * NJ % XW == 0 && 6 * IX <= 64 && TJ % 16 == 0, "units over the term waves");
    const uint32_t w = ((threadIdx.x >> 6) + (blockIdx.x >> 8)) % (BS / 64);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t k0 = it * IX;
    const uint32_t tiles = (n + TJ - 1) / TJ;
    const bool adds = w == XW;
    // term waves: unit u = w UPW + k is particle u / NJ, j sub-tile u % NJ
    uint32_t iu[UPW], js[UPW];
    double pi[UPW][6];
    double4 ja[UPW], jb[UPW];
    double acc = 0.0;
    if (!adds) {
#pragma unroll
        for (uint32_t k = 0; k < UPW; ++k) {
            const uint32_t u = w * UPW + k, a = k0 + u / NJ;
            iu[k] = mv[a < nact ? a : nact - 1];
            js[k] = (u % NJ) * 64 + lane;
            load_predictor(s, iu[k], pi[k]);
            const uint32_t j = j_begin + min(js[k], n - 1);
            ja[k] = s.pp[j];
            jb[k] = s.pv[j];
        }
    }
    for (uint32_t t = 0; t <= tiles; ++t) {
        if (!adds) {
            if (t < tiles) {
                double *buf = lds + (t & 1u) * (6 * IX * TS);
#pragma unroll
                for (uint32_t k = 0; k < UPW; ++k) {
                    const double4 a = ja[k], b = jb[k];
                    const uint32_t j = t * TJ + js[k];
                    if (t + 1 < tiles) {  // the next tile's records, under this one's terms
                        const uint32_t jn = j_begin + min(j + TJ, n - 1);
                        ja[k] = s.pp[jn];
                        jb[k] = s.pv[jn];
                    }
                    double tm[6];
                    terms_exact(pi[k], a.x, a.y, a.z, b.x, b.y, b.z, a.w, e2, tm);
                    double *row = buf + 6 * ((w * UPW + k) / NJ) * TS + js[k];
                    const bool me = j_begin + j == iu[k];
                    if (__ballot(me))  // (one tile in n / TJ)
                        for (uint32_t q = 0; q < 6; ++q) tm[q] = me ? 0.0 : tm[q];
                    for (uint32_t q = 0; q < 6; ++q) row[q * TS] = tm[q];
                }
            }
        } else if (t > 0 && lane < 6 * IX) {
            const double *row = lds + ((t - 1) & 1u) * (6 * IX * TS) + lane * TS;
            const uint32_t jn = min(TJ, n - (t - 1) * TJ);
            constexpr uint32_t U = 16;  // terms in flight from LDS ahead of the adds
            if (jn == TJ) {
                double2 cur[U / 2], nxt[U / 2];
                const double2 *r2 = reinterpret_cast<const double2 *>(row);
                for (uint32_t k = 0; k < U / 2; ++k) cur[k] = r2[k];
#pragma unroll
                for (uint32_t j = 0; j < TJ; j += U) {
                    if (j + U < TJ)
                        for (uint32_t k = 0; k < U / 2; ++k) nxt[k] = r2[(j + U) / 2 + k];
                    for (uint32_t k = 0; k < U / 2; ++k) {
                        acc += cur[k].x;
                        acc += cur[k].y;
                    }
                    for (uint32_t k = 0; k < U / 2; ++k) cur[k] = nxt[k];
                }
            } else {
                for (uint32_t j = 0; j < jn; ++j) acc += row[j];
            }
        }
        __syncthreads();
    }
    if (adds && lane < 6 * IX) {
        const uint32_t a = k0 + lane / 6;
        if (a < nact) s.f[lane % 6][mv[a]] = acc;
    }
}

// One lane per active particle (BS of them per item), its own adds the
// chain.
__device__ __forceinline__ void exact_item_wide(const Soa &s, const uint32_t *mv, uint32_t nact,
                                                uint32_t it, uint32_t j_begin, uint32_t n,
                                                double e2, double4 *tile) {
    const double4 *sp = tile, *sv = tile + JT;
    const uint32_t k = it * BS + threadIdx.x;
    const bool act = k < nact;
    const uint32_t i = act ? mv[k] : mv[0];
    const uint32_t j_end = j_begin + n;
    double pi[6];
    load_predictor(s, i, pi);
    double fo[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (uint32_t j0 = j_begin; j0 < j_end; j0 += JT) {
        __syncthreads();
        load_jtile(s, j0, tile, threadIdx.x);
        __syncthreads();
        const uint32_t jn = min((uint32_t)JT, j_end - j0);
        for (uint32_t jj = 0; jj < jn; ++jj) {
            const double4 a = sp[jj], b = sv[jj];
            if (j0 + jj != i) {
                double tm[6];
                terms_exact(pi, a.x, a.y, a.z, b.x, b.y, b.z, a.w, e2, tm);
                for (int q = 0; q < 6; ++q) fo[q] += tm[q];
            }
        }
    }
    __syncthreads();  // the next item may write the tile as its term buffer
    if (act)
        for (int q = 0; q < 6; ++q) s.f[q][i] = fo[q];
}

// Workgroups stride over the plan's items (exact_iw particles each) and
// write f[i] directly.
__global__ __launch_bounds__(BS) void k_update_exact(Soa s, Ens e, const uint32_t *move,
                                                    double e2) {
    constexpr uint32_t L1 = exact_lds<1, 192>(), L3 = exact_lds<3, 64>();
    constexpr uint32_t LX = L1 > L3 ? L1 : L3, LM = LX > 8 * JT ? LX : 8 * JT;
    __shared__ __align__(32) double lds[LM];
    const bool single = e.K == 1;
    unsigned long long total = 0;
    ClPlan pl0{};
    if (single)
        pl0 = plan_single(e, H4H_FP64_EXACT, total);
    else
        total = e.ctl->items;
    for (unsigned long long item = blockIdx.x; item < total; item += gridDim.x) {
        const uint32_t c = single ? 0u : find_cluster(e.items_pre, e.K, item);
        const uint32_t it = (uint32_t)(item - (single ? 0ull : e.items_pre[c]));
        const uint32_t iw = single ? pl0.iw : e.plan[c].iw;
        const uint32_t nact = e.cs[c].nact, off = e.off[c], n = e.cnt[c];
        const uint32_t *mv = move + off;
        // (every item ends with a barrier after its last read of lds)
        if (iw == 1)
            exact_item<1, 192>(s, mv, nact, it, off, n, e2, lds);
        else if (iw == 3)
            exact_item<3, 64>(s, mv, nact, it, off, n, e2, lds);
        else
            exact_item_wide(s, mv, nact, it, off, n, e2, reinterpret_cast<double4 *>(lds));
    }
}

// One work item of the FP64 / mixed update: i tile `it` of a cluster
// against j chunk `sc`.  With one chunk the result goes to f[i]; with
// several, the chunk sums go to partial[partial_at(pl, comp, sc, k)] and
// the finish pass adds them in chunk order.
template <int IW, bool MIXED>
__device__ __forceinline__ void update_item(const Soa &s, const ClPlan &pl, uint32_t jt_begin,
                                            uint32_t jt_end, uint32_t it, uint32_t sc,
                                            const uint32_t *mv, const double4 *cr, size_t np,
                                            uint32_t nact, double *partial, double e2,
                                            double4 *lA, double4 *lB, double *red) {
    const uint32_t il = threadIdx.x % IW;
    const uint32_t js = subgroup<IW>(threadIdx.x);
    uint32_t k = it * IW + il;
    bool act = k < nact;
    uint32_t t0 = jt_begin + sc * pl.tpc;
    uint32_t t1 = min(jt_end, t0 + pl.tpc);
    // FP64 wide groups keep their tile as interleaved (position, velocity)
    // record pairs: every LDS read of the pair loop then fits the
    // instructions' offset field, with no extra address arithmetic (0.5 %
    // on the full step; the mixed kernel runs as fast with two arrays).
    constexpr uint32_t ES = (IW >= 64 && !MIXED) ? 2u : 1u;
    // jrun: record j of a tile is stored where sub-group j / 64 reads its
    // (j % 64)th (a second pair loop for it made the mixed kernel 12
    // registers larger and 0.5 % slower).
    constexpr bool RUNS = IW == 64 && MIXED;
    auto place = [&](uint32_t j) { return RUNS && pl.jrun ? (j % 64) * (JT / 64) + j / 64 : j; };
    const uint32_t at = place(threadIdx.x);
    // The first j tile is requested before the i particles, whose loads wait
    // for their indices, so the two memory latencies overlap: narrow groups
    // start its copy into lA (once the previous item is done with lA: tiles
    // or red), wide groups load it into registers.
    [[maybe_unused]] double4 ja, jb;
    if constexpr (IW < 64) {
        __syncthreads();
        dma_jtile(s, t0 * JT, lA);
    } else {
        ja = s.pp[t0 * JT + threadIdx.x];
        jb = s.pv[t0 * JT + threadIdx.x];
    }
    // The i particles' predictors: from the selection's records in
    // active-list order when it wrote them (cr; then their loads wait for
    // no index), else through the active list.
    uint32_t i = act ? mv[k] : mv[0];
    double pi[6];
    if (cr) {
        const uint32_t kk = act ? k : 0u;
        const double4 a = cr[kk], b = cr[np + kk];
        pi[0] = a.x;
        pi[1] = a.y;
        pi[2] = a.z;
        pi[3] = b.x;
        pi[4] = b.y;
        pi[5] = b.z;
    } else {
        load_predictor(s, i, pi);
    }
    double fo[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    auto tile = [&](const double4 *buf, uint32_t tt) {
        const uint32_t j0 = tt * JT;
        const bool self = (i - j0) < (uint32_t)JT;
        const double4 *sv = ES == 2 ? buf + 1 : buf + JT;
        if (__ballot(self))
            tile_pairs<IW, true, MIXED, ES>(pi, RUNS && self ? j0 + place(i - j0) : i, j0, js, buf,
                                            sv, e2, fo);
        else
            tile_pairs<IW, false, MIXED, ES>(pi, i, j0, js, buf, sv, e2, fo);
    };
    // Narrow lane groups (few pairs per lane and tile): double-buffered
    // tiles, the copy of tile tt + 1 in flight while tile tt is computed, one
    // barrier per tile.  The loop is written out for the two buffers so that
    // the compiler sees the copy's target and the tile being read as
    // different LDS objects and does not wait for the copy before each
    // read.  red overlays lA, whose last reader has passed a barrier before
    // reduce_subgroups.
    if constexpr (IW < 64) {
        __syncthreads();  // the first tile's copy has landed
        for (uint32_t tt = t0; tt < t1; tt += 2) {
            if (tt + 1 < t1) dma_jtile(s, (tt + 1) * JT, lB);
            tile(lA, tt);
            __syncthreads();
            if (tt + 1 >= t1) break;
            if (tt + 2 < t1) dma_jtile(s, (tt + 2) * JT, lA);
            tile(lB, tt + 1);
            __syncthreads();
        }
    } else {
        // Wide lane groups do 64-256 pairs per lane and tile: the copy is
        // a small share of the time and one buffer keeps registers free.
        __syncthreads();  // the previous item is done with lA (tiles or red)
        lA[ES * at] = ja;
        lA[ES == 2 ? 2 * at + 1 : JT + at] = jb;
        __syncthreads();
        tile(lA, t0);
        for (uint32_t tt = t0 + 1; tt < t1; ++tt) {
            __syncthreads();
            load_jtile<ES>(s, tt * JT, lA, at);
            __syncthreads();
            tile(lA, tt);
        }
    }
    reduce_subgroups<IW>(fo, red, threadIdx.x);
    if constexpr (IW == BS) {
        constexpr double scale = MIXED ? 1.0 : PAIR_SCALE;  // pair_fp64's 3 sqrt(3)
        if (act) {
            if (pl.S == 1) {
                const size_t fs = s.f[1] - s.f[0];  // (columns equally spaced)
                double *fi = s.f[0] + i;
                for (int q = 0; q < 6; ++q) fi[q * fs] = fo[q] * scale;
            } else {
                // partial_at(pl, q, sc, k), with the layout's strides
                const size_t kst = pl.cmaj ? pl.S : 1u, cst = pl.cmaj ? 1u : pl.rows;
                double *pq = partial + (size_t)sc * cst + (size_t)k * kst;
                const size_t qs = (size_t)pl.S * pl.rows;
                for (int q = 0; q < 6; ++q) pq[q * qs] = fo[q] * scale;
            }
        }
    }
}

// The sums of an item of less than BS slots, one thread per slot and
// component (consecutive slots on consecutive threads): the waves' sums in
// order from red, to f[i] or the item's partials.
template <bool MIXED>
__device__ __forceinline__ void store_item(const Soa &s, const ClPlan &pl, uint32_t it, uint32_t sc,
                                           const uint32_t *mv, uint32_t nact, double *partial,
                                           const double *red) {
    constexpr double scale = MIXED ? 1.0 : PAIR_SCALE;
    const uint32_t iw = pl.iw, lw = 31u - (uint32_t)__clz(iw);
    const size_t kst = pl.cmaj ? pl.S : 1u, cst = pl.cmaj ? 1u : pl.rows;
    const size_t qs = (size_t)pl.S * pl.rows;
    for (uint32_t x = threadIdx.x; x < 6 * iw; x += BS) {
        const uint32_t q = x >> lw, sl = x & (iw - 1), ks = it * iw + sl;
        if (ks >= nact) continue;
        double f = red[sl * 6 + q];
        for (uint32_t g = 1; g < BS / 64; ++g) f += red[(g * iw + sl) * 6 + q];
        f *= scale;
        if (pl.S == 1)
            s.f[0][(size_t)q * (s.f[1] - s.f[0]) + mv[ks]] = f;  // (columns equally spaced)
        else
            partial[(size_t)sc * cst + (size_t)ks * kst + q * qs] = f;
    }
}

// FP64 and mixed precision: persistent workgroups over the plan's work
// items of all clusters; each item's lane-group width comes from the plan,
// so one launch serves every active-set size.
template <bool MIXED>
__device__ __forceinline__ void update_items(const Soa &s, const Ens &e, const uint32_t *move,
                                             double *partial, double e2, uint32_t compact) {
    __shared__ double4 lA[2 * JT];
    __shared__ double4 lB[2 * JT];
    static_assert(BS * 6 * sizeof(double) <= sizeof(lA), "red overlays lA");
    double *red = reinterpret_cast<double *>(lA);
    const bool single = e.K == 1;
    unsigned long long total = 0;
    const ClPlan pl0 = single ? plan_single(e, MIXED ? H4H_MIXED : H4H_FP64, total) : ClPlan{};
    if (!single) total = e.ctl->items;
    // The first gridDim.x items go one to each workgroup; a workgroup that
    // has finished one takes the next unclaimed item from the queue counter,
    // so faster CUs and XCDs take more.  The last workgroup to leave the
    // queue zeroes it for the next launch.
    __shared__ unsigned long long claimed;
    unsigned long long item = blockIdx.x;
    while (item < total) {
        const uint32_t c = single ? 0u : find_cluster(e.items_pre, e.K, item);
        const ClPlan pl = single ? pl0 : e.plan[c];
        const uint32_t li = (uint32_t)(item - (single ? 0ull : e.items_pre[c]));
        // j-chunk major: items taken at about the same time share their j
        // tiles (one chunk per XCD L2 rather than S of them)
        const uint32_t sc = li / pl.n_it;
        const uint32_t it = li - sc * pl.n_it;
        const uint32_t nact = e.cs[c].nact;
        const uint32_t jt_begin = e.off[c] / JT;
        const uint32_t jt_end = jt_begin + ntiles(e, c);
        const uint32_t *mv = move + e.off[c];
        const double4 *cr = compact ? e.arec + e.off[c] : nullptr;
        const size_t np = (size_t)e.nblk * JT;
        double *part = partial + (single ? 0ull : e.part_pre[c]);
        switch (pl.iw) {
            case 4:
                update_item<4, MIXED>(s, pl, jt_begin, jt_end, it, sc, mv, cr, np, nact, part, e2,
                                      lA, lB, red);
                break;
            case 16:
                update_item<16, MIXED>(s, pl, jt_begin, jt_end, it, sc, mv, cr, np, nact, part, e2,
                                       lA, lB, red);
                break;
            case 64:
                update_item<64, MIXED>(s, pl, jt_begin, jt_end, it, sc, mv, cr, np, nact, part, e2,
                                       lA, lB, red);
                break;
            default:
                update_item<256, MIXED>(s, pl, jt_begin, jt_end, it, sc, mv, cr, np, nact, part, e2,
                                        lA, lB, red);
                break;
        }
        if (pl.iw < BS) store_item<MIXED>(s, pl, it, sc, mv, nact, part, red);
        if (total <= gridDim.x) break;
        __syncthreads();  // every lane has read the previous claim
        if (threadIdx.x == 0) claimed = gridDim.x + atomicAdd(&e.ctl->qnext, 1ull);
        __syncthreads();
        item = claimed;
    }
    // Every workgroup claims until it draws an index >= total and then
    // counts itself out; when all have, no claim of this launch remains.
    if (total > gridDim.x && threadIdx.x == 0 &&
        atomicAdd(&e.ctl->qdone, 1u) == gridDim.x - 1) {
        atomicExch(&e.ctl->qnext, 0ull);
        atomicExch(&e.ctl->qdone, 0u);
    }
}

// The four lane-group variants in one kernel would take 144 VGPRs (3 waves
// per SIMD); each alone needs <= 126, so the FP64 kernel is held to 128
// (4 waves per SIMD; a few per-item values spill to scratch, none inside
// the tile or pair loops).  The mixed kernel fits in 120 by itself.
// compact: the step's selection wrote the active particles' records
// (k_select PS_COMPACT).
__global__ __launch_bounds__(BS, 4) void k_update_fp64(Soa s, Ens e, const uint32_t *move,
                                                      double *partial, double e2,
                                                      uint32_t compact) {
    update_items<false>(s, e, move, partial, e2, compact);
}

__global__ __launch_bounds__(BS) void k_update_mixed(Soa s, Ens e, const uint32_t *move,
                                                    double *partial, double e2,
                                                    uint32_t compact) {
    update_items<true>(s, e, move, partial, e2, compact);
}

// ---------------------------------------------------------------------------
// Corrector + Aarseth timestep + block quantisation
// ---------------------------------------------------------------------------

// NbodyUtils::get_magnitude (NbodyUtils.cpp:331-334).
__device__ __forceinline__ double magnitude(double x, double y, double z) {
#pragma clang fp contract(off)
    return sqrt(x * x + y * y + z * z);
}

// Whether block time t is commensurate with twice the step (the condition of
// NbodyUtils::normalize_dt for doubling it).
__device__ __forceinline__ bool dt_doubles(double old_dt, double t) {
#pragma clang fp contract(off)
    const double val = t / (2 * old_dt);
    return ceil(val) == val;
}

// NbodyUtils::normalize_dt (NbodyUtils.cpp:371-424), bounds as arguments;
// doubles() gives dt_doubles(old_dt, t).
template <class F>
__device__ __forceinline__ double normalize_dt(double new_dt, double old_dt, F doubles,
                                               double dt_min, double dt_max) {
#pragma clang fp contract(off)
    // (selects from the last branch to the first; NaN keeps the old step)
    double res = old_dt;
    if (2 * old_dt < new_dt) res = doubles() ? 2.0 * old_dt : old_dt;
    res = old_dt / 2 < new_dt && new_dt <= old_dt ? old_dt / 2 : res;
    res = old_dt / 4 < new_dt && new_dt <= old_dt / 2 ? old_dt / 4 : res;
    res = old_dt / 8 < new_dt && new_dt <= old_dt / 4 ? old_dt / 8 : res;
    new_dt = new_dt <= old_dt / 8 ? dt_min : res;
    return new_dt < dt_min ? dt_min : new_dt > dt_max ? dt_max : new_dt;
}

// Hermite4CPU::correction_pos_vel (Hermite4CPU.cpp:370-411) with
// NbodyUtils::get_timestep_normal (NbodyUtils.cpp:337-365) of one particle
// at block time itime: old forces o, new forces f, predictor pr (position,
// velocity), step dt1, ETA (the reference's float, widened exactly).  Writes
// the corrected position rn and velocity vn and a2, a3; returns the new step.
__device__ __forceinline__ double correct_vals(const double o[6], const double f[6],
                                               const double pr[6], double dt1, double itime,
                                               double eta, double dt_min, double dt_max,
                                               double rn[3], double vn[3], double a2[3],
                                               double a3[3]) {
#pragma clang fp contract(off)
    double dt2 = dt1 * dt1;
    double dt3 = dt2 * dt1;
    double dt4 = dt2 * dt2;
    double dt5 = dt4 * dt1;
    for (int c = 0; c < 3; ++c)
        a2[c] = (-6 * (o[c] - f[c]) - dt1 * (4 * o[3 + c] + 2 * f[3 + c])) / dt2;
    for (int c = 0; c < 3; ++c)
        a3[c] = (12 * (o[c] - f[c]) + 6 * dt1 * (o[3 + c] + f[3 + c])) / dt3;
    for (int c = 0; c < 3; ++c) {
        rn[c] = pr[c] + (dt4 / 24) * a2[c] + (dt5 / 120) * a3[c];
        vn[c] = pr[3 + c] + (dt3 / 6) * a2[c] + (dt4 / 24) * a3[c];
    }
    double ax1_2 = a2[0] + dt1 * a3[0];
    double ay1_2 = a2[1] + dt1 * a3[1];
    double az1_2 = a2[2] + dt1 * a3[2];
    double abs_a1 = magnitude(f[0], f[1], f[2]);
    double abs_j1 = magnitude(f[3], f[4], f[5]);
    double abs_j12 = abs_j1 * abs_j1;
    double abs_a1_3 = magnitude(a3[0], a3[1], a3[2]);
    double abs_a1_2 = magnitude(ax1_2, ay1_2, az1_2);
    double abs_a1_22 = abs_a1_2 * abs_a1_2;
    double normal_dt = sqrt(eta * ((abs_a1 * abs_a1_2 + abs_j12) /
                                   (abs_j1 * abs_a1_3 + abs_a1_22)));
    return normalize_dt(normal_dt, dt1, [&] { return dt_doubles(dt1, itime); }, dt_min, dt_max);
}

// The corrector of one particle on 8 consecutive lanes of a wave (all lanes
// active): lane c + 4 vel has component c (0..2; lane 3 repeats 2) of the
// position and a2 (vel = 0) or of the velocity and a3 (vel = 1).  The same
// operations as correct_vals, value by value, so the same bits; on one lane
// they are ~600 instructions, 18 of them IEEE divisions and square roots one
// after the other (5900 cycles in a one-workgroup step), here a chain of two
// divisions and two square roots.
struct Corr8 {
    double dt1, den, k1, k2;
    bool doubles;
};
// What depends on the step and the block time only.
__device__ __forceinline__ Corr8 corr8_coef(double dt1, double itime, bool vel) {
#pragma clang fp contract(off)
    const double dt2 = dt1 * dt1;
    const double dt3 = dt2 * dt1;
    const double dt4 = dt2 * dt2;
    const double dt5 = dt4 * dt1;
    Corr8 k;
    k.dt1 = dt1;
    k.den = vel ? dt3 : dt2;
    k.k1 = (vel ? dt3 : dt4) / (vel ? 6.0 : 24.0);
    k.k2 = (vel ? dt4 : dt5) / (vel ? 24.0 : 120.0);
    k.doubles = dt_doubles(dt1, itime);
    return k;
}
// o0, o1 and f0, f1: component c of the old and new acceleration and jerk;
// pr: of the predicted position or velocity.  x: the corrected one, ad: a2
// or a3 of the component; returns the new step (every lane).
__device__ __forceinline__ double corr8(const Corr8 &k, bool vel, double o0, double o1, double f0,
                                        double f1, double pr, double eta, double dt_min,
                                        double dt_max, double &x, double &ad) {
#pragma clang fp contract(off)
    const double dt1 = k.dt1;
    const double n2 = -6 * (o0 - f0) - dt1 * (4 * o1 + 2 * f1);
    const double n3 = 12 * (o0 - f0) + 6 * dt1 * (o1 + f1);
    ad = (vel ? n3 : n2) / k.den;
    const double other = xor4(ad);
    const double a2 = vel ? other : ad, a3 = vel ? ad : other;
    x = pr + k.k1 * a2 + k.k2 * a3;
    // squared lengths: acceleration and jerk (vel = 0); a3 and the second
    // derivative at the new time (vel = 1), one square root per lane
    const double a1_2 = a2 + dt1 * a3;
    const double p = vel ? a3 : f0, q = vel ? a1_2 : f1;
    const double p2 = p * p, q2 = q * q;
    const double sp = quad_lane<0>(p2) + quad_lane<1>(p2) + quad_lane<2>(p2);
    const double sq = quad_lane<0>(q2) + quad_lane<1>(q2) + quad_lane<2>(q2);
    const double m = sqrt((threadIdx.x & 1u) ? sq : sp);
    const double mp = quad_lane<0>(m), mq = quad_lane<1>(m);
    const double op = dpp<DPP_QUADS>(mp, mp), oq = dpp<DPP_QUADS>(mq, mq);
    const double abs_a1 = vel ? op : mp, abs_j1 = vel ? oq : mq;
    const double abs_a1_3 = vel ? mp : op, abs_a1_2 = vel ? mq : oq;
    const double abs_j12 = abs_j1 * abs_j1;
    const double abs_a1_22 = abs_a1_2 * abs_a1_2;
    const double normal_dt = sqrt(eta * ((abs_a1 * abs_a1_2 + abs_j12) /
                                         (abs_j1 * abs_a1_3 + abs_a1_22)));
    return normalize_dt(normal_dt, dt1, [&] { return k.doubles; }, dt_min, dt_max);
}

// The corrector of particle i at block time itime, given its new forces
// f[6] (old forces in s.old, predictor in s.pp / s.pv), on the state in
// HBM.  Returns the new dt.
__device__ __forceinline__ double correct_store(const Soa &s, uint32_t i, const double o[6],
                                                const double pr[6], double dt1, const double f[6],
                                                double itime, float eta, double dt_min,
                                                double dt_max) {
    double rn[3], vn[3], a2[3], a3[3];
    const double dt_new =
        correct_vals(o, f, pr, dt1, itime, eta, dt_min, dt_max, rn, vn, a2, a3);
    for (int c = 0; c < 3; ++c) {
        s.r[c][i] = rn[c];
        s.v[c][i] = vn[c];
        s.a2[c][i] = a2[c];
        s.a3[c][i] = a3[c];
    }
    s.t[i] = itime;
    s.dt[i] = dt_new;
    return dt_new;
}

__device__ __forceinline__ double correct_one(const Soa &s, uint32_t i, const double f[6],
                                              double itime, float eta, double dt_min,
                                              double dt_max) {
    double o[6], pr[6];
    for (int c = 0; c < 6; ++c) o[c] = s.old[c][i];
    load_predictor(s, i, pr);
    return correct_store(s, i, o, pr, s.dt[i], f, itime, eta, dt_min, dt_max);
}

// The corrector's inputs of the particle at place k of the step's active
// list from the selection's records (Ens::arec): old forces o, predictor
// pr, step dt1.
__device__ __forceinline__ void load_arec(const Ens &e, size_t k, double o[6], double pr[6],
                                          double &dt1) {
    const size_t np = (size_t)e.nblk * JT;
    const double4 p = e.arec[k], q = e.arec[np + k], a = e.arec[2 * np + k],
                  j = e.arec[3 * np + k];
    pr[0] = p.x;
    pr[1] = p.y;
    pr[2] = p.z;
    pr[3] = q.x;
    pr[4] = q.y;
    pr[5] = q.z;
    o[0] = a.x;
    o[1] = a.y;
    o[2] = a.z;
    o[3] = j.x;
    o[4] = j.y;
    o[5] = j.z;
    dt1 = a.w;
}

// Standalone corrector of cluster 0's active list at itime (the ABI call
// h4h_correction_pos_vel): forces from s.f.
__global__ __launch_bounds__(BS) void k_correct(Soa s, Ens e, const uint32_t *move, double itime,
                                               float eta, double dt_min, double dt_max) {
    const uint32_t nact = e.cs[0].nact;
    for (uint32_t k = blockIdx.x * BS + threadIdx.x; k < nact; k += gridDim.x * BS) {
        uint32_t i = move[k];
        double f[6];
        for (int c = 0; c < 6; ++c) f[c] = s.f[c][i];
        correct_one(s, i, f, itime, eta, dt_min, dt_max);
    }
}


// Sum of active particle k's S j-chunk partials (plan pl, partials of its
// cluster at part) on the group of L = pl.lanes consecutive lanes of one
// wave that share it: lane sl adds chunks sl, sl + L, ... in that order,
// then a fixed xor butterfly over the group, so the order is fixed for a
// given plan and results are deterministic.  With one chunk the update
// stored the forces in f[i].  Every lane of the group gets the sums.
__device__ __forceinline__ void chunk_sums(const Soa &s, const ClPlan &pl, const double *part,
                                           uint32_t k, uint32_t i, bool valid, double f[6]) {
    const uint32_t L = pl.lanes;
    const uint32_t sl = threadIdx.x % L;
    if (pl.S == 1) {
        for (int q = 0; q < 6; ++q) f[q] = valid ? s.f[q][i] : 0.0;
        return;
    }
    // The loads of a round of U chunks of all six components are issued
    // together (a few memory latencies per round instead of one per chunk;
    // S <= 1024 takes two rounds at L = 64).
    constexpr uint32_t U = 8;
    // stride between consecutive chunks and between components (partial_at)
    const size_t cs = pl.cmaj ? 1 : pl.rows;
    const size_t qs = (size_t)pl.S * pl.rows;
    const double *pk = part + (pl.cmaj ? (size_t)k * pl.S : (size_t)k);
    double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (valid) {
        for (uint32_t s0 = sl; s0 < pl.S; s0 += U * L) {
            double v[6][U];
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (uint32_t u = 0; u < U; ++u) {
                    const uint32_t sc = s0 + u * L;
                    v[q][u] = sc < pl.S ? pk[q * qs + (size_t)sc * cs] : 0.0;
                }
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (uint32_t u = 0; u < U; ++u)
                    if (s0 + u * L < pl.S) acc[q] += v[q][u];
        }
    }
    for (int q = 0; q < 6; ++q) f[q] = lanes_sum(acc[q], L);
}

// Finish pass of an update: adds the j-chunk partials of each active
// particle (chunk_sums) and stores the forces.  A particle's chunk sums are
// spread over L = pl.lanes lanes, so a workgroup finishes BS/L particles with
// no barrier.
__global__ __launch_bounds__(BS) void k_finish(Soa s, Ens e, const uint32_t *move,
                                              const double *partial) {
    const unsigned long long total = e.ctl->fin_units;
    for (unsigned long long u = blockIdx.x; u < total; u += gridDim.x) {
        const uint32_t c = find_cluster(e.fin_pre, e.K, u);
        const ClPlan pl = e.plan[c];
        if (pl.S == 1) continue;  // the update stored them
        const uint32_t L = pl.lanes;
        const uint32_t lu = (uint32_t)(u - e.fin_pre[c]);
        const uint32_t k = lu * (BS / L) + threadIdx.x / L;
        const bool valid = k < e.cs[c].nact;
        const uint32_t i = valid ? move[e.off[c] + k] : 0u;
        double f[6];
        chunk_sums(s, pl, partial + e.part_pre[c], k, i, valid, f);
        if (valid && threadIdx.x % L == 0)
            for (int q = 0; q < 6; ++q) s.f[q][i] = f[q];
    }
}

// The same, with the corrector at the cluster's block time: the finish of a
// block step of an ensemble of many blocks (finish_by_blocks), after a selection
// that wrote the active particles' records, whose loads go out with those of
// the partials.
__global__ __launch_bounds__(BS) void k_finish_correct(Soa s, Ens e, const uint32_t *move,
                                                      const double *partial, float eta,
                                                      double dt_min, double dt_max) {
    const unsigned long long total = e.ctl->fin_units;
    for (unsigned long long u = blockIdx.x; u < total; u += gridDim.x) {
        const uint32_t c = find_cluster(e.fin_pre, e.K, u);
        const ClPlan pl = e.plan[c];
        const uint32_t L = pl.lanes;
        const uint32_t lu = (uint32_t)(u - e.fin_pre[c]);
        const double T = e.cs[c].atime;
        const uint32_t k = lu * (BS / L) + threadIdx.x / L;
        const bool valid = k < e.cs[c].nact;
        const uint32_t i = valid ? move[e.off[c] + k] : 0u;
        double o[6], pr[6], dt1 = 0.0;
        if (valid) load_arec(e, (size_t)e.off[c] + k, o, pr, dt1);
        double f[6];
        chunk_sums(s, pl, partial + e.part_pre[c], k, i, valid, f);
        if (valid && threadIdx.x % L == 0) {
            correct_store(s, i, o, pr, dt1, f, T, eta, dt_min, dt_max);
            if (pl.S > 1)
                for (int q = 0; q < 6; ++q) s.f[q][i] = f[q];
        }
    }
}

// ---------------------------------------------------------------------------
// Block times
// ---------------------------------------------------------------------------

__device__ __forceinline__ double block_min(double v, double *red) {
    v = wave_min(v);
    uint32_t w = threadIdx.x >> 6;
    if (__lane_id() == 0) red[w] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t k = 1; k < BS / 64; ++k) v = fmin(v, red[k]);
    }
    return v;  // valid in thread 0
}

// Minimum of v over the block and the number of threads that have it (within
// find_particles_to_move's tolerance; BCNT_MANY if a value within the
// tolerance of the minimum is not equal to it, which the one-workgroup-per-
// tile steps leave to the others).  Valid in thread 0.
constexpr uint32_t BCNT_MANY = 0xffffffu;
__device__ __forceinline__ double block_min_count(double v, double *red, uint32_t *cnt,
                                                  uint32_t &n) {
    const uint32_t w = threadIdx.x >> 6;
    double m = wave_min(v);
    const uint32_t at = (uint32_t)__popcll(__ballot(v == m));
    const bool close = __ballot(v != m && fabs(m - v) < 2 * DBL_EPSILON) != 0;
    if (__lane_id() == 0) {
        red[w] = m;
        cnt[w] = close ? BCNT_MANY : at;
    }
    __syncthreads();
    n = 0;
    if (threadIdx.x == 0) {
        for (uint32_t k = 1; k < BS / 64; ++k) m = vmin(m, red[k]);
        for (uint32_t k = 0; k < BS / 64; ++k)
            n += red[k] == m ? cnt[k] : fabs(m - red[k]) < 2 * DBL_EPSILON ? BCNT_MANY : 0u;
    }
    return m;
}

// min(t + dt) of one JT block (padding has dt = +inf).
__device__ __forceinline__ double block_tmin(const Soa &s, uint32_t b, double *red) {
    uint32_t i = b * JT + threadIdx.x;
    double v = s.t[i] + s.dt[i];
    double m = block_min(v, red);
    return m;  // valid in thread 0
}

// Finish pass of a block step, one block with active particles per workgroup
// (the dirty list k_select made for the step's parity: block, first place in
// the cluster's active list, count): the chunk sums and the corrector with
// NbodyUtils::get_timestep_normal and normalize_dt (Hermite4CPU.cpp:370-411,
// NbodyUtils.cpp:337-424) of the block's active particles, then the block's
// min(t + dt), from which the loop tail takes the next block time
// (Hermite4::next_integration_time, Hermite4.cpp:90-102).  The sums are
// chunk_sums', so the forces are k_finish's bit for bit.  The step of every
// live cluster is recorded for its loop tail (ClState tail_*), which the next
// launch that needs the next block time makes, and the active count of the
// next step starts from zero.
//
// A small step's pass is one chain: list, partials, sums, corrector, minimum.
// With at most 32 active particles in the block the corrector runs on 8 lanes
// each (corr8); with that and DPP sums the average launch of an N = 10007 run
// takes 6.9 us instead of 8.5, of an N = 65536 run 6.2 instead of 8.2.  For an
// ensemble it replaces a pass over the active particles with one-lane
// correctors and one over the blocks (k_finish_correct, k_blockmin_dirty; 64
// clusters of 4096: 12.1 us instead of 8.7 + 4.3), unless it has many blocks
// (finish_by_blocks).
template <bool SINGLE>
__global__ __launch_bounds__(BS) void k_finish_blocks(Soa s, Ens e, const uint32_t *move,
                                                     const double *partial, float eta,
                                                     double dt_min, double dt_max, uint32_t par) {
    __shared__ double red[BS / 64];
    __shared__ double tnew[JT];  // t + dt of the block's corrected particles (NaN: not active)
    constexpr uint32_t C8 = BS / 8;  // particles of one corr8 pass
    __shared__ double fs[6 * C8];    // their forces
    __shared__ uint32_t cnts[BS / 64];
    const uint32_t *dl = e.dirty + (size_t)par * 3 * e.nblk;
    // What the first block needs is requested at once: the list's count and
    // this workgroup's list entry (read before the count is known: the list
    // has nblk entries and the grid is at most nblk; an entry beyond the count
    // is not used), and for a single system the loop's stop flag, the plan and
    // the block time.
    const uint32_t nd = e.ctl->ndirty[par];
    uint32_t w = blockIdx.x;
    uint32_t b = dl[3 * w], k0 = dl[3 * w + 1], cnt = dl[3 * w + 2];
    ClPlan pl{};
    double T = 0.0;
    if constexpr (SINGLE) {
        const uint32_t done = e.cs[0].done;
        pl = e.plan[0];
        T = e.cs[0].atime;
        if (done) return;  // the loop stopped at this step's selection
    }
    // the other list's count, for the next step's selection
    if (blockIdx.x == 0 && threadIdx.x == 0) e.ctl->ndirty[par ^ 1] = 0;
    // the step's loop tail, for the next step's selection (k_select PS_TAIL),
    // k_small_run or k_tail to make
    for (uint32_t c = blockIdx.x * BS + threadIdx.x; c < e.K; c += gridDim.x * BS) {
        ClState *cs = &e.cs[c];
        if (!SINGLE && cs->done) continue;
        cs->tail_t = SINGLE ? T : cs->atime;
        cs->tail_nact = cs->nact;
        cs->tail_steps = cs->steps;
        cs->tail_pend = 1;
        cs->nact = 0;
    }
    for (; w < nd; w += gridDim.x) {
        if (w != blockIdx.x) {
            b = dl[3 * w];
            k0 = dl[3 * w + 1];
            cnt = dl[3 * w + 2];
        }
        const double *part = partial;
        uint32_t off = 0;  // of the cluster's active list
        if constexpr (!SINGLE) {
            const uint32_t c = cluster_of_block(e, b);
            pl = e.plan[c];
            T = e.cs[c].atime;
            part = partial + e.part_pre[c];
            off = e.off[c];
        }
        const uint32_t L = pl.lanes, per = BS / L;
        // t + dt of the block as it stands, loaded ahead of the corrector
        const uint32_t j = b * JT + threadIdx.x;
        const double tdt = s.t[j] + s.dt[j];
        if (cnt <= C8) {
            // The corrector of the kk-th active particle on lanes 8 kk ... + 7
            // (beyond one pass of that, one lane each: 3 times fewer
            // instructions).  Its inputs from the selection's records: their
            // loads go out ahead of the partials'.
            const uint32_t kk = threadIdx.x / 8, lane = threadIdx.x & 7u;
            const bool mine = kk < cnt, vel = lane >= 4;
            const uint32_t c = min(lane & 3u, 2u), q = c + (vel ? 3u : 0u);
            const uint32_t ka = off + k0 + (mine ? kk : 0u);
            const double *ar = reinterpret_cast<const double *>(e.arec);
            const size_t np = (size_t)e.nblk * JT;
            const double pr = ar[4 * ((vel ? np : 0) + ka) + c];
            const double o0 = ar[4 * (2 * np + ka) + c], o1 = ar[4 * (3 * np + ka) + c];
            const double dt1 = ar[4 * (2 * np + ka) + 3];
            const uint32_t i = move[ka];
            __syncthreads();  // red, tnew and fs of the previous block have been read
            tnew[threadIdx.x] = NAN;
            for (uint32_t base = 0; base < cnt; base += per) {
                const uint32_t ks = base + threadIdx.x / L;
                const bool valid = ks < cnt;
                const uint32_t k = k0 + (valid ? ks : 0u);
                double f[6];
                chunk_sums(s, pl, part, k, pl.S == 1 ? move[off + k] : 0u, valid, f);
                if (valid && threadIdx.x % L == 0)
                    for (int y = 0; y < 6; ++y) fs[6 * ks + y] = f[y];
            }
            __syncthreads();
            if (threadIdx.x / 64 * 8 < cnt) {  // (whole waves)
                const Corr8 ck = corr8_coef(dt1, T, vel);
                const double f0 = fs[6 * (mine ? kk : 0u) + c], f1 = fs[6 * (mine ? kk : 0u) + 3 + c];
                double x, ad;
                const double dtn =
                    corr8(ck, vel, o0, o1, f0, f1, pr, eta, dt_min, dt_max, x, ad);
                if (mine && (lane & 3u) < 3u) {
                    double *col = s.r[0] + i;
                    col[(q + (vel ? COL_R + 1 : COL_R)) * np] = x;  // (m between r and v)
                    if (pl.S > 1) col[(q + COL_F) * np] = vel ? f1 : f0;
                    col[(q + COL_A2) * np] = ad;
                    if (lane == 0) {
                        col[COL_T * np] = T;
                        col[COL_DT * np] = dtn;
                        tnew[i - b * JT] = T + dtn;
                    }
                }
            }
        } else {
            __syncthreads();  // red, tnew and fs of the previous block have been read
            tnew[threadIdx.x] = NAN;
            __syncthreads();
            for (uint32_t base = 0; base < cnt; base += per) {
                const uint32_t kk = base + threadIdx.x / L;
                const bool valid = kk < cnt;
                const uint32_t k = k0 + (valid ? kk : 0u);
                const uint32_t i = move[off + k];
                // the corrector's inputs from the selection's records: their
                // loads go out with those of the partials
                double o[6], pr[6], dt1 = 0.0;
                if (valid) load_arec(e, off + k, o, pr, dt1);
                double f[6];
                chunk_sums(s, pl, part, k, i, valid, f);
                if (valid && threadIdx.x % L == 0) {
                    const double dtn = correct_store(s, i, o, pr, dt1, f, T, eta, dt_min, dt_max);
                    if (pl.S > 1)
                        for (int q = 0; q < 6; ++q) s.f[q][i] = f[q];
                    tnew[i - b * JT] = T + dtn;
                }
            }
        }
        __syncthreads();
        const double tn = tnew[threadIdx.x];
        uint32_t nm;
        const double m = block_min_count(isnan(tn) ? tdt : tn, red, cnts, nm);
        if (threadIdx.x == 0) {
            e.bmin[b] = m;
            e.bcnt[b] = nm;
        }
    }
}

// After k_finish_correct: the minima of the blocks of dirty list `par` (the
// others did not change), and what k_finish_blocks leaves for the next step.
__global__ __launch_bounds__(BS) void k_blockmin_dirty(Soa s, Ens e, uint32_t par) {
    __shared__ double red[BS / 64];
    if (blockIdx.x == 0 && threadIdx.x == 0) e.ctl->ndirty[par ^ 1] = 0;
    for (uint32_t c = blockIdx.x * BS + threadIdx.x; c < e.K; c += gridDim.x * BS) {
        ClState *cs = &e.cs[c];
        if (cs->done) continue;
        cs->tail_t = cs->atime;
        cs->tail_nact = cs->nact;
        cs->tail_steps = cs->steps;
        cs->tail_pend = 1;
        cs->nact = 0;
    }
    const uint32_t *dl = e.dirty + (size_t)par * 3 * e.nblk;
    uint32_t b = dl[3 * blockIdx.x];  // (read with the count, as k_finish_blocks does)
    const uint32_t nd = e.ctl->ndirty[par];
    for (uint32_t w = blockIdx.x; w < nd; w += gridDim.x) {
        if (w != blockIdx.x) b = dl[3 * w];
        __syncthreads();  // red of the previous block has been read
        const double m = block_tmin(s, b, red);
        if (threadIdx.x == 0) e.bmin[b] = m;
    }
}

__global__ __launch_bounds__(BS) void k_blockmin_all(Soa s, Ens e) {
    __shared__ double red[BS / 64];
    __shared__ uint32_t cnts[BS / 64];
    for (uint32_t b = blockIdx.x; b < e.nblk; b += gridDim.x) {
        __syncthreads();
        const uint32_t i = b * JT + threadIdx.x;
        uint32_t nm;
        const double m = block_min_count(s.t[i] + s.dt[i], red, cnts, nm);
        if (threadIdx.x == 0) {
            e.bmin[b] = m;
            e.bcnt[b] = nm;
        }
    }
}

// Hermite4::next_integration_time (Hermite4.cpp:90-102) per cluster:
// min(t_i + dt_i) into the cluster's tmin_key (one workgroup per block).
__global__ __launch_bounds__(BS) void k_next_time(Soa s, Ens e) {
    __shared__ double red[BS / 64];
    for (uint32_t b = blockIdx.x; b < e.nblk; b += gridDim.x) {
        __syncthreads();
        double m = block_tmin(s, b, red);
        if (threadIdx.x == 0) atomicMin(&e.cs[cluster_of_block(e, b)].tmin_key, dkey(m));
    }
}

// Hermite4::init_dt (Hermite4.cpp:108-140) per particle, plus the cluster
// minimum of dt in tmin_key.  Non-positive, infinite or NaN ETA|a|/|j|
// map to dt_min (the reference's x86 outcome of its undefined int cast).
__global__ __launch_bounds__(BS) void k_init_dt(Soa s, Ens e, float eta, double itime,
                                               double dt_min, double dt_max) {
#pragma clang fp contract(off)
    __shared__ double red[BS / 64];
    for (uint32_t b = blockIdx.x; b < e.nblk; b += gridDim.x) {
        const uint32_t c = cluster_of_block(e, b);
        const uint32_t i = b * JT + threadIdx.x;
        double mn = INFINITY;
        if (i - e.off[c] < e.cnt[c]) {
            double a2 = magnitude(s.f[0][i], s.f[1][i], s.f[2][i]);
            double j2 = magnitude(s.f[3][i], s.f[4][i], s.f[5][i]);
            double tmp_dt = eta * (a2 / j2);
            double d;
            if (!(tmp_dt > 0.0) || isinf(tmp_dt)) {
                d = dt_min;
            } else {
                int ex = (int)(ceil(log(tmp_dt) / log(2.0)) - 1);
                d = ldexp(1.0, ex);
                if (d < dt_min)
                    d = dt_min;
                else if (d > dt_max)
                    d = dt_max;
            }
            s.dt[i] = d;
            s.t[i] = itime;
            mn = d;
        }
        __syncthreads();
        mn = block_min(mn, red);
        if (threadIdx.x == 0) atomicMin(&e.cs[c].tmin_key, dkey(mn));
    }
}

// ---------------------------------------------------------------------------
// Step-loop control
// ---------------------------------------------------------------------------

// Arms the device step loop of every cluster.  set0: cluster 0 takes
// (itime0, atime0) first.  A cluster whose ITIME is not < t_end is done
// at once (the reference's loop test, Hermite4CPU_integration.cpp:81).
// team_rest: k_team_run leaves that many steps alone first, team_fails teams in
// a row not having formed.
__global__ __launch_bounds__(BS) void k_run_setup(Ens e, double t_end, double t_stop,
                                                 unsigned long long max_steps, uint32_t set0,
                                                 double itime0, double atime0,
                                                 unsigned long long team_rest,
                                                 uint32_t team_fails) {
    __shared__ uint32_t cnt[BS / 64];
    uint32_t nd = 0;
    for (uint32_t c = threadIdx.x; c < e.K; c += BS) {
        ClState &cs = e.cs[c];
        if (set0 && c == 0) {
            cs.itime = itime0;
            cs.atime = atime0;
        }
        cs.steps = 0;
        cs.interactions = 0;
        cs.nsteps = 0;
        cs.small_steps = 0;
        cs.nact = 0;
        cs.tail_pend = 0;
        cs.done = (cs.itime < t_end) ? 0u : 1u;
        nd += cs.done;
    }
    for (int o = 32; o > 0; o >>= 1) nd += __shfl_xor(nd, o);
    if (__lane_id() == 0) cnt[threadIdx.x >> 6] = nd;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (uint32_t k = 0; k < BS / 64; ++k) t += cnt[k];
        RunCtl &ctl = *e.ctl;
        ctl.t_end = t_end;
        ctl.t_stop = t_stop;
        ctl.max_steps = max_steps;
        ctl.ndirty[0] = ctl.ndirty[1] = 0;
        ctl.ndone = t;
        ctl.team_retry = team_rest;
        ctl.team_fails = team_fails;
        ctl.team_steps = 0;
        ctl.team_err = 0;
        ctl.items = 0;
        ctl.fin_units = 0;
    }
}

// Stores and loads of this wave so far are done.
__device__ __forceinline__ void wait_memory() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// What a step made without a device loop leaves in the cluster's record, as the
// loop of one step does: later calls start from it (h4h_ensemble_run, its
// ITIME and ATIME; h4h_correction_pos_vel, the size of the active list).
// Stored after the result, for which the host waits (before it: 0.4 us more a
// step): the launches that read it come after this one.
__device__ __forceinline__ void step_state(ClState *cs, double itime, double atime, uint32_t nact,
                                           uint32_t n, unsigned long long small) {
    cs->itime = itime;
    cs->atime = atime;
    cs->nact = 0;
    cs->tail_pend = 0;
    cs->steps = 1;
    cs->interactions = (unsigned long long)nact * n;
    cs->nsteps = nact;
    cs->small_steps = small;
    cs->done = 1;
}

// The result of one h4h_step, to the pinned record the host waits at: its
// fields, and when they are there `done`.  (Waiting for the launch itself
// takes 5 us more, of a step of 18 to 28.)  next: the next block step's
// active count (tail_nact there; BCNT_MANY or more: not known).
enum : uint32_t { STEP_DONE = 1, STEP_LEFT = 2, STEP_FAILED = 3, STEP_ALONE = 4 };
template <class T>
__device__ __forceinline__ void host_store(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void step_result(ClState *host, double atime, uint32_t nact, uint32_t n,
                                            unsigned long long small, uint32_t next) {
    host_store(&host->atime, atime);
    host_store(&host->nsteps, (unsigned long long)nact);
    host_store(&host->interactions, (unsigned long long)nact * n);
    host_store(&host->small_steps, small);
    host_store(&host->tail_nact, next);
    wait_memory();
    host_store(&host->done, (uint32_t)STEP_DONE);
}

// The loop tail a single system's last block step left (k_finish_blocks),
// when no further step of the loop makes it: after one h4h_step, whose
// result goes to the pinned record `host`, or at the end of a loop's step
// budget (null; the loop may have stopped before).
__global__ __launch_bounds__(BS) void k_tail(Ens e, ClState *host) {
    __shared__ double red[BS / 64];
    __shared__ uint32_t next;
    ClState *cs = &e.cs[0];
    if (!host && cs->done) return;
    double mn = INFINITY;
    for (uint32_t b = threadIdx.x; b < e.nblk; b += BS) mn = fmin(mn, e.bmin[b]);
    mn = block_min(mn, red);
    if (threadIdx.x == 0) {
        red[0] = mn;
        next = 0;
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < e.nblk; b += BS)
        if (e.bmin[b] == red[0]) atomicAdd(&next, min(e.bcnt[b], BCNT_MANY));
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long steps = cs->tail_steps + 1;
        record_tail(e, 0, cs->tail_t, cs->tail_nact, steps, mn,
                    loop_stops(*e.ctl, cs->tail_t, steps, mn));
        cs->tail_pend = 0;
        if (host) step_result(host, mn, cs->tail_nact, e.cnt[0], 0, next);
    }
}

// ---------------------------------------------------------------------------
// Small systems: whole block steps in one workgroup
// ---------------------------------------------------------------------------

constexpr uint32_t SN = 1024;            // largest N k_small_run takes
constexpr uint32_t SB = 512;             // its threads
constexpr uint32_t SP = SN / SB;         // particles per thread
constexpr uint32_t SW = SB / 64;         // waves
constexpr uint32_t SC = SN / 64;         // chunks of 64 particles
constexpr uint32_t SMALL_MAX_ACT = 256;  // largest active set k_small_run takes
static_assert(SB % JT == 0 && SC == 16, "a row of 16 lanes holds the chunks");

// p (a global-memory pointer), as a value the compiler cannot hoist out of
// a loop: stores through it inside the loop address SGPR base + VGPR offset
// instead of holding one 64-bit VGPR address per array for the whole loop.
// Typed as a global pointer so that they are global (not flat) stores: a
// flat store also counts against the LDS wait of the next barrier.
template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T *in_loop(T *p) {
    asm volatile("" : "+s"(p));
    return (__attribute__((address_space(1))) T *)p;
}

// Sum of c over the 16 lanes of the row.
__device__ __forceinline__ uint32_t row_sum(uint32_t c) {
    auto add = [&](int o) { c += (uint32_t)o; };
    add(__builtin_amdgcn_update_dpp(0, (int)c, DPP_XOR1, 0xf, 0xf, false));
    add(__builtin_amdgcn_update_dpp(0, (int)c, DPP_XOR2, 0xf, 0xf, false));
    add(__builtin_amdgcn_update_dpp(0, (int)c, DPP_QUADS, 0xf, 0xf, false));
    add(__builtin_amdgcn_update_dpp(0, (int)c, DPP_EIGHTS, 0xf, 0xf, false));
    return c;
}

// Exclusive prefix sum of c over the wave, and the total.
__device__ __forceinline__ uint32_t wave_scan(uint32_t c, uint32_t &total) {
    uint32_t x = c;  // inclusive, in the row of 16 first (row_shr 1, 2, 4, 8)
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, true);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, true);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, true);
    const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)x, 15);
    const uint32_t r1 = r0 + (uint32_t)__builtin_amdgcn_readlane((int)x, 31);
    const uint32_t r2 = r1 + (uint32_t)__builtin_amdgcn_readlane((int)x, 47);
    total = r2 + (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
    const uint32_t row = __lane_id() >> 4;
    return x - c + (row == 0 ? 0u : row == 1 ? r0 : row == 2 ? r1 : r2);
}

// Number of particles of the workgroup with their flag set (particle
// tid + k SB: flag[k] of thread tid), and (for those) the count below them
// in particle order.  Ends after a barrier.
__device__ __forceinline__ uint32_t small_count(const bool flag[SP], uint32_t *wcnt,
                                                uint32_t below[SP]) {
    const uint32_t lane = __lane_id(), w = threadIdx.x >> 6;
    unsigned long long mask[SP];
    for (uint32_t k = 0; k < SP; ++k) {
        mask[k] = __ballot(flag[k]);
        if (lane == 0) wcnt[k * SW + w] = (uint32_t)__popcll(mask[k]);
    }
    __syncthreads();
    const uint32_t c = wcnt[lane % SC];
    for (uint32_t k = 0; k < SP; ++k)
        below[k] = row_sum(lane % SC < k * SW + w ? c : 0u) +
                   (uint32_t)__popcll(mask[k] & ((1ull << lane) - 1ull));
    return row_sum(c);
}

// Minimum over the workgroup (every thread gets it).  Ends after a barrier;
// wmin is free again after the next one.
__device__ __forceinline__ double small_min(const double x[SP], double *wmin) {
    double v = x[0];
    for (uint32_t k = 1; k < SP; ++k) v = vmin(v, x[k]);
    v = wave_min(v);
    if (__lane_id() == 0) wmin[threadIdx.x >> 6] = v;
    __syncthreads();
    return wave_min(wmin[__lane_id() % SW]);
}

// Pairs of particle i (record pi) with j = g, g + G, ... < n, added to fo;
// MIXED: FP32 sums of 32 pairs at a time.
template <bool MIXED>
__device__ __forceinline__ void small_pairs(const double pi[6], uint32_t i, uint32_t g, uint32_t G,
                                            uint32_t n, const double4 *lpp, const double4 *lpv,
                                            double e2, uint32_t self_zero, double fo[6]) {
    if constexpr (!MIXED) {
        if (self_zero) {
            // two j at a time (a missing second one without mass): most lanes
            // have 2 to 16, and one at a time their latency is the phase
#pragma unroll 2
            for (uint32_t j = g; j < n; j += 2 * G) {
                const uint32_t k = min(j + G, n - 1);
                const double4 a = lpp[j], b = lpv[j], a2 = lpp[k], b2 = lpv[k];
                pair_fp64(pi, a.x, a.y, a.z, b.x, b.y, b.z, a.w, e2, fo);
                pair_fp64(pi, a2.x, a2.y, a2.z, b2.x, b2.y, b2.z, j + G < n ? a2.w : 0.0, e2, fo);
            }
        } else {
            for (uint32_t j = g; j < n; j += G) {
                const double4 a = lpp[j], b = lpv[j];
                const bool me = j == i;
                pair_fp64(pi, me ? pi[0] + 1.0 : a.x, a.y, a.z, b.x, b.y, b.z, me ? 0.0 : a.w, e2,
                          fo);
            }
        }
    } else {
        const float e2f = (float)e2;
        for (uint32_t j0 = g; j0 < n; j0 += 32 * G) {
            const uint32_t j1 = min(n, j0 + 32 * G);
            float t6[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (self_zero) {
#pragma unroll 4
                for (uint32_t j = j0; j < j1; j += G) {
                    const double4 a = lpp[j], b = lpv[j];
                    pair_mixed(pi, a.x, a.y, a.z, b.x, b.y, b.z, (float)a.w, e2f, t6);
                }
            } else {
                for (uint32_t j = j0; j < j1; j += G) {
                    const double4 a = lpp[j], b = lpv[j];
                    const bool me = j == i;
                    pair_mixed(pi, me ? pi[0] + 1.0 : a.x, a.y, a.z, b.x, b.y, b.z,
                               me ? 0.f : (float)a.w, e2f, t6);
                }
            }
            for (int k = 0; k < 6; ++k) fo[k] += (double)t6[k];
        }
    }
}

// One block step at `itime` without a device loop (h4h_step): the kernels
// that make whole steps take the loop's state from here instead of the loop
// control and the cluster record, and write the step's result to the pinned
// record `host` (STEP_LEFT if they leave the step to others, STEP_ALONE if the
// workgroups of a team did not come together), so that such a
// step is one launch and no copy.
struct OneStep {
    double itime;
    ClState *host;  // null: a device loop
};

// Block steps of systems of n <= SN particles, workgroup c of SB threads for
// cluster c (a larger cluster's workgroup returns at once), up to max_run
// steps per launch; clusters are independent, so the workgroups never wait
// for each other.  Thread t owns particles t and t + SB of its cluster and
// keeps their position, velocity, forces, time and step in registers for the
// whole launch; the threads exchange the predictor records and the active
// list through LDS, and the state goes to HBM as it changes (stores
// that nothing in the launch reads back).  Each step is the device loop's
// step: predictor of all particles at the block time T, the particles with
// t + dt = T (Hermite4::find_particles_to_move), their old forces, the pair
// sums, the corrector and new step, the next block time min(t + dt) and the
// loop tail (the record_tail of each step; the counters go out at the end).
// The active set of the next step is counted before its predictor; when it
// is empty or larger than max_act the launch ends and leaves that step to
// the multi-workgroup kernels.
//
// Pair sums: P = nact rounded up to a power of two i slots and G groups of
// lanes; a lane of group g takes one slot and j = g, g + G, ...  P < 64:
// G = SB / P, a wave's groups summed by halving (slot_sums: neighbouring
// groups first, so a lane's group is its slot-free bits reversed), the waves'
// sums in order through LDS.  P >= 64: G = 1024 / P in two passes, one j per
// wave (an LDS broadcast), summed in group order.  A fixed order for a given
// nact.  The mixed path folds its FP32 runs into FP64 every 32 pairs, as the
// main kernel does.  The corrector of slot k runs on 8 lanes (corr8), slots
// 0-7 on the first wave; waves without one take the minima of the particles
// that are not active.  The next block time is the minimum over those and
// the new steps; with at most 64 active particles every wave reads the new
// steps itself and makes the next active list without another barrier: three
// barriers per step.
//
// What bounds a step is the chain of these phases on one CU, at n = 1024 also
// its pairs.  Cycles per step, of the form before (1024 threads, shuffles, a
// one-lane corrector of 5900 cycles, counters read back from memory, 8
// barriers) and of this one: n = 256 14300 and 7600, n = 1024 21400 and
// 13900.  512 threads of two particles each have 256 registers: 1024 threads
// spilled 62 around the pair loop, 5000 cycles of a step at n = 1024.  On exit
// the per-block minima of t + dt are stored, and the step left to the
// multi-workgroup kernels is predicted and selected from the registers, which
// saves it k_select's launch (1.8 us here; 5.4 us and a launch gap there).
template <bool MIXED>
__global__ __launch_bounds__(SB) void k_small_run(Soa s, Ens e, uint32_t max_run,
                                                  uint32_t max_act, double e2, double eta,
                                                  double dt_min, double dt_max,
                                                  uint32_t self_zero, uint32_t par,
                                                  uint32_t *move, OneStep one) {
#pragma clang fp contract(off)
    __shared__ double4 lpp[SN], lpv[SN];          // predictor records
    __shared__ __align__(16) double red[6 * SN];  // pair sums per (group, slot)
    __shared__ double stg[7 * SMALL_MAX_ACT];     // old forces and step per active slot
    __shared__ double outs[13 * SMALL_MAX_ACT];   // new forces, position, velocity, step
    // t + dt (inf: active, or no particle), behind the sums of a step with
    // P < 64
    double *rest = red + 4 * SN;
    static_assert(6 * 32 * SW <= 4 * SN, "sums of 32 slots");
    __shared__ uint32_t lact[SN];                 // active list
    __shared__ double wmin[SC], cmin[SW];         // minimum of rest per chunk
    __shared__ unsigned long long wmask[SC];      // the particles that have it
    __shared__ uint32_t wcnt[SC];

    const uint32_t tid = threadIdx.x, lane = __lane_id(), w = tid >> 6;
    const uint32_t c = blockIdx.x;
    ClState *cs = &e.cs[c];
    const uint32_t n = e.cnt[c];
    if (n > SN) return;
    const uint32_t off = e.off[c];  // first particle of the cluster
    if (max_act > SMALL_MAX_ACT) max_act = SMALL_MAX_ACT;
    const bool loop = one.host == nullptr;
    if (loop && cs->done) return;
    const double t_end = loop ? e.ctl->t_end : (double)INFINITY;
    const double t_stop = loop ? e.ctl->t_stop : -(double)INFINITY;
    const unsigned long long max_steps = loop ? e.ctl->max_steps : 1ull;
    unsigned long long steps = loop ? cs->steps : 0ull;
    unsigned long long inter = loop ? cs->interactions : 0ull, nst = loop ? cs->nsteps : 0ull;
    uint32_t hk = (uint32_t)(steps % e.hist_cap);  // history slot of the next step
    double T = loop ? cs->atime : one.itime;
    // self_zero (set by the host, self_pair_is_zero): a particle's pair with
    // itself (r = 0, v = 0) has a finite weight m / e2^1.5 for every mass of
    // the context, so it adds exact zeros and the j loop needs no test for it.

    bool in[SP], act[SP];
    double r[SP][3], v[SP][3], f[SP][6], ti[SP], dti[SP], tdt[SP];
    float mf[SP];
#pragma unroll
    for (uint32_t k = 0; k < SP; ++k) {
        in[k] = tid + k * SB < n;
        for (int q = 0; q < 3; ++q) r[k][q] = v[k][q] = 0.0;
        for (int q = 0; q < 6; ++q) f[k][q] = 0.0;
        ti[k] = dti[k] = 0.0;
        mf[k] = 0.0f;
        if (in[k]) {
            const uint32_t gi = off + tid + k * SB;
            for (int q = 0; q < 3; ++q) {
                r[k][q] = s.r[q][gi];
                v[k][q] = s.v[q][gi];
            }
            for (int q = 0; q < 6; ++q) f[k][q] = s.f[q][gi];
            ti[k] = s.t[gi];
            dti[k] = s.dt[gi];
            mf[k] = (float)s.m[gi];
        }
        tdt[k] = in[k] ? ti[k] + dti[k] : (double)INFINITY;
    }
    if (tid < SC) {  // (chunks without a particle are never minimised)
        wmin[tid] = INFINITY;
        wmask[tid] = 0;
    }
    // The loop tail the cluster's last multi-workgroup step left comes
    // first; its next block time is the minimum of t + dt, which these
    // threads hold.
    if (loop && cs->tail_pend) {
        const double Tp = cs->tail_t;
        const uint32_t np = cs->tail_nact;
        steps = cs->tail_steps + 1;
        const double mn = small_min(tdt, cmin);
        const bool last = loop_stops(*e.ctl, Tp, steps, mn);
        if (tid == 0) {
            record_tail(e, c, Tp, np, steps, mn, last);
            cs->tail_pend = 0;
        }
        if (last) return;  // (the block minima are the finish pass's)
        inter += (unsigned long long)np * n;
        nst += np;
        hk = (uint32_t)(steps % e.hist_cap);
        T = mn;
    }
    uint32_t k_act[SP];  // the particles' places in the active list
    for (uint32_t k = 0; k < SP; ++k)
        act[k] = in[k] && fabs(T - tdt[k]) < 2 * DBL_EPSILON;
    uint32_t nact = small_count(act, wcnt, k_act);

    uint32_t it = 0;
    bool stop = false;
    double t_last = 0.0;
    const size_t np = (size_t)e.nblk * JT;  // the state's columns are np apart
    // Corrector lanes: slot k on lanes 8 (k % 8) ... + 7 of wave k / 8 (the
    // first waves, which the SIMDs issue first, prepare it before their pairs).
    const bool vel = (lane & 4u) != 0;
    const uint32_t cc = min(lane & 3u, 2u), cq = cc + (vel ? 3u : 0u);
    for (; !stop && it < max_run && nact >= 1 && nact <= max_act; ++it) {
        // Predictor of every particle at T; active list.
#pragma unroll
        for (uint32_t k = 0; k < SP; ++k) {
            const uint32_t i = tid + k * SB;
            if (in[k]) {
                double4 a, b;
                predict_vals(r[k], v[k], f[k], T - ti[k], mf[k], a, b);
                lpp[i] = a;
                lpv[i] = b;
            }
            if (act[k]) {
                lact[k_act[k]] = i;
                double *st = stg + 7 * k_act[k];
                for (int q = 0; q < 6; ++q) st[q] = f[k][q];
                st[6] = dti[k];
            }
            if (nact <= 32) rest[i] = act[k] ? (double)INFINITY : tdt[k];
        }
        __syncthreads();

        const uint32_t lp = nact > 1 ? 32u - (uint32_t)__clz(nact - 1) : 0u;
        const uint32_t P = 1u << lp;
        const bool corr = 8 * w < nact;  // this wave has corrector slots
        Corr8 ck{};
        double o0 = 0.0, o1 = 0.0, pr = 0.0;
        auto corr_prepare = [&](uint32_t k) {
            const double *st = stg + 7 * k;
            const uint32_t ia = lact[k];
            o0 = st[cc];
            o1 = st[3 + cc];
            ck = corr8_coef(st[6], T, vel);
            pr = reinterpret_cast<const double *>(vel ? lpv + ia : lpp + ia)[cc];
        };
        if (corr) corr_prepare(min(8 * w + lane / 8, nact - 1));

        // Pair sums.
        {
            const uint32_t slot = tid & (P - 1);
            const uint32_t i = lact[min(slot, nact - 1)];
            double pi[6];
            {
                const double4 a = lpp[i], b = lpv[i];
                pi[0] = a.x;
                pi[1] = a.y;
                pi[2] = a.z;
                pi[3] = b.x;
                pi[4] = b.y;
                pi[5] = b.z;
            }
            double fo[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            if (P < 64) {
                const uint32_t g = w * (64 >> lp) + (__brev(lane >> lp) >> (26 + lp));
                small_pairs<MIXED>(pi, i, g, SB >> lp, n, lpp, lpv, e2, self_zero, fo);
                slot_sums(fo, P, red + (w * P + slot) * 6);
            } else {
                const uint32_t G = SN >> lp;
                for (uint32_t g = tid >> lp; g < G; g += SB >> lp) {
                    for (int k = 0; k < 6; ++k) fo[k] = 0.0;
                    small_pairs<MIXED>(pi, i, g, G, n, lpp, lpv, e2, self_zero, fo);
                    double2 *row = reinterpret_cast<double2 *>(red + (g * P + slot) * 6);
                    row[0] = make_double2(fo[0], fo[1]);
                    row[1] = make_double2(fo[2], fo[3]);
                    row[2] = make_double2(fo[4], fo[5]);
                }
            }
        }
        __syncthreads();

        auto rest_min = [&](uint32_t q, double x) {
            const double m = wave_min(x);
            const unsigned long long mask = __ballot(fabs(m - x) < 2 * DBL_EPSILON);
            if (lane == 0) {
                wmin[q] = m;
                wmask[q] = mask;
            }
        };
        const uint32_t chunks = (n + 63) / 64;
        const uint32_t corr_waves = (nact + 7) / 8;  // (P < 64: at most 4 of SW)
        if (corr) {
            for (uint32_t k0 = 8 * w; k0 < nact; k0 += 8 * SW) {
                const uint32_t k = min(k0 + lane / 8, nact - 1);
                if (k0 != 8 * w) corr_prepare(k);
                // groups in order: 8 (P < 64), else 1024 / P = 16, 8 or 4
                double fq = 0.0;
                const double *rk = red + k * 6 + cq;
                if (P < 64) {
                    double x8[SW];  // (all loads under way before the first sum)
#pragma unroll
                    for (uint32_t q = 0; q < SW; ++q) x8[q] = rk[q * P * 6];
#pragma unroll
                    for (uint32_t q = 0; q < SW; ++q) fq += x8[q];
                } else {
                    const uint32_t ngrp = SN >> lp;
                    for (uint32_t q0 = 0; q0 < ngrp; q0 += 4) {
#pragma unroll
                        for (uint32_t q = 0; q < 4; ++q) fq += rk[(q0 + q) * P * 6];
                    }
                }
                if (!MIXED) fq *= PAIR_SCALE;
                const double fx = xor4(fq);
                double x, ad;
                const double dtn = corr8(ck, vel, o0, o1, vel ? fx : fq, vel ? fq : fx, pr, eta,
                                         dt_min, dt_max, x, ad);
                if (k0 + lane / 8 < nact && (lane & 3u) < 3u) {
                    double *out = outs + 13 * k;
                    out[cq] = fq;
                    out[6 + cq] = x;
                    const uint32_t gi = off + lact[k];
                    auto *col = in_loop(s.r[0]) + gi;  // one base: one SGPR pair
                    col[(cq + (vel ? COL_R + 1 : COL_R)) * np] = x;  // (m between r and v)
                    col[(cq + COL_F) * np] = fq;
                    col[(cq + COL_OLD) * np] = vel ? o1 : o0;
                    col[(cq + COL_A2) * np] = ad;
                    if ((lane & 7u) == 0) {
                        out[12] = dtn;
                        col[COL_T * np] = T;
                        col[COL_DT * np] = dtn;
                    }
                }
            }
        } else if (P < 64) {
            for (uint32_t q = w - corr_waves; q < chunks; q += SW - corr_waves)
                rest_min(q, rest[64 * q + lane]);
        }
        if (P >= 64)
#pragma unroll
            for (uint32_t k = 0; k < SP; ++k)
                rest_min(k * SW + w, act[k] ? (double)INFINITY : tdt[k]);
        __syncthreads();

        // (what the next time needs is read before the owners' state, so that
        // the reads' latencies overlap)
        const double wv = wmin[lane % SC];
        const uint32_t wc = (uint32_t)__popcll(wmask[lane % SC]);
        const double x = lane < nact && nact <= 64 ? T + outs[13 * min(lane, nact - 1) + 12]
                                                   : (double)INFINITY;
        // The owners take their corrected state.
#pragma unroll
        for (uint32_t k = 0; k < SP; ++k)
            if (act[k]) {
                const double *o = outs + 13 * k_act[k];
                for (int q = 0; q < 6; ++q) f[k][q] = o[q];
                for (int q = 0; q < 3; ++q) {
                    r[k][q] = o[6 + q];
                    v[k][q] = o[9 + q];
                }
                ti[k] = T;
                dti[k] = o[12];
                tdt[k] = T + o[12];
            }

        // Next block time (Hermite4::next_integration_time): the minimum over
        // the not-active minima and the active slots' new times, and the
        // particles that have it.  A time that is not the minimum but within
        // find_particles_to_move's tolerance of it (steps below 2^-50) sends
        // every wave to the counting below.
        double mn;
        bool close;
        uint32_t cnt = 0;
        if (nact <= 64) {
            mn = wave_min(vmin(x, wv));
            close = __ballot((wv != mn && fabs(mn - wv) < 2 * DBL_EPSILON) ||
                             (x != mn && fabs(mn - x) < 2 * DBL_EPSILON)) != 0;
            const unsigned long long cm = __ballot(x == mn && lane < nact);
            const unsigned long long at = __ballot(wv == mn);  // bit q: chunk q has the minimum
            const uint32_t mine = wv == mn ? wc : 0u;
            const uint32_t base = (uint32_t)__popcll(cm);
            cnt = base + row_sum(mine);
#pragma unroll
            for (uint32_t k = 0; k < SP; ++k) {
                const uint32_t q = k * SW + w;
                const unsigned long long mask = wmask[q];
                const uint32_t below = row_sum(lane % SC < q ? mine : 0u);
                if (act[k]) {
                    act[k] = (cm >> k_act[k]) & 1ull;
                    k_act[k] = (uint32_t)__popcll(cm & ((1ull << k_act[k]) - 1ull));
                } else {
                    act[k] = ((at >> q) & 1ull) && ((mask >> lane) & 1ull);
                    k_act[k] = base + below + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
                }
            }
        } else {
            mn = small_min(tdt, cmin);
            close = true;
        }

        // Loop tail.
        steps += 1;
        stop = T >= t_stop || steps >= max_steps || !(T < t_end) || !(mn > T);
        inter += (unsigned long long)nact * n;
        nst += nact;
        if (c == 0 && tid == 0) {
            e.hist_t[hk] = T;
            e.hist_n[hk] = nact;
        }
        t_last = T;
        T = mn;
        if (++hk == e.hist_cap) hk = 0;
        if (close) {  // (uniform over the workgroup)
            for (uint32_t k = 0; k < SP; ++k)
                act[k] = in[k] && fabs(T - tdt[k]) < 2 * DBL_EPSILON;
            cnt = small_count(act, wcnt, k_act);
        }
        nact = cnt;
    }

    // Loop state and predictor records of the last step made; per-block
    // minima of t + dt.
    if (it > 0) {
        if (tid == 0 && loop) {
            cs->itime = t_last;
            cs->atime = T;
            cs->steps = steps;
            cs->interactions = inter;
            cs->nsteps = nst;
            cs->small_steps += it;
            if (stop) {
                cs->done = 1;
                atomicAdd(&e.ctl->ndone, 1u);
            }
        }
        if (stop || !loop)
            for (uint32_t k = 0; k < SP; ++k)
                if (in[k]) {
                    s.pp[off + tid + k * SB] = lpp[tid + k * SB];
                    s.pv[off + tid + k * SB] = lpv[tid + k * SB];
                }
    }
    // The step left is selected here, from the registers: what k_select does
    // with PS_COMPACT, in particle order, so that each block's active
    // particles are neighbours in the list.
    if (loop && !stop) {
        __syncthreads();  // wcnt may be being read
        nact = small_count(act, wcnt, k_act);
        for (uint32_t k = 0; k < SP; ++k) {
            const uint32_t gi = off + tid + k * SB, slot = off + k_act[k];
            double4 a, b;
            if (in[k]) {
                predict_vals(r[k], v[k], f[k], T - ti[k], mf[k], a, b);
                s.pp[gi] = a;
                s.pv[gi] = b;
            }
            if (act[k]) {
                move[slot] = gi;
                auto *col = in_loop(s.r[0]) + gi;
                for (int q = 0; q < 6; ++q) col[(COL_OLD + q) * np] = f[k][q];
                e.arec[slot] = a;
                e.arec[np + slot] = b;
                e.arec[2 * np + slot] = make_double4(f[k][0], f[k][1], f[k][2], dti[k]);
                e.arec[3 * np + slot] = make_double4(f[k][3], f[k][4], f[k][5], 0.0);
            }
        }
        if (w == 0) {  // block `lane` of the cluster: the list entry
            constexpr uint32_t WPB = JT / 64;
            uint32_t below = 0, cnt = 0;
            for (uint32_t q = 0; q < SC; ++q) {
                const uint32_t x = wcnt[q];
                below += q / WPB < lane ? x : 0u;
                cnt += q / WPB == lane ? x : 0u;
            }
            const unsigned long long has = __ballot(cnt != 0);
            uint32_t d = 0;
            if (lane == 0) {
                const uint32_t total = (uint32_t)__popcll(has);
                if (e.K == 1)
                    e.ctl->ndirty[par] = total;
                else
                    d = atomicAdd(&e.ctl->ndirty[par], total);
                cs->nact = nact;
            }
            d = (uint32_t)__builtin_amdgcn_readfirstlane((int)d) +
                (uint32_t)__popcll(has & ((1ull << lane) - 1ull));
            if (cnt) {
                uint32_t *dl = e.dirty + ((size_t)par * e.nblk + d) * 3;
                dl[0] = off / JT + lane;
                dl[1] = below;
                dl[2] = cnt;
            }
        }
    }
    __syncthreads();  // wmin is rewritten below
    // (block_min_count's, block by block)
    for (uint32_t k = 0; k < SP; ++k) {
        const double m = wave_min(tdt[k]);
        const bool near = __ballot(tdt[k] != m && fabs(m - tdt[k]) < 2 * DBL_EPSILON) != 0;
        const uint32_t at = (uint32_t)__popcll(__ballot(tdt[k] == m));
        if (lane == 0) {
            wmin[k * SW + w] = m;
            wcnt[k * SW + w] = near ? BCNT_MANY : at;
        }
    }
    __syncthreads();
    constexpr uint32_t WPB = JT / 64;  // chunks per block
    if (tid < ntiles(e, c)) {
        const uint32_t w0 = tid * WPB;
        double m = wmin[w0];
        uint32_t at = 0;
        for (uint32_t k = 1; k < WPB; ++k) m = vmin(m, wmin[w0 + k]);
        for (uint32_t k = 0; k < WPB; ++k)
            at += wmin[w0 + k] == m ? wcnt[w0 + k]
                  : fabs(m - wmin[w0 + k]) < 2 * DBL_EPSILON ? BCNT_MANY : 0u;
        e.bmin[off / JT + tid] = m;
        e.bcnt[off / JT + tid] = at;
    }
    if (loop) return;
    wait_memory();
    __syncthreads();  // the step's stores are done
    if (tid) return;
    if (it > 0) {
        step_result(one.host, T, (uint32_t)nst, n, 1, nact);
        step_state(cs, one.itime, T, (uint32_t)nst, n, 1);
    } else {
        host_store(&one.host->done, (uint32_t)STEP_LEFT);
    }
}

// ---------------------------------------------------------------------------
// Mid-size systems: whole block steps in one workgroup per j tile or two
// ---------------------------------------------------------------------------

constexpr uint32_t TB = 2 * BS;         // threads of k_team_run
// Largest active set of a team with tpw tiles per workgroup.  Its pairs keep a
// workgroup one tile each: at 256 and one tile 15 us, where the launches of a
// larger step take 45; with two tiles what they take.
constexpr uint32_t team_act(uint32_t tpw) { return tpw == 1 ? 256u : 128u; }
constexpr uint32_t ONE_ACT = 128;       // of a single step (h4h_step)
constexpr uint32_t TEAM_ONE = 128;      // tiles up to which a workgroup has one (else two)
constexpr uint32_t TEAM_WGS = TEAM_TILES / 2;
// Steps left to the launches after a team did not form: that one, and twice as
// many each time in a row, up to 64.  (One launch in some thousand after the GPU
// was idle, and now and then a kernel's first, starts its last workgroup too
// late; that step takes 80 to 140 us.  With the CUs held by other work every
// launch does.)
__host__ __device__ inline uint64_t team_backoff(uint32_t fails) { return 1ull << (fails < 6 ? fails : 6); }
static_assert(TEAM_ONE <= TEAM_WGS && TEAM_WGS == 128, "workgroups of a team");

// What the workgroups of a team exchange, in device memory.  Every 64-bit
// word is written and read with agent-scope relaxed atomics (they go past
// the XCDs' L2s, so no fence is needed: an agent acquire fence per step
// measured 10 to 35 us) and holds SENT until it is written, so that reading a
// word is also waiting for it.
struct Team {
    uint32_t *sync;             // decision, number of workgroups that have left
    const uint32_t *plan;       // [team_act + 1]: log2 of the lane-group width | log2 of the
                                // finish lanes << 16, of the plan for nact (0: not one chunk
                                // per tile)
    unsigned long long *hdr;    // [3][workgroups][8]: min(t + dt) of the workgroup's tiles;
                                // number of particles that have it | first one's index << 32;
                                // its predicted position and velocity there
    unsigned long long *rec;    // [3][workgroups][team_act][8]: the others' position, velocity,
                                // index
    unsigned long long *part;   // [team_act][6][tiles]: the tiles' partial sums per active particle
                                // and component (the reader's lanes take consecutive tiles)
};
constexpr unsigned long long SENT = 0x7FF4A5A55A5A7E57ull;  // a signalling NaN: no sum's value
enum : uint32_t { TS_DECISION = 0, TS_LEFT = 32, TS_WORDS = 64 };
enum : uint32_t { TEAM_GO = 1, TEAM_NO = 2 };

template <class T>
__device__ __forceinline__ T agent_load(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void agent_store(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long bits(double x) {
    return __builtin_bit_cast(unsigned long long, x);
}
__device__ __forceinline__ double from_bits(unsigned long long u) {
    return __builtin_bit_cast(double, u);
}
// The word at p once it is written (SENT if it did not come).  Every writer
// of a formed team is resident, so the wait is short; POLLS (about a second)
// only bounds it.  Before (decision not null): some 200 us, and no longer
// than until somebody has given up.
constexpr uint32_t POLLS = 1u << 20, POLLS_FORM = 256;
__device__ __forceinline__ unsigned long long wait_word(const unsigned long long *p,
                                                        const uint32_t *decision) {
    unsigned long long v = agent_load(p);
    const uint32_t polls = decision ? POLLS_FORM : POLLS;
    for (uint32_t k = 1; v == SENT && k < polls; ++k) {
        v = agent_load(p);
        if (decision && k % 32 == 0 && agent_load(decision) == TEAM_NO) break;
    }
    return v;
}

// i tile `it` (IW slots, thread t of a group of BS) against a tile in LDS:
// the work item of the update kernel for one chunk of one tile, the same
// sums in the same order.  Leaves each wave's sums of the slots in red.
template <int IW, bool MIXED>
__device__ __forceinline__ void team_item(uint32_t it, uint32_t t, uint32_t nact, uint32_t j0,
                                          const double4 *tile, const double *irec,
                                          const uint32_t *ii, double e2, double *red) {
    const uint32_t k = it * IW + t % IW, kk = k < nact ? k : 0u;
    double pi[6];
    for (int q = 0; q < 6; ++q) pi[q] = irec[6 * kk + q];
    const uint32_t i = ii[kk], js = subgroup<IW>(t);
    double fo[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (__ballot((i - j0) < (uint32_t)JT))
        tile_pairs<IW, true, MIXED, 1>(pi, i, j0, js, tile, tile + JT, e2, fo);
    else
        tile_pairs<IW, false, MIXED, 1>(pi, i, j0, js, tile, tile + JT, e2, fo);
    double *row = red + ((it * (BS / 64) + (t >> 6)) * IW + t % IW) * 6;
    if constexpr (IW < 64)
        slot_sums(fo, IW, row);
    else
        for (int q = 0; q < 6; ++q) row[q] = fo[q];
}

// Block steps of a single system of 5 to TEAM_TILES j tiles, one workgroup
// per TPW tiles, up to max_run steps per launch: the device loop's steps with
// at most team_act active particles whose plan has one chunk per tile, with the
// same operations in the same order as the selection, update and finish
// launches, so a step has the same bits whichever makes it.  A step of those
// is three launches of 5-7 us each at least; here it is two exchanges:
//
// (1) every workgroup publishes its tiles' min(t + dt) and the particles that
//     have it, already predicted to that time; all read all of them, and know
//     the next block time T and the active particles.
// (2) every workgroup predicts its particles to T, sums the pairs of the
//     active particles with them and publishes the sums; the workgroups that
//     own active particles add the tiles' sums and apply the corrector.
//
// What bounds a step is the chain from one next time to the next on a
// workgroup that owns an active particle, two exchanges of 2-3 us each in it;
// about 7.5 us at 16 and 40 tiles, 10 us at 256.  Average block steps of runs
// (start to several hundred steps, all active sets): N = 4096 21.5 -> 10.9 us,
// 10007 26.0 -> 15.3, 65536 46.0 -> 37.6.  Up to TEAM_ONE
// tiles a workgroup has one, its two groups of BS threads take turns at the
// i tiles (N = 20000: 24.8 us, 27.1 with two tiles each); beyond, two, as 256
// workgroups exchange more slowly than 128.  Steps with more active particles
// want the whole chip for their pairs.
//
// Buffers: (1) goes round three slots; a workgroup clears its words of the
// slot before the last exchange when that exchange is complete (then every
// other one has read them) and before it publishes in the next (which the
// others wait for before they look at the cleared slot again).  The sums of
// (2) have one reader each, which clears them before it publishes.  The last
// workgroup to leave clears the last slot.
//
// Nothing here may wait for a workgroup that is not running.  The team forms
// if the first exchange is complete within a bounded wait: whoever sees it
// complete sets the decision to GO, whoever does not to NO, and the first
// setting holds; after GO all are resident until they end.  After NO
// everybody leaves without having changed anything, and so they do when the
// next step is not one of theirs: the launches after this one make it.
//
// ONE: a single step at `one.itime` (h4h_step), the first exchange and the
// sums; the last workgroup to leave clears what was published, takes the next
// time from the block minima and writes the result (a third exchange took 2 us
// more of 23).
template <bool MIXED, uint32_t TPW, bool ONE>
__global__ __launch_bounds__(TB) void k_team_run(Soa s, Ens e, Team tm, uint32_t max_run,
                                                 double e2, double eta, double dt_min,
                                                 double dt_max, OneStep one) {
#pragma clang fp contract(off)
    constexpr uint32_t TM_ACT = ONE ? ONE_ACT : team_act(TPW);
    constexpr uint32_t RED = 25 * TM_ACT;  // a tile's sums: 24 doubles per slot (<= 133 or 256)
    __shared__ double4 tile[TPW][2 * JT];  // predictor records
    __shared__ __align__(16) double red[TPW * RED];  // pair sums; then fs, outs
    __shared__ double hw[8 * TEAM_WGS];    // headers, word by word
    __shared__ double irec[6 * TM_ACT];    // active particles: position, velocity
    __shared__ uint32_t ii[TM_ACT], lst[TM_ACT];  // index; workgroup | place in its list << 16
    __shared__ double stg[7 * TM_ACT];     // own active particles: old forces, step
    __shared__ uint32_t lact[TM_ACT];      // their threads
    __shared__ uint32_t plans[TM_ACT + 1];
    __shared__ double wmn[TB / 64];
    __shared__ uint32_t wct[TB / 64], s_dec, s_bad;
    double *fs = red, *outs = red + 6 * TM_ACT;  // (19 per own active particle)
    constexpr uint32_t NQ = TEAM_WGS / 64;
    constexpr uint32_t OW = TPW * (BS / 64);  // waves that own particles

    const uint32_t tid = threadIdx.x, lane = __lane_id(), w = tid >> 6;
    const uint32_t b = blockIdx.x, M = gridDim.x, tiles = e.nblk;
    const uint32_t n = e.cnt[0];
    const uint32_t i = b * TPW * JT + tid;
    const bool in = tid < TPW * JT && i < n;
    // The state's loads go out with those of the check below.
    double r[3] = {0.0, 0.0, 0.0}, v[3] = {0.0, 0.0, 0.0};
    double f[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    double ti = 0.0, dti = 0.0, tdt = INFINITY;
    float mf = 0.0f;
    if (in) {
        for (int k = 0; k < 3; ++k) {
            r[k] = s.r[k][i];
            v[k] = s.v[k][i];
        }
        for (int k = 0; k < 6; ++k) f[k] = s.f[k][i];
        ti = s.t[i];
        dti = s.dt[i];
        mf = (float)s.m[i];
        tdt = ti + dti;
    }
    if (tid <= TM_ACT) plans[tid] = tm.plan[tid];
    ClState *cs = e.cs;
    RunCtl *ctl = e.ctl;
    constexpr bool loop = !ONE;
    const bool pend = loop && cs->tail_pend != 0;
    const double Tp = cs->tail_t, atime = loop ? cs->atime : one.itime;
    const uint32_t np_tail = cs->tail_nact;
    unsigned long long steps = !loop ? 0ull : pend ? cs->tail_steps + 1 : cs->steps;
    unsigned long long inter = loop ? cs->interactions : 0ull, nst = loop ? cs->nsteps : 0ull;
    const double t_end = loop ? ctl->t_end : (double)INFINITY;
    const double t_stop = loop ? ctl->t_stop : -(double)INFINITY;
    const unsigned long long max_steps = loop ? ctl->max_steps : 1ull;
    if (loop && (cs->done || steps < ctl->team_retry)) return;
    if (pend) {
        inter += (unsigned long long)np_tail * n;
        nst += np_tail;
    }
    double T;
    {
        // Whether the next step is one of a team's, from the block minima.
        constexpr uint32_t BQ = TEAM_TILES / 64;
        double x[BQ], m = INFINITY;
        uint32_t xc[BQ], c = 0;
        for (uint32_t q = 0; q < BQ; ++q) {
            const uint32_t k = 64 * q + lane;
            x[q] = k < tiles ? e.bmin[k] : (double)INFINITY;
            xc[q] = k < tiles ? e.bcnt[k] : 0u;
        }
        for (uint32_t q = 0; q < BQ; ++q) m = vmin(m, x[q]);
        T = wave_min(m);
        bool close = false;
        for (uint32_t q = 0; q < BQ; ++q) {
            c += x[q] == T ? min(xc[q], BCNT_MANY) : 0u;
            close |= __ballot(x[q] != T && fabs(T - x[q]) < 2 * DBL_EPSILON) != 0;
        }
        c = row_sum(c);
        const uint32_t nact = (uint32_t)__builtin_amdgcn_readlane((int)c, 0) +
                              (uint32_t)__builtin_amdgcn_readlane((int)c, 16) +
                              (uint32_t)__builtin_amdgcn_readlane((int)c, 32) +
                              (uint32_t)__builtin_amdgcn_readlane((int)c, 48);
        __syncthreads();  // plans
        if (close || nact < 1 || nact > TM_ACT || !plans[nact] ||
            (pend ? loop_stops(*ctl, Tp, steps, T) : T != atime)) {
            if (!loop && b == 0 && tid == 0) host_store(&one.host->done, (uint32_t)STEP_LEFT);
            return;
        }
    }

    bool go = false, stop = false, act = false;
    uint32_t it = 0, slot = 0, hk = (uint32_t)(steps % e.hist_cap);
    uint32_t nact = 0, cnt = 0, cnt_before = 0;  // published in this and the last exchange
    double t_last = 0.0;
    if (tid == 0) s_bad = 0;
    // corrector lanes
    const bool vel = (lane & 4u) != 0;
    const uint32_t cc = min(lane & 3u, 2u), cq = cc + (vel ? 3u : 0u);
    // The state after a step, while the others publish: the old forces and
    // the derivatives are still in stg and outs (place `was` of the list).
    uint32_t was = 0;
    auto store_state = [&] {
        if (!act) return;
        const size_t np = (size_t)tiles * JT;  // the state's columns are np apart
        auto *col = in_loop(s.r[0]) + i;
        for (int k = 0; k < 3; ++k) col[(COL_R + k) * np] = r[k];
        for (int k = 0; k < 3; ++k) col[(COL_R + 4 + k) * np] = v[k];
        for (int k = 0; k < 6; ++k) col[(COL_F + k) * np] = f[k];
        for (int k = 0; k < 6; ++k) col[(COL_OLD + k) * np] = stg[7 * was + k];
        for (int k = 0; k < 6; ++k) col[(COL_A2 + k) * np] = outs[19 * was + 13 + k];
        col[COL_T * np] = ti;
        col[COL_DT * np] = dti;
    };
    for (;;) {
        // (1) The next time of this workgroup's particles, and those that
        // have it.  (A wave whose minimum is within the selection's tolerance
        // of the time but not equal to it makes the count BCNT_MANY.)
        unsigned long long mask = 0;
        if (w < OW) {
            const double m = wave_min(tdt);
            mask = __ballot(in && fabs(m - tdt) < 2 * DBL_EPSILON);
            if (lane == 0) {
                wmn[w] = m;
                wct[w] = (uint32_t)__popcll(mask);
            }
        }
        __syncthreads();
        double t_own = wmn[0];
        for (uint32_t k = 1; k < OW; ++k) t_own = vmin(t_own, wmn[k]);
        cnt_before = cnt;
        cnt = 0;
        uint32_t rank = (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
        for (uint32_t k = 0; k < OW; ++k) {
            const uint32_t c = wmn[k] == t_own ? wct[k]
                               : fabs(t_own - wmn[k]) < 2 * DBL_EPSILON ? BCNT_MANY : 0u;
            rank += k < w && wmn[k] == t_own ? c : 0u;  // (there always is a rank 0)
            cnt += c;
        }
        const bool cand = w < OW && wmn[w] == t_own && ((mask >> lane) & 1ull);
        unsigned long long *hd = tm.hdr + ((size_t)slot * M + b) * 8;
        if (cand && rank < TM_ACT && (loop || rank == 0 || t_own == T)) {
            double4 pa, pb;
            predict_vals(r, v, f, t_own - ti, mf, pa, pb);
            unsigned long long *o =
                rank ? tm.rec + (((size_t)slot * M + b) * TM_ACT + rank) * 8 : hd + 2;
            agent_store(o + 0, bits(pa.x));
            agent_store(o + 1, bits(pa.y));
            agent_store(o + 2, bits(pa.z));
            agent_store(o + 3, bits(pb.x));
            agent_store(o + 4, bits(pb.y));
            agent_store(o + 5, bits(pb.z));
            if (rank) {
                agent_store(o + 6, (unsigned long long)i);
            } else {
                agent_store(hd + 1, (unsigned long long)cnt | (unsigned long long)i << 32);
                agent_store(hd, bits(t_own));
            }
        }
        if (!cnt && tid == 0) {  // (no finite time)
            for (int k = 1; k < 8; ++k) agent_store(hd + k, 0ull);
            agent_store(hd, bits((double)INFINITY));
        }
        // The step before's state, to HBM while the others publish.
        if (loop) store_state();
        // All workgroups'.
        for (uint32_t k = tid; k < 8 * M; k += TB) {
            const unsigned long long u =
                wait_word(
                tm.hdr + (size_t)slot * M * 8 + k, go ? nullptr : tm.sync + TS_DECISION);
            if (u == SENT) s_bad = 1;
            hw[k % 8 * TEAM_WGS + k / 8] = from_bits(u);
        }
        __syncthreads();
        if (!go) {
            if (tid == 0) {
                const uint32_t want = s_bad ? TEAM_NO : TEAM_GO;
                const uint32_t d = atomicCAS(&tm.sync[TS_DECISION], 0u, want);
                s_dec = d ? d : want;
                // (all were there, though this one's wait ran out: it goes on)
                if (s_dec == TEAM_GO) s_bad = 0;
            }
            __syncthreads();
            go = s_dec == TEAM_GO;
            if (!go) break;
            for (uint32_t k = tid; k < 8 * M; k += TB)
                if (bits(hw[k % 8 * TEAM_WGS + k / 8]) == SENT) {  // (this wait had missed it)
                    const unsigned long long u = wait_word(tm.hdr + k, nullptr);
                    if (u == SENT) s_bad = 1;
                    hw[k % 8 * TEAM_WGS + k / 8] = from_bits(u);
                }
            __syncthreads();
            if (pend && b == 0 && tid == 0) {
                record_tail(e, 0, Tp, np_tail, steps, T, false);
                cs->tail_pend = 0;
            }
        }
        if (s_bad) break;
        // The next block time, the workgroups that have it, and the places of
        // their particles in the active list (workgroup by workgroup); every
        // wave for itself.
        double x[NQ], m = INFINITY;
        for (uint32_t q = 0; q < NQ; ++q) {
            x[q] = 64 * q + lane < M ? hw[64 * q + lane] : (double)INFINITY;
            m = vmin(m, x[q]);
        }
        const double mn = wave_min(m);
        bool close = false;
        const uint32_t last_nact = nact;
        uint32_t place[NQ], c[NQ], heads = 0;
        nact = 0;
        for (uint32_t q = 0; q < NQ; ++q) {
            close |= __ballot(x[q] != mn && fabs(mn - x[q]) < 2 * DBL_EPSILON) != 0;
            const bool at = x[q] == mn && 64 * q + lane < M;
            c[q] = at ? (uint32_t)bits(hw[TEAM_WGS + 64 * q + lane]) : 0u;
            heads += (uint32_t)__popcll(__ballot(c[q] != 0));
            uint32_t sum;
            place[q] = nact + wave_scan(c[q], sum);
            nact += sum;
        }
        const uint32_t mine = b < 64 ? (uint32_t)__builtin_amdgcn_readlane((int)c[0], (int)(b & 63))
                                     : (uint32_t)__builtin_amdgcn_readlane((int)c[NQ - 1], (int)(b & 63));
        const uint32_t k0 = b < 64
                                ? (uint32_t)__builtin_amdgcn_readlane((int)place[0], (int)(b & 63))
                                : (uint32_t)__builtin_amdgcn_readlane((int)place[NQ - 1], (int)(b & 63));
        static_assert(NQ == 2, "two masks of workgroups");
        if (it > 0) {
            // The slot of the exchange before is read by all.
            const uint32_t prev = slot == 0 ? 2u : slot - 1u;
            if (tid < 8) agent_store(tm.hdr + ((size_t)prev * M + b) * 8 + tid, SENT);
            unsigned long long *pr = tm.rec + ((size_t)prev * M + b) * TM_ACT * 8;
            for (uint32_t k = 8 + tid; k < 8 * min(cnt_before, TM_ACT); k += TB)
                agent_store(pr + k, SENT);
            // Loop tail of the step made before this exchange.
            steps += 1;
            inter += (unsigned long long)last_nact * n;
            nst += last_nact;
            stop = t_last >= t_stop || steps >= max_steps || !(t_last < t_end) || !(mn > t_last);
            if (b == 0 && tid == 0) {
                e.hist_t[hk] = t_last;
                e.hist_n[hk] = last_nact;
            }
            if (++hk == e.hist_cap) hk = 0;
        }
        T = mn;
        if (close) nact = BCNT_MANY;  // (not counted)
        if (stop || it >= max_run || nact < 1 || nact > TM_ACT) break;
        const uint32_t plan = __builtin_amdgcn_readfirstlane(plans[nact]);
        if (!plan) break;
        const uint32_t lw = plan & 0xffffu, iw = 1u << lw, ll = plan >> 16, L = 1u << ll;
        // (2) The active particles (the last wave: the headers' and the list of
        // the others), and this workgroup's at T.
        if (w == TB / 64 - 1)
            for (uint32_t q = 0; q < NQ; ++q)
                if (c[q]) {
                    const double *h = hw + 64 * q + lane;
                    for (int y = 0; y < 6; ++y) irec[6 * place[q] + y] = h[(2 + y) * TEAM_WGS];
                    ii[place[q]] = (uint32_t)(bits(h[TEAM_WGS]) >> 32);
                    for (uint32_t l = 0; l < c[q]; ++l) lst[place[q] + l] = (64 * q + lane) | l << 16;
                }
        act = mine && cand;
        if (tid < TPW * JT) {
            double4 pa = make_double4(PAD_POS, PAD_POS, PAD_POS, 0.0);
            double4 pb = make_double4(0.0, 0.0, 0.0, mass_bits(0.0f));
            if (in) predict_vals(r, v, f, T - ti, mf, pa, pb);
            tile[tid / JT][tid % JT] = pa;
            tile[tid / JT][JT + tid % JT] = pb;
            if (act) {
                lact[rank] = tid;
                for (int q = 0; q < 6; ++q) stg[7 * rank + q] = f[q];
                stg[7 * rank + 6] = dti;
            }
        }
        __syncthreads();
        if (nact > heads) {
            const uint32_t l = tid < nact ? lst[tid] >> 16 : 0u;
            if (l) {
                const unsigned long long *o =
                    tm.rec + (((size_t)slot * M + (lst[tid] & 0xffffu)) * TM_ACT + l) * 8;
                unsigned long long u[7];
                bool wait = true;
                for (uint32_t polls = 0; wait && polls < POLLS; ++polls) {
                    wait = false;
#pragma unroll
                    for (int q = 0; q < 7; ++q) u[q] = agent_load(o + q);
#pragma unroll
                    for (int q = 0; q < 7; ++q) wait |= u[q] == SENT;
                }
                if (wait) s_bad = 1;
#pragma unroll
                for (int q = 0; q < 6; ++q) irec[6 * tid + q] = from_bits(u[q]);
                ii[tid] = (uint32_t)u[6];
            }
            __syncthreads();
        }
        {
            const uint32_t grp = tid / BS, t = tid % BS, nit = (nact + iw - 1) >> lw;
            const uint32_t tl = TPW == 2 ? grp : 0u;
            const uint32_t j0 = (b * TPW + tl) * JT;
            for (uint32_t a = TPW == 2 ? 0u : grp; a < nit; a += TPW == 2 ? 1u : 2u) {
                if (iw == 4)
                    team_item<4, MIXED>(a, t, nact, j0, tile[tl], irec, ii, e2, red + tl * RED);
                else if (iw == 16)
                    team_item<16, MIXED>(a, t, nact, j0, tile[tl], irec, ii, e2, red + tl * RED);
                else
                    team_item<64, MIXED>(a, t, nact, j0, tile[tl], irec, ii, e2, red + tl * RED);
            }
        }
        wait_memory();  // the cleared words are clear (before anything is published again)
        __syncthreads();
        // The waves' sums in order, as the update's work item adds them.
        for (uint32_t y = tid; y < TPW * 6 * nact; y += TB) {
            constexpr double scale = MIXED ? 1.0 : PAIR_SCALE;
            const uint32_t tl = TPW == 2 && y >= 6 * nact ? 1u : 0u;
            const uint32_t yy = y - tl * 6 * nact, k = yy / 6, q = yy % 6;
            if (b * TPW + tl >= tiles) continue;  // (an odd last tile's partner)
            const uint32_t st = 6 << lw;
            const double *row =
                red + tl * RED + (((k >> lw) * (BS / 64) << lw) + (k & (iw - 1))) * 6 + q;
            double acc = row[0];
            for (uint32_t g = 1; g < BS / 64; ++g) acc += row[g * st];
            agent_store(tm.part + (size_t)yy * tiles + b * TPW + tl, bits(acc * scale));
        }
        if (mine) {
            __syncthreads();  // red is read: fs and outs go there
            // The tiles' sums of this workgroup's active particles, as the
            // finish pass adds them (chunk_sums): lane sl of L takes tiles sl,
            // sl + L, ...
            const uint32_t sl = tid & (L - 1);
            for (uint32_t base = 0; base < mine; base += TB >> ll) {
                const uint32_t kk = base + (tid >> ll);
                const bool valid = kk < mine;
                double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                if (valid) {
                    unsigned long long *pk = tm.part + 6 * (size_t)(k0 + kk) * tiles;
                    constexpr uint32_t U = 4;  // tiles of one wait
                    for (uint32_t s0 = sl; s0 < tiles; s0 += U * L) {
                        unsigned long long u[U][6];
                        bool wait = true;
                        for (uint32_t polls = 0; wait && polls < POLLS; ++polls) {
                            wait = false;
#pragma unroll
                            for (uint32_t y = 0; y < U; ++y) {
                                // (past the end: the lane's first tile again)
                                const uint32_t sc = s0 + y * L < tiles ? s0 + y * L : s0;
#pragma unroll
                                for (int q = 0; q < 6; ++q)
                                    u[y][q] = agent_load(pk + q * tiles + sc);
                            }
#pragma unroll
                            for (uint32_t y = 0; y < U; ++y)
#pragma unroll
                                for (int q = 0; q < 6; ++q) wait |= u[y][q] == SENT;
                        }
                        if (wait) s_bad = 1;
#pragma unroll
                        for (uint32_t y = 0; y < U; ++y)
                            if (s0 + y * L < tiles) {
#pragma unroll
                                for (int q = 0; q < 6; ++q) {
                                    agent_store(pk + q * tiles + s0 + y * L, SENT);
                                    acc[q] += from_bits(u[y][q]);
                                }
                            }
                    }
                }
                for (int q = 0; q < 6; ++q) acc[q] = lanes_sum(acc[q], L);
                if (valid && sl == 0)
                    for (int q = 0; q < 6; ++q) fs[6 * kk + q] = acc[q];
            }
            __syncthreads();
            for (uint32_t p0 = 0; p0 < mine; p0 += TB / 8) {
                if (p0 + 8 * w >= mine) continue;  // (whole waves)
                const uint32_t kk = min(p0 + tid / 8, mine - 1);
                const double *st = stg + 7 * kk, *fk = fs + 6 * kk;
                const uint32_t la = lact[kk];
                const double pr = reinterpret_cast<const double *>(
                    tile[la / JT] + la % JT + (vel ? (uint32_t)JT : 0u))[cc];
                const Corr8 ck = corr8_coef(st[6], T, vel);
                const double f0 = fk[cc], f1 = fk[3 + cc];
                double xn, ad;
                const double dtn = corr8(ck, vel, st[cc], st[3 + cc], f0, f1, pr, eta, dt_min,
                                         dt_max, xn, ad);
                if (p0 + tid / 8 < mine && (lane & 3u) < 3u) {
                    double *o = outs + 19 * kk;
                    o[cq] = vel ? f1 : f0;
                    o[6 + cq] = xn;
                    o[13 + cq] = ad;
                    if ((lane & 7u) == 0) o[12] = dtn;
                }
            }
            wait_memory();  // the cleared sums are clear
            __syncthreads();
            if (act) {
                const double *o = outs + 19 * rank;
                was = rank;
                for (int q = 0; q < 6; ++q) f[q] = o[q];
                for (int q = 0; q < 3; ++q) {
                    r[q] = o[6 + q];
                    v[q] = o[9 + q];
                }
                ti = T;
                dti = o[12];
                tdt = ti + dti;
            }
        }
        t_last = T;
        ++it;
        if (!loop) {
            nst = nact;
            store_state();
            break;
        }
        slot = slot == 2 ? 0u : slot + 1u;
    }
    // Loop state, predictor records of the last step, block minima.
    if (it > 0) {
        if (b == 0 && tid == 0 && loop) {
            cs->itime = t_last;
            cs->atime = T;
            cs->steps = steps;
            cs->interactions = inter;
            cs->nsteps = nst;
            ctl->team_steps += it;
            ctl->team_fails = 0;
            if (stop) {
                cs->done = 1;
                atomicAdd(&ctl->ndone, 1u);
            }
        }
        if (in) {
            s.pp[i] = tile[tid / JT][tid % JT];
            s.pv[i] = tile[tid / JT][JT + tid % JT];
        }
        // (block_min_count's, tile by tile)
        double m = INFINITY;
        if (w < OW) {
            m = wave_min(tdt);
            const bool near = __ballot(tdt != m && fabs(m - tdt) < 2 * DBL_EPSILON) != 0;
            const uint32_t at = (uint32_t)__popcll(__ballot(tdt == m));
            if (lane == 0) {
                wmn[w] = m;
                wct[w] = near ? BCNT_MANY : at;
            }
        }
        __syncthreads();
        if (tid < TPW && b * TPW + tid < tiles) {
            const uint32_t w0 = tid * (BS / 64);
            uint32_t at = 0;
            m = wmn[w0];
            for (uint32_t k = 1; k < BS / 64; ++k) m = vmin(m, wmn[w0 + k]);
            for (uint32_t k = 0; k < BS / 64; ++k)
                at += wmn[w0 + k] == m ? wct[w0 + k]
                      : fabs(m - wmn[w0 + k]) < 2 * DBL_EPSILON ? BCNT_MANY : 0u;
            if (loop) {
                e.bmin[b * TPW + tid] = m;
                e.bcnt[b * TPW + tid] = at;
            } else {  // (read by the last one out)
                agent_store(reinterpret_cast<unsigned long long *>(e.bmin) + b * TPW + tid, bits(m));
                agent_store(e.bcnt + b * TPW + tid, at);
            }
        }
    }
    // This workgroup's further records of the last exchange (nobody reads
    // them), and its header if no team formed.
    unsigned long long *rc = tm.rec + ((size_t)slot * M + b) * TM_ACT * 8;
    if (loop || !it)
        for (uint32_t k = 8 + tid; k < 8 * min(cnt, TM_ACT); k += TB) agent_store(rc + k, SENT);
    if (!go && tid < 8) agent_store(tm.hdr + (size_t)b * 8 + tid, SENT);
    if (go && s_bad && tid == 0) agent_store(&ctl->team_err, 1u);
    wait_memory();
    __syncthreads();
    if (tid == 0) s_dec = atomicAdd(&tm.sync[TS_LEFT], 1u) == M - 1;
    __syncthreads();
    if (!s_dec) return;
    // The last one out.
    if (go)
        for (uint32_t k = tid; k < 8 * M; k += TB)
            agent_store(tm.hdr + (size_t)slot * M * 8 + k, SENT);
    else if (tid == 0 && loop) {
        const uint32_t fails = ctl->team_fails;
        ctl->team_retry = steps + team_backoff(fails);
        ctl->team_fails = fails + 1;
    }
    if (tid == 0) {
        agent_store(&tm.sync[TS_DECISION], 0u);
        agent_store(&tm.sync[TS_LEFT], 0u);
    }
    if (loop) return;
    double x = INFINITY, mn = INFINITY;
    uint32_t xc = 0;
    if (it > 0) {
        for (uint32_t k = tid; k < 8 * nact; k += TB)  // the active particles' records
            if (const uint32_t l = lst[k / 8] >> 16)
                agent_store(tm.rec + ((size_t)(lst[k / 8] & 0xffffu) * TM_ACT + l) * 8 + k % 8, SENT);
        if (tid < tiles) {
            x = from_bits(agent_load(reinterpret_cast<unsigned long long *>(e.bmin) + tid));
            xc = min(agent_load(e.bcnt + tid), BCNT_MANY);
        }
        const double m = wave_min(x);
        if (lane == 0) wmn[w] = m;
        if (tid == 0) lact[0] = 0;
        __syncthreads();
        for (uint32_t k = 0; k < TB / 64; ++k) mn = vmin(mn, wmn[k]);
        if (x != mn) xc = fabs(mn - x) < 2 * DBL_EPSILON ? BCNT_MANY : 0u;
        if (xc) atomicAdd(&lact[0], xc);
    }
    wait_memory();
    __syncthreads();
    if (tid) return;
    if (agent_load(&ctl->team_err))
        host_store(&one.host->done, (uint32_t)STEP_FAILED);
    else if (it > 0) {
        step_result(one.host, mn, (uint32_t)nst, n, 0, lact[0]);
        step_state(cs, one.itime, mn, (uint32_t)nst, n, 0);
    } else {
        host_store(&one.host->done, (uint32_t)(go ? STEP_LEFT : STEP_ALONE));
    }
}

// The decision of the next team made ahead (h4h_refuse_team).
__global__ void k_team_refuse(Team tm) { agent_store(&tm.sync[TS_DECISION], (uint32_t)TEAM_NO); }

// Every word of a team's buffers waiting (context creation).
__global__ __launch_bounds__(BS) void k_team_clear(Team tm, size_t words) {
    for (size_t k = blockIdx.x * (size_t)BS + threadIdx.x; k < words; k += (size_t)gridDim.x * BS)
        tm.hdr[k] = SENT;
    if (blockIdx.x == 0 && threadIdx.x < TS_WORDS) tm.sync[threadIdx.x] = 0;
}

// Single-cluster ABI helpers.
__global__ void k_set_nact0(Ens e, uint32_t nact) { e.cs[0].nact = nact; }
__global__ void k_reset_tmin(Ens e) {
    for (uint32_t c = 0; c < e.K; ++c) e.cs[c].tmin_key = dkey(INFINITY);
}
__global__ void k_reset_select(Ens e) {
    for (uint32_t c = 0; c < e.K; ++c) e.cs[c].nact = 0;
}
// After init_dt: every cluster at t = itime with ATIME = its minimum dt.
__global__ void k_set_times_from_tmin(Ens e, double itime) {
    for (uint32_t c = 0; c < e.K; ++c) {
        e.cs[c].itime = itime;
        e.cs[c].atime = dkey_inv(e.cs[c].tmin_key);
    }
}

// ---------------------------------------------------------------------------
// Energy: sum 1/2 m v^2 - sum_{i<j} m_i m_j / |r_ij| (unsoftened) of one
// cluster, NbodyUtils::get_energy (NbodyUtils.cpp:427-529).  1/|r_ij| from
// v_rsq_f64 and one Newton step (relative error below 2^-47 and of one
// sign, against the reference's division by sqrt): a lane sums
// 2 m_j / |r_ij| over one j chunk in plain FP64 (at most 256 terms of one
// sign, so at most 256 roundings of the partial sum: 3e-14 relative),
// multiplies by m_i / 2 and adds that into its Neumaier-compensated sum;
// then per workgroup, then over workgroups in index order (deterministic
// for a fixed n).  A coincident pair (r = 0) makes the Newton step NaN; such
// a chunk is summed again with 1/0 = inf, so coincident particles give -inf
// as in the reference.
// ---------------------------------------------------------------------------

// Neumaier-compensated sum += x.  Once the sum is infinite (coincident
// particles in the unsoftened energy) the compensation is left alone, so
// the result is the infinity a plain sum gives rather than inf - inf.
__device__ __forceinline__ void neumaier(double &sum, double &comp, double x) {
#pragma clang fp contract(off)
    double t = sum + x;
    if (isfinite(t)) {
        if (fabs(sum) >= fabs(x))
            comp += (sum - t) + x;
        else
            comp += (x - t) + sum;
    }
    sum = t;
}

__device__ __forceinline__ void block_sum2(double &a, double &b, double *red) {
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o);
        b += __shfl_xor(b, o);
    }
    uint32_t w = threadIdx.x >> 6;
    __syncthreads();
    if (__lane_id() == 0) {
        red[2 * w] = a;
        red[2 * w + 1] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t k = 1; k < BS / 64; ++k) {
            a += red[2 * k];
            b += red[2 * k + 1];
        }
    }
}

// Cluster c0 + blockIdx.y of the cluster tables offs / cnts: items are pairs
// of an i block (ENERGY_I particles, EI per lane) and a j chunk (jc
// particles, EnergyItems) that reaches past the block's first particle,
// numbered row by row (i block by i block), a contiguous run of them per
// workgroup; out[4 (blockIdx.y gridDim.x + blockIdx.x)] = {epot, epot_comp,
// ekin, ekin_comp} of the run.
//
// VALU bound at 14 issue slots per pair (3 sub, 3 for r^2, 4 for v_rsq_f64,
// 4 for the Newton step and the sum) if each j record read from LDS serves
// EI pairs: one pair per read took the 16 cycles that a CU's LDS needs to
// return a broadcast double4 to a wave as often as its SIMDs took 60 to use
// it, four SIMDs per LDS (N = 262144: 1.72e12 pairs/s).
constexpr uint32_t EI = ENERGY_I / BS;

__device__ __forceinline__ double energy_term(const double4 &q, double xi, double yi, double zi,
                                              double sum, bool guard) {
    const double rx = q.x - xi, ry = q.y - yi, rz = q.z - zi;
    const double r2 = __builtin_fma(rx, rx, __builtin_fma(ry, ry, rz * rz));
    const double y = __builtin_amdgcn_rsq(r2);
    double w = __builtin_fma(-(r2 * y), y, 3.0);  // y w = 2 / r
    if (guard && !(r2 > 0.0)) w = INFINITY;       // (y is +inf there too)
    return __builtin_fma(q.w * y, w, sum);
}

__global__ __launch_bounds__(BS) void k_energy(Soa s, const uint32_t *offs, const uint32_t *cnts,
                                              uint32_t c0, double *out) {
#pragma clang fp contract(off)
    __shared__ double4 sr[2][JT];
    __shared__ double red[2 * (BS / 64)];
    const uint32_t off = offs[c0 + blockIdx.y], n = cnts[c0 + blockIdx.y];
    const EnergyItems ei = energy_items(n);
    const uint32_t R = ENERGY_I / ei.jc;  // a row starts R chunks after the one before
    double ep = 0.0, epc = 0.0, ek = 0.0, ekc = 0.0;
    if (blockIdx.x < ei.wgs) {
        const uint64_t first = ei.items * blockIdx.x / ei.wgs;
        const uint64_t last = ei.items * (blockIdx.x + 1) / ei.wgs;
        uint32_t row = 0;
        uint64_t rem = first;
        while (rem >= ei.chunks - row * R) {
            rem -= ei.chunks - row * R;
            ++row;
        }
        auto load_j = [&](uint32_t ch) {  // (past the end: zero mass, far away)
            const uint32_t lj = ch * ei.jc + threadIdx.x, j = off + lj;
            if (threadIdx.x < ei.jc && lj < n)
                return make_double4(s.r[0][j], s.r[1][j], s.r[2][j], s.m[j]);
            return make_double4(PAD_POS, PAD_POS, PAD_POS, 0.0);
        };
        double xi[EI], yi[EI], zi[EI], mi[EI];
        double4 nj = load_j(row * R + (uint32_t)rem);
        bool fresh = true;  // a new row's i particles are to be loaded
        for (uint64_t item = first; item < last; ++item) {
            const uint32_t ch = row * R + (uint32_t)rem;
            const uint32_t li0 = row * ENERGY_I + threadIdx.x;
            double4 *tile = sr[item & 1];
            tile[threadIdx.x] = nj;
            if (fresh)
                for (uint32_t k = 0; k < EI; ++k) {
                    const uint32_t li = li0 + k * BS, i = off + li;
                    const bool in = li < n;
                    xi[k] = in ? s.r[0][i] : -PAD_POS;
                    yi[k] = in ? s.r[1][i] : -PAD_POS;
                    zi[k] = in ? s.r[2][i] : -PAD_POS;
                    mi[k] = in ? s.m[i] : 0.0;
                    if (rem == 0 && in) {  // the row's first item counts its kinetic energy
                        const double vx = s.v[0][i], vy = s.v[1][i], vz = s.v[2][i];
                        const double vv2 = vx * vx + vy * vy + vz * vz;
                        neumaier(ek, ekc, 0.5 * mi[k] * vv2);
                    }
                }
            // the next item, its j chunk requested under this one's pairs
            const bool diag = rem < R;
            fresh = ++rem >= ei.chunks - row * R;
            if (fresh) {
                rem = 0;
                ++row;
            }
            if (item + 1 < last) nj = load_j(row * R + (uint32_t)rem);
            __syncthreads();  // (the other tile's readers passed the last one)
            double sum[EI];
            for (uint32_t k = 0; k < EI; ++k) sum[k] = 0.0;
            if (!diag) {
#pragma unroll 4
                for (uint32_t jj = 0; jj < ei.jc; ++jj) {
                    const double4 q = tile[jj];
#pragma unroll
                    for (uint32_t k = 0; k < EI; ++k)
                        sum[k] = energy_term(q, xi[k], yi[k], zi[k], sum[k], false);
                }
            }
            for (uint32_t k = 0; k < EI; ++k) {
                const uint32_t li = li0 + k * BS, jd = li + 1;
                const uint32_t jb = jd > ch * ei.jc ? jd - ch * ei.jc : 0u;  // j > i
                if (diag)
                    for (uint32_t jj = jb; jj < ei.jc; ++jj)
                        sum[k] = energy_term(tile[jj], xi[k], yi[k], zi[k], sum[k], false);
                if (isnan(sum[k])) {
                    sum[k] = 0.0;
                    for (uint32_t jj = jb; jj < ei.jc; ++jj)
                        sum[k] = energy_term(tile[jj], xi[k], yi[k], zi[k], sum[k], true);
                }
                if (li < n) neumaier(ep, epc, -(0.5 * mi[k] * sum[k]));
            }
        }
    }
    block_sum2(ep, epc, red);
    __syncthreads();
    block_sum2(ek, ekc, red);
    if (threadIdx.x == 0) {
        double *o = out + 4 * ((size_t)blockIdx.y * gridDim.x + blockIdx.x);
        o[0] = ep;
        o[1] = epc;
        o[2] = ek;
        o[3] = ekc;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Context
// ---------------------------------------------------------------------------

namespace {
constexpr uint32_t RUN_CHUNK = 32;    // block steps per captured graph
constexpr uint32_t SMALL_RUN = 255;   // k_small_run steps per launch
constexpr uint32_t SMALL_SLOTS = 8;   // (k_small_run + block step) pairs per captured graph
static_assert(RUN_CHUNK % 2 == 0 && SMALL_SLOTS % 2 == 0,
              "a step's dirty list is its slot in the chunk mod 2; chunks follow each other");
constexpr uint32_t SMALL_ACT = 64;    // default largest active set k_small_run takes (one system)
constexpr uint32_t HIST_CAP = 2048;   // per-step history ring of cluster 0
static_assert(HIST_CAP >= RUN_CHUNK && HIST_CAP >= SMALL_SLOTS * (SMALL_RUN + 1),
              "history ring shorter than the steps of one graph");
constexpr int N_SOA = 35;           // doubles per particle in `state`

// Downloads go through pinned slots, written by k_rows_out over the bus and
// copied to the caller's arrays by the calling thread and, for more than a few
// pieces, others, two slots each.  From DL_MIN doubles (4 MB): 4 threads and
// 512 KB slots, as one thread's copies and its page faults on arrays not
// touched before take longer than the bus: 28 doubles of 262144 particles 8.1
// -> 3.9 ms into new arrays, 3.4 -> 1.8 ms into used ones (the pieces alone: 2
// threads 3.2 and 1.7 ms, 4 2.4 and 1.6, 8 1.8 and 1.7; slots of 256 KB: 2.7).
// Below: 256 KB slots, 1 MB in all, which is had in 15 to 40 us (2 MB: 270); a
// gather, a copy and a wait per array took 0.30 ms at n = 1024 and 0.67 at n =
// 4096.  From DL_TWO doubles (1 MB) 2 threads, whose start takes as long as one
// copies 0.5 MB: r of 25000 particles (0.8 MB) 54 us with one, 72 with two, r of
// 50000 91 and 98, all of 15000 (3.4 MB) into new arrays 0.20 and 0.19 ms.
constexpr uint32_t DL_THREADS = 4, DL_SLOTS = 2 * DL_THREADS;
constexpr uint32_t DL_SLOT = 1u << 16, DL_SLOT_SMALL = 1u << 15;  // doubles
constexpr size_t DL_MIN = 8 * (size_t)DL_SLOT, DL_TWO = 4 * (size_t)DL_SLOT_SMALL;
}  // namespace

struct h4h_ctx {
    uint32_t K = 0;       // clusters
    uint32_t n = 0;       // particles (all clusters)
    uint32_t n_dev = 0;   // padded device particles
    uint32_t nblk = 0;    // JT blocks
    std::vector<uint32_t> off, cnt, hoff;
    double e2 = 0.0;
    float eta = 0.0f;
    double dt_min = 0.0, dt_max = 0.0;
    int precision = H4H_FP64;
    int device = 0;
    uint32_t grid = DEFAULT_GRID;      // requested persistent workgroups
    uint32_t max_split = DEFAULT_MAX_SPLIT;
    uint32_t iw_fill = DEFAULT_IW_FILL;  // pick_iw fill rule (sixteenths)
    bool uploaded = false;
    bool timing = false;
    bool bm_valid = false;   // per-block minima match t + dt
    bool small_ok = false;   // the device can launch k_small_run
    uint32_t small_act = SMALL_ACT;  // k_small_run takes active sets up to this (0: off)
    uint32_t nact_host = 0;  // size of cluster 0's active list (single-system calls)
    uint32_t next_nact = 0;  // active count of the step at next_time, told by the last h4h_step
    double next_time = 0.0;  // (while the block minima stay valid; 0: not known)
    double mass_max = 0.0;   // largest |float mass| of the uploaded state (+inf: not finite)

    hipStream_t stream = nullptr;
    char *arena = nullptr;       // device memory of all the pointers below but partial
    double *state = nullptr;     // all SoA arrays
    double *staging = nullptr;   // n * 8 doubles
    double *partial = nullptr;   // j-split partials
    size_t partial_len = 0;
    uint32_t *move = nullptr;
    // cluster tables
    uint32_t *d_off = nullptr, *d_cnt = nullptr, *d_hoff = nullptr, *d_bcl = nullptr;
    ClState *d_cs = nullptr;  // behind d_ctl
    ClPlan *d_plan = nullptr;
    unsigned long long *d_pre = nullptr;  // items_pre | fin_pre | part_pre
    RunCtl *d_ctl = nullptr;
    uint32_t *d_dirty = nullptr;
    double *d_bmin = nullptr;    // [nblk], then u32 x nblk counts
    Team team{};                 // exchange buffers of k_team_run (behind d_arec)
    bool team_ok = false;        // the system has a team's number of tiles, and the device room
    double4 *d_arec = nullptr;   // the step's active particles' records (Ens::arec)
    uint32_t *d_tune = nullptr;  // [64] tuning table
    // pinned host memory: energy per-workgroup sums, mirrors
    double *pinned = nullptr;
    double *eout = nullptr;
    RunCtl *ctl_host = nullptr;
    ClState *cs_host = nullptr;
    double *hist_t_host = nullptr;   // step history, written by the device (Ens::hist_t): a
    uint32_t *hist_n_host = nullptr; // copy of it after each chunk took 5 us and a gap
    uint32_t *team_plan_host = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    bool graphs = true;          // device loops replay captured chunks
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    double *dl_pin = nullptr;    // pinned slots of downloads (download_rows), made by the first
    size_t dl_len = 0;           // one that needs them: doubles
    hipEvent_t dl_ev[DL_SLOTS] = {};
    Soa s{};
    Ens e{};
    h4h_stats stats{};
    uint64_t team_steps = 0;     // block steps made by k_team_run
    uint64_t team_rest = 0;      // coming steps it leaves alone, since its workgroups were
                                 // not all running,
    uint32_t team_fails = 0;     // so many times in a row (team_backoff)
};

namespace {

int check_ctx(h4h_ctx *ctx, bool need_upload = true) {
    if (!ctx) return fail(H4H_EINVAL, "null context");
    if (need_upload && !ctx->uploaded)
        return fail(H4H_ESTATE, "no state uploaded (call h4h_upload first)");
    return H4H_OK;
}

int check_single(h4h_ctx *ctx) {
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (ctx->K != 1)
        return fail(H4H_EINVAL, "this call acts on one system; use the h4h_ensemble_* calls");
    return H4H_OK;
}

uint32_t blocks_for(size_t n) { return (uint32_t)((n + BS - 1) / BS); }

// Largest number of update work items any active-set size can produce for
// one cluster of n particles (the persistent grid of a single-system
// context is capped by it, so small systems do not launch idle
// workgroups).
uint32_t max_items(uint32_t n, uint32_t grid, uint32_t max_split, uint32_t fill16) {
    uint32_t n_jt = (n + JT - 1) / JT;
    uint32_t best = 1;
    for (uint32_t nact = 1;; nact = (nact < 64 ? nact + 1 : nact * 2)) {
        uint32_t k = nact > n ? n : nact;
        // (narrower groups make at least as many items)
        const LaneGroup lg = lane_group(k, fill16, std::min(n_jt, max_split), false);
        best = std::max(best, decompose(k, lg.iw, n_jt, grid, max_split).n_items);
        if (nact >= n) break;
    }
    return best;
}

void drop_graph(h4h_ctx *ctx) {
    if (ctx->graph_exec) (void)hipGraphExecDestroy(ctx->graph_exec);
    if (ctx->graph) (void)hipGraphDestroy(ctx->graph);
    ctx->graph_exec = nullptr;
    ctx->graph = nullptr;
}

// A single system of 5 to TEAM_TILES j tiles makes its small steps in
// k_team_run.  Fewer tiles: k_small_run, whose one workgroup needs no
// exchange.  More: a tile per workgroup would not leave every workgroup a CU.
bool team_size(const h4h_ctx *ctx) { return ctx->K == 1 && ctx->nblk > 4 && ctx->nblk <= TEAM_TILES; }

uint32_t team_act(const h4h_ctx *ctx) { return team_act(ctx->nblk > TEAM_ONE ? 2u : 1u); }

auto *team_kernel(bool two, bool mixed, bool one) {
    return one ? (two ? (mixed ? k_team_run<true, 2, true> : k_team_run<false, 2, true>)
                      : (mixed ? k_team_run<true, 1, true> : k_team_run<false, 1, true>))
               : (two ? (mixed ? k_team_run<true, 2, false> : k_team_run<false, 2, false>)
                      : (mixed ? k_team_run<true, 1, false> : k_team_run<false, 1, false>));
}
uint32_t team_wgs(uint32_t nblk) { return nblk > TEAM_ONE ? (nblk + 1) / 2 : nblk; }

// Whether all workgroups of a team of the context's size can run at once on
// the device (one per CU at least, so a full MI355X holds any; a partition
// of it may not).
bool team_fits(const h4h_ctx *ctx) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess)
        return false;
    for (uint32_t k = 0; k < 4; ++k) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, team_kernel(ctx->nblk > TEAM_ONE, k & 1, k & 2), TB, 0) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        if ((uint64_t)per_cu * cus < team_wgs(ctx->nblk)) return false;
    }
    return true;
}

// The plans of the active counts a team takes (0: not one chunk per tile,
// or a tuning table is set).
int configure_team(h4h_ctx *ctx) {
    if (!ctx->team_ok) return H4H_OK;
    for (uint32_t k = 0; k <= team_act(ctx); ++k) {
        uint32_t plan = 0;
        if (k >= 1 && k <= ctx->n && !ctx->e.tuned) {
            const LaneGroup lg = lane_group(k, ctx->iw_fill, std::min(ctx->nblk, ctx->max_split),
                                            ctx->precision == H4H_MIXED);
            const Decomp d = decompose(k, lg.iw, ctx->nblk, ctx->e.grid, ctx->max_split);
            if (lg.iw <= 64 && !lg.jrun && d.S == ctx->nblk)
                plan = (uint32_t)__builtin_ctz(lg.iw) |
                       (uint32_t)__builtin_ctz(finish_lanes(d.S, k)) << 16;
        }
        ctx->team_plan_host[k] = plan;
    }
    H4H_HIP(hipMemcpyAsync(const_cast<uint32_t *>(ctx->team.plan), ctx->team_plan_host,
                           (team_act(ctx) + 1) * sizeof(uint32_t), hipMemcpyHostToDevice,
                           ctx->stream));
    return H4H_OK;
}

// (Re)sizes the j-split partials for the current grid and updates the
// launch fields of the cluster table.
int configure_launch(h4h_ctx *ctx) {
    uint32_t g = ctx->grid;
    if (ctx->K == 1)
        g = std::min(g, max_items(ctx->cnt[0], ctx->grid, ctx->max_split, ctx->iw_fill));
    ctx->e.grid = g;
    // queue target of the plans: an upper bound of their work items
    const uint32_t target = ctx->grid * QUEUE_FACTOR;
    ctx->e.max_split = ctx->max_split;
    ctx->e.iw_fill = ctx->iw_fill;
    drop_graph(ctx);
    int rc = configure_team(ctx);
    if (rc) return rc;
    // j-split partials for any plan of any step (partial_bound).
    size_t need;
    if (ctx->K == 1) {
        need = partial_bound(ctx->cnt[0], target);
    } else {
        unsigned long long n_total = 0, per_cluster = 0;
        for (uint32_t c = 0; c < ctx->K; ++c) {
            n_total += ctx->cnt[c];
            per_cluster += partial_bound(ctx->cnt[c], target);
        }
        need = std::min(per_cluster, ensemble_partial_bound(ctx->K, n_total, target));
    }
    if (ctx->partial && ctx->partial_len >= need) return H4H_OK;
    if (ctx->partial) H4H_HIP(hipFree(ctx->partial));
    ctx->partial = nullptr;
    H4H_HIP(hipMalloc(&ctx->partial, need * sizeof(double)));
    ctx->partial_len = need;
    return H4H_OK;
}

uint32_t finish_grid(h4h_ctx *ctx) { return std::min<uint32_t>(1024, std::max<uint32_t>(64, ctx->nblk)); }

// Workgroups of the exact update for up to n active particles: its items
// stride over them, and up to 3 are resident on each CU.
uint32_t exact_grid(uint32_t n) { return std::min<uint32_t>(n, 1024); }

// Pair kernel of the current precision over the plan's items.  compact:
// the step's selection wrote the active particles' records.
int launch_update(h4h_ctx *ctx, bool compact = false) {
    if (ctx->precision == H4H_FP64_EXACT) {
        hipLaunchKernelGGL(k_update_exact, dim3(exact_grid(ctx->n)), dim3(BS), 0, ctx->stream,
                           ctx->s, ctx->e, ctx->move, ctx->e2);
    } else {
        auto *kern = ctx->precision == H4H_MIXED ? k_update_mixed : k_update_fp64;
        hipLaunchKernelGGL(kern, dim3(ctx->e.grid), dim3(BS), 0, ctx->stream, ctx->s, ctx->e,
                           ctx->move, ctx->partial, ctx->e2, compact ? 1u : 0u);
    }
    H4H_LAUNCHED();
    return H4H_OK;
}

int launch_finish(h4h_ctx *ctx) {
    hipLaunchKernelGGL(k_finish, dim3(finish_grid(ctx)), dim3(BS), 0, ctx->stream, ctx->s, ctx->e,
                       ctx->move, ctx->partial);
    H4H_LAUNCHED();
    return H4H_OK;
}

int launch_select(h4h_ctx *ctx, uint32_t flags, double itime, uint32_t par = 0) {
    hipLaunchKernelGGL(k_select, dim3(ctx->nblk), dim3(BS), 0, ctx->stream, ctx->s, ctx->e,
                       flags, itime, par, ctx->move);
    H4H_LAUNCHED();
    return H4H_OK;
}

int launch_plan(h4h_ctx *ctx) {
    hipLaunchKernelGGL(k_plan, dim3(1), dim3(BS), 0, ctx->stream, ctx->e,
                       ctx->precision);
    H4H_LAUNCHED();
    return H4H_OK;
}

// Whether the device can launch k_small_run (SB threads, 157 KiB of LDS).
bool small_fits(int device) {
    int lds = 0;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device) != hipSuccess)
        return false;
    for (const void *k : {reinterpret_cast<const void *>(&k_small_run<false>),
                          reinterpret_cast<const void *>(&k_small_run<true>)}) {
        hipFuncAttributes fa{};
        if (hipFuncGetAttributes(&fa, k) != hipSuccess) return false;
        if (fa.sharedSizeBytes > (size_t)lds || fa.maxThreadsPerBlock < (int)SB) return false;
    }
    return true;
}

// Device loops of this context start each step slot with k_small_run: every
// cluster has at most SN particles.  (With larger clusters beside them, the
// small clusters' runs of up to SMALL_RUN steps would hold up the larger
// clusters' steps, which wait for the launch to end.)
bool small_path(const h4h_ctx *ctx) {
    return ctx->small_ok && ctx->small_act > 0 && ctx->precision != H4H_FP64_EXACT &&
           *std::max_element(ctx->cnt.begin(), ctx->cnt.end()) <= SN;
}

// Whether the pair loop of `precision` may add a particle's pair with itself
// (r = 0, v = 0) untested: its weight 3 sqrt(3) m / r^3 at r^2 = e2 (FP64;
// m / r^3 in FP32 for the mixed kernel) must be finite for the largest
// float mass mmax of the context, and e2 inside the range where the
// hardware rsqrt (refined in FP64) keeps its accuracy.  Then the pair's terms are
// finite times zero, exact zeros.  mmax is +inf when a mass is not finite.
bool self_pair_is_zero(int precision, double e2, double mmax) {
    if (precision == H4H_MIXED) {
        const float e2f = (float)e2;
        return e2f >= 0x1p-60f && mmax * std::pow((double)e2f, -1.5) < 0x1p120;
    }
    return e2 >= 0x1p-600 && mmax * std::pow(e2, -1.5) < 0x1p1016;
}

// One workgroup per cluster.
int launch_small(h4h_ctx *ctx, uint32_t max_run, uint32_t par, OneStep one = {}) {
    auto *kern = ctx->precision == H4H_MIXED ? k_small_run<true> : k_small_run<false>;
    hipLaunchKernelGGL(kern, dim3(ctx->K), dim3(SB), 0, ctx->stream, ctx->s, ctx->e, max_run,
                       ctx->small_act, ctx->e2, (double)ctx->eta, ctx->dt_min, ctx->dt_max,
                       self_pair_is_zero(ctx->precision, ctx->e2, ctx->mass_max) ? 1u : 0u, par,
                       ctx->move, one);
    H4H_LAUNCHED();
    return H4H_OK;
}

bool team_path(const h4h_ctx *ctx) {
    return ctx->team_ok && !ctx->e.tuned && ctx->precision != H4H_FP64_EXACT;
}

int launch_team(h4h_ctx *ctx, uint32_t max_run, OneStep one = {}) {
    auto *kern = team_kernel(ctx->nblk > TEAM_ONE, ctx->precision == H4H_MIXED, one.host != nullptr);
    hipLaunchKernelGGL(kern, dim3(team_wgs(ctx->nblk)), dim3(TB), 0, ctx->stream,
                       ctx->s, ctx->e, ctx->team, max_run, ctx->e2, (double)ctx->eta, ctx->dt_min,
                       ctx->dt_max, one);
    H4H_LAUNCHED();
    return H4H_OK;
}

// After a loop's (or one step's) state is read back: whether a wait inside a
// team ran out (the state is then between two steps).
int check_team(h4h_ctx *ctx, bool failed) {
    if (!failed) return H4H_OK;
    ctx->team_ok = false;
    drop_graph(ctx);
    return fail(H4H_EHIP, "a wait between workgroups ran out; upload the state again");
}

// The result of h4h_step's launches: when it is in the pinned record, or
// (with timing events, or if it does not come soon) after them.
int await_step(h4h_ctx *ctx) {
    if (!ctx->timing) {
        const uint32_t *done = &ctx->cs_host[0].done;
        const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
        do {
            for (int k = 0; k < 64; ++k) {
                if (__atomic_load_n(done, __ATOMIC_ACQUIRE)) return H4H_OK;
                __builtin_ia32_pause();
            }
        } while (std::chrono::steady_clock::now() < until);
    }
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    return H4H_OK;
}

int ensure_blockmin(h4h_ctx *ctx) {
    if (ctx->bm_valid) return H4H_OK;
    hipLaunchKernelGGL(k_blockmin_all, dim3(std::min<uint32_t>(ctx->nblk, 1024)), dim3(BS), 0,
                       ctx->stream, ctx->s, ctx->e);
    H4H_LAUNCHED();
    ctx->bm_valid = true;
    return H4H_OK;
}

// One block step of every live cluster, device-driven: selection with the
// fused predictor and save-old (after the loop tail of each cluster's last
// step), work plan, update, finish (chunk sums + corrector) and the
// per-block minima of the touched blocks; each cluster's loop tail is made
// by the next launch that needs its next block time (the next step's
// selection, k_small_run, or k_tail after h4h_step), so in a device loop
// that ends, the step after the last one finds the loop stopped.  One
// system: three launches (its update makes its own plan); an ensemble: four,
// or five (finish_by_blocks).
// par: the step's slot in its captured chunk, mod 2 (its dirty list); select
// false: k_small_run has made the selection.  Optional HIP events bracket the update kernel.
int enqueue_step(h4h_ctx *ctx, bool events, uint32_t par, bool select = true) {
    int rc;
    if (select &&
        (rc = launch_select(ctx,
                            PS_PREDICT | PS_SELECT | PS_SAVE_OLD | PS_DEVTIME | PS_DIRTY | PS_TAIL |
                                PS_COMPACT,
                            0.0, par)))
        return rc;
    // (a single-system context's update kernel makes its own plan)
    if (ctx->K > 1 && (rc = launch_plan(ctx))) return rc;
    if (events) H4H_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
    if ((rc = launch_update(ctx, true))) return rc;
    if (events) H4H_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
    const dim3 grid(std::min<uint32_t>(ctx->nblk, 1024));
    if (!finish_by_blocks(ctx->K, ctx->nblk)) {
        hipLaunchKernelGGL(k_finish_correct, dim3(finish_grid(ctx)), dim3(BS), 0, ctx->stream,
                           ctx->s, ctx->e, ctx->move, ctx->partial, ctx->eta, ctx->dt_min,
                           ctx->dt_max);
        H4H_LAUNCHED();
        hipLaunchKernelGGL(k_blockmin_dirty, grid, dim3(BS), 0, ctx->stream, ctx->s, ctx->e, par);
    } else {
        hipLaunchKernelGGL(ctx->K == 1 ? k_finish_blocks<true> : k_finish_blocks<false>, grid,
                           dim3(BS), 0, ctx->stream, ctx->s, ctx->e, ctx->move, ctx->partial,
                           ctx->eta, ctx->dt_min, ctx->dt_max, par);
    }
    H4H_LAUNCHED();
    return H4H_OK;
}

// One chunk of the device loop: RUN_CHUNK block steps, or for a small or
// mid-size system SMALL_SLOTS slots of k_small_run or k_team_run (up to
// SMALL_RUN steps with small active sets) followed by one block step of the
// multi-workgroup kernels (the step it left, if any).  At most HIST_CAP steps.
int enqueue_chunk(h4h_ctx *ctx) {
    int rc = H4H_OK;
    const bool small = small_path(ctx);
    if (small || team_path(ctx)) {
        for (uint32_t k = 0; k < SMALL_SLOTS && rc == H4H_OK; ++k) {
            rc = small ? launch_small(ctx, SMALL_RUN, k & 1) : launch_team(ctx, SMALL_RUN);
            if (rc == H4H_OK) rc = enqueue_step(ctx, false, k & 1, !small);
        }
    } else {
        for (uint32_t k = 0; k < RUN_CHUNK && rc == H4H_OK; ++k) rc = enqueue_step(ctx, false, k & 1);
    }
    return rc;
}

// Captures one chunk into a graph (once per configuration).  The graph
// holds kernel nodes only.
int ensure_graph(h4h_ctx *ctx) {
    if (ctx->graph_exec) return H4H_OK;
    H4H_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    int rc = enqueue_chunk(ctx);
    hipGraph_t g = nullptr;
    hipError_t err = hipStreamEndCapture(ctx->stream, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (err != hipSuccess)
        return fail(H4H_EHIP, std::string("graph capture: ") + hipGetErrorString(err));
    ctx->graph = g;
    H4H_HIP(hipGraphInstantiate(&ctx->graph_exec, ctx->graph, nullptr, nullptr, 0));
    return H4H_OK;
}

// (The loop control and the cluster states are neighbours, on the device and
// in the pinned mirror: one copy.)
int read_state(h4h_ctx *ctx) {
    H4H_HIP(hipMemcpyAsync(ctx->ctl_host, ctx->d_ctl, sizeof(RunCtl) + ctx->K * sizeof(ClState),
                           hipMemcpyDeviceToHost, ctx->stream));
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    return H4H_OK;
}

// Update pass of the single-method calls (plan already on the device).
int update_pass(h4h_ctx *ctx) {
    if (ctx->timing) H4H_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
    int rc = launch_update(ctx);
    if (rc) return rc;
    if (ctx->timing) H4H_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
    if ((rc = launch_finish(ctx))) return rc;
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    if (ctx->timing) {
        float ms = 0.f;
        H4H_HIP(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
        ctx->stats.update_ms += ms;
        ctx->stats.update_launches += 1;
    }
    return H4H_OK;
}

int upload_cols(h4h_ctx *ctx, const double *src, uint32_t ncols, Cols dst) {
    H4H_HIP(hipMemcpyAsync(ctx->staging, src, (size_t)ctx->n * ncols * sizeof(double),
                           hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_aos_to_soa, dim3(blocks_for(ctx->n_dev)), dim3(BS), 0, ctx->stream,
                       ctx->staging, ncols, dst, ctx->e);
    H4H_LAUNCHED();
    return H4H_OK;
}

int download_cols(h4h_ctx *ctx, double *dst, uint32_t ncols, Cols src) {
    hipLaunchKernelGGL(k_soa_to_aos, dim3(blocks_for(ctx->n_dev)), dim3(BS), 0, ctx->stream, src,
                       ncols, ctx->staging, ctx->e);
    H4H_LAUNCHED();
    H4H_HIP(hipMemcpyAsync(dst, ctx->staging, (size_t)ctx->n * ncols * sizeof(double),
                           hipMemcpyDeviceToHost, ctx->stream));
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    return H4H_OK;
}

// `slots` slots of `len` doubles; false: not to be had, with the error cleared.
bool make_slots(h4h_ctx *ctx, uint32_t slots, size_t len) {
    for (uint32_t k = 0; k < slots; ++k) {
        hipEvent_t &ev = ctx->dl_ev[k];
        if (!ev && hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
            ev = nullptr;
            (void)hipGetLastError();
            return false;
        }
    }
    if (ctx->dl_len >= slots * len) return true;
    if (ctx->dl_pin) (void)hipHostFree(ctx->dl_pin);  // (no download is under way)
    ctx->dl_len = slots * len;
    if (hipHostMalloc((void **)&ctx->dl_pin, ctx->dl_len * sizeof(double)) != hipSuccess) {
        ctx->dl_pin = nullptr;
        ctx->dl_len = 0;
        (void)hipGetLastError();
        return false;
    }
    return true;
}

// The doubles of t (t.at[t.n] of them) to the arrays dst, slot by slot: each
// thread takes the next piece that nobody has, has the device write it, and
// copies it on while the device writes its other slot.  The caller is one of
// the threads, so that the call ends without the others too.
int download_rows(h4h_ctx *ctx, const RowArrays &t, double *const *dst, uint32_t threads,
                  uint32_t size) {
    const unsigned long long total = t.at[t.n], pieces = (total + size - 1) / size;
    std::atomic<unsigned long long> next{0};
    std::atomic<int> err{(int)hipSuccess};
    auto work = [&](uint32_t w) {
        unsigned long long piece[2];
        auto slot = [&](uint32_t k) { return ctx->dl_pin + (size_t)(2 * w + k) * size; };
        auto length = [&](unsigned long long p) {
            return (uint32_t)std::min<unsigned long long>(size, total - p * size);
        };
        auto check = [&](hipError_t rc) {
            if (rc != hipSuccess) err = (int)rc;
            return rc == hipSuccess;
        };
        auto issue = [&](uint32_t k) {
            piece[k] = err == (int)hipSuccess ? next.fetch_add(1) : pieces;
            if (piece[k] >= pieces) return;
            const uint32_t len = length(piece[k]);
            hipLaunchKernelGGL(k_rows_out, dim3(blocks_for(len)), dim3(BS), 0, ctx->stream,
                               ctx->s.r[0], t, ctx->e, piece[k] * size, len, slot(k));
            check(hipGetLastError());
            check(hipEventRecord(ctx->dl_ev[2 * w + k], ctx->stream));
        };
        if (w && !check(hipSetDevice(ctx->device))) return;
        issue(0);
        issue(1);
        for (uint32_t k = 0; piece[k] < pieces; k ^= 1) {
            if (!check(hipEventSynchronize(ctx->dl_ev[2 * w + k])) || err != (int)hipSuccess) return;
            const unsigned long long b = piece[k] * size, end = b + length(piece[k]);
            for (uint32_t a = 0; a < t.n; ++a) {
                const unsigned long long lo = std::max(b, t.at[a]), hi = std::min(end, t.at[a + 1]);
                if (lo < hi)
                    std::memcpy(dst[a] + (lo - t.at[a]), slot(k) + (lo - b), (hi - lo) * sizeof(double));
            }
            issue(k);
        }
    };
    std::thread th[DL_THREADS];
    try {
        for (uint32_t w = 1; w < threads; ++w) th[w] = std::thread(work, w);
    } catch (...) {  // fewer threads
    }
    work(0);
    for (std::thread &x : th)
        if (x.joinable()) x.join();
    if (err != (int)hipSuccess) {
        (void)hipStreamSynchronize(ctx->stream);
        H4H_HIP((hipError_t)err.load());
    }
    return H4H_OK;
}

int upload_scalar(h4h_ctx *ctx, const double *src, double *dst) {
    H4H_HIP(hipMemcpyAsync(ctx->staging, src, (size_t)ctx->n * sizeof(double),
                           hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_scalar_to_soa, dim3(blocks_for(ctx->n_dev)), dim3(BS), 0, ctx->stream,
                       ctx->staging, dst, ctx->e);
    H4H_LAUNCHED();
    return H4H_OK;
}

int download_scalar(h4h_ctx *ctx, const double *src, double *dst) {
    hipLaunchKernelGGL(k_soa_to_scalar, dim3(blocks_for(ctx->n_dev)), dim3(BS), 0, ctx->stream,
                       src, ctx->staging, ctx->e);
    H4H_LAUNCHED();
    H4H_HIP(hipMemcpyAsync(dst, ctx->staging, (size_t)ctx->n * sizeof(double),
                           hipMemcpyDeviceToHost, ctx->stream));
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    return H4H_OK;
}

bool valid_precision(int p) { return p == H4H_FP64 || p == H4H_FP64_EXACT || p == H4H_MIXED; }

// Workgroup sums the energy buffer of a context holds: one system's, or
// ENERGY_OUT for an ensemble.
size_t eout_len(const h4h_ctx *ctx) {
    return ctx->K > 1 ? ENERGY_OUT : energy_items(ctx->cnt[0]).wgs;
}

// Energies of clusters c0 .. c0 + count - 1, in launches of as many
// clusters as fit the sums of eout (64 clusters of 1024 to 32768 particles:
// 4 launches; 48, each waited for, with a buffer for one system's
// workgroups), then per cluster a host Neumaier sum of its workgroup sums
// in order.  The workgroups write their sums, 32 bytes each, to the pinned
// host buffer themselves, which takes no copy call.
int energies_of(h4h_ctx *ctx, uint32_t c0, uint32_t count, double *ekin, double *epot) {
    // Neumaier sum of the per-workgroup (sum, compensation) pairs (an
    // infinite sum leaves the compensation alone, as on the device).
    auto add = [](double &s, double &c2, double x) {
        double t = s + x;
        if (std::isfinite(t)) {
            if (std::fabs(s) >= std::fabs(x))
                c2 += (s - t) + x;
            else
                c2 += (x - t) + s;
        }
        s = t;
    };
    auto wgs = [&](uint32_t c) { return energy_items(ctx->cnt[c]).wgs; };
    const size_t most = eout_len(ctx);
    for (uint32_t b0 = c0; b0 < c0 + count;) {
        uint32_t gx = wgs(b0), kb = 1;
        while (b0 + kb < c0 + count) {
            const uint32_t g2 = std::max(gx, wgs(b0 + kb));
            if ((uint64_t)(kb + 1) * g2 > most) break;
            gx = g2;
            ++kb;
        }
        hipLaunchKernelGGL(k_energy, dim3(gx, kb), dim3(BS), 0, ctx->stream, ctx->s, ctx->d_off,
                           ctx->d_cnt, b0, ctx->eout);
        H4H_LAUNCHED();
        H4H_HIP(hipStreamSynchronize(ctx->stream));
        for (uint32_t k = 0; k < kb; ++k) {
            double sp = 0.0, cp = 0.0, sk = 0.0, ck = 0.0;
            const double *hk = ctx->eout + (size_t)k * gx * 4;
            for (uint32_t b = 0; b < wgs(b0 + k); ++b) {
                add(sp, cp, hk[4 * b + 0]);
                add(sp, cp, hk[4 * b + 1]);
                add(sk, ck, hk[4 * b + 2]);
                add(sk, ck, hk[4 * b + 3]);
            }
            if (ekin) ekin[b0 - c0 + k] = sk + ck;
            if (epot) epot[b0 - c0 + k] = sp + cp;
        }
        b0 += kb;
    }
    return H4H_OK;
}

int create_impl(h4h_ctx **out, uint32_t K, const uint32_t *sizes, double e2, float eta,
                double dt_min, double dt_max, int precision) {
    if (!out) return fail(H4H_EINVAL, "out is null");
    *out = nullptr;
    if (K < 1 || !sizes) return fail(H4H_EINVAL, "need at least one cluster");
    if (K > (1u << 20)) return fail(H4H_EINVAL, "too many clusters");
    uint64_t total = 0, total_dev = 0;
    for (uint32_t c = 0; c < K; ++c) {
        if (sizes[c] < 1) return fail(H4H_EINVAL, "every cluster needs n >= 1");
        total += sizes[c];
        total_dev += (sizes[c] + JT - 1) / JT * JT;
    }
    if (total_dev > (1u << 30)) return fail(H4H_EINVAL, "n too large");
    if (!(e2 >= 0.0) || !std::isfinite(e2)) return fail(H4H_EINVAL, "e2 must be finite and >= 0");
    if (!(eta > 0.0f) || !std::isfinite(eta)) return fail(H4H_EINVAL, "eta must be > 0");
    if (!(dt_min > 0.0) || !(dt_max >= dt_min) || !std::isfinite(dt_max))
        return fail(H4H_EINVAL, "need 0 < dt_min <= dt_max");
    if (!valid_precision(precision)) return fail(H4H_EINVAL, "unknown precision");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return fail(H4H_ENODEV, "no HIP device available");

    h4h_ctx *ctx = new (std::nothrow) h4h_ctx();
    if (!ctx) return fail(H4H_ENOMEM, "host allocation failed");
    ctx->K = K;
    ctx->n = (uint32_t)total;
    ctx->n_dev = (uint32_t)total_dev;
    ctx->nblk = ctx->n_dev / JT;
    ctx->e2 = e2;
    ctx->eta = eta;
    ctx->dt_min = dt_min;
    ctx->dt_max = dt_max;
    ctx->precision = precision;
    ctx->off.resize(K);
    ctx->cnt.resize(K);
    ctx->hoff.resize(K);
    std::vector<uint32_t> bcl(ctx->nblk);
    uint32_t o = 0, h = 0;
    for (uint32_t c = 0; c < K; ++c) {
        ctx->off[c] = o;
        ctx->cnt[c] = sizes[c];
        ctx->hoff[c] = h;
        uint32_t nb = (sizes[c] + JT - 1) / JT;
        for (uint32_t b = 0; b < nb; ++b) bcl[o / JT + b] = c;
        o += nb * JT;
        h += sizes[c];
    }

    auto cleanup = [&](int rc) {
        std::string keep = g_err;
        h4h_destroy(ctx);
        g_err = keep;
        return rc;
    };
    if (hipGetDevice(&ctx->device) != hipSuccess) return cleanup(fail(H4H_EHIP, "hipGetDevice failed"));
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess)
        return cleanup(fail(H4H_EHIP, "hipStreamCreate failed"));
    size_t np = ctx->n_dev;
    ctx->team_ok = team_size(ctx) && team_fits(ctx);
    const size_t tm_hdr = 3 * (size_t)ctx->nblk * 8,
                 tm_rec = 3 * (size_t)ctx->nblk * 8 * team_act(ctx),
                 tm_part = (size_t)ctx->nblk * team_act(ctx) * 6, tm_words = tm_hdr + tm_rec + tm_part,
                 tm_plan = TS_WORDS + team_act(ctx) + 2;  // u32
    const size_t team_bytes =
        ctx->team_ok ? tm_words * sizeof(double) + tm_plan * sizeof(uint32_t) : 0;
    // One device allocation for everything but the partials (17 of them took
    // half of the time of a small context's creation); what starts at zero is
    // at its front, the four cluster tables are neighbours.
    struct Piece {
        void **p;
        size_t bytes;
    };
    const size_t tables = 3 * (size_t)K + ctx->nblk;
    const Piece pieces[] = {
        {(void **)&ctx->d_ctl, sizeof(RunCtl) + K * sizeof(ClState)},
        {(void **)&ctx->d_tune, 64 * sizeof(uint32_t)},
        {(void **)&ctx->d_pre, 3 * (size_t)(K + 1) * sizeof(unsigned long long)},
        {(void **)&ctx->state, np * N_SOA * sizeof(double)},
        {(void **)&ctx->staging, (size_t)ctx->n * 8 * sizeof(double)},
        {(void **)&ctx->move, np * sizeof(uint32_t)},
        {(void **)&ctx->d_off, tables * sizeof(uint32_t)},
        {(void **)&ctx->d_plan, K * sizeof(ClPlan)},
        {(void **)&ctx->d_dirty, 6 * (size_t)ctx->nblk * sizeof(uint32_t)},
        {(void **)&ctx->d_bmin, ctx->nblk * (sizeof(double) + sizeof(uint32_t))},
        {(void **)&ctx->d_arec, 4 * np * sizeof(double4) + team_bytes},
    };
    size_t bytes = 0, zeroed = 0;
    for (const Piece &x : pieces) {
        bytes += (x.bytes + 255) / 256 * 256;
        if (x.p == (void **)&ctx->state) zeroed = bytes;
    }
    if (hipMalloc(&ctx->arena, bytes) != hipSuccess)
        return cleanup(fail(H4H_ENOMEM, "device allocation failed"));
    bytes = 0;
    for (const Piece &x : pieces) {
        *x.p = ctx->arena + bytes;
        bytes += (x.bytes + 255) / 256 * 256;
    }
    ctx->d_cnt = ctx->d_off + K;
    ctx->d_hoff = ctx->d_cnt + K;
    ctx->d_bcl = ctx->d_hoff + K;
    ctx->d_cs = reinterpret_cast<ClState *>(ctx->d_ctl + 1);
    // One pinned allocation for all host mirrors (each costs ~0.2 ms).
    static_assert(sizeof(RunCtl) % 8 == 0 && sizeof(ClState) % 8 == 0, "carved in doubles");
    const size_t eo = eout_len(ctx) * 4, ct = sizeof(RunCtl) / 8, cst = K * sizeof(ClState) / 8;
    const size_t pl = team_act(ctx) / 2 + 1;
    if (hipHostMalloc(&ctx->pinned, (eo + ct + cst + HIST_CAP + HIST_CAP / 2 + pl) * sizeof(double),
                      hipHostMallocDefault) != hipSuccess)
        return cleanup(fail(H4H_ENOMEM, "pinned allocation failed"));
    ctx->eout = ctx->pinned;
    ctx->ctl_host = reinterpret_cast<RunCtl *>(ctx->eout + eo);
    ctx->cs_host = reinterpret_cast<ClState *>(ctx->eout + eo + ct);
    ctx->hist_t_host = ctx->eout + eo + ct + cst;
    ctx->hist_n_host = reinterpret_cast<uint32_t *>(ctx->hist_t_host + HIST_CAP);
    ctx->team_plan_host = ctx->hist_n_host + HIST_CAP;
    for (int k = 0; k < 4; ++k)
        if (hipEventCreate(&ctx->ev[k]) != hipSuccess)
            return cleanup(fail(H4H_EHIP, "hipEventCreate failed"));
    std::vector<uint32_t> tab(ctx->off);
    tab.insert(tab.end(), ctx->cnt.begin(), ctx->cnt.end());
    tab.insert(tab.end(), ctx->hoff.begin(), ctx->hoff.end());
    tab.insert(tab.end(), bcl.begin(), bcl.end());
    bool ok = hipMemcpyAsync(ctx->d_off, tab.data(), tables * sizeof(uint32_t),
                             hipMemcpyHostToDevice, ctx->stream) == hipSuccess &&
              hipMemsetAsync(ctx->arena, 0, zeroed, ctx->stream) == hipSuccess;
    if (!ok) return cleanup(fail(H4H_EHIP, "initialisation failed"));

    Ens &e = ctx->e;
    e.K = K;
    e.nblk = ctx->nblk;
    e.off = ctx->d_off;
    e.cnt = ctx->d_cnt;
    e.hoff = ctx->d_hoff;
    e.bcl = ctx->d_bcl;
    e.cs = ctx->d_cs;
    e.plan = ctx->d_plan;
    e.items_pre = ctx->d_pre;
    e.fin_pre = ctx->d_pre + (K + 1);
    e.part_pre = ctx->d_pre + 2 * (size_t)(K + 1);
    e.ctl = ctx->d_ctl;
    e.dirty = ctx->d_dirty;
    e.bmin = ctx->d_bmin;
    e.bcnt = reinterpret_cast<uint32_t *>(ctx->d_bmin + ctx->nblk);
    e.arec = ctx->d_arec;
    e.hist_t = ctx->hist_t_host;
    e.hist_n = ctx->hist_n_host;
    e.hist_cap = HIST_CAP;
    e.tuned = 0;
    e.tune = ctx->d_tune;
    if (ctx->team_ok) {
        unsigned long long *tb = reinterpret_cast<unsigned long long *>(ctx->d_arec + 4 * np);
        Team &tm = ctx->team;
        tm.hdr = tb;
        tm.rec = tb + tm_hdr;
        tm.part = tb + tm_hdr + tm_rec;
        tm.sync = reinterpret_cast<uint32_t *>(tb + tm_words);
        tm.plan = tm.sync + TS_WORDS;
        hipLaunchKernelGGL(k_team_clear, dim3(256), dim3(BS), 0, ctx->stream, tm, tm_words);
        if (hipGetLastError() != hipSuccess) return cleanup(fail(H4H_EHIP, "kernel launch"));
    }
    int rc = configure_launch(ctx);
    if (rc) return cleanup(rc);
    ctx->small_ok = small_fits(ctx->device);
    // An ensemble's other clusters keep the rest of the chip busy, so a
    // larger step in a cluster's own workgroup costs the others nothing.
    ctx->small_act = K > 1 ? SMALL_MAX_ACT : SMALL_ACT;

    double *b = ctx->state;
    Soa &s = ctx->s;
    auto take = [&]() {
        double *p = b;
        b += np;
        return p;
    };
    for (int c = 0; c < 3; ++c) s.r[c] = take();
    s.m = take();
    for (int c = 0; c < 3; ++c) s.v[c] = take();
    for (int c = 0; c < 6; ++c) s.f[c] = take();
    for (int c = 0; c < 6; ++c) s.old[c] = take();
    for (int c = 0; c < 3; ++c) s.a2[c] = take();
    for (int c = 0; c < 3; ++c) s.a3[c] = take();
    s.t = take();
    s.dt = take();
    s.pp = reinterpret_cast<double4 *>(take());  // 4 columns each
    for (int c = 0; c < 3; ++c) (void)take();
    s.pv = reinterpret_cast<double4 *>(take());
    for (int c = 0; c < 3; ++c) (void)take();
    if (b != ctx->state + (size_t)np * N_SOA || s.v[0] != s.r[0] + COL_V * np ||
        s.f[0] != s.r[0] + COL_F * np || s.old[0] != s.r[0] + COL_OLD * np ||
        s.a2[0] != s.r[0] + COL_A2 * np || s.a3[0] != s.r[0] + COL_A3 * np ||
        s.t != s.r[0] + COL_T * np || s.dt != s.r[0] + COL_DT * np)
        return cleanup(fail(H4H_EINVAL, "state layout"));
    ok = hipStreamSynchronize(ctx->stream) == hipSuccess;
    if (!ok) return cleanup(fail(H4H_EHIP, "initialisation failed"));
    *out = ctx;
    return H4H_OK;
}

// ---------------------------------------------------------------------------
// Context-free update with a static device buffer (h4h_update_acc_jrk_static)
// ---------------------------------------------------------------------------
//
// Everything the update and finish kernels need beyond the caller's inputs
// and outputs lives in `scratch`, one file-scope device array per GPU (the
// loader gives each device its own copy): tables of one cluster, the
// active list (range-checked copy), the predictor records and the forces in
// the kernels' layouts, and the j-split partial sums.  Offsets in doubles,
// each a multiple of 32 (256 bytes).
//
// Partial sums: for n <= STATIC_MAX_N with the default launch (grid <= 2048
// workgroups, queue target 16 items per workgroup, at most 256 i slots per
// item), a plan with S > 1 chunks has S <= max(s_fill, s_tiles) where
// s_fill = ceil(grid / n_it) and s_tiles = floor(n_jt / CHUNK_TILES) <= 16
// (n_jt <= 256, so the large-set chunk rule does not apply):
// S n_it iw <= (grid + n_it - 1) iw <= grid BS + n + BS - 1 in the first
// case and S rows <= 16 (n + BS - 1) in the second, so 6 S rows <=
// ST_PART doubles.  The call also checks its own plan against ST_PART.
constexpr uint32_t STATIC_MAX_N = 65536;
static_assert(STATIC_MAX_N == H4H_STATIC_MAX_N, "header and library agree");
constexpr size_t st_round32(size_t x) { return (x + 31) / 32 * 32; }
constexpr size_t ST_PART_ROWS_FILL = (size_t)DEFAULT_GRID * BS + STATIC_MAX_N + BS - 1;
constexpr size_t ST_PART_ROWS_TILES =
    (size_t)(STATIC_MAX_N / JT / CHUNK_TILES) * (STATIC_MAX_N + BS - 1);
constexpr size_t ST_PART =
    st_round32(6 * (ST_PART_ROWS_FILL > ST_PART_ROWS_TILES ? ST_PART_ROWS_FILL : ST_PART_ROWS_TILES));
constexpr size_t ST_CTL = 0, ST_CS = 16, ST_PLAN = 32, ST_PRE = 40, ST_TAB = 48, ST_BAD = 64;  // header
constexpr size_t ST_MOVE = 128;                                   // u32 x STATIC_MAX_N
constexpr size_t ST_PP = ST_MOVE + STATIC_MAX_N / 2;              // double4 x STATIC_MAX_N
constexpr size_t ST_PV = ST_PP + 4 * (size_t)STATIC_MAX_N;
constexpr size_t ST_F = ST_PV + 4 * (size_t)STATIC_MAX_N;         // 6 columns
constexpr size_t ST_PARTIAL = ST_F + 6 * (size_t)STATIC_MAX_N;
constexpr size_t ST_TOTAL = ST_PARTIAL + ST_PART;
static_assert(ST_TOTAL * sizeof(double) == H4H_STATIC_SCRATCH_BYTES, "header states the size");
static_assert(sizeof(RunCtl) <= 16 * sizeof(double) && sizeof(ClState) <= 16 * sizeof(double) &&
                  sizeof(ClPlan) <= 8 * sizeof(double),
              "header block of the static buffer");
static_assert(ST_MOVE % 32 == 0 && ST_PP % 32 == 0 && ST_PV % 32 == 0 && ST_F % 32 == 0 &&
                  ST_PARTIAL % 32 == 0,
              "256-byte sections");

// ST_TAB holds off, cnt, hoff of the one cluster, ST_BAD whether the list
// held an index >= n, one word for each ST_LIST entries of it.
enum : uint32_t { TAB_OFF = 0, TAB_CNT = 1, TAB_HOFF = 2 };
constexpr uint32_t ST_LIST = 4 * BS;
static_assert(STATIC_MAX_N / ST_LIST <= 64 && ST_BAD + 32 <= ST_MOVE, "a wave reads the words");

// Predictor records of p6 (n x 6: r, v) and pm (float masses).
__device__ __forceinline__ void static_record(const double *p6, const float *pm, uint32_t n,
                                              uint32_t i, double4 &a, double4 &b) {
    if (i < n) {
        const float mf = pm[i];
        const double *p = p6 + (size_t)i * 6;
        a = make_double4(p[0], p[1], p[2], (double)mf);
        b = make_double4(p[3], p[4], p[5], mass_bits(mf));
    } else {
        a = make_double4(PAD_POS, PAD_POS, PAD_POS, 0.0);
        b = make_double4(0.0, 0.0, 0.0, mass_bits(0.0f));
    }
}

// The records in the tile layout, zero-mass padding up to n_pad; the active
// list copied with every index >= n replaced by 0 and flagged; the tables of
// one cluster of n particles with nact active, and the work-queue counters at
// zero.
__global__ __launch_bounds__(BS) void k_static_pack(const double *p6, const float *pm, uint32_t n,
                                                   uint32_t n_pad, const uint32_t *move_in,
                                                   uint32_t nact, uint32_t *move, Soa s, Ens e,
                                                   uint32_t *tab, uint32_t *bad) {
    const uint32_t i = blockIdx.x * BS + threadIdx.x;
    if (i == 0) {
        ClState c{};
        c.nact = nact;
        e.cs[0] = c;
        *e.ctl = RunCtl{};
        tab[TAB_OFF] = 0;
        tab[TAB_CNT] = n;
        tab[TAB_HOFF] = 0;
    }
    if (i < n_pad) {
        double4 a, b;
        static_record(p6, pm, n, i, a, b);
        s.pp[i] = a;
        s.pv[i] = b;
    }
    if (blockIdx.x * ST_LIST < nact) {
        int out = 0;
        for (uint32_t q = 0; q < ST_LIST / BS; ++q) {
            const uint32_t k = blockIdx.x * ST_LIST + q * BS + threadIdx.x;
            if (k >= nact) break;
            const uint32_t j = move_in[k];
            out |= j >= n;
            move[k] = j < n ? j : 0u;
        }
        out = __syncthreads_or(out);
        if (threadIdx.x == 0) bad[blockIdx.x] = out ? 1u : 0u;
    }
}

// The finish pass: chunk sums as k_finish, to rows move_in[k] of f6 (n x 6);
// every row NaN if the list held an index >= n (those indices are skipped).
__global__ __launch_bounds__(BS) void k_static_finish(Soa s, Ens e, const uint32_t *move,
                                                     const double *partial,
                                                     const uint32_t *move_in, uint32_t n,
                                                     uint32_t nact, const uint32_t *bad,
                                                     double *f6) {
    const ClPlan pl = e.plan[0];
    const uint32_t L = pl.lanes, per = BS / L;
    const uint32_t word = __lane_id() * ST_LIST < nact ? bad[__lane_id()] : 0u;
    const bool nan = __ballot(word != 0) != 0;
    for (uint32_t u = blockIdx.x; u * per < nact; u += gridDim.x) {
        const uint32_t k = u * per + threadIdx.x / L;
        const bool valid = k < nact;
        const uint32_t i = valid ? move_in[k] : n;
        double f[6];
        chunk_sums(s, pl, partial, k, i < n ? i : 0u, valid, f);
        if (i < n && threadIdx.x % L == 0)
            for (int q = 0; q < 6; ++q) f6[(size_t)i * 6 + q] = nan ? (double)NAN : f[q];
    }
}

// The whole call in one launch where the plan has one j chunk of at most
// ONE_TILES tiles and at most BS active particles: each workgroup takes IW of
// them (a work item of the plan), reads the particles straight from p6 and pm,
// all tiles at once, and writes its rows, so nothing passes between
// workgroups.  Same tiles, sub-groups and sums as update_item: the same bits.
// Bound by its launch and one trip to memory: n = 1024, nact = 24 takes 10.3 us a
// call in a row (4 of them issuing the pairs) instead of 22.3 with five launches.
constexpr uint32_t ONE_TILES = 4;
template <int IW, bool MIXED>
__device__ __forceinline__ void static_item(const double *p6, const float *pm, uint32_t n,
                                            const uint32_t *move_in, uint32_t nact, double e2,
                                            double *f6, double4 *tiles, double *red) {
    const uint32_t n_jt = (n + JT - 1) / JT;
    const uint32_t mine = threadIdx.x < nact ? move_in[threadIdx.x] : 0u;
    double4 a[ONE_TILES], b[ONE_TILES];
#pragma unroll
    for (uint32_t q = 0; q < ONE_TILES; ++q)
        if (q < n_jt) static_record(p6, pm, n, q * JT + threadIdx.x, a[q], b[q]);
    const uint32_t k = blockIdx.x * IW + threadIdx.x % IW;
    uint32_t i = move_in[k < nact ? k : 0u];
    if (i >= n) i = 0;
    double pi[6];
    for (int q = 0; q < 6; ++q) pi[q] = p6[(size_t)i * 6 + q];
#pragma unroll
    for (uint32_t q = 0; q < ONE_TILES; ++q)
        if (q < n_jt) {
            tiles[2 * JT * q + threadIdx.x] = a[q];
            tiles[2 * JT * q + JT + threadIdx.x] = b[q];
        }
    const bool nan = __syncthreads_or(mine >= n) != 0;
    const uint32_t js = subgroup<IW>(threadIdx.x);
    double fo[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (uint32_t tt = 0; tt < n_jt; ++tt) {
        const double4 *sp = tiles + 2 * JT * tt;
        if (__ballot(i - tt * JT < (uint32_t)JT))
            tile_pairs<IW, true, MIXED, 1>(pi, i, tt * JT, js, sp, sp + JT, e2, fo);
        else
            tile_pairs<IW, false, MIXED, 1>(pi, i, tt * JT, js, sp, sp + JT, e2, fo);
    }
    reduce_subgroups<IW>(fo, red, threadIdx.x);
    constexpr double scale = MIXED ? 1.0 : PAIR_SCALE;
    for (uint32_t x = threadIdx.x; x < 6 * IW; x += BS) {
        const uint32_t sl = x / 6, q = x - 6 * sl, ks = blockIdx.x * IW + sl;
        if (ks >= nact) continue;
        const uint32_t is = move_in[ks];
        if (is >= n) continue;
        double f = red[sl * 6 + q];
        for (uint32_t g = 1; g < BS / 64; ++g) f += red[(g * IW + sl) * 6 + q];
        f *= scale;
        f6[(size_t)is * 6 + q] = nan ? (double)NAN : f;
    }
}
template <bool MIXED>
__global__ __launch_bounds__(BS) void k_static_one(const double *p6, const float *pm, uint32_t n,
                                                  const uint32_t *move_in, uint32_t nact,
                                                  uint32_t iw, double e2, double *f6) {
    __shared__ double4 tiles[2 * JT * ONE_TILES];
    __shared__ double red[6 * BS];
    if (iw == 4)
        static_item<4, MIXED>(p6, pm, n, move_in, nact, e2, f6, tiles, red);
    else if (iw == 16)
        static_item<16, MIXED>(p6, pm, n, move_in, nact, e2, f6, tiles, red);
    else
        static_item<64, MIXED>(p6, pm, n, move_in, nact, e2, f6, tiles, red);
}

}  // namespace

// The static buffer (one per GPU).  Host code uses the device address
// from hipGetSymbolAddress, never this name.
static __device__ __align__(256) double scratch[ST_TOTAL];

namespace {

std::mutex g_static_mu;
constexpr int STATIC_MAX_DEVICES = 256;
double *g_static_ptr[STATIC_MAX_DEVICES] = {};

// Device address of `scratch` on the current device, looked up once per
// device (the first call there).
int static_scratch(double **out) {
    int dev = 0;
    H4H_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= STATIC_MAX_DEVICES) return fail(H4H_ENODEV, "device index out of range");
    std::lock_guard<std::mutex> lock(g_static_mu);
    if (!g_static_ptr[dev]) {
        void *p = nullptr;
        H4H_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(H4H_EHIP, "hipGetSymbolAddress returned null");
        g_static_ptr[dev] = static_cast<double *>(p);
    }
    *out = g_static_ptr[dev];
    return H4H_OK;
}

}  // namespace

extern "C" {

int h4h_abi_version(void) { return 107; }

const char *h4h_last_error(void) { return g_err.c_str(); }

int h4h_create(h4h_ctx **out, uint32_t n, double e2, float eta, double dt_min, double dt_max,
               int precision) {
    if (n < 1) {
        if (out) *out = nullptr;
        return fail(H4H_EINVAL, "n must be >= 1");
    }
    return create_impl(out, 1, &n, e2, eta, dt_min, dt_max, precision);
}

int h4h_create_ensemble(h4h_ctx **out, uint32_t nclusters, const uint32_t *sizes, double e2,
                        float eta, double dt_min, double dt_max, int precision) {
    return create_impl(out, nclusters, sizes, e2, eta, dt_min, dt_max, precision);
}

int h4h_destroy(h4h_ctx *ctx) {
    if (!ctx) return H4H_OK;
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    drop_graph(ctx);
    for (int k = 0; k < 4; ++k)
        if (ctx->ev[k]) (void)hipEventDestroy(ctx->ev[k]);
    for (void *p : {(void *)ctx->arena, (void *)ctx->partial})
        if (p) (void)hipFree(p);
    for (hipEvent_t ev : ctx->dl_ev)
        if (ev) (void)hipEventDestroy(ev);
    if (ctx->dl_pin) (void)hipHostFree(ctx->dl_pin);
    if (ctx->pinned) (void)hipHostFree(ctx->pinned);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return H4H_OK;
}

int h4h_set_precision(h4h_ctx *ctx, int precision) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    if (!valid_precision(precision)) return fail(H4H_EINVAL, "unknown precision");
    if (precision == ctx->precision) return H4H_OK;
    drop_graph(ctx);
    ctx->precision = precision;
    return configure_team(ctx);
}

int h4h_set_launch(h4h_ctx *ctx, uint32_t workgroups, uint32_t max_jsplit) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    if (workgroups > 65536) return fail(H4H_EINVAL, "workgroups > 65536");
    ctx->grid = workgroups ? workgroups : DEFAULT_GRID;
    ctx->max_split = max_jsplit ? max_jsplit : DEFAULT_MAX_SPLIT;
    return configure_launch(ctx);
}

int h4h_upload(h4h_ctx *ctx, const double *r4, const double *v4, const double *f6,
               const double *t, const double *dt) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    if (!r4 || !v4) return fail(H4H_EINVAL, "r4 and v4 are required");
    const Soa &s = ctx->s;
    // Zero everything first (init_data semantics), then fill.
    H4H_HIP(hipMemsetAsync(ctx->state, 0, (size_t)ctx->n_dev * N_SOA * sizeof(double), ctx->stream));
    // Largest pair weight's mass (Predictor::m is the float mass): it decides
    // whether the one-workgroup step may skip its self-pair test, a kernel
    // argument of the captured graphs.
    double mmax = 0.0;
    for (uint32_t i = 0; i < ctx->n; ++i) {
        const double m = std::fabs((double)(float)r4[4 * (size_t)i + 3]);
        mmax = std::isfinite(m) ? std::max(mmax, m) : (double)INFINITY;
    }
    if (self_pair_is_zero(ctx->precision, ctx->e2, mmax) !=
        self_pair_is_zero(ctx->precision, ctx->e2, ctx->mass_max))
        drop_graph(ctx);
    ctx->mass_max = mmax;
    Cols c{};
    c.c[0] = s.r[0]; c.c[1] = s.r[1]; c.c[2] = s.r[2]; c.c[3] = s.m;
    if ((rc = upload_cols(ctx, r4, 4, c))) return rc;
    Cols cv{};
    cv.c[0] = s.v[0]; cv.c[1] = s.v[1]; cv.c[2] = s.v[2];
    if ((rc = upload_cols(ctx, v4, 4, cv))) return rc;
    if (f6) {
        Cols cf{};
        for (int k = 0; k < 6; ++k) cf.c[k] = s.f[k];
        if ((rc = upload_cols(ctx, f6, 6, cf))) return rc;
    }
    if (t && (rc = upload_scalar(ctx, t, s.t))) return rc;
    if (dt && (rc = upload_scalar(ctx, dt, s.dt))) return rc;
    hipLaunchKernelGGL(k_init_predictor, dim3(blocks_for(ctx->n_dev)), dim3(BS), 0, ctx->stream,
                       ctx->s, ctx->e);
    H4H_LAUNCHED();
    H4H_HIP(hipMemsetAsync(ctx->d_cs, 0, ctx->K * sizeof(ClState), ctx->stream));
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    ctx->nact_host = 0;
    ctx->bm_valid = false;
    ctx->uploaded = true;
    return H4H_OK;
}

int h4h_download(h4h_ctx *ctx, double *r4, double *v4, double *f6, double *time, double *dt,
                 double *old6, double *a2, double *a3) {
    int rc = check_ctx(ctx);
    if (rc) return rc;
    RowArrays t{};
    double *to[8];
    auto rows = [&](double *p, uint32_t nc, uint32_t col, uint32_t fourth) {
        if (!p) return;
        to[t.n] = p;
        t.nc[t.n] = nc;
        t.col[t.n] = col;
        t.fourth[t.n] = fourth;
        t.at[t.n + 1] = t.at[t.n] + (unsigned long long)nc * ctx->n;
        ++t.n;
    };
    rows(r4, 4, COL_R, COL_M);
    rows(v4, 4, COL_V, NO_COL);
    rows(f6, 6, COL_F, NO_COL);
    rows(old6, 6, COL_OLD, NO_COL);
    rows(a2, 3, COL_A2, NO_COL);
    rows(a3, 3, COL_A3, NO_COL);
    rows(time, 1, COL_T, NO_COL);
    rows(dt, 1, COL_DT, NO_COL);
    if (t.at[t.n]) {
        int current = 0;  // the slots' events are of the context's device
        H4H_HIP(hipGetDevice(&current));
        if (current != ctx->device) H4H_HIP(hipSetDevice(ctx->device));
        const bool large = t.at[t.n] >= DL_MIN;
        const uint32_t size = large ? DL_SLOT : DL_SLOT_SMALL;
        const uint32_t threads =
            std::min(large ? DL_THREADS : t.at[t.n] >= DL_TWO ? 2u : 1u,
                     std::max(1u, std::thread::hardware_concurrency()));
        const bool slots = make_slots(ctx, 2 * threads, size);
        rc = slots ? download_rows(ctx, t, to, threads, size) : H4H_OK;
        if (current != ctx->device) H4H_HIP(hipSetDevice(current));
        if (slots) return rc;
    }
    const Soa &s = ctx->s;
    if (r4) {
        Cols c{};
        c.c[0] = s.r[0]; c.c[1] = s.r[1]; c.c[2] = s.r[2]; c.c[3] = s.m;
        if ((rc = download_cols(ctx, r4, 4, c))) return rc;
    }
    if (v4) {
        Cols c{};
        c.c[0] = s.v[0]; c.c[1] = s.v[1]; c.c[2] = s.v[2]; c.c[3] = nullptr;
        if ((rc = download_cols(ctx, v4, 4, c))) return rc;
    }
    if (f6) {
        Cols c{};
        for (int k = 0; k < 6; ++k) c.c[k] = s.f[k];
        if ((rc = download_cols(ctx, f6, 6, c))) return rc;
    }
    if (old6) {
        Cols c{};
        for (int k = 0; k < 6; ++k) c.c[k] = s.old[k];
        if ((rc = download_cols(ctx, old6, 6, c))) return rc;
    }
    if (a2) {
        Cols c{};
        for (int k = 0; k < 3; ++k) c.c[k] = s.a2[k];
        if ((rc = download_cols(ctx, a2, 3, c))) return rc;
    }
    if (a3) {
        Cols c{};
        for (int k = 0; k < 3; ++k) c.c[k] = s.a3[k];
        if ((rc = download_cols(ctx, a3, 3, c))) return rc;
    }
    if (time && (rc = download_scalar(ctx, s.t, time))) return rc;
    if (dt && (rc = download_scalar(ctx, s.dt, dt))) return rc;
    return H4H_OK;
}

int h4h_download_predictor(h4h_ctx *ctx, double *p6, float *pm) {
    int rc = check_ctx(ctx);
    if (rc) return rc;
    const Soa &s = ctx->s;
    if (p6) {
        Cols c{};
        for (int k = 0; k < 3; ++k) {
            c.c[k] = &s.pp[0].x + k;
            c.c[3 + k] = &s.pv[0].x + k;
            c.stride[k] = c.stride[3 + k] = 4;
        }
        if ((rc = download_cols(ctx, p6, 6, c))) return rc;
    }
    if (pm) {
        std::vector<double> tmp(ctx->n);
        Cols c{};
        c.c[0] = &s.pp[0].w;
        c.stride[0] = 4;
        if ((rc = download_cols(ctx, tmp.data(), 1, c))) return rc;
        for (uint32_t i = 0; i < ctx->n; ++i) pm[i] = (float)tmp[i];
    }
    return H4H_OK;
}

int h4h_upload_predictor(h4h_ctx *ctx, const double *p6, const float *pm) {
    int rc = check_ctx(ctx);
    if (rc) return rc;
    const Soa &s = ctx->s;
    if (p6) {
        Cols c{};
        for (int k = 0; k < 3; ++k) {
            c.c[k] = &s.pp[0].x + k;
            c.c[3 + k] = &s.pv[0].x + k;
            c.stride[k] = c.stride[3 + k] = 4;
        }
        if ((rc = upload_cols(ctx, p6, 6, c))) return rc;
    }
    if (pm) {
        // pp.w = the mass as a double, pv.w = its float bit pattern
        std::vector<double> tmp(2 * (size_t)ctx->n);
        for (uint32_t i = 0; i < ctx->n; ++i) {
            tmp[2 * i] = (double)pm[i];
            tmp[2 * i + 1] = mass_bits(pm[i]);
        }
        Cols c{};
        c.c[0] = &s.pp[0].w;
        c.c[1] = &s.pv[0].w;
        c.stride[0] = c.stride[1] = 4;
        if ((rc = upload_cols(ctx, tmp.data(), 2, c))) return rc;
    }
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    return H4H_OK;
}

int h4h_set_active(h4h_ctx *ctx, const uint32_t *move, uint32_t nact) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (nact > ctx->n) return fail(H4H_EINVAL, "nact > n");
    if (nact && !move) return fail(H4H_EINVAL, "move is null");
    for (uint32_t k = 0; k < nact; ++k)
        if (move[k] >= ctx->n) return fail(H4H_EINVAL, "active index out of range");
    if (nact)
        H4H_HIP(hipMemcpyAsync(ctx->move, move, nact * sizeof(uint32_t), hipMemcpyHostToDevice,
                               ctx->stream));
    hipLaunchKernelGGL(k_set_nact0, dim3(1), dim3(1), 0, ctx->stream, ctx->e, nact);
    H4H_LAUNCHED();
    if ((rc = launch_plan(ctx))) return rc;
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    ctx->nact_host = nact;
    return H4H_OK;
}

int h4h_get_active(h4h_ctx *ctx, uint32_t *move, uint32_t *nact) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (!nact) return fail(H4H_EINVAL, "nact is null");
    *nact = ctx->nact_host;
    if (move && ctx->nact_host) {
        H4H_HIP(hipMemcpyAsync(move, ctx->move, ctx->nact_host * sizeof(uint32_t),
                               hipMemcpyDeviceToHost, ctx->stream));
        H4H_HIP(hipStreamSynchronize(ctx->stream));
        std::sort(move, move + ctx->nact_host);
    }
    return H4H_OK;
}

// Initial forces of every cluster: each active list = the whole cluster.
int h4h_init_acc_jrk(h4h_ctx *ctx) {
    int rc = check_ctx(ctx);
    if (rc) return rc;
    hipLaunchKernelGGL(k_identity_active, dim3(blocks_for(ctx->n_dev)), dim3(BS), 0, ctx->stream,
                       ctx->move, ctx->e);
    H4H_LAUNCHED();
    if ((rc = launch_plan(ctx))) return rc;
    if ((rc = update_pass(ctx))) return rc;
    ctx->nact_host = ctx->K == 1 ? ctx->cnt[0] : 0;
    return H4H_OK;
}

static int init_dt_impl(h4h_ctx *ctx, float eta, double itime) {
    hipLaunchKernelGGL(k_reset_tmin, dim3(1), dim3(1), 0, ctx->stream, ctx->e);
    H4H_LAUNCHED();
    hipLaunchKernelGGL(k_init_dt, dim3(std::min<uint32_t>(ctx->nblk, 1024)), dim3(BS), 0,
                       ctx->stream, ctx->s, ctx->e, eta, itime, ctx->dt_min, ctx->dt_max);
    H4H_LAUNCHED();
    hipLaunchKernelGGL(k_set_times_from_tmin, dim3(1), dim3(1), 0, ctx->stream, ctx->e, itime);
    H4H_LAUNCHED();
    ctx->bm_valid = false;
    return read_state(ctx);
}

int h4h_init_dt(h4h_ctx *ctx, double *ctime, float eta, double itime) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (!ctime) return fail(H4H_EINVAL, "ctime is null");
    if ((rc = init_dt_impl(ctx, eta, itime))) return rc;
    double mn = dkey_inv(ctx->cs_host[0].tmin_key);
    if (mn < *ctime) *ctime = mn;
    return H4H_OK;
}

int h4h_find_particles_to_move(h4h_ctx *ctx, double itime, uint32_t *nact) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (!nact) return fail(H4H_EINVAL, "nact is null");
    hipLaunchKernelGGL(k_reset_select, dim3(1), dim3(1), 0, ctx->stream, ctx->e);
    H4H_LAUNCHED();
    if ((rc = launch_select(ctx, PS_SELECT, itime))) return rc;
    if ((rc = launch_plan(ctx))) return rc;
    if ((rc = read_state(ctx))) return rc;
    ctx->nact_host = ctx->cs_host[0].nact;
    *nact = ctx->nact_host;
    return H4H_OK;
}

int h4h_save_old_acc_jrk(h4h_ctx *ctx) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (!ctx->nact_host) return H4H_OK;
    uint32_t grid = std::max<uint32_t>(1, std::min<uint32_t>(blocks_for(ctx->nact_host), 1024));
    hipLaunchKernelGGL(k_save_old, dim3(grid), dim3(BS), 0, ctx->stream, ctx->s, ctx->e, ctx->move);
    H4H_LAUNCHED();
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    return H4H_OK;
}

int h4h_predicted_pos_vel(h4h_ctx *ctx, double itime) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if ((rc = launch_select(ctx, PS_PREDICT, itime))) return rc;
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    return H4H_OK;
}

int h4h_update_acc_jrk(h4h_ctx *ctx, uint32_t nact) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (nact != ctx->nact_host)
        return fail(H4H_EINVAL, "nact differs from the current active list size");
    if (nact && (rc = update_pass(ctx))) return rc;
    ctx->stats.block_steps += 1;
    ctx->stats.interactions += (uint64_t)nact * ctx->n;
    ctx->stats.nsteps += nact;
    return H4H_OK;
}

int h4h_correction_pos_vel(h4h_ctx *ctx, double itime, uint32_t nact) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (nact != ctx->nact_host)
        return fail(H4H_EINVAL, "nact differs from the current active list size");
    uint32_t grid = std::max<uint32_t>(1, std::min<uint32_t>(blocks_for(nact), 1024));
    hipLaunchKernelGGL(k_correct, dim3(grid), dim3(BS), 0, ctx->stream, ctx->s, ctx->e, ctx->move,
                       itime, ctx->eta, ctx->dt_min, ctx->dt_max);
    H4H_LAUNCHED();
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    ctx->bm_valid = false;
    return H4H_OK;
}

int h4h_next_integration_time(h4h_ctx *ctx, double *atime) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (!atime) return fail(H4H_EINVAL, "atime is null");
    hipLaunchKernelGGL(k_reset_tmin, dim3(1), dim3(1), 0, ctx->stream, ctx->e);
    H4H_LAUNCHED();
    hipLaunchKernelGGL(k_next_time, dim3(std::min<uint32_t>(ctx->nblk, 1024)), dim3(BS), 0,
                       ctx->stream, ctx->s, ctx->e);
    H4H_LAUNCHED();
    if ((rc = read_state(ctx))) return rc;
    *atime = dkey_inv(ctx->cs_host[0].tmin_key);
    return H4H_OK;
}

int h4h_step(h4h_ctx *ctx, double itime, uint32_t *nact, double *atime) {
    int rc = check_single(ctx);
    if (rc) return rc;
    // The step the device loop would make: k_small_run or k_team_run when they
    // take it, which the host looks at before it launches the others (most
    // steps are theirs, and the launches cost more than a look).  A step that
    // the last one has counted and found too large for them is spared the look
    // (18 us of 50).
    const bool small = small_path(ctx);
    const bool large = ctx->bm_valid && itime == ctx->next_time && ctx->next_nact < BCNT_MANY &&
                       ctx->next_nact > (small ? std::min(ctx->small_act, SMALL_MAX_ACT) : ONE_ACT);
    const bool team = team_path(ctx) && !ctx->team_rest;
    if (ctx->team_rest) --ctx->team_rest;
    ctx->next_nact = 0;
    if ((rc = ensure_blockmin(ctx))) return rc;
    if (ctx->timing) H4H_HIP(hipEventRecord(ctx->ev[2], ctx->stream));
    ctx->cs_host[0] = ClState{};
    if (!large && (small || team)) {
        const OneStep one{itime, ctx->cs_host};
        if ((rc = small ? launch_small(ctx, 1, 0, one) : launch_team(ctx, 1, one))) return rc;
        if (ctx->timing) H4H_HIP(hipEventRecord(ctx->ev[3], ctx->stream));
        if ((rc = await_step(ctx))) return rc;
        if ((rc = check_team(ctx, ctx->cs_host[0].done == STEP_FAILED))) return rc;
        // (this step and the ones after it, as in a loop)
        if (ctx->cs_host[0].done == STEP_ALONE)
            ctx->team_rest = team_backoff(ctx->team_fails++) - 1;
    }
    const bool launches = ctx->cs_host[0].done != STEP_DONE;
    if (!launches && !small) {
        ctx->team_steps += 1;
        ctx->team_fails = 0;
    }
    if (launches) {
        ctx->cs_host[0].done = 0;
        // One-step loop: ATIME = itime, stop after the step.
        hipLaunchKernelGGL(k_run_setup, dim3(1), dim3(BS), 0, ctx->stream, ctx->e, (double)INFINITY,
                           -INFINITY, 1ull, 1u, -INFINITY, itime, 0ull, 0u);
        H4H_LAUNCHED();
        if ((rc = enqueue_step(ctx, ctx->timing, 0))) return rc;
        hipLaunchKernelGGL(k_tail, dim3(1), dim3(BS), 0, ctx->stream, ctx->e, ctx->cs_host);
        H4H_LAUNCHED();
        if (ctx->timing) H4H_HIP(hipEventRecord(ctx->ev[3], ctx->stream));
        if ((rc = await_step(ctx))) return rc;
    }
    if (ctx->timing) {
        float ms = 0.f;
        H4H_HIP(hipEventElapsedTime(&ms, ctx->ev[2], ctx->ev[3]));
        ctx->stats.step_ms += ms;
        if (launches) {
            H4H_HIP(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
            ctx->stats.update_ms += ms;
            ctx->stats.update_launches += 1;
        }
    }
    const ClState &cs = ctx->cs_host[0];
    uint32_t k = (uint32_t)cs.nsteps;  // the step's nact (counters were reset)
    ctx->nact_host = 0;
    ctx->next_nact = cs.tail_nact;
    ctx->next_time = cs.atime;
    ctx->stats.block_steps += 1;
    ctx->stats.interactions += cs.interactions;
    ctx->stats.nsteps += k;
    ctx->stats.small_steps += cs.small_steps;
    if (nact) *nact = k;
    if (atime) *atime = cs.atime;
    return H4H_OK;
}

// Replays captured chunks of RUN_CHUNK steps until every cluster's loop has
// stopped; copies cluster 0's per-step history when asked.
static int run_chunks(h4h_ctx *ctx, double *step_time, uint32_t *step_nact, uint64_t cap) {
    ctx->next_nact = 0;
    int rc = H4H_OK;
    uint64_t seen = 0, made = 0;  // steps copied out, steps made
    const bool plain = ctx->K == 1 && !small_path(ctx) && !team_path(ctx);
    bool hist = (step_time || step_nact) && ctx->K == 1;
    if (ctx->timing) H4H_HIP(hipEventRecord(ctx->ev[2], ctx->stream));
    for (;;) {
        if (plain && made < cap && cap - made <= RUN_CHUNK) {
            // the last steps of the budget, and their loop tail: a chunk's
            // steps beyond it are three empty launches each (a run that ends
            // with a chunk needed another one of 32 for its last loop tail:
            // 0.18 ms)
            for (uint64_t k = 0; k < cap - made; ++k)
                if ((rc = enqueue_step(ctx, false, k & 1))) return rc;
            hipLaunchKernelGGL(k_tail, dim3(1), dim3(BS), 0, ctx->stream, ctx->e,
                               (ClState *)nullptr);
            H4H_LAUNCHED();
        } else if (ctx->graphs) {
            if ((rc = ensure_graph(ctx))) return rc;
            H4H_HIP(hipGraphLaunch(ctx->graph_exec, ctx->stream));
        } else if ((rc = enqueue_chunk(ctx))) {
            return rc;
        }
        H4H_HIP(hipMemcpyAsync(ctx->ctl_host, ctx->d_ctl, sizeof(RunCtl) + sizeof(ClState),
                               hipMemcpyDeviceToHost, ctx->stream));
        H4H_HIP(hipStreamSynchronize(ctx->stream));
        if ((rc = check_team(ctx, ctx->ctl_host->team_err != 0))) return rc;
        if (hist) {
            uint64_t steps = ctx->cs_host[0].steps;
            for (uint64_t k = seen; k < steps && k < cap; ++k) {
                if (step_time) step_time[k] = ctx->hist_t_host[k % HIST_CAP];
                if (step_nact) step_nact[k] = ctx->hist_n_host[k % HIST_CAP];
            }
            seen = steps;
        }
        made = ctx->cs_host[0].steps + (ctx->cs_host[0].tail_pend ? 1 : 0);
        if (ctx->ctl_host->ndone >= ctx->K) break;
    }
    if (ctx->timing) {
        H4H_HIP(hipEventRecord(ctx->ev[3], ctx->stream));
        H4H_HIP(hipEventSynchronize(ctx->ev[3]));
        float ms = 0.f;
        H4H_HIP(hipEventElapsedTime(&ms, ctx->ev[2], ctx->ev[3]));
        ctx->stats.step_ms += ms;
    }
    if ((rc = read_state(ctx))) return rc;
    const RunCtl &ctl = *ctx->ctl_host;
    const uint64_t steps = ctx->cs_host[0].steps;
    ctx->team_steps += ctl.team_steps;
    ctx->team_rest = ctl.team_retry > steps ? ctl.team_retry - steps : 0;
    ctx->team_fails = ctl.team_fails;
    return H4H_OK;
}

int h4h_run(h4h_ctx *ctx, double t_end, double t_stop, uint64_t max_steps, h4h_run_info *io,
            double *step_time, uint32_t *step_nact) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (!io) return fail(H4H_EINVAL, "io is null");
    if (max_steps == 0) return fail(H4H_EINVAL, "max_steps must be >= 1");
    if ((rc = ensure_blockmin(ctx))) return rc;
    hipLaunchKernelGGL(k_run_setup, dim3(1), dim3(BS), 0, ctx->stream, ctx->e, t_end, t_stop,
                       (unsigned long long)max_steps, 1u, io->itime, io->atime,
                       (unsigned long long)ctx->team_rest, ctx->team_fails);
    H4H_LAUNCHED();
    if ((rc = run_chunks(ctx, step_time, step_nact, max_steps))) return rc;
    const ClState &d = ctx->cs_host[0];
    io->itime = d.itime;
    io->atime = d.atime;
    io->steps = d.steps;
    io->interactions = d.interactions;
    io->nsteps = d.nsteps;
    const uint32_t last = d.steps ? ctx->hist_n_host[(d.steps - 1) % HIST_CAP] : 0u;
    io->last_nact = last;
    if (d.steps && d.itime >= t_stop)
        io->stopped = H4H_STOP_OUTPUT;
    else if (d.steps >= max_steps)
        io->stopped = H4H_STOP_MAXSTEPS;
    else
        io->stopped = H4H_STOP_END;
    ctx->nact_host = 0;
    ctx->stats.block_steps += d.steps;
    ctx->stats.interactions += d.interactions;
    ctx->stats.nsteps += d.nsteps;
    ctx->stats.small_steps += d.small_steps;
    return H4H_OK;
}

int h4h_get_energy(h4h_ctx *ctx, double *ekin, double *epot) {
    int rc = check_single(ctx);
    if (rc) return rc;
    return energies_of(ctx, 0, 1, ekin, epot);
}

int h4h_ensemble_init(h4h_ctx *ctx, float eta_s) {
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if ((rc = h4h_init_acc_jrk(ctx))) return rc;
    return init_dt_impl(ctx, eta_s, 0.0);
}

int h4h_ensemble_run(h4h_ctx *ctx, double t_end, double t_stop, uint64_t max_steps,
                     h4h_cluster_info *info) {
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (max_steps == 0) return fail(H4H_EINVAL, "max_steps must be >= 1");
    if ((rc = ensure_blockmin(ctx))) return rc;
    hipLaunchKernelGGL(k_run_setup, dim3(1), dim3(BS), 0, ctx->stream, ctx->e, t_end, t_stop,
                       (unsigned long long)max_steps, 0u, 0.0, 0.0, (unsigned long long)ctx->team_rest,
                       ctx->team_fails);
    H4H_LAUNCHED();
    if ((rc = run_chunks(ctx, nullptr, nullptr, 0))) return rc;
    for (uint32_t c = 0; c < ctx->K; ++c) {
        const ClState &d = ctx->cs_host[c];
        ctx->stats.block_steps += d.steps;
        ctx->stats.interactions += d.interactions;
        ctx->stats.nsteps += d.nsteps;
        ctx->stats.small_steps += d.small_steps;
        if (info) {
            info[c].itime = d.itime;
            info[c].atime = d.atime;
            info[c].steps = d.steps;
            info[c].interactions = d.interactions;
            info[c].nsteps = d.nsteps;
            info[c].stopped = d.steps && d.itime >= t_stop ? H4H_STOP_OUTPUT
                              : d.steps >= max_steps    ? H4H_STOP_MAXSTEPS
                                                        : H4H_STOP_END;
        }
    }
    ctx->nact_host = 0;
    return H4H_OK;
}

int h4h_ensemble_energy(h4h_ctx *ctx, double *ekin, double *epot) {
    int rc = check_ctx(ctx);
    if (rc) return rc;
    return energies_of(ctx, 0, ctx->K, ekin, epot);
}

int h4h_ensemble_sizes(h4h_ctx *ctx, uint32_t *nclusters, uint32_t *sizes) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    if (nclusters) *nclusters = ctx->K;
    if (sizes)
        for (uint32_t c = 0; c < ctx->K; ++c) sizes[c] = ctx->cnt[c];
    return H4H_OK;
}

int h4h_set_tuning(h4h_ctx *ctx, const uint32_t *grid32, const uint32_t *iw32) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    uint32_t table[64] = {0};
    for (int b = 0; b < 32; ++b) {
        uint32_t g = grid32 ? grid32[b] : 0u;
        uint32_t w = iw32 ? iw32[b] : 0u;
        if (w != 0 && w != 4 && w != 16 && w != 64 && w != 256)
            return fail(H4H_EINVAL, "lane-group width must be 0, 4, 16, 64 or 256");
        if (g > 65536) return fail(H4H_EINVAL, "workgroup share > 65536");
        table[b] = g;
        table[32 + b] = w;
    }
    H4H_HIP(hipMemcpyAsync(ctx->d_tune, table, sizeof(table), hipMemcpyHostToDevice, ctx->stream));
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    ctx->e.tuned = (grid32 || iw32) ? 1u : 0u;
    drop_graph(ctx);
    return configure_team(ctx);
}

// Measures the update kernel for nact = 2^b (b = 0 .. log2 n, plus n) with
// evenly spaced active particles, for every candidate workgroup share and
// lane-group width, and installs the fastest per bucket.  The active list
// is left empty.
int h4h_autotune(h4h_ctx *ctx, uint32_t reps, uint32_t *grid32, uint32_t *iw32) {
    int rc = check_single(ctx);
    if (rc) return rc;
    if (reps < 1) reps = 1;
    const uint32_t n = ctx->n;
    const uint32_t gmax = ctx->e.grid;
    uint32_t best_g[32] = {0}, best_w[32] = {0};
    std::vector<uint32_t> move;
    for (uint32_t b = 0; b < 32; ++b) {
        uint64_t want = 1ull << b;
        if (want > n) break;
        uint32_t nact = (2 * want > n) ? n : (uint32_t)want;  // top bucket: all n
        move.resize(nact);
        for (uint32_t k = 0; k < nact; ++k) move[k] = (uint32_t)((uint64_t)k * n / nact);
        if ((rc = h4h_set_active(ctx, move.data(), nact))) return rc;
        std::vector<uint32_t> gs, ws;
        for (uint32_t g = 64; g <= gmax; g *= 2) gs.push_back(g);
        if (gs.empty() || gs.back() != gmax) gs.push_back(gmax);
        const uint32_t wopt[4] = {4, 16, 64, 256};
        for (uint32_t w : wopt)
            if (w <= 4 * std::max<uint32_t>(nact, 1) || w == 256) ws.push_back(w);
        float best = 1e30f;
        for (uint32_t w : ws) {
            for (uint32_t g : gs) {
                uint32_t gt[32] = {0}, wt[32] = {0};
                std::copy(best_g, best_g + 32, gt);
                std::copy(best_w, best_w + 32, wt);
                gt[b] = g;
                wt[b] = w;
                if ((rc = h4h_set_tuning(ctx, gt, wt))) return rc;
                if ((rc = launch_plan(ctx))) return rc;
                if ((rc = launch_update(ctx))) return rc;  // warm
                H4H_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
                for (uint32_t r = 0; r < reps; ++r)
                    if ((rc = launch_update(ctx))) return rc;
                H4H_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
                H4H_HIP(hipEventSynchronize(ctx->ev[1]));
                float ms = 0.f;
                H4H_HIP(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
                if (ms < best) {
                    best = ms;
                    best_g[b] = g;
                    best_w[b] = w;
                }
            }
        }
    }
    if ((rc = h4h_set_tuning(ctx, best_g, best_w))) return rc;
    if (grid32) std::copy(best_g, best_g + 32, grid32);
    if (iw32) std::copy(best_w, best_w + 32, iw32);
    hipLaunchKernelGGL(k_set_nact0, dim3(1), dim3(1), 0, ctx->stream, ctx->e, 0u);
    H4H_LAUNCHED();
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    ctx->nact_host = 0;
    return H4H_OK;
}

// Launch autotuner: every candidate (persistent workgroups x largest j
// split x lane-group fill rule) runs the same `steps` device block steps
// from the context's current state, which is saved once and restored
// before each trial and at the end; the fastest is installed.
int h4h_tune_launch(h4h_ctx *ctx, uint32_t steps, h4h_launch_choice *choice) {
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (steps < 1 || steps > (1u << 20)) return fail(H4H_EINVAL, "steps must be in [1, 2^20]");
    const size_t sbytes = (size_t)ctx->n_dev * N_SOA * sizeof(double);
    const size_t cbytes = (size_t)ctx->K * sizeof(ClState);
    char *save = nullptr;
    if (hipMalloc(&save, sbytes + cbytes) != hipSuccess) {
        (void)hipGetLastError();
        return fail(H4H_ENOMEM, "tune_launch: no device memory for the state copy");
    }
    auto copy_state = [&](bool store) -> int {
        if (store) {
            H4H_HIP(hipMemcpyAsync(save, ctx->state, sbytes, hipMemcpyDeviceToDevice, ctx->stream));
            H4H_HIP(hipMemcpyAsync(save + sbytes, ctx->d_cs, cbytes, hipMemcpyDeviceToDevice,
                                   ctx->stream));
        } else {
            H4H_HIP(hipMemcpyAsync(ctx->state, save, sbytes, hipMemcpyDeviceToDevice, ctx->stream));
            H4H_HIP(hipMemcpyAsync(ctx->d_cs, save + sbytes, cbytes, hipMemcpyDeviceToDevice,
                                   ctx->stream));
            ctx->bm_valid = false;
        }
        return H4H_OK;
    };
    const h4h_stats stats0 = ctx->stats;
    const uint64_t team0 = ctx->team_steps;
    const uint32_t g0 = ctx->grid, s0 = ctx->max_split, f0 = ctx->iw_fill;
    const uint32_t grids[5] = {256, 512, 1024, 2048, 4096};
    const uint32_t splits[4] = {16, 64, 256, 1024};
    const uint32_t fills[3] = {8, 12, 15};
    float best = 1e30f;
    uint32_t bg = g0, bs = s0, bf = f0;
    rc = copy_state(true);
    for (uint32_t gi = 0; gi < 5 && !rc; ++gi)
        for (uint32_t si = 0; si < 4 && !rc; ++si)
            for (uint32_t fi = 0; fi < 3 && !rc; ++fi) {
                ctx->grid = grids[gi];
                ctx->max_split = splits[si];
                ctx->iw_fill = fills[fi];
                if ((rc = configure_launch(ctx))) break;
                // untimed run: graph capture and first-touch costs
                if ((rc = copy_state(false))) break;
                if ((rc = h4h_ensemble_run(ctx, INFINITY, INFINITY, std::min<uint32_t>(steps, RUN_CHUNK),
                                           nullptr)))
                    break;
                if ((rc = copy_state(false))) break;
                if (hipEventRecord(ctx->ev[0], ctx->stream) != hipSuccess) { rc = fail(H4H_EHIP, "event"); break; }
                if ((rc = h4h_ensemble_run(ctx, INFINITY, INFINITY, steps, nullptr))) break;
                float ms = 0.f;
                if (hipEventRecord(ctx->ev[1], ctx->stream) != hipSuccess ||
                    hipEventSynchronize(ctx->ev[1]) != hipSuccess ||
                    hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]) != hipSuccess) {
                    rc = fail(H4H_EHIP, "tune_launch: event timing failed");
                    break;
                }
                if (ms < best) {
                    best = ms;
                    bg = grids[gi];
                    bs = splits[si];
                    bf = fills[fi];
                }
            }
    ctx->grid = rc ? g0 : bg;
    ctx->max_split = rc ? s0 : bs;
    ctx->iw_fill = rc ? f0 : bf;
    int rc2 = configure_launch(ctx);
    if (!rc2) rc2 = copy_state(false);
    if (!rc2 && hipStreamSynchronize(ctx->stream) != hipSuccess) rc2 = fail(H4H_EHIP, "sync");
    (void)hipFree(save);
    ctx->stats = stats0;
    ctx->team_steps = team0;
    if (rc) return rc;
    if (rc2) return rc2;
    if (choice) {
        choice->workgroups = bg;
        choice->max_jsplit = bs;
        choice->iw_fill16 = bf;
        choice->ms_per_step = best / (float)steps;
    }
    return H4H_OK;
}

int h4h_set_launch_choice(h4h_ctx *ctx, const h4h_launch_choice *choice) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    if (!choice) return fail(H4H_EINVAL, "choice is null");
    if (choice->workgroups < 1 || choice->workgroups > 65536)
        return fail(H4H_EINVAL, "workgroups must be in [1, 65536]");
    if (choice->max_jsplit < 1) return fail(H4H_EINVAL, "max_jsplit must be >= 1");
    if (choice->iw_fill16 < 1 || choice->iw_fill16 > 16)
        return fail(H4H_EINVAL, "iw_fill16 must be in [1, 16]");
    ctx->grid = choice->workgroups;
    ctx->max_split = choice->max_jsplit;
    ctx->iw_fill = choice->iw_fill16;
    return configure_launch(ctx);
}

int h4h_set_graphs(h4h_ctx *ctx, int enable) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    ctx->graphs = enable != 0;
    drop_graph(ctx);
    return H4H_OK;
}

int h4h_set_small_path(h4h_ctx *ctx, uint32_t max_active) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    ctx->small_act = max_active;
    drop_graph(ctx);
    return H4H_OK;
}

int h4h_set_timing(h4h_ctx *ctx, int enable) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    ctx->timing = enable != 0;
    return H4H_OK;
}

int h4h_get_stats(h4h_ctx *ctx, h4h_stats *out, int reset) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    if (out) *out = ctx->stats;
    if (reset) ctx->stats = h4h_stats{};
    return H4H_OK;
}

int h4h_refuse_team(h4h_ctx *ctx) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    if (!ctx->team_ok) return H4H_OK;
    hipLaunchKernelGGL(k_team_refuse, dim3(1), dim3(1), 0, ctx->stream, ctx->team);
    H4H_LAUNCHED();
    return H4H_OK;
}

int h4h_team_steps(h4h_ctx *ctx, uint64_t *steps, int reset) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    if (steps) *steps = ctx->team_steps;
    if (reset) ctx->team_steps = 0;
    return H4H_OK;
}

int h4h_synchronize(h4h_ctx *ctx) {
    int rc = check_ctx(ctx, false);
    if (rc) return rc;
    H4H_HIP(hipStreamSynchronize(ctx->stream));
    return H4H_OK;
}

int h4h_update_acc_jrk_static(const double *d_p6, const float *d_pm, uint32_t n,
                              const uint32_t *d_move, uint32_t nact, double e2, int precision,
                              double *d_f6, void *stream) {
    if (n > STATIC_MAX_N) return fail(H4H_EINVAL, "n exceeds H4H_STATIC_MAX_N (65536)");
    if (nact > n) return fail(H4H_EINVAL, "nact > n");
    if (!(e2 >= 0.0) || !std::isfinite(e2)) return fail(H4H_EINVAL, "e2 must be finite and >= 0");
    if (!valid_precision(precision)) return fail(H4H_EINVAL, "unknown precision");
    if (nact && (!d_p6 || !d_pm || !d_move || !d_f6))
        return fail(H4H_EINVAL, "null device pointer");
    double *base = nullptr;
    int rc = static_scratch(&base);
    if (rc) return rc;
    if (nact == 0) return H4H_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint32_t n_pad = (n + JT - 1) / JT * JT;

    // The plan of a default single-system context of n particles.  (Its grid
    // is DEFAULT_GRID at most, and one j chunk at a larger grid is one at a
    // smaller.)
    const bool mixed = precision == H4H_MIXED;
    const uint32_t n_jt = n_pad / JT;
    const LaneGroup lg =
        lane_group(nact, DEFAULT_IW_FILL, std::min(n_jt, DEFAULT_MAX_SPLIT), mixed);
    // The forces may be written over the particles (d_f6 on d_p6 or d_pm): the one
    // launch reads those while it writes.
    auto over = [&](const void *p, size_t bytes) {
        const uintptr_t f = (uintptr_t)d_f6, x = (uintptr_t)p;
        return f < x + bytes && x < f + (size_t)n * 48;
    };
    const bool apart = !over(d_p6, (size_t)n * 48) && !over(d_pm, (size_t)n * 4);
    if (precision != H4H_FP64_EXACT && n_jt <= ONE_TILES && nact <= BS && lg.iw <= 64 && !lg.jrun &&
        apart) {
        const Decomp d = decompose(nact, lg.iw, n_jt, DEFAULT_GRID, DEFAULT_MAX_SPLIT);
        if (d.S == 1) {
            hipLaunchKernelGGL(mixed ? k_static_one<true> : k_static_one<false>, dim3(d.n_it),
                               dim3(BS), 0, st, d_p6, d_pm, n, d_move, nact, lg.iw, e2, d_f6);
            H4H_LAUNCHED();
            return H4H_OK;
        }
    }
    const uint32_t grid = std::min(DEFAULT_GRID, max_items(n, DEFAULT_GRID, DEFAULT_MAX_SPLIT,
                                                           DEFAULT_IW_FILL));
    if (precision != H4H_FP64_EXACT) {
        const Decomp d = decompose(nact, lg.iw, n_jt, grid, DEFAULT_MAX_SPLIT);
        if (d.S > 1 && 6ull * d.S * d.rows > ST_PART)
            return fail(H4H_EINVAL, "work plan exceeds the static buffer");
    }
    Soa s{};
    s.pp = reinterpret_cast<double4 *>(base + ST_PP);
    s.pv = reinterpret_cast<double4 *>(base + ST_PV);
    for (int q = 0; q < 6; ++q) s.f[q] = base + ST_F + (size_t)q * STATIC_MAX_N;
    uint32_t *tab = reinterpret_cast<uint32_t *>(base + ST_TAB);
    uint32_t *move = reinterpret_cast<uint32_t *>(base + ST_MOVE);
    unsigned long long *pre = reinterpret_cast<unsigned long long *>(base + ST_PRE);
    double *partial = base + ST_PARTIAL;
    Ens e{};
    e.K = 1;
    e.nblk = n_pad / JT;
    e.off = tab + TAB_OFF;
    e.cnt = tab + TAB_CNT;
    e.hoff = tab + TAB_HOFF;
    e.cs = reinterpret_cast<ClState *>(base + ST_CS);
    e.plan = reinterpret_cast<ClPlan *>(base + ST_PLAN);
    e.items_pre = pre;
    e.fin_pre = pre + 2;
    e.part_pre = pre + 4;
    e.ctl = reinterpret_cast<RunCtl *>(base + ST_CTL);
    e.grid = grid;
    e.max_split = DEFAULT_MAX_SPLIT;
    e.iw_fill = DEFAULT_IW_FILL;
    e.tuned = 0;

    uint32_t *bad = reinterpret_cast<uint32_t *>(base + ST_BAD);
    hipLaunchKernelGGL(k_static_pack, dim3(n_pad / BS), dim3(BS), 0, st, d_p6, d_pm, n, n_pad,
                       d_move, nact, move, s, e, tab, bad);
    H4H_LAUNCHED();
    if (precision == H4H_FP64_EXACT) {
        hipLaunchKernelGGL(k_update_exact, dim3(exact_grid(nact)), dim3(BS), 0, st, s, e, move, e2);
    } else {
        auto *kern = precision == H4H_MIXED ? k_update_mixed : k_update_fp64;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(BS), 0, st, s, e, move, partial, e2, 0u);
    }
    H4H_LAUNCHED();
    hipLaunchKernelGGL(k_static_finish, dim3(std::min<uint32_t>(1024, std::max<uint32_t>(64, e.nblk))),
                       dim3(BS), 0, st, s, e, move, partial, d_move, n, nact, bad, d_f6);
    H4H_LAUNCHED();
    return H4H_OK;
}

}  // extern "C"
