// Refinement on gfx950: projection, label propagation with per-vertex
// part-connectivity tables in LDS, afterburner priority filter, exact
// incremental cut/load updates, deterministic capacity repair and the
// capacity-complementary exchange.  Restates src/refine.cu and
// src/refinement/*.cuh of the reference; order-dependent steps follow the
// canonical vertex-id order.
#include "gp_metrics.hpp"
#include "gp_refine.hpp"
#include "gp_rows.hpp"

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstdio>
#include <type_traits>

namespace gp {
namespace {

constexpr int kBalanceBuckets = 50;
constexpr int kBalanceSections = 16;
constexpr int kBalanceWidth = kBalanceBuckets * kBalanceSections;

// Slot of bucket b = (gain bucket, section) in a part's row of the counts
// array: section-major, so the sections of one gain bucket (the donors of a
// part with similar gains, often most of them) sit kBalanceBuckets words
// apart, in different cache lines, and their atomics spread over memory
// channels instead of queueing on one line.
__host__ __device__ constexpr int count_slot(int b) {
    return (b % kBalanceSections) * kBalanceBuckets + b / kBalanceSections;
}
constexpr int kJointSeeds = 128;
constexpr int kJointSide = 4;
constexpr int kJointArchive = 4;

// Counter slots (device array of u64).  Those that many blocks of one launch
// add to lie in cache lines of their own: atomics on one line queue up (12 ns
// each from different waves), on several lines they run side by side.
constexpr int kCtrLine = 16;  // words of a 128-byte line
enum Ctr {
    kFrontier = 0,
    kCand = kCtrLine,
    kTier = 2 * kCtrLine,  // two slots: medium, heavy
    kMovers = 3 * kCtrLine,
    kDelta = 4 * kCtrLine,
    kDonors = 5 * kCtrLine,
    kRowSum = 6 * kCtrLine,  // profiling: entries of the rows scanned by the last LP proposal sweep
    // Tier list counters of the second and third sweep of a round, so that
    // one clear of the whole block at the round start serves all three.
    kTierB = 7 * kCtrLine,
    kTierC = 8 * kCtrLine,
    // (entries, rows) handled by the afterburner, update and repair-proposal
    // sweeps, counted only when the context profiles kernel classes.
    kEntAfter = 9 * kCtrLine,
    kEntUpdate = kEntAfter + 2,
    kEntRepair = kEntAfter + 4,
    // What a repair iteration's donor selection hands on (written, not added
    // to; a read-back that clears the counters before it leaves it): eligible
    // donors, the same when one tail launch takes them (else 0), all donors.
    kSelected = 10 * kCtrLine,
    kCtrCount = 11 * kCtrLine
};
constexpr int kCtrClear = kSelected;

// Part ids inside refinement: k <= 128 fits a byte, which keeps the label
// array of a level small enough for the neighbour gathers to hit in cache.
using Label = std::uint8_t;

struct RepairSample {
    unsigned long long loss;    // modular sum of -gain
    unsigned long long weight;
};

// 1.5^j for j = -23..24 at index j + 23, by repeated exact-IEEE products
// and quotients (compile-time evaluation rounds like the run-time ops).
struct Pow15 {
    double p[48];
};
constexpr Pow15 make_pow15() {
    Pow15 t{};
    t.p[23] = 1.0;
    for (int j = 1; j <= 24; ++j) t.p[23 + j] = t.p[22 + j] * 1.5;
    for (int j = 1; j <= 23; ++j) t.p[23 - j] = t.p[24 - j] / 1.5;
    return t;
}
__constant__ Pow15 kPow15 = make_pow15();

// One byte lane of the packed per-vertex state word (indexing like an
// array of T; the four lanes of a vertex share one 32-bit word).
template <typename T>
struct StateLane {
    T* base;
    __host__ __device__ T& operator[](std::int64_t v) const { return base[4 * v]; }
};

// Per-vertex refinement state, one 32-bit word per vertex: target part
// (signed byte, -1 none) in byte 0, moving flag in byte 1, frontier
// membership in byte 2, the label with the lock as its top bit in byte 3.  The
// afterburner and the update sweep read a neighbour's whole state with one
// gather; the label array, which the histograms gather (a quarter the size,
// so that it stays in L2), holds the same labels.  With the label gathered from
// that array beside the word, an update of R-MAT scale 22 took 92 us on its
// medium rows and an afterburner 271, now 66 and 217.
constexpr int kStateTarget = 0, kStateFlag = 1, kStateMember = 2, kStateOwn = 3;
constexpr int kLockBit = 0x80;
__host__ __device__ inline int state_label(std::uint32_t st) { return (int)((st >> (8 * kStateOwn)) & (kLockBit - 1)); }
static_assert(kMaxParts <= kLockBit, "a label leaves the lock its bit");

struct RefArgs {
    std::int64_t n;
    const std::int32_t* off;
    const std::int32_t* nbr;
    const std::uint32_t* ew;
    const std::uint32_t* vw;
    int k;
    std::uint64_t cap;
    // Null on levels without edge weights, else nonzero when some edge weighs
    // more than 1 (the proposal filter's constant, incremental.cuh:897-899).
    const unsigned long long* heavy_edge;
    Label* labels;
    unsigned long long* loads;
    const double* prices;  // null unless vertex weights exceed n
    std::uint32_t* state;  // packed lanes below
    StateLane<std::int8_t> targets;  // -1: none
    std::int64_t* gains;
    // When every row of the level weighs less than 2^31, the gains are kept
    // in 32 bits here instead (gains is null): the afterburner gathers half
    // the bytes from an array half the size.
    std::int32_t* gains32;
    StateLane<std::uint8_t> own;     // label and lock
    StateLane<std::uint8_t> flags;
    StateLane<std::uint8_t> member;
    unsigned long long* ctr;
    RepairSample* samples;
    // repair
    const unsigned long long* loads0;
    std::int32_t* bucket;
    unsigned long long* counts;
};

// Part-connectivity table of one vertex in team-private LDS; returns the
// incident weight excluding self loops (src/refinement/affinity.cuh:9-66).
// Bin: the table's word (32 bits when no row of the level weighs 2^32).
template <class Team, class Bin = unsigned long long>
__device__ inline std::uint64_t team_histogram(const Team& t, const RefArgs& a, std::int64_t v, Bin* hist) {
    t.sync();  // earlier readers of the table are done
    for (int p = t.rank(); p < a.k; p += Team::size) hist[p] = 0;
    t.sync();
    std::uint64_t total = 0;
    struct Rec {
        int label;  // -1 for a self loop
        std::uint32_t w;
    };
    row_batches(
        t, a.off[v], a.off[v + 1],
        [&](std::int64_t x) {
            const std::int32_t u = a.nbr[(std::uint32_t)x];
            return Rec{u == v ? -1 : a.labels[(std::uint32_t)u], (std::uint32_t)ew_at(a.ew, x)};
        },
        [&](std::int64_t, const Rec& r) {
            if (r.label < 0) return;
            atomicAdd(&hist[r.label], (Bin)r.w);
            total += r.w;
        });
    t.sync();
    return t.sum(total);
}

// Heavy rows: one block, so each wave adds into its own table (hub rows
// put most of their entries into a few parts, and one shared table would
// serialise the whole block on those bins); the wave tables are then summed
// into hist[0, k).  The block's scratch holds 1 + waves tables.
constexpr int kHeavyTables = 1 + BlockTeam::size / kWave;
template <class Bin = unsigned long long>
__device__ inline std::uint64_t team_histogram(const BlockTeam& t, const RefArgs& a, std::int64_t v, Bin* hist) {
    constexpr int kWaves = BlockTeam::size / kWave;
    Bin* mine = hist + (threadIdx.x / kWave + 1) * a.k;
    t.sync();  // earlier readers of the table are done
    for (int i = t.rank(); i < kHeavyTables * a.k; i += BlockTeam::size) hist[i] = 0;
    t.sync();
    std::uint64_t total = 0;
    struct Rec {
        int label;  // -1 for a self loop
        std::uint32_t w;
    };
    row_batches(
        t, a.off[v], a.off[v + 1],
        [&](std::int64_t x) {
            const std::int32_t u = a.nbr[(std::uint32_t)x];
            return Rec{u == v ? -1 : a.labels[(std::uint32_t)u], (std::uint32_t)ew_at(a.ew, x)};
        },
        [&](std::int64_t, const Rec& r) {
            if (r.label < 0) return;
            atomicAdd(&mine[r.label], (Bin)r.w);
            total += r.w;
        });
    t.sync();
    for (int p = t.rank(); p < a.k; p += BlockTeam::size) {
        Bin sum = 0;
        for (int w = 1; w <= kWaves; ++w) sum += hist[w * a.k + p];
        hist[p] = sum;
    }
    t.sync();
    return t.sum(total);
}

// Short rows (light teams of at most 16 lanes, at most kTierLight entries):
// the row's labels stay in registers and only their bins are touched, so a
// table that starts zero is left zero and no per-row clear of all k bins is
// needed.  The light kernel zeroes the tables once at start.
template <int W>
struct LightRow {
    static constexpr int kPer = kTierLight / W;
    static constexpr int kWords = (kPer + 3) / 4;
    unsigned packed[kWords];  // four byte labels per word; 0xff: no entry or a self loop
    __device__ int lab(int j) const { return (int)((packed[j >> 2] >> (8 * (j & 3))) & 0xffu); }
};

template <int W, class Bin>
__device__ inline std::uint64_t light_histogram(const GroupTeam<W>& t, const RefArgs& a, std::int64_t v, Bin* hist,
                                                LightRow<W>& r) {
    const std::int64_t b = a.off[v], e = a.off[v + 1];
    std::uint64_t total = 0;
#pragma unroll
    for (int q = 0; q < LightRow<W>::kWords; ++q) r.packed[q] = 0xffffffffu;
    t.sync();  // the previous row's clean-up is done
    // Four entries per lane in flight; iterations beyond the longest row of
    // the wave are skipped as a whole (t.wave_rows_max is wave-uniform).
#pragma unroll
    for (int q = 0; q < LightRow<W>::kWords; ++q) {
        if (q * 4 * W >= t.wave_rows_max) break;
        int lab[4];
        std::uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const std::int64_t x = b + t.rank() + (q * 4 + i) * W;
            const bool in = x < e;
            const std::int32_t u = in ? a.nbr[(std::uint32_t)x] : (std::int32_t)v;
            lab[i] = u != v ? (int)a.labels[(std::uint32_t)u] : 0xff;
            w[i] = in ? (std::uint32_t)ew_at(a.ew, x) : 0u;
        }
        unsigned word = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (lab[i] != 0xff) {
                atomicAdd(&hist[lab[i]], static_cast<Bin>(w[i]));
                total += w[i];
            }
            word |= (unsigned)lab[i] << (8 * i);
        }
        r.packed[q] = word;
    }
    t.sync();
    return t.sum(total);
}

template <int W, class Bin>
__device__ inline void light_clear(const GroupTeam<W>& t, Bin* hist, const LightRow<W>& r) {
    t.sync();  // all reads of the row's bins are done
#pragma unroll
    for (int j = 0; j < LightRow<W>::kPer; ++j) {
        const int l = r.lab(j);
        if (l != 0xff) hist[l] = 0;
    }
}

template <class Team>
struct IsLight : std::false_type {};
template <int W>
struct IsLight<GroupTeam<W>> : std::integral_constant<bool, (W <= 16)> {};

// estimated_repair_cost (src/refinement/incremental.cuh:156-159).
__device__ inline double repair_cost(const RefArgs& a, int part, std::uint64_t weight) {
    const std::uint64_t slack = a.cap - a.loads[part];
    return weight > slack ? a.prices[part] * (double)(weight - slack) : 0.0;
}

struct Cand {
    int p;
    std::uint64_t conn;
    double score;
};

__device__ inline bool cand_better(const Cand& x, const Cand& y, bool priced) {
    if (x.p < 0) return false;
    if (y.p < 0) return true;
    if (priced) return x.score > y.score || (x.score == y.score && x.p < y.p);
    return x.conn > y.conn || (x.conn == y.conn && x.p < y.p);
}

template <int W>
__device__ inline Cand cand_group_reduce(Cand c, bool priced) {
    // Shuffles: with lane exchanges here the proposals of medium rows took
    // 46 us instead of 39 (R-MAT scale 18), for their registers.
    for (int d = W / 2; d; d >>= 1) {
        Cand o;
        o.p = __shfl_xor(c.p, d, W);
        o.conn = __shfl_xor(c.conn, d, W);
        o.score = __shfl_xor(c.score, d, W);
        if (cand_better(o, c, priced)) c = o;
    }
    return c;
}
template <int W>
__device__ inline Cand team_reduce(const GroupTeam<W>&, Cand c, bool priced) {
    return cand_group_reduce<W>(c, priced);
}
__device__ inline Cand team_reduce(const BlockTeam& t, Cand c, bool priced) {
    c = cand_group_reduce<kWave>(c, priced);
    __syncthreads();
    const int w = threadIdx.x / kWave;
    if (lane_id() == 0) {
        t.red[3 * w] = (unsigned long long)(long long)c.p;
        t.red[3 * w + 1] = c.conn;
        t.red[3 * w + 2] = __double_as_longlong(c.score);
    }
    __syncthreads();
    Cand r{(int)(long long)t.red[0], t.red[1], __longlong_as_double((long long)t.red[2])};
    for (int i = 1; i < BlockTeam::size / kWave; ++i) {
        Cand o{(int)(long long)t.red[3 * i], t.red[3 * i + 1], __longlong_as_double((long long)t.red[3 * i + 2])};
        if (cand_better(o, r, priced)) r = o;
    }
    __syncthreads();
    return r;
}

// Stores a vertex's proposal gain in the level's gain array (32 or 64 bits;
// the "none" value INT64_MIN is stored as INT32_MIN in 32 bits).
__device__ inline void set_gain(const RefArgs& a, std::int64_t v, std::int64_t g) {
    if (a.gains32)
        a.gains32[v] = g == INT64_MIN ? INT32_MIN : (std::int32_t)g;
    else
        a.gains[v] = g;
}

struct RowBody {
    RefArgs a;
    __device__ std::int64_t degree(std::int32_t v) const { return a.off[v + 1] - a.off[v]; }
};

// LP proposal (incremental.cuh:166-198, 229-296).  Bin is the bin type of
// the part tables: 32 bits when no row of the level weighs 2^32 or more
// (short rows: half the LDS per team, twice the resident teams; longer rows:
// one bank per LDS atomic instead of two), else 64.
template <class Bin>
struct LpProposeBody : RowBody {
    using LightBin = Bin;
    // With prices, the scored candidates read (cap - load, price) of their
    // part from an LDS copy of the part table.
    __host__ __device__ int part_words() const { return a.prices ? 2 * a.k : 0; }
    __device__ void stage(unsigned long long* t) const {
        for (int p = threadIdx.x; p < a.k; p += blockDim.x) {
            t[2 * p] = a.cap - a.loads[p];
            t[2 * p + 1] = (unsigned long long)__double_as_longlong(a.prices[p]);
        }
    }
    // estimated_repair_cost (src/refinement/incremental.cuh:156-159).
    __device__ double cost(const unsigned long long* part, int p, std::uint64_t w) const {
        const std::uint64_t slack = part ? part[2 * p] : a.cap - a.loads[p];
        const double price = part ? __longlong_as_double((long long)part[2 * p + 1]) : a.prices[p];
        return w > slack ? price * (double)(w - slack) : 0.0;
    }
    template <class Team>
    __device__ RowOut operator()(const Team& t, std::int32_t v, unsigned long long* hist) const {
        const int own = a.own[v], s = own & (kLockBit - 1);
        t.sync();
        if (t.leader()) {
            a.targets[v] = -1;
            set_gain(a, v, INT64_MIN);
            a.flags[v] = 0;
            a.own[v] = (std::uint8_t)s;
        }
        if (own & kLockBit) return RowOut{false, 0};
        const bool priced = a.prices != nullptr;
        const std::uint64_t w = a.vw[v];
        Cand best{-1, 0, 0.0};
        std::uint64_t total, current;
        auto consider = [&](int p, std::uint64_t c) {
            if (p == s || !c) return;
            Cand x{p, c, priced ? (double)c - cost(t.part, p, w) : 0.0};
            if (cand_better(x, best, priced)) best = x;
        };
        if constexpr (IsLight<Team>::value) {
            LightRow<Team::size> r;
            Bin* lh = reinterpret_cast<Bin*>(hist);
            total = light_histogram(t, a, v, lh, r);
            current = lh[s];
            if (current != total)
#pragma unroll
                for (int j = 0; j < LightRow<Team::size>::kPer; ++j) {
                    const int l = r.lab(j);
                    if (l != 0xff) consider(l, lh[l]);
                }
            best = team_reduce(t, best, priced);
            light_clear(t, lh, r);
        } else {
            Bin* bh = reinterpret_cast<Bin*>(hist);
            total = team_histogram(t, a, v, bh);
            current = bh[s];
            if (current != total)
                for (int p = t.rank(); p < a.k; p += Team::size) consider(p, bh[p]);
            best = team_reduce(t, best, priced);
        }
        if (current == total) return RowOut{false, degree(v)};
        const double filter = a.heavy_edge && *a.heavy_edge ? 0.75 : 0.25;
        const bool accept = best.p >= 0 && (best.conn >= current ||
                                            current - best.conn < (std::uint64_t)(filter * (double)current));
        if (accept && t.leader()) {
            a.targets[v] = best.p;
            set_gain(a, v, best.conn >= current ? (std::int64_t)(best.conn - current) : -(std::int64_t)(current - best.conn));
        }
        return RowOut{accept, degree(v)};
    }
};

// Afterburner (incremental.cuh:361-438).  G: the level's gain word
// (std::int32_t: gains32, else gains).
template <class G>
struct AfterBody : RowBody {
    __device__ std::int64_t gain(std::int64_t u) const {
        if constexpr (sizeof(G) == 4) {
            const std::int32_t g = a.gains32[u];
            return g == INT32_MIN ? INT64_MIN : (std::int64_t)g;
        } else {
            return a.gains[u];
        }
    }
    template <class Team>
    __device__ RowOut operator()(const Team& t, std::int32_t v, unsigned long long*) const {
        const int s = a.labels[v], tv = a.targets[v];
        const std::int64_t gv = gain(v);
        std::int64_t corr = 0;
        struct Rec {
            std::int32_t u;
            std::uint32_t st;
            std::int64_t gu;
        };
        row_batches(
            t, a.off[v], a.off[v + 1],
            [&](std::int64_t x) {
                const std::int32_t u = a.nbr[(std::uint32_t)x];
                const std::uint32_t uu = (std::uint32_t)u;
                // The gain is gathered beside the state rather than after
                // it: one round trip per batch instead of two.
                return Rec{u, a.state[uu], gain(uu)};
            },
            [&](std::int64_t x, const Rec& r) {
                const int tu = (int)(std::int8_t)((r.st >> (8 * kStateTarget)) & 0xff), lu = state_label(r.st);
                if (r.u == v || tu < 0) return;
                if (!(r.gu > gv || (r.gu == gv && r.u < v))) return;
                corr += (std::int64_t)ew_at(a.ew, x) * ((tu == tv) - (tu == s) - (lu == tv) + (lu == s));
            });
        corr = t.sum(corr);
        bool keep;
        if (a.prices) {
            const std::uint64_t w = a.vw[v];
            const double adj = repair_cost(a, s, w) - repair_cost(a, tv, w);
            keep = (double)(gv + corr) + adj >= 0;
        } else
            keep = gv + corr >= 0;
        if (t.leader()) a.flags[v] = keep;
        return RowOut{keep, 0};
    }
};

// Exact cut delta (incremental.cuh:440-547): an undirected edge is owned by
// the endpoint that moves alone, or by the larger id when both move.
struct UpdateBody : RowBody {
    bool samples;
    template <class Team>
    __device__ RowOut operator()(const Team& t, std::int32_t v, unsigned long long*) const {
        const int s = a.labels[v], tv = a.targets[v];
        std::int64_t gain = 0;
        struct Rec {
            std::int32_t u;
            std::uint32_t st;
        };
        row_batches(
            t, a.off[v], a.off[v + 1],
            [&](std::int64_t x) {
                const std::int32_t u = a.nbr[(std::uint32_t)x];
                const std::uint32_t uu = (std::uint32_t)u;
                return Rec{u, a.state[uu]};
            },
            [&](std::int64_t x, const Rec& r) {
                if (r.u == v) return;
                const int old_u = state_label(r.st), tu = (int)(std::int8_t)((r.st >> (8 * kStateTarget)) & 0xff);
                const bool moves = ((r.st >> (8 * kStateFlag)) & 0xff) != 0;
                // Most neighbours are already in the frontier: skip the
                // scattered byte store for them.
                if (!((r.st >> (8 * kStateMember)) & 0xff)) a.member[r.u] = 1;
                const int new_u = moves ? tu : old_u;
                if (!moves || r.u > v) gain += (std::int64_t)ew_at(a.ew, x) * ((s != old_u) - (tv != new_u));
            });
        gain = t.sum(gain);
        // The commit adds it to the price samples (a mover's gain word is free
        // until its next proposal resets it).
        if (samples && t.leader()) set_gain(a, v, gain);
        return RowOut{false, gain};
    }
};

// Boundary test for the frontier (incremental.cuh:214-225).
struct BoundaryBody : RowBody {
    template <class Team>
    __device__ RowOut operator()(const Team& t, std::int32_t v, unsigned long long*) const {
        const int s = a.labels[v];
        // Batches of kBatch entries per lane, with a team-wide test after
        // each: most rows of a cut graph meet another part in their first
        // batch and stop there.  The loop bound is the same for the whole
        // team, so every lane takes part in each test.
        const std::int64_t b = a.off[v], e = a.off[v + 1];
        int any = 0;
        for (std::int64_t x0 = b; x0 < e && !any; x0 += kBatch * Team::size) {
            bool other[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const std::int64_t x = x0 + t.rank() + j * Team::size;
                other[j] = false;
                if (x < e) {
                    const std::int32_t u = a.nbr[(std::uint32_t)x];
                    other[j] = u != v && a.labels[(std::uint32_t)u] != s;
                }
            }
            int mine = 0;
#pragma unroll
            for (int j = 0; j < kBatch; ++j) mine |= other[j];
            any = t.sum(mine);
        }
        if (t.leader()) {
            a.member[v] = any != 0;
            a.targets[v] = -1;
            set_gain(a, v, INT64_MIN);
            a.flags[v] = 0;
            a.own[v] = (std::uint8_t)s;
        }
        return RowOut{false, 0};
    }
};

// ------------------------------------------------- device LP loop control
// The LP round loop of one level decided on the device (the rules of the
// host loop, incremental.cuh:911-961, which lp_graph.cuh:57-92 records as a
// GPU-controlled loop), so the host can issue rounds ahead instead of reading
// counters back after each.  Its words sit behind the part loads in the
// counter block; the best loads (k words) follow them.
enum LoopWord {
    kRun = 0,      // 1 while rounds run; a round issued after the stop does nothing
    kPhase,        // rounds run
    kStale,
    kEmpty,
    kCut,
    kBestCut,
    kLpMoves,
    kReason,       // LoopReason of the stop
    kImproved,     // the last round set a new best cut: checkpoint its labels
    kAccFrontier,  // profiled runs: rows and entries of the three sweeps, summed
    kAccRowSum,
    kAccAfterE,
    kAccAfterR,
    kAccUpdateE,
    kAccUpdateR,
    kLoopWords
};
enum LoopReason { kRunning = 0, kEnded = 1, kNeedRepair = 2, kCutUnderflow = 3, kDeferred = 4 };
// Words of the loop state mirrored into the host mailbox after each round.
constexpr int kMailWords = kImproved + 1;

struct LoopParams {
    int k;
    int rounds;
    int stale_rounds;
    int graph_mode;  // stale rule in integers (graph loop) or long double
    int light_only;  // no medium launch: a deferred row is an error
    int profiling;
    std::uint64_t cap;
    std::uint64_t m0999;  // 64-bit significand of the long double 0.999, scaled by 2^64
};

// (long double)cut < 0.999L * (long double)best exactly as x87 extended
// precision evaluates it (64-bit significands, round to nearest even), in
// integers: 0.999L = m0999 / 2^64, so the product is best * m0999 / 2^64
// rounded to 64 significant bits.
__host__ __device__ inline bool below_0999(std::uint64_t cut, std::uint64_t best, std::uint64_t m0999) {
    using u128 = unsigned __int128;
    u128 p = (u128)best * m0999;
    const std::uint64_t hi = (std::uint64_t)(p >> 64);
    const int len = hi ? 128 - __builtin_clzll(hi) : 0;
    if (len > 64) {
        const int s = len - 64;
        const u128 q = p >> s;
        const u128 rem = p - (q << s);
        const u128 half = (u128)1 << (s - 1);
        const u128 r = (rem > half || (rem == half && (q & 1))) ? q + 1 : q;
        p = r << s;
    }
    return ((u128)cut << 64) < p;
}

// 0.999L as m / 2^64 (0.999L lies in [1/2, 1), so m has 64 bits).
inline std::uint64_t significand_0999() { return static_cast<std::uint64_t>(std::ldexp(0.999L, 64)); }

// Loop state at the start of a run of device-controlled rounds; clears the
// counter block; copy_best: the best loads take the current loads.
__global__ void k_lp_arm(unsigned long long* ctr, int k, unsigned long long run, unsigned long long phase,
                         unsigned long long stale, unsigned long long empty, unsigned long long cut,
                         unsigned long long best, unsigned long long lp_moves, int copy_best) {
    unsigned long long* loads = ctr + kCtrCount;
    unsigned long long* L = loads + k;
    for (int i = threadIdx.x; i < kCtrCount; i += blockDim.x) ctr[i] = 0;
    if (copy_best)
        for (int p = threadIdx.x; p < k; p += blockDim.x) L[kLoopWords + p] = loads[p];
    if (threadIdx.x == 0) {
        L[kRun] = run;
        L[kPhase] = phase;
        L[kStale] = stale;
        L[kEmpty] = empty;
        L[kCut] = cut;
        L[kBestCut] = best;
        L[kLpMoves] = lp_moves;
        L[kReason] = kRunning;
        L[kImproved] = 0;
        for (int i = kAccFrontier; i < kLoopWords; ++i) L[i] = 0;
    }
}

// What the last block of a commit does once every block is through: nothing,
// the end of an LP round (lp_decide), or the read-back of the counters and
// loads.  (A launch of its own for either took 5 us and the gap before it,
// once per round and per repair iteration.)
enum RoundEndMode { kEndNothing = 0, kEndDecide = 1, kEndRead = 2 };
struct RoundEnd {
    int mode;
    LoopParams P;
    unsigned int* ticket;
    unsigned long long* host;  // mailbox or read-back buffer
    unsigned long long* flag;
    unsigned long long seq;
    Label* keep;  // kEndDecide: see lp_decide
    bool vec;
    int words;    // kEndRead: words of the counter block on, the first kCtrClear of them cleared
};

// Copies n bytes by one block; vec: both arrays are 16-byte aligned.
__device__ inline void copy_labels(const Label* from, Label* to, std::int64_t n, bool vec) {
    const std::int64_t words = vec ? n / 16 : 0;
    for (std::int64_t i = threadIdx.x; i < words; i += blockDim.x)
        reinterpret_cast<uint4*>(to)[i] = reinterpret_cast<const uint4*>(from)[i];
    for (std::int64_t v = words * 16 + threadIdx.x; v < n; v += blockDim.x) to[v] = from[v];
}

// End of one LP round, by one block: the movers, cut delta and part loads of
// the round decide whether the loop goes on; the counter block is cleared for
// the next round and the state is mirrored to the host mailbox.
// keep: non-null on levels of at most kKeepInline vertices, where this block
// also checkpoints the labels of an improving round (n bytes from labels to
// keep) instead of a separate k_lp_keep launch.
constexpr std::int64_t kKeepInline = 131072;
__device__ inline void lp_decide(unsigned long long* ctr, const LoopParams& P, unsigned long long* mailbox,
                                 unsigned long long* flag, unsigned long long seq, const Label* labels, Label* keep,
                                 bool vec, std::int64_t n) {
    unsigned long long* loads = ctr + kCtrCount;
    unsigned long long* L = loads + P.k;
    __shared__ int s_run, s_improved, s_stop;
    __shared__ unsigned long long s_words[kLoopWords];
    __shared__ unsigned long long s_max[1024 / kWave];
    // Largest part load, by every thread.
    unsigned long long mx = 0;
    for (int p = threadIdx.x; p < P.k; p += blockDim.x) mx = loads[p] > mx ? loads[p] : mx;
    mx = wave_max(mx);
    if (lane_id() == 0) s_max[threadIdx.x / kWave] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (unsigned i = 1; i < blockDim.x / kWave; ++i) mx = s_max[i] > mx ? s_max[i] : mx;
        s_run = L[kRun] != 0;
        s_improved = 0;
        s_stop = 0;
        L[kImproved] = 0;
        if (s_run) {
            const std::uint64_t phase = L[kPhase] + 1;
            std::uint64_t stale = L[kStale], empty = L[kEmpty], cut = L[kCut], best = L[kBestCut];
            const std::uint64_t movers = ctr[kMovers];
            const std::int64_t delta = (std::int64_t)ctr[kDelta];
            int reason = kRunning;
            if (P.profiling) {
                L[kAccFrontier] += ctr[kFrontier];
                L[kAccRowSum] += ctr[kRowSum];
                L[kAccAfterE] += ctr[kEntAfter];
                L[kAccAfterR] += ctr[kEntAfter + 1];
                L[kAccUpdateE] += ctr[kEntUpdate];
                L[kAccUpdateR] += ctr[kEntUpdate + 1];
            }
            if (P.light_only && (ctr[kTier] || ctr[kTierB] || ctr[kTierC])) {
                reason = kDeferred;
            } else if (!movers) {
                if (++empty >= 2)
                    reason = kEnded;
                else
                    ++stale;
            } else {
                empty = 0;
                if (delta >= 0 && (std::uint64_t)delta > cut) {
                    reason = kCutUnderflow;
                } else {
                    cut = delta >= 0 ? cut - (std::uint64_t)delta : cut + (std::uint64_t)(-delta);
                    L[kLpMoves] += movers;
                    if (mx > P.cap) {
                        reason = kNeedRepair;  // the host repairs and finishes the round
                    } else {
                        ++stale;
                        if (cut < best) {
                            if (P.graph_mode ? best - cut > best / 1000 : below_0999(cut, best, P.m0999)) stale = 0;
                            best = cut;
                            s_improved = 1;
                            L[kImproved] = 1;
                        }
                    }
                }
            }
            if (reason == kRunning && !(phase < (std::uint64_t)P.rounds && stale < (std::uint64_t)P.stale_rounds))
                reason = kEnded;
            L[kPhase] = phase;
            L[kStale] = stale;
            L[kEmpty] = empty;
            L[kCut] = cut;
            L[kBestCut] = best;
            L[kReason] = reason;
            if (reason != kRunning) {
                L[kRun] = 0;
                s_stop = 1;
            }
            for (int i = 0; i < kLoopWords; ++i) s_words[i] = L[i];
        }
    }
    __syncthreads();
    if (!s_run) {
        publish_to_host(flag, seq);
        return;
    }
    // Running: the first kMailWords loop words to the mailbox; stopped:
    // every loop word, then the loads and the best loads.
    for (int i = threadIdx.x; i < (s_stop ? (int)kLoopWords : kMailWords); i += blockDim.x) mailbox[i] = s_words[i];
    for (int p = threadIdx.x; p < P.k; p += blockDim.x) {
        const unsigned long long load = loads[p];
        const unsigned long long best = s_improved ? load : L[kLoopWords + p];
        if (s_improved) L[kLoopWords + p] = load;
        if (s_stop) {
            mailbox[kLoopWords + p] = load;
            mailbox[kLoopWords + P.k + p] = best;
        }
    }
    publish_to_host(flag, seq);
    for (int i = threadIdx.x; i < kCtrCount; i += blockDim.x) ctr[i] = 0;
    if (keep && s_improved) copy_labels(labels, keep, n, vec);
}

// incremental_commit (incremental.cuh:532-547) with per-block load deltas;
// with samples also the repair's price samples, from the gains the update
// sweep left at the movers.  Sums per part meet in LDS and reach global memory
// once per block, and the blocks are few and large (kCommitBlocks): k atomics
// per block on k words queue up, 40 ns a block at k = 64.  (The samples were
// two global atomics per mover in the update sweep, 77 us of its 90 on the
// repairs of R-MAT scale 19 at k = 32.)
constexpr int kCommitThreads = 1024;
constexpr int kCommitBlocks = 128;
//
// donors: null, or the donor list of the repair iteration, of selected[2]
// entries: those that were not admitted lose their target
// (rebalance_graph.cuh:155) unless the reservation is still to come (not
// settled, and more eligible donors, selected[0], than one tail launch takes,
// selected[1]).
__global__ void __launch_bounds__(kCommitThreads) k_commit(RefArgs a, const std::int32_t* list,
                                                           const unsigned long long* count_ptr, bool lp, bool samples,
                                                           const std::int32_t* donors,
                                                           const unsigned long long* selected, bool settled,
                                                           RoundEnd end) {
    __shared__ unsigned long long delta[kMaxParts], loss[kMaxParts], weight[kMaxParts];
    const std::int64_t count = (std::int64_t)*count_ptr;
    if (donors && (settled || selected[0] == selected[1])) {
        const std::int64_t nd = (std::int64_t)selected[2];
        for (std::int64_t i = blockIdx.x * (std::int64_t)kCommitThreads + threadIdx.x; i < nd;
             i += (std::int64_t)gridDim.x * kCommitThreads) {
            const std::int32_t v = donors[i];
            if (!a.flags[v]) a.targets[v] = -1;
        }
    }
    if (blockIdx.x * (std::int64_t)kCommitThreads < count) {
        for (int p = threadIdx.x; p < a.k; p += kCommitThreads) {
            delta[p] = 0;
            loss[p] = 0;
            weight[p] = 0;
        }
        __syncthreads();
        for (std::int64_t i = blockIdx.x * (std::int64_t)kCommitThreads + threadIdx.x; i < count;
             i += (std::int64_t)gridDim.x * kCommitThreads) {
            const std::int32_t v = list[i];
            const int s = a.labels[v], t = a.targets[v];
            const unsigned long long w = a.vw[v];
            atomicAdd(&delta[s], 0ULL - w);
            atomicAdd(&delta[t], w);
            if (samples) {
                const std::int64_t gain = a.gains32 ? (std::int64_t)a.gains32[v] : a.gains[v];
                atomicAdd(&loss[s], (unsigned long long)(-gain));
                atomicAdd(&weight[s], w);
            }
            a.labels[v] = (Label)t;
            a.own[v] = (std::uint8_t)((lp ? kLockBit : a.own[v] & kLockBit) | t);
            a.member[v] = 1;
        }
        __syncthreads();
        for (int p = threadIdx.x; p < a.k; p += kCommitThreads) {
            if (delta[p]) atomicAdd(&a.loads[p], delta[p]);
            if (loss[p]) atomicAdd(&a.samples[p].loss, loss[p]);
            if (weight[p]) atomicAdd(&a.samples[p].weight, weight[p]);
        }
    }
    if (end.mode == kEndNothing || !block_is_last(end.ticket)) return;
    if (end.mode == kEndDecide) {
        lp_decide(a.ctr, end.P, end.host, end.flag, end.seq, a.labels, end.keep, end.vec, a.n);
    } else {
        for (int i = threadIdx.x; i < end.words; i += kCommitThreads) {
            end.host[i] = a.ctr[i];
            if (i < kCtrClear) a.ctr[i] = 0;
        }
        publish_to_host(end.flag, end.seq);
    }
}

// Clears the moving flag and the target of every vertex and takes over its
// label (restored from a checkpoint by the host).
__global__ void k_clear_moves(std::uint32_t* state, const Label* labels, std::int64_t n) {
    const std::uint32_t keep = (0xffu << (8 * kStateMember)) | ((std::uint32_t)kLockBit << (8 * kStateOwn));
    for (std::int64_t v = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < n;
         v += (std::int64_t)gridDim.x * blockDim.x)
        state[v] = (state[v] & keep) | (0xffu << (8 * kStateTarget)) | ((std::uint32_t)labels[v] << (8 * kStateOwn));
}

// Frontier list from member flags (order irrelevant: per-vertex decisions).
// Each wave reads kScanRounds x 64 consecutive flags before appending them.
constexpr int kScanRounds = 8;
// Large blocks: each reserves its part of the list with one atomic.
constexpr int kCompactThreads = 1024;
constexpr int kCompactTile = kCompactThreads * kScanRounds;
// gate: null, or a device word; when it is zero the launch does nothing (a
// round of a device-controlled loop that has ended).
template <typename F>
__global__ void __launch_bounds__(kCompactThreads) k_compact_flags(std::int64_t n, F flags, std::int32_t* out,
                                                                   unsigned long long* count,
                                                                   const unsigned long long* gate) {
    if (gate && !*gate) return;
    __shared__ std::int32_t sb[kCompactThreads / kWave][kStage];
    Stage st{sb[threadIdx.x / kWave], out, count, 0};
    const std::int64_t wave = (blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x) / kWave;
    const std::int64_t waves = (std::int64_t)gridDim.x * blockDim.x / kWave;
    for (std::int64_t base = wave * (kWave * kScanRounds); base < n; base += waves * (kWave * kScanRounds)) {
        bool f[kScanRounds];
#pragma unroll
        for (int r = 0; r < kScanRounds; ++r) {
            const std::int64_t v = base + r * kWave + lane_id();
            f[r] = v < n && flags[v] != 0;
        }
#pragma unroll
        for (int r = 0; r < kScanRounds; ++r) st.push(f[r], (std::int32_t)(base + r * kWave + lane_id()));
    }
    block_flush<1>({&st}, 0, nullptr);
}

// ------------------------------------------------------------- repair
// pow15: the table kPow15 (the block's LDS copy: the search is a chain of six
// loads).
__device__ inline int gain_bucket(const double* pow15, double gain) {
    if (gain > 0) return 0;
    if (gain == 0) return 1;
    // First j in -23..23 with x <= 1.5^j gives bucket 25 + j (at least 2);
    // beyond the table, 49.  Equivalently 2 + #{table entries below x}.
    const double x = -gain;
    int lo = 0, hi = 47;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (pow15[mid] < x)
            lo = mid + 1;
        else
            hi = mid;
    }
    return 2 + lo;
}

// Donor flags, resets (flags, bucket) on frozen loads.
// With counts set it also starts the repair iteration: the bucket weights
// cleared and loads0 = loads, as k_repair_begin does but for the counter
// block, which the caller knows to be zero.  The donor test then reads the
// part loads themselves, the values loads0 is given.
__global__ void __launch_bounds__(kCompactThreads) k_repair_donors(RefArgs a, std::int32_t* donors,
                                                                   unsigned long long* count,
                                                                   unsigned long long* loads0,
                                                                   unsigned long long* counts, std::int64_t ncounts) {
    __shared__ std::int32_t sb[kCompactThreads / kWave][kStage];
    if (counts)
        for (std::int64_t i = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; i < ncounts;
             i += (std::int64_t)gridDim.x * blockDim.x) {
            counts[i] = 0;
            if (i < a.k) loads0[i] = a.loads[i];
        }
    const unsigned long long* frozen = counts ? a.loads : a.loads0;
    Stage st{sb[threadIdx.x / kWave], donors, count, 0};
    const std::int64_t wave = (blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x) / kWave;
    const std::int64_t waves = (std::int64_t)gridDim.x * blockDim.x / kWave;
    for (std::int64_t base = wave * (kWave * kScanRounds); base < a.n; base += waves * (kWave * kScanRounds)) {
        int lab[kScanRounds];
#pragma unroll
        for (int r = 0; r < kScanRounds; ++r) {
            const std::int64_t v = base + r * kWave + lane_id();
            lab[r] = v < a.n ? (int)a.labels[v] : -1;
        }
#pragma unroll
        for (int r = 0; r < kScanRounds; ++r) {
            const std::int64_t v = base + r * kWave + lane_id();
            bool d = false;
            if (lab[r] >= 0) {
                a.flags[v] = 0;
                a.bucket[v] = -1;
                d = frozen[lab[r]] > a.cap;
            }
            st.push(d, (std::int32_t)v);
        }
    }
    block_flush<1>({&st}, 0, nullptr);
}

struct RepairPick {
    int p;
    std::uint64_t conn, slack;
};
__device__ inline bool pick_better(const RepairPick& x, const RepairPick& y) {
    if (x.p < 0) return false;
    if (y.p < 0) return true;
    return x.conn > y.conn || (x.conn == y.conn && (x.slack > y.slack || (x.slack == y.slack && x.p < y.p)));
}
template <int W>
__device__ inline RepairPick pick_group_reduce(RepairPick c) {
    for (int d = W / 2; d; d >>= 1) {  // shuffles, as in cand_group_reduce
        RepairPick o;
        o.p = __shfl_xor(c.p, d, W);
        o.conn = __shfl_xor(c.conn, d, W);
        o.slack = __shfl_xor(c.slack, d, W);
        if (pick_better(o, c)) c = o;
    }
    return c;
}
template <int W>
__device__ inline RepairPick team_reduce(const GroupTeam<W>&, RepairPick c) {
    return pick_group_reduce<W>(c);
}
__device__ inline RepairPick team_reduce(const BlockTeam& t, RepairPick c) {
    c = pick_group_reduce<kWave>(c);
    __syncthreads();
    const int w = threadIdx.x / kWave;
    if (lane_id() == 0) {
        t.red[3 * w] = (unsigned long long)(long long)c.p;
        t.red[3 * w + 1] = c.conn;
        t.red[3 * w + 2] = c.slack;
    }
    __syncthreads();
    RepairPick r{(int)(long long)t.red[0], t.red[1], t.red[2]};
    for (int i = 1; i < BlockTeam::size / kWave; ++i) {
        RepairPick o{(int)(long long)t.red[3 * i], t.red[3 * i + 1], t.red[3 * i + 2]};
        if (pick_better(o, r)) r = o;
    }
    __syncthreads();
    return r;
}

// enumerate_repair_destination (rebalance_select.cuh:8-75) on frozen loads,
// then the gain bucket (incremental.cuh:559-626).
// load0: the frozen part loads (the block's LDS copy where it has one).
// Block-level table of repair bucket sums in LDS: kAggSlots keys (u32 count
// slots, all ones when free) packed two per word, then kAggSlots u64 sums.
// Linear probing over at most kAggProbes slots; a sum that finds no slot goes
// to global memory directly.  Sums are order-independent, so the counts are
// the same with or without the table.
constexpr int kAggSlots = 512;
constexpr int kAggProbes = 8;
constexpr int kAggWords = kAggSlots / 2 + kAggSlots;

__device__ inline bool agg_add(unsigned long long* agg, std::uint32_t key, unsigned long long w) {
    std::uint32_t* keys = reinterpret_cast<std::uint32_t*>(agg);
    unsigned long long* sums = agg + kAggSlots / 2;
    std::uint32_t h = mix32(key) & (kAggSlots - 1);
    for (int probe = 0; probe < kAggProbes; ++probe) {
        const std::uint32_t old = atomicCAS(&keys[h], 0xffffffffu, key);
        if (old == 0xffffffffu || old == key) {
            atomicAdd(&sums[h], w);
            return true;
        }
        h = (h + 1) & (kAggSlots - 1);
    }
    return false;
}

// Words of the table a repair-proposal block stages in LDS: frozen loads, the
// bucket sums above, prefix sums of the parts' room in part order, their
// total, the smallest room of a part with any, and the powers of 1.5.
struct RepairTable {
    int k;
    __host__ __device__ int rooms() const { return k + kAggWords; }
    __host__ __device__ int total() const { return rooms() + k; }
    __host__ __device__ int smallest() const { return total() + 1; }  // 0: room sums might wrap
    __host__ __device__ int pow15() const { return total() + 2; }
    __host__ __device__ int words() const { return pow15() + 48; }
};

// Destination of a donor without an admissible connected part: a hash picks a
// unit of room among the parts that can take its weight (in part order).
// The sum and the search go over all parts, so they are split over the team's
// lanes; a donor no heavier than the smallest room (every donor of unit
// weight) can go to any part with room, and the table's prefix sums answer it
// with a binary search.  One lane walking the k parts twice was most of the
// light proposal sweep at k = 128: most donors of an overloaded part lie in
// its inside (300,007 weighted vertices: 55 us a sweep, now 29).
template <int W>
__device__ inline int repair_route(const RefArgs& a, std::int64_t v, int s, std::uint64_t w,
                                   const unsigned long long* tab, int lg) {
    const RepairTable at{a.k};
    const std::uint32_t h = mix32((std::uint32_t)v);
    auto ticket_of = [&](std::uint64_t tot) {
        return tot <= 0xffffffffULL ? (std::uint64_t)(h % (std::uint32_t)tot) : (std::uint64_t)h % tot;
    };
    if (w <= tab[at.smallest()] && tab[at.smallest()]) {
        const std::uint64_t tot = tab[at.total()];
        if (!tot) return -1;
        const std::uint64_t ticket = ticket_of(tot);
        int lo = 0, hi = a.k - 1;  // the last part whose prefix is at or below the ticket
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (tab[at.rooms() + mid] <= ticket)
                lo = mid;
            else
                hi = mid - 1;
        }
        return lo;
    }
    const int per = (a.k + W - 1) / W, p0 = lg * per, p1 = p0 + per < a.k ? p0 + per : a.k;
    auto room = [&](int p) {
        const std::uint64_t l = tab[p];
        return p != s && l < a.cap && w <= a.cap - l ? a.cap - l : 0;
    };
    std::uint64_t own = 0;  // saturating, as the ticket range is
    for (int p = p0; p < p1; ++p) {
        const std::uint64_t sl = room(p);
        own = ~0ULL - own < sl ? ~0ULL : own + sl;
    }
    std::uint64_t inc = own;
    for (int d = 1; d < W; d <<= 1) {
        const std::uint64_t y = __shfl_up(inc, d, W);
        if (lg >= d) inc = ~0ULL - inc < y ? ~0ULL : inc + y;
    }
    const std::uint64_t before = __shfl_up(inc, 1, W);
    const std::uint64_t exc = lg ? before : 0;
    const std::uint64_t tot = __shfl(inc, W - 1, W);
    if (!tot) return -1;
    std::uint64_t ticket = ticket_of(tot);
    int pick = -1;
    if (ticket >= exc && ticket - exc < own) {
        ticket -= exc;
        for (int p = p0; p < p1; ++p) {
            const std::uint64_t sl = room(p);
            if (ticket < sl) {
                pick = p;
                break;
            }
            ticket -= sl;
        }
    }
    for (int d = W / 2; d; d >>= 1) {
        const int o = __shfl_xor(pick, d, W);
        pick = o > pick ? o : pick;
    }
    return pick;
}

// Called by every lane of the team; W lanes share the routing (lg: the lane
// among them) and one writes.
template <int W>
__device__ inline void repair_finish(const RefArgs& a, std::int64_t v, int s, std::uint64_t w, std::uint64_t current,
                                     RepairPick best, unsigned long long* tab, int lg, bool writer) {
    if (best.p < 0) {
        best.conn = 0;
        best.p = repair_route<W>(a, v, s, w, tab, lg);
    }
    if (!writer) return;
    a.targets[v] = best.p;
    if (best.p < 0) return;
    const RepairTable at{a.k};
    const double gain = best.conn >= current ? (double)(best.conn - current) : -(double)(current - best.conn);
    const std::uint64_t excess = tab[s] - a.cap;
    const std::uint64_t relief = w < excess ? w : excess;
    const double gpw = gain / (double)relief;
    const int lb = gain_bucket(reinterpret_cast<const double*>(tab + at.pow15()), gpw) * kBalanceSections +
                   (int)(mix32((std::uint32_t)v) % kBalanceSections);
    a.bucket[v] = s * kBalanceWidth + lb;
    const std::uint32_t slot = (std::uint32_t)(s * kBalanceWidth + count_slot(lb));
    if (!agg_add(tab + a.k, slot, (unsigned long long)w)) atomicAdd(&a.counts[slot], (unsigned long long)w);
}

template <class Bin>
struct RepairProposeBody : RowBody {
    using LightBin = Bin;
    // Frozen part loads in LDS for the destination scan, then the block's
    // table of bucket sums: the donors of one part mostly share a few
    // buckets, so each block adds its sums to the global counts once.
    __host__ __device__ int part_words() const { return RepairTable{a.k}.words(); }
    __device__ void stage(unsigned long long* t) const {
        const RepairTable at{a.k};
        for (int p = threadIdx.x; p < a.k; p += blockDim.x) t[p] = a.loads0[p];
        for (int i = threadIdx.x; i < kAggWords; i += blockDim.x) t[a.k + i] = i < kAggSlots / 2 ? ~0ULL : 0ULL;
        for (int i = threadIdx.x; i < 48; i += blockDim.x)
            t[at.pow15() + i] = (unsigned long long)__double_as_longlong(kPow15.p[i]);
        if (threadIdx.x < kWave) {
            std::uint64_t sum = 0, smallest = ~0ULL;
            for (int p0 = 0; p0 < a.k; p0 += kWave) {
                const int p = p0 + lane_id();
                const std::uint64_t l = p < a.k ? a.loads0[p] : a.cap;
                const std::uint64_t room = l < a.cap ? a.cap - l : 0;
                if (room && room < smallest) smallest = room;
                const std::uint64_t inc = wave_inclusive_scan<PlusOp>(room);
                if (p < a.k) t[at.rooms() + p] = sum + inc - room;
                sum += __shfl(inc, kWave - 1);
            }
            smallest = ~wave_max(~smallest);
            if (lane_id() == 0) {
                t[at.total()] = sum;
                t[at.smallest()] = a.cap < (1ULL << 55) ? smallest : 0;  // at most 128 rooms below 2^63
            }
        }
    }
    __device__ void flush(const unsigned long long* t) const {
        const std::uint32_t* keys = reinterpret_cast<const std::uint32_t*>(t + a.k);
        const unsigned long long* sums = t + a.k + kAggSlots / 2;
        for (int i = threadIdx.x; i < kAggSlots; i += blockDim.x)
            if (keys[i] != 0xffffffffu && sums[i]) atomicAdd(&a.counts[keys[i]], sums[i]);
    }
    template <class Team>
    __device__ RowOut operator()(const Team& t, std::int32_t v, unsigned long long* hist) const {
        const int s = a.labels[v];
        const std::uint64_t w = a.vw[v];
        RepairPick best{-1, 0, 0};
        unsigned long long* tab = const_cast<unsigned long long*>(t.part);
        const unsigned long long* load0 = tab;
        auto consider = [&](int p, std::uint64_t c) {
            if (p == s || !c || load0[p] >= a.cap || w > a.cap - load0[p]) return;
            RepairPick x{p, c, a.cap - load0[p]};
            if (pick_better(x, best)) best = x;
        };
        std::uint64_t total, current;
        if constexpr (IsLight<Team>::value) {
            LightRow<Team::size> r;
            Bin* lh = reinterpret_cast<Bin*>(hist);
            total = light_histogram(t, a, v, lh, r);
            current = lh[s];
            if (current != total)
#pragma unroll
                for (int j = 0; j < LightRow<Team::size>::kPer; ++j) {
                    const int l = r.lab(j);
                    if (l != 0xff) consider(l, lh[l]);
                }
            best = team_reduce(t, best);
            light_clear(t, lh, r);
        } else {
            Bin* bh = reinterpret_cast<Bin*>(hist);
            total = team_histogram(t, a, v, bh);
            current = bh[s];
            if (current != total)
                for (int p = t.rank(); p < a.k; p += Team::size) consider(p, bh[p]);
            best = team_reduce(t, best);
        }
        // A block team's waves all find the same route; one thread writes.
        constexpr int kRouteLanes = Team::size < kWave ? Team::size : kWave;
        repair_finish<kRouteLanes>(a, v, s, w, current, best, tab, t.rank() % kRouteLanes, t.leader());
        return RowOut{false, 0};
    }
};

// Per overloaded part: exclusive prefix over the 800 buckets and the bucket
// that contains the excess threshold (balance_scan_buckets, incremental.cuh:628-652).
// One block per part; the first bucket whose range contains the excess is
// the minimum over buckets that satisfy the test.
__global__ void __launch_bounds__(kScanThreads) k_bucket_scan(RefArgs a, unsigned long long* prefix,
                                                             std::int32_t* bstar, unsigned long long* excess) {
    __shared__ unsigned long long wsum[kScanThreads / kWave];
    __shared__ int star;
    const int p = blockIdx.x;
    if (!(a.loads0[p] > a.cap)) {
        if (threadIdx.x == 0) {
            bstar[p] = -1;
            excess[p] = 0;
        }
        return;
    }
    const unsigned long long ex = a.loads0[p] - a.cap;
    if (threadIdx.x == 0) star = kBalanceWidth;
    __syncthreads();
    unsigned long long carry = 0;
    for (int b0 = 0; b0 < kBalanceWidth; b0 += kScanThreads) {
        const int b = b0 + threadIdx.x;
        const unsigned long long cnt = b < kBalanceWidth ? a.counts[p * kBalanceWidth + count_slot(b)] : 0;
        unsigned long long inc, exc, tot;
        block_scan<PlusOp>(cnt, wsum, inc, exc, tot);
        const unsigned long long sum = carry + exc;
        if (b < kBalanceWidth) {
            prefix[p * kBalanceWidth + b] = sum;
            if (cnt && sum < ex && ex <= sum + cnt) atomicMin(&star, b);
        }
        carry += tot;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        bstar[p] = star;
        excess[p] = ex;
    }
}

// Position of the calling lane among the team's lanes with pred set, and
// their number (every lane of the team calls it).
template <int W>
__device__ inline int team_ballot_prefix(const GroupTeam<W>& t, bool pred, int& total) {
    const unsigned long long m = __ballot(pred);
    const unsigned long long bits = W == kWave ? m : (m >> (lane_id() & ~(W - 1))) & ((1ULL << W) - 1ULL);
    total = __popcll(bits);
    return __popcll(bits & ((1ULL << t.lg) - 1ULL));
}
__device__ inline int team_ballot_prefix(const BlockTeam& t, bool pred, int& total) {
    constexpr int kWaves = BlockTeam::size / kWave;
    const unsigned long long m = __ballot(pred);
    const int w = threadIdx.x / kWave;
    __syncthreads();
    if (lane_id() == 0) t.red[w] = (unsigned long long)__popcll(m);
    __syncthreads();
    int before = 0;
    total = 0;
    for (int i = 0; i < kWaves; ++i) {
        if (i < w) before += (int)t.red[i];
        total += (int)t.red[i];
    }
    __syncthreads();
    return before + __popcll(m & ((1ULL << lane_id()) - 1ULL));
}

// Sparse connection rows: the parts a listed donor connects to, in part
// order, as (weight, part) pairs in slots [0, nnz) of its k slots, by the
// row tiers over the positions [0, ne) of the donor list E (the tier
// kernels hand the position over as the row id): short rows take 4-lane
// teams, hub rows whole blocks; team ballots give each nonzero part's slot.
template <class Bin>
struct ConnBody : RowBody {
    using LightBin = Bin;
    const std::int32_t* E;
    const std::uint8_t* skip;  // null, or nonzero for donors whose row is not needed
    unsigned long long* vals;
    std::uint8_t* parts;
    std::uint8_t* nnz;
    __device__ std::int64_t degree(std::int32_t i) const {
        const std::int32_t v = E[i];
        return a.off[v + 1] - a.off[v];
    }
    template <class Team>
    __device__ void emit(const Team& t, std::int64_t i, const Bin* bh) const {
        int base = 0;
        for (int p0 = 0; p0 < a.k; p0 += Team::size) {
            const int p = p0 + t.rank();
            const unsigned long long c = p < a.k ? (unsigned long long)bh[p] : 0ULL;
            int cnt = 0;
            const int pos = team_ballot_prefix(t, c != 0, cnt);
            if (c) {
                const std::int64_t j = i * a.k + base + pos;
                vals[j] = c;
                parts[j] = static_cast<std::uint8_t>(p);
            }
            base += cnt;
        }
        if (t.leader()) nnz[i] = static_cast<std::uint8_t>(base);
    }
    template <class Team>
    __device__ RowOut operator()(const Team& t, std::int32_t i, unsigned long long* hist) const {
        if (skip && skip[i]) return RowOut{false, 0};
        const std::int32_t v = E[i];
        Bin* bh = reinterpret_cast<Bin*>(hist);
        if constexpr (IsLight<Team>::value) {
            LightRow<Team::size> r;
            light_histogram(t, a, v, bh, r);
            emit(t, i, bh);
            light_clear(t, bh, r);
        } else {
            team_histogram(t, a, v, bh);
            emit(t, i, bh);
        }
        return RowOut{false, 0};
    }
};


// Receiver reservation (rebalance_graph.cuh:86-156) in canonical order:
// requesters of one part are ranked by vertex id on top of the part's
// request total at the start of the attempt.  A rank is an exclusive
// weighted prefix among earlier items with the same key, computed without
// sorting: per-tile key sums, a per-key scan over tiles, then in-tile
// prefixes from wave scans per distinct key.
constexpr int kKeyTile = 1024;
constexpr int kKeyRounds = kKeyTile / kTierThreads;

// Exclusive weighted prefix among lanes with the same key (lower lanes
// first); wt[key] receives the wave's total for every key present.  key < 0
// marks a lane without a key; keys are below kMaxParts.  All lanes of the wave
// call it.  The lanes are put in (key, lane) order by seven ballots and one
// permute, scanned once, and read their key's first prefix back: about 20
// lane moves whatever the keys.  A scan per distinct key, the earlier form,
// took eight dependent moves for each of them: with some fifty parts asked for
// in a wave (weighted graph, k = 128) the reservation tail took 50 us on
// average and takes 38; the admission on R-MAT scale 18 (k = 64) 24 and 11.
__device__ inline std::uint64_t wave_keyed_exclusive(int key, std::uint32_t w, unsigned long long* wt) {
    static_assert(kMaxParts <= 128, "seven key bits");
    const unsigned long long lt = (1ULL << lane_id()) - 1ULL;
    const unsigned long long valid = __ballot(key >= 0);
    unsigned long long peers = valid;  // lanes with a key equal in the bits seen
    int less = 0;                      // lanes with a smaller key
#pragma unroll
    for (int b = 6; b >= 0; --b) {
        const bool bit = (key >> b) & 1;
        const unsigned long long ones = __ballot(bit);
        less += bit ? __popcll(peers & ~ones) : 0;
        peers &= bit ? ones : ~ones;
    }
    const int before = __popcll(peers & lt);
    const int pos = key >= 0 ? less + before : __popcll(valid) + __popcll(~valid & lt);
    const std::uint32_t mine = (std::uint32_t)__builtin_amdgcn_ds_permute(pos * 4, key >= 0 ? (int)w : 0);
    const std::uint64_t inc = wave_inclusive_scan<PlusOp>((std::uint64_t)mine);
    const std::uint64_t exc = inc - mine;
    const std::uint64_t at = __shfl(exc, pos);
    const std::uint64_t first = __shfl(exc, key >= 0 ? less : 0);
    const std::uint64_t end = __shfl(inc, key >= 0 ? less + __popcll(peers) - 1 : 0);
    if (key < 0) return 0;
    if (before == 0) wt[key] = end - first;
    return at - first;
}

// Per-key exclusive scan over tiles (one wave per key, four keys a block);
// with requests, ranks start at the request totals and the totals advance by
// this attempt's requests.
__global__ void __launch_bounds__(kTierThreads) k_keyed_scan(unsigned long long* S, int nb, int k,
                                                            unsigned long long* requests) {
    const int lane = lane_id();
    const int c = blockIdx.x * (kTierThreads / kWave) + threadIdx.x / kWave;
    if (c >= k) return;
    unsigned long long carry = requests ? requests[c] : 0;
    for (int b0 = 0; b0 < nb; b0 += kWave) {
        const int b = b0 + lane;
        const unsigned long long own = b < nb ? S[(std::int64_t)c * nb + b] : 0;
        const std::uint64_t x = wave_inclusive_scan<PlusOp>((std::uint64_t)own);
        if (b < nb) S[(std::int64_t)c * nb + b] = carry + x - own;
        carry += __shfl(x, kWave - 1);
    }
    if (requests && lane == 0) requests[c] = carry;
}

// In-tile ranks in index order; f(i, key, weight, rank) returns whether i
// is appended to the stage list.
template <class F>
__global__ void __launch_bounds__(kTierThreads) k_keyed_apply(const std::int32_t* keys, std::int64_t n,
                                                             const unsigned long long* S, int nb, F f,
                                                             std::int32_t* list, unsigned long long* count) {
    __shared__ unsigned long long wt[kTierThreads / kWave][kMaxParts];
    __shared__ unsigned long long run[kMaxParts];
    __shared__ std::int32_t sb[kTierThreads / kWave][kStage];
    const int w = threadIdx.x / kWave;
    Stage st{sb[w], list, count, 0};
    for (int c = threadIdx.x; c < kMaxParts; c += kTierThreads) {
        run[c] = 0;
        for (int i = 0; i < kTierThreads / kWave; ++i) wt[i][c] = 0;
    }
    __syncthreads();
    const std::int64_t base = blockIdx.x * (std::int64_t)kKeyTile;
    for (int r = 0; r < kKeyRounds; ++r) {
        const std::int64_t i = base + r * kTierThreads + threadIdx.x;
        const int key = i < n ? keys[i] : -1;
        const std::uint32_t wgt = key >= 0 ? f.weight(i) : 0;
        const std::uint64_t ex = wave_keyed_exclusive(key, wgt, wt[w]);
        __syncthreads();
        bool append = false;
        if (key >= 0) {
            std::uint64_t rank = S[(std::int64_t)key * nb + blockIdx.x] + run[key] + ex;
            for (int j = 0; j < w; ++j) rank += wt[j][key];
            append = f(i, key, wgt, rank);
        }
        st.push(append, append ? f.vertex(i) : 0);
        __syncthreads();
        for (int c = threadIdx.x; c < kMaxParts; c += kTierThreads) {
            unsigned long long add = 0;
            for (int j = 0; j < kTierThreads / kWave; ++j) {
                add += wt[j][c];
                wt[j][c] = 0;
            }
            run[c] += add;
        }
        __syncthreads();
    }
    st.flush();
}

// Per-tile key weight sums (S is key-major: S[key * nb + tile]).
template <class F>
__device__ inline void tile_key_sums(const std::int32_t* keys, std::int64_t n, int k, int nb, const F& f,
                                     unsigned long long* acc, unsigned long long* S) {
    __syncthreads();
    const std::int64_t base = blockIdx.x * (std::int64_t)kKeyTile;
    for (int r = 0; r < kKeyRounds; ++r) {
        const std::int64_t i = base + r * kTierThreads + threadIdx.x;
        if (i < n && keys[i] >= 0) atomicAdd(&acc[keys[i]], (unsigned long long)f.weight(i));
    }
    __syncthreads();
    for (int c = threadIdx.x; c < k; c += kTierThreads) S[(std::int64_t)c * nb + blockIdx.x] = acc[c];
}

// Donor selection of a repair iteration (rebalance_graph.cuh:86-110): of the
// donors in vertex order, those whose bucket lies below their part's boundary
// bucket, and those inside it while the weight of earlier donors of that
// bucket stays under the excess.  Three launches over tiles of consecutive
// vertices, none of which the host waits for: each tile's weights inside the
// boundary buckets; the eligible donors, ranked on top of the earlier tiles'
// weights, and their number per tile; the list E of them with the state the
// reservation starts from.  (Flags, a four-launch compaction, a read-back,
// keys, a scan, ranks, a second compaction and read-back and the set-up took
// its place before: 14 launches and two host waits, of 20 and three in the
// whole iteration.)
constexpr int kSelectWaves = kSelectThreads / kWave;

// A live donor as the attempts read it: index into the eligible list, the
// vertex, its weight and label (one 16-byte load per donor).
struct DonorInfo {
    std::int32_t e;
    std::int32_t v;
    std::uint32_t w;
    std::int32_t label;
};

struct SelectState {
    const std::int32_t* bstar;          // boundary bucket per part, -1 when not overloaded
    const unsigned long long* prefix;   // weight below each bucket of its part
    const unsigned long long* excess;   // weight a part has to lose
    unsigned long long* S;              // tiles x k boundary weights
    std::int32_t* counts;               // eligible donors per tile
    std::uint8_t* elig;                 // n
    // The reservation's start: eligible donors (n), the records and cleared
    // state (done, tried bits) of the first tail_limit of them, each part's
    // room and request total.
    std::int32_t* E;
    DonorInfo* live;
    std::uint8_t* done;
    unsigned long long* tried;
    unsigned long long* slack;
    unsigned long long* requests;
    unsigned long long* selected;       // kSelected words
    unsigned long long tail_limit;      // donors one tail launch takes
};

__device__ inline void donor_start(const RefArgs& a, std::int64_t j, std::int32_t v, DonorInfo* live,
                                   std::uint8_t* done, unsigned long long* tried) {
    live[j] = DonorInfo{static_cast<std::int32_t>(j), v, a.vw[v], (std::int32_t)a.labels[v]};
    done[j] = 0;
    tried[2 * j] = 0;
    tried[2 * j + 1] = 0;
}
// With more donors than one tail launch takes, k_donor_start lays their state
// out once the host knows how many: arrays for all n vertices would take 33
// bytes each at the peak of the finest level.
__device__ inline void select_place(const RefArgs& a, const SelectState& q, std::int64_t j, std::int32_t v) {
    q.E[j] = v;
    if ((unsigned long long)j < q.tail_limit) donor_start(a, j, v, q.live, q.done, q.tried);
}
__global__ void k_donor_start(RefArgs a, const std::int32_t* E, std::int64_t ne, DonorInfo* live, std::uint8_t* done,
                              unsigned long long* tried) {
    for (std::int64_t j = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; j < ne;
         j += (std::int64_t)gridDim.x * blockDim.x)
        donor_start(a, j, E[j], live, done, tried);
}
__device__ inline void select_parts(const RefArgs& a, const SelectState& q) {
    for (int p = threadIdx.x; p < a.k; p += blockDim.x) {
        q.slack[p] = a.loads0[p] < a.cap ? a.cap - a.loads0[p] : 0;
        q.requests[p] = 0;
    }
}
// One thread, once the number of eligible donors is known.
__device__ inline void select_counts(const RefArgs& a, const SelectState& q, unsigned long long ne) {
    q.selected[0] = ne;
    q.selected[1] = ne <= q.tail_limit ? ne : 0;
    q.selected[2] = a.ctr[kDonors];
}

__global__ void __launch_bounds__(kSelectThreads) k_select_weights(RefArgs a, SelectState q, int rounds) {
    __shared__ unsigned long long acc[kMaxParts];
    __shared__ std::int32_t star[kMaxParts];
    for (int p = threadIdx.x; p < a.k; p += kSelectThreads) {
        acc[p] = 0;
        star[p] = q.bstar[p];
    }
    __syncthreads();
    const std::int64_t base = (std::int64_t)blockIdx.x * rounds * kSelectThreads + threadIdx.x;
    for (int r = 0; r < rounds; ++r) {
        const std::int64_t v = base + (std::int64_t)r * kSelectThreads;
        const int b = v < a.n ? a.bucket[v] : -1;
        if (b >= 0 && b % kBalanceWidth == star[b / kBalanceWidth])
            atomicAdd(&acc[b / kBalanceWidth], (unsigned long long)a.vw[v]);
    }
    __syncthreads();
    for (int p = threadIdx.x; p < a.k; p += kSelectThreads) q.S[(std::int64_t)blockIdx.x * a.k + p] = acc[p];
}

__global__ void __launch_bounds__(kSelectThreads) k_select_eligible(RefArgs a, SelectState q, int rounds) {
    __shared__ unsigned long long run[kMaxParts];
    __shared__ unsigned long long wt[kSelectWaves][kMaxParts];
    __shared__ std::int32_t star[kMaxParts];
    __shared__ int count;
    const int t = threadIdx.x, w = t / kWave;
    for (int i = t; i < kSelectWaves * kMaxParts; i += kSelectThreads) wt[i / kMaxParts][i % kMaxParts] = 0;
    if (t < kMaxParts) {
        run[t] = 0;
        star[t] = t < a.k ? q.bstar[t] : -1;
    }
    if (t == 0) count = 0;
    __syncthreads();
    // Boundary weights of the earlier tiles, eight threads per part.
    const int p = t % kMaxParts;
    if (p < a.k && star[p] >= 0) {
        unsigned long long sum = 0;
        for (int tile = t / kMaxParts; tile < (int)blockIdx.x; tile += kSelectThreads / kMaxParts)
            sum += q.S[(std::int64_t)tile * a.k + p];
        if (sum) atomicAdd(&run[p], sum);
    }
    __syncthreads();
    const std::int64_t base = (std::int64_t)blockIdx.x * rounds * kSelectThreads + t;
    int mine = 0;
    for (int r = 0; r < rounds; ++r) {
        const std::int64_t v = base + (std::int64_t)r * kSelectThreads;
        const int b = v < a.n ? a.bucket[v] : -1;
        int key = -1;
        bool el = false;
        std::uint32_t wgt = 0;
        if (b >= 0) {
            const int s = b / kBalanceWidth, lb = b % kBalanceWidth;
            el = lb < star[s];
            if (lb == star[s]) {
                key = s;
                wgt = a.vw[v];
            }
        }
        if (__syncthreads_or(key >= 0)) {
            const std::uint64_t ex = wave_keyed_exclusive(key, wgt, wt[w]);
            __syncthreads();
            if (key >= 0) {
                std::uint64_t rank = run[key] + ex;
                for (int j = 0; j < w; ++j) rank += wt[j][key];
                el = q.prefix[b] + rank < q.excess[key];
            }
            __syncthreads();
            if (t < a.k) {
                unsigned long long add = 0;
                for (int j = 0; j < kSelectWaves; ++j) {
                    add += wt[j][t];
                    wt[j][t] = 0;
                }
                run[t] += add;
            }
        }
        if (v < a.n) q.elig[v] = el;
        mine += __popcll(__ballot(el));
    }
    if (lane_id() == 0 && mine) atomicAdd(&count, mine);
    __syncthreads();
    if (t == 0) q.counts[blockIdx.x] = count;
}

__global__ void __launch_bounds__(kSelectThreads) k_select_place(RefArgs a, SelectState q, int rounds) {
    if (blockIdx.x == 0) select_parts(a, q);
    const std::int64_t at = select_tile(q.elig, a.n, rounds, q.counts, [&](std::int64_t j, std::int64_t v) {
        select_place(a, q, j, (std::int32_t)v);
    });
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) select_counts(a, q, (unsigned long long)at);
}

// Donor selection of a repair iteration on a level of at most
// kSelectSmallMax vertices, in one block: the flagged donors (bucket at or
// below the part's boundary bucket) in vertex order, then their eligibility
// (below the boundary bucket, or inside it while the weighted rank among
// earlier donors of that bucket stays under the excess), placed as the
// three launches above do.
constexpr int kDonorThreads = 1024;
constexpr int kDonorWaves = kDonorThreads / kWave;

__global__ void __launch_bounds__(kDonorThreads) k_donors_small(RefArgs a, SelectState q) {
    const std::int32_t* bstar = q.bstar;
    const unsigned long long* prefix = q.prefix;
    const unsigned long long* excess = q.excess;
    __shared__ std::int32_t L[kSelectSmallMax];
    __shared__ unsigned long long wt[kDonorWaves][kMaxParts];
    __shared__ unsigned long long run[kMaxParts];
    __shared__ int wsum[kDonorWaves];
    __shared__ int base;
    const int t = threadIdx.x, w = t / kWave, lane = lane_id();
    const unsigned long long lt = (1ULL << lane) - 1ULL;
    for (int c = t; c < kMaxParts; c += kDonorThreads) {
        run[c] = 0;
        for (int j = 0; j < kDonorWaves; ++j) wt[j][c] = 0;
    }
    if (t == 0) base = 0;
    __syncthreads();
    select_parts(a, q);
    // Stable compaction of `mine` over one round: place(base + rank).
    auto compact = [&](bool mine, auto place) {
        const unsigned long long m = __ballot(mine);
        if (lane == 0) wsum[w] = __popcll(m);
        __syncthreads();
        int pre = base, total = 0;
        for (int j = 0; j < kDonorWaves; ++j) {
            pre += j < w ? wsum[j] : 0;
            total += wsum[j];
        }
        if (mine) place(pre + __popcll(m & lt));
        __syncthreads();
        if (t == 0) base += total;
        __syncthreads();
    };
    for (std::int64_t r = 0; r < a.n; r += kDonorThreads) {
        const std::int64_t v = r + t;
        bool f = false;
        if (v < a.n) {
            const int b = a.bucket[v];
            f = b >= 0 && (b % kBalanceWidth) <= bstar[b / kBalanceWidth];
        }
        compact(f, [&](int j) { L[j] = static_cast<std::int32_t>(v); });
    }
    const int nl = base;
    __syncthreads();
    if (t == 0) base = 0;
    __syncthreads();
    for (int r = 0; r < nl; r += kDonorThreads) {
        const int i = r + t;
        int key = -1, b = 0;
        bool el = false;
        std::int32_t v = 0;
        std::uint32_t wgt = 0;
        if (i < nl) {
            v = L[i];
            b = a.bucket[v];
            const int s = b / kBalanceWidth, lb = b % kBalanceWidth;
            if (lb == bstar[s]) {
                key = s;
                wgt = a.vw[v];
            }
            el = lb < bstar[s];
        }
        const std::uint64_t ex = wave_keyed_exclusive(key, wgt, wt[w]);
        __syncthreads();
        if (key >= 0) {
            std::uint64_t rank = run[key] + ex;
            for (int j = 0; j < w; ++j) rank += wt[j][key];
            el = prefix[b] + rank < excess[key];
        }
        __syncthreads();
        for (int c = t; c < kMaxParts; c += kDonorThreads) {
            unsigned long long add = 0;
            for (int j = 0; j < kDonorWaves; ++j) {
                add += wt[j][c];
                wt[j][c] = 0;
            }
            run[c] += add;
        }
        compact(el, [&](int j) { select_place(a, q, j, v); });
    }
    if (t == 0) select_counts(a, q, (unsigned long long)base);
}

struct ReserveState {
    const std::int32_t* E;           // eligible donors in vertex order
    std::int64_t ne;
    const unsigned long long* conn;  // ne x k sparse rows: weights
    const std::uint8_t* conn_part;   // ne x k: their parts
    const std::uint8_t* conn_nnz;    // ne: entries per row
    unsigned long long* requests;    // k, request totals
    const unsigned long long* slack; // k
    std::uint8_t* done;              // 1 admitted, 2 without a part left
    unsigned long long* tried;       // ne x 2
    const DonorInfo* live;           // donors still choosing, ascending
    std::int64_t nlive;
    const unsigned long long* nlive_dev;  // null, or where the device keeps nlive (the tail launch only)
};

// Choices of one attempt, one 4-lane group per live donor (many donors in
// flight per wave: the per-donor loads form a dependent chain).  Attempt 0
// requests the proposed target; later attempts the untried part with the
// most connection, then the most room left at the start of the attempt,
// then the lowest id.  Room only shrinks (request totals only grow) and
// tried parts stay tried, so a donor without a choice in some attempt has
// none in any later one: it is marked done (2) and leaves the live list.
struct Choice {
    int p;
    unsigned long long conn, room;
};
__device__ inline bool choice_better(const Choice& x, const Choice& y) {
    if (x.p < 0) return false;
    if (y.p < 0) return true;
    return x.conn > y.conn || (x.conn == y.conn && (x.room > y.room || (x.room == y.room && x.p < y.p)));
}

// A part without connection to the donor (conn 0) loses to every connected
// one, and among unconnected parts the order is (room desc, id asc): the
// scan walks the connected parts of the sparse row, and only when none is
// open falls back to the first untried part in that block-wide order (open
// when its room admits the donor; rooms after it are no larger).
constexpr int kChooseLanes = 4;
// Entries of a connection row per lane loaded before the first is judged.
constexpr int kChooseBatch = 4;
__global__ void __launch_bounds__(kTierThreads) k_choose(RefArgs a, ReserveState r, int attempt, std::int32_t* keys,
                                                        unsigned long long* active) {
    constexpr int W = kChooseLanes;
    __shared__ unsigned long long room[kMaxParts];  // start-of-attempt room per part
    __shared__ std::uint8_t order[kMaxParts];       // parts by (room desc, id asc)
    const int lg = threadIdx.x % W;
    const int gbase = (threadIdx.x % kWave) / W * W;
    if (attempt > 0) {
        for (int p = threadIdx.x; p < a.k; p += kTierThreads)
            room[p] = r.requests[p] < r.slack[p] ? r.slack[p] - r.requests[p] : 0;
        __syncthreads();
        for (int p = threadIdx.x; p < a.k; p += kTierThreads) {
            int rank = 0;
            for (int q = 0; q < a.k; ++q) rank += room[q] > room[p] || (room[q] == room[p] && q < p);
            order[rank] = static_cast<std::uint8_t>(p);
        }
        __syncthreads();
    }
    const std::int64_t groups = (std::int64_t)gridDim.x * (kTierThreads / W);
    unsigned long long cnt = 0;
    for (std::int64_t i = (blockIdx.x * (std::int64_t)kTierThreads + threadIdx.x) / W; i < r.nlive; i += groups) {
        const DonorInfo d = r.live[i];
        const std::int64_t e = d.e;
        Choice best{-1, 0, 0};
        bool open = !r.done[e];
        if (open) {
            const std::int32_t v = d.v;
            if (attempt == 0)
                best.p = a.targets[v];
            else {
                const std::uint64_t w = d.w;
                const int lv = d.label;
                const unsigned long long tried0 = r.tried[2 * e], tried1 = r.tried[2 * e + 1];
                auto closed = [&](int p) { return p == lv || ((((p >> 6) ? tried1 : tried0) >> (p & 63)) & 1ULL); };
                const int cnt = r.conn_nnz[e];
                for (int j0 = lg; j0 < cnt; j0 += W * kChooseBatch) {
                    std::uint8_t part[kChooseBatch];
                    unsigned long long conn[kChooseBatch];
#pragma unroll
                    for (int q = 0; q < kChooseBatch; ++q) {
                        const int j = j0 + q * W;
                        const std::int64_t x = e * a.k + (j < cnt ? j : cnt - 1);
                        part[q] = r.conn_part[x];
                        conn[q] = r.conn[x];
                    }
#pragma unroll
                    for (int q = 0; q < kChooseBatch; ++q) {
                        const int p = part[q];
                        if (j0 + q * W >= cnt || closed(p) || room[p] < w) continue;
                        const Choice x{p, conn[q], room[p]};
                        if (choice_better(x, best)) best = x;
                    }
                }
                for (int d = W / 2; d; d >>= 1) {
                    const Choice o{__shfl_xor(best.p, d, W), __shfl_xor(best.conn, d, W), __shfl_xor(best.room, d, W)};
                    if (choice_better(o, best)) best = o;
                }
                if (best.p < 0) {
                    for (int q0 = 0; q0 < a.k; q0 += W) {
                        const int q = q0 + lg;
                        const bool open = q < a.k && !closed(order[q]);
                        const unsigned sub = static_cast<unsigned>((__ballot(open) >> gbase) & ((1ULL << W) - 1));
                        if (sub) {
                            const int p = order[q0 + __ffs(sub) - 1];
                            if (room[p] >= w) best = Choice{p, 0, room[p]};
                            break;
                        }
                    }
                }
            }
        }
        if (lg == 0) {
            keys[i] = best.p;
            cnt += best.p >= 0;
            if (open && attempt > 0 && best.p < 0) r.done[e] = 2;
        }
    }
    cnt = wave_sum(cnt);
    if (lane_id() == 0 && cnt) atomicAdd(active, cnt);
}

struct DonorWeight {
    const DonorInfo* live;
    __device__ std::uint32_t weight(std::int64_t i) const { return live[i].w; }
};

template <class F>
__global__ void __launch_bounds__(kTierThreads) k_keyed_sums(const std::int32_t* keys, std::int64_t n, int k, int nb,
                                                            F f, unsigned long long* S) {
    __shared__ unsigned long long acc[kMaxParts];
    for (int c = threadIdx.x; c < kMaxParts; c += kTierThreads) acc[c] = 0;
    tile_key_sums(keys, n, k, nb, f, acc, S);
}

// Admission: the request fits when it ends within the receiver's slack.
struct AdmitFn {
    RefArgs a;
    ReserveState r;
    __device__ std::uint32_t weight(std::int64_t i) const { return r.live[i].w; }
    __device__ std::int32_t vertex(std::int64_t i) const { return r.live[i].v; }
    __device__ bool operator()(std::int64_t i, int c, std::uint64_t w, std::uint64_t begin) const {
        const std::int64_t e = r.live[i].e;
        r.tried[2 * e + (c >> 6)] |= 1ULL << (c & 63);
        if (begin <= r.slack[c] && w <= r.slack[c] - begin) {
            const std::int32_t v = r.live[i].v;
            a.targets[v] = c;
            a.flags[v] = 1;
            r.done[e] = 1;
            return true;
        }
        return false;
    }
};

// The remaining attempts of a reservation whose live donors fit one block
// (at most kTailDonors), looped inside one launch: per attempt the same
// start-of-attempt room and part order, the same choice per donor (attempt 0:
// the proposed target), the same ranks (exclusive weight prefix per requested
// part in donor order on top of the part's request total) and admissions as
// the per-attempt launches; the loop stops after an attempt with no chooser.
// Connection rows must be built before the launch.
//
// Bound: the latency of an attempt, up to k of them in a chain.  While more
// donors wait than the block has threads, an attempt goes over them in rounds
// and their state stays in memory.  Once each has a thread of its own (most
// launches start there) the rest runs with the donor's record, its tried parts
// and the first kRowCache entries of its connection row in registers, and the
// parts' totals in LDS, so that an attempt touches memory only for longer rows
// and admissions; the part order is made only in attempts where a donor has no
// open connected part.  Average launch with all state in memory and in this
// form: weighted graph at k = 128 38 and 18 us, R-MAT scale 18 at k = 64 86
// and 69, a grid at k = 16 11 and 8.
constexpr int kTailThreads = 1024;
constexpr int kTailDonors = 4096;  // donors per launch: rounds of kTailThreads
constexpr int kRowCache = 4;

struct TailShared {
    static constexpr int kWaves = kTailThreads / kWave;
    unsigned long long room[kMaxParts];
    unsigned long long requests[kMaxParts];
    unsigned long long slack[kMaxParts];
    unsigned long long run[kMaxParts];  // this attempt's requests of earlier rounds
    unsigned long long wt[kWaves][kMaxParts];
    int rank[kMaxParts];
    std::uint8_t order[kMaxParts];
    std::int32_t stage[kWaves][kStage];
    // Positions in r.live of the donors still choosing, ascending: donors
    // that were admitted or found no part are dropped after each attempt
    // (they would choose nothing again), so later attempts visit only the
    // waiting ones.  Ranks are weight prefixes over choosing donors in
    // list order, which dropping non-choosers leaves unchanged.
    std::uint16_t pos[kTailDonors];
    int wcount[kWaves];
};

// order[] = the parts by (room desc, id asc); the rooms are in place and the
// whole block calls it.  Eight threads count each part's rank.
__device__ inline void tail_order(TailShared& s, int k) {
    constexpr int kSplit = kTailThreads / kMaxParts;
    const int t = threadIdx.x, p = t % kMaxParts;
    if (t < kMaxParts) s.rank[t] = 0;
    __syncthreads();
    if (p < k) {
        const unsigned long long mine = s.room[p];
        int rank = 0;
        for (int q = t / kMaxParts; q < k; q += kSplit) rank += s.room[q] > mine || (s.room[q] == mine && q < p);
        atomicAdd(&s.rank[p], rank);
    }
    __syncthreads();
    if (t < k) s.order[s.rank[t]] = static_cast<std::uint8_t>(t);
    __syncthreads();
}

__device__ inline bool part_closed(int p, int label, unsigned long long tried0, unsigned long long tried1) {
    return p == label || ((((p >> 6) ? tried1 : tried0) >> (p & 63)) & 1ULL);
}

// The first part in the block's order that is not closed, if the weight fits.
__device__ inline int tail_fallback(const TailShared& s, int k, std::uint64_t w, int label, unsigned long long tried0,
                                    unsigned long long tried1) {
    for (int q = 0; q < k; ++q) {
        const int p = s.order[q];
        if (part_closed(p, label, tried0, tried1)) continue;
        return s.room[p] >= w ? p : -1;
    }
    return -1;
}

// Attempts from `attempt` on with one donor per thread (s.pos[0, nl), at most
// kTailThreads of them).
__device__ inline void tail_resident(TailShared& s, const RefArgs& a, const ReserveState& r, int attempt, int nl,
                                     Stage& st) {
    const int t = threadIdx.x, w = t / kWave, k = a.k;
    const int waves = (nl + kWave - 1) / kWave;
    DonorInfo d{-1, 0, 0, 0};
    bool alive = false;
    unsigned long long tried0 = 0, tried1 = 0;
    int cnt = 0;
    std::uint8_t part[kRowCache];
    unsigned long long conn[kRowCache];
    std::int64_t row = 0;
#pragma unroll
    for (int q = 0; q < kRowCache; ++q) {
        part[q] = 0;
        conn[q] = 0;
    }
    if (t < nl) {
        d = r.live[s.pos[t]];
        row = (std::int64_t)d.e * k;
        alive = !r.done[d.e];
        tried0 = r.tried[2 * (std::int64_t)d.e];
        tried1 = r.tried[2 * (std::int64_t)d.e + 1];
        cnt = r.conn_nnz[d.e];
#pragma unroll
        for (int q = 0; q < kRowCache; ++q)
            if (q < cnt) {
                part[q] = r.conn_part[row + q];
                conn[q] = r.conn[row + q];
            }
    }
    const std::uint64_t wd = d.w;
    for (; attempt < k; ++attempt) {
        if (t < k) s.room[t] = s.requests[t] < s.slack[t] ? s.slack[t] - s.requests[t] : 0;
        __syncthreads();
        int key = -1;
        if (attempt == 0) {
            if (alive) key = a.targets[d.v];
        } else {
            Choice best{-1, 0, 0};
            auto consider = [&](int p, unsigned long long c) {
                if (part_closed(p, d.label, tried0, tried1) || s.room[p] < wd) return;
                const Choice x{p, c, s.room[p]};
                if (choice_better(x, best)) best = x;
            };
            if (alive) {
#pragma unroll
                for (int q = 0; q < kRowCache; ++q)
                    if (q < cnt) consider(part[q], conn[q]);
                for (int j0 = kRowCache; j0 < cnt; j0 += kChooseBatch) {
                    std::uint8_t pp[kChooseBatch];
                    unsigned long long cc[kChooseBatch];
#pragma unroll
                    for (int q = 0; q < kChooseBatch; ++q) {
                        const std::int64_t x = row + (j0 + q < cnt ? j0 + q : cnt - 1);
                        pp[q] = r.conn_part[x];
                        cc[q] = r.conn[x];
                    }
#pragma unroll
                    for (int q = 0; q < kChooseBatch; ++q)
                        if (j0 + q < cnt) consider(pp[q], cc[q]);
                }
            }
            const bool lost = alive && best.p < 0;
            if (__syncthreads_or(lost)) {
                tail_order(s, k);
                if (lost) best.p = tail_fallback(s, k, wd, d.label, tried0, tried1);
            }
            if (best.p < 0) alive = false;  // rooms only shrink: it never chooses again
            key = best.p;
        }
        const std::uint64_t ex = wave_keyed_exclusive(key, key >= 0 ? d.w : 0, s.wt[w]);
        if (!__syncthreads_or(key >= 0)) break;
        bool admit = false;
        if (key >= 0) {
            std::uint64_t rank = s.requests[key] + ex;
            for (int j = 0; j < w; ++j) rank += s.wt[j][key];
            (key >> 6 ? tried1 : tried0) |= 1ULL << (key & 63);
            if (rank <= s.slack[key] && wd <= s.slack[key] - rank) {
                a.targets[d.v] = key;
                a.flags[d.v] = 1;
                alive = false;
                admit = true;
            }
        }
        st.push(admit, d.v);
        if (!__syncthreads_or(alive)) break;
        if (t < k) {
            unsigned long long add = 0;
            for (int j = 0; j < waves; ++j) {
                add += s.wt[j][t];
                s.wt[j][t] = 0;
            }
            s.requests[t] += add;
        }
    }
}

__global__ void __launch_bounds__(kTailThreads) k_reserve_tail(RefArgs a, ReserveState r, int attempt0,
                                                               std::int32_t* movers, unsigned long long* mcount) {
    constexpr int kWaves = TailShared::kWaves;
    __shared__ TailShared s;
    const int t = threadIdx.x, w = t / kWave;
    Stage st{s.stage[w], movers, mcount, 0};
    for (int i = t; i < kWaves * kMaxParts; i += kTailThreads) s.wt[i / kMaxParts][i % kMaxParts] = 0;
    int nl = static_cast<int>(r.nlive_dev ? *r.nlive_dev : r.nlive);
    if (nl == 0) return;
    for (int i = t; i < nl; i += kTailThreads) s.pos[i] = static_cast<std::uint16_t>(i);
    if (t < a.k) {
        s.requests[t] = r.requests[t];
        s.slack[t] = r.slack[t];
    }
    __syncthreads();
    int attempt = attempt0;
    for (; attempt < a.k && nl > kTailThreads; ++attempt) {
        if (t < a.k) {
            s.room[t] = s.requests[t] < s.slack[t] ? s.slack[t] - s.requests[t] : 0;
            s.run[t] = 0;
        }
        __syncthreads();
        tail_order(s, a.k);
        bool any = false;
        for (int base = 0; base < nl; base += kTailThreads) {
            const int i = base + t;
            int key = -1;
            DonorInfo d{-1, 0, 0, 0};
            if (i < nl) {
                d = r.live[s.pos[i]];
                const std::int64_t e = d.e;
                // Independent loads first: the donor's state, then its row in
                // batches.
                const std::uint8_t done = r.done[e];
                const unsigned long long tried0 = r.tried[2 * e], tried1 = r.tried[2 * e + 1];
                const int cnt = attempt ? r.conn_nnz[e] : 0;
                if (!done && attempt == 0) {
                    key = a.targets[d.v];
                } else if (!done) {
                    const std::uint64_t wd = d.w;
                    Choice best{-1, 0, 0};
                    for (int j0 = 0; j0 < cnt; j0 += kChooseBatch) {
                        std::uint8_t part[kChooseBatch];
                        unsigned long long conn[kChooseBatch];
#pragma unroll
                        for (int q = 0; q < kChooseBatch; ++q) {
                            const std::int64_t x = e * a.k + (j0 + q < cnt ? j0 + q : cnt - 1);
                            part[q] = r.conn_part[x];
                            conn[q] = r.conn[x];
                        }
#pragma unroll
                        for (int q = 0; q < kChooseBatch; ++q) {
                            const int p = part[q];
                            if (j0 + q >= cnt || part_closed(p, d.label, tried0, tried1) || s.room[p] < wd) continue;
                            const Choice x{p, conn[q], s.room[p]};
                            if (choice_better(x, best)) best = x;
                        }
                    }
                    if (best.p < 0) best.p = tail_fallback(s, a.k, wd, d.label, tried0, tried1);
                    if (best.p < 0) r.done[e] = 2;
                    key = best.p;
                }
            }
            const std::uint32_t wgt = key >= 0 ? d.w : 0;
            const std::uint64_t ex = wave_keyed_exclusive(key, wgt, s.wt[w]);
            __syncthreads();
            bool admit = false;
            if (key >= 0) {
                any = true;
                std::uint64_t rank = s.requests[key] + s.run[key] + ex;
                for (int j = 0; j < w; ++j) rank += s.wt[j][key];
                const std::int64_t e = d.e;
                r.tried[2 * e + (key >> 6)] |= 1ULL << (key & 63);
                if (rank <= s.slack[key] && wgt <= s.slack[key] - rank) {
                    a.targets[d.v] = key;
                    a.flags[d.v] = 1;
                    r.done[e] = 1;
                    admit = true;
                }
            }
            st.push(admit, d.v);
            __syncthreads();
            if (t < a.k) {
                unsigned long long add = 0;
                for (int j = 0; j < kWaves; ++j) {
                    add += s.wt[j][t];
                    s.wt[j][t] = 0;
                }
                s.run[t] += add;
            }
            __syncthreads();
        }
        if (t < a.k) s.requests[t] += s.run[t];
        if (!__syncthreads_or(any)) {
            nl = 0;
            break;
        }
        // Stable compaction of the waiting donors: thread t keeps its
        // kPer consecutive positions in registers, a block scan of the
        // counts gives where they go.
        constexpr int kPer = kTailDonors / kTailThreads;
        std::uint16_t q[kPer];
        bool waiting[kPer];
        int keep = 0;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int i = t * kPer + j;
            q[j] = i < nl ? s.pos[i] : 0;
            waiting[j] = i < nl && !r.done[r.live[q[j]].e];
            keep += waiting[j];
        }
        const int inc = wave_inclusive_scan<PlusOp>(keep);
        if (lane_id() == kWave - 1) s.wcount[w] = inc;
        __syncthreads();  // every position has been read
        int at = inc - keep, total = 0;
        for (int j = 0; j < kWaves; ++j) {
            if (j < w) at += s.wcount[j];
            total += s.wcount[j];
        }
#pragma unroll
        for (int j = 0; j < kPer; ++j)
            if (waiting[j]) s.pos[at++] = q[j];
        nl = total;
        __syncthreads();
    }
    if (nl > 0) tail_resident(s, a, r, attempt, nl, st);
    st.flush();
}

__global__ void k_live_flags(const DonorInfo* live, std::int64_t count, const std::uint8_t* done, std::uint8_t* flags) {
    for (std::int64_t j = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; j < count;
         j += (std::int64_t)gridDim.x * blockDim.x)
        flags[j] = done[live[j].e] == 0;
}

__global__ void k_gather_info(const DonorInfo* src, const std::int32_t* idx, std::int64_t count, DonorInfo* dst) {
    for (std::int64_t j = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; j < count;
         j += (std::int64_t)gridDim.x * blockDim.x)
        dst[j] = src[idx[j]];
}

// One word per part handed to a kernel by value: no copy and no host wait.
struct PartWords {
    unsigned long long w[kMaxParts];
};
inline PartWords part_words(const std::vector<std::uint64_t>& v) {
    PartWords p{};
    for (std::size_t i = 0; i < v.size() && i < kMaxParts; ++i) p.w[i] = v[i];
    return p;
}
__global__ void k_set_parts(PartWords in, unsigned long long* out, int k) {
    for (int p = threadIdx.x; p < k; p += blockDim.x) out[p] = in.w[p];
}

// Start of a refinement level in one launch: clears the counter block, the
// heavy-edge flag and (when the level has prices) the prices, and sets the
// part loads.  (An upload with its host wait and three fills before.)
__global__ void k_level_begin(unsigned long long* ctr, PartWords loads, unsigned long long* loads_out, int k,
                              unsigned long long* heavy_edge, double* prices) {
    for (int i = threadIdx.x; i < kCtrCount; i += blockDim.x) ctr[i] = 0;
    for (int p = threadIdx.x; p < k; p += blockDim.x) {
        loads_out[p] = loads.w[p];
        if (prices) prices[p] = 0.0;
    }
    if (threadIdx.x == 0) *heavy_edge = 0;
}

// Raises the flag when some weight is above 1; blocks stop once it is up.
// The proposals read it on the device: the largest weight was read back to
// the host before, one more wait per level.
__global__ void __launch_bounds__(256) k_heavy_edge(std::int64_t m, const std::uint32_t* ew, unsigned long long* flag) {
    const std::int64_t stride = (std::int64_t)gridDim.x * blockDim.x;
    for (std::int64_t base = blockIdx.x * (std::int64_t)blockDim.x; base < m; base += 8 * stride) {
        if (__syncthreads_or(threadIdx.x == 0 && *(volatile unsigned long long*)flag)) return;
        bool heavy = false;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const std::int64_t x = base + j * stride + threadIdx.x;
            heavy |= x < m && ew[x] > 1;
        }
        if (__syncthreads_or(heavy)) {
            if (threadIdx.x == 0) *(volatile unsigned long long*)flag = 1;
            return;
        }
    }
}

// Start of a repair iteration in one launch: freezes the part loads
// (loads0 = loads), clears the bucket weights and the counter block.
__global__ void k_repair_begin(RefArgs a, unsigned long long* loads0, unsigned long long* counts, std::int64_t ncounts,
                               unsigned long long* ctr, int nctr) {
    for (std::int64_t i = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; i < ncounts;
         i += (std::int64_t)gridDim.x * blockDim.x) {
        counts[i] = 0;
        if (i < a.k) loads0[i] = a.loads[i];
        if (i < nctr) ctr[i] = 0;
    }
}

// New repair prices from the samples of the last repair (parts without a
// sample keep their price): loss / weight for a positive loss, else 0.  The
// samples are cleared for the next repair.
__global__ void k_publish_prices(RepairSample* samples, double* prices, int k) {
    for (int p = threadIdx.x; p < k; p += blockDim.x) {
        const RepairSample x = samples[p];
        samples[p] = RepairSample{0, 0};
        if (!x.weight) continue;
        const long long loss = (long long)x.loss;
        prices[p] = loss > 0 ? (double)loss / (double)x.weight : 0.0;
    }
}

// Checkpoint of the labels of a round that set a new best cut.
// vec: both arrays are 16-byte aligned (copied in 16-byte words).
__global__ void k_lp_keep(const unsigned long long* flag, const Label* labels, Label* best, std::int64_t n, bool vec) {
    if (!*flag) return;
    const std::int64_t words = vec ? n / 16 : 0;
    const uint4* src = reinterpret_cast<const uint4*>(labels);
    uint4* dst = reinterpret_cast<uint4*>(best);
    for (std::int64_t i = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; i < words;
         i += (std::int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
    for (std::int64_t v = words * 16 + blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < n;
         v += (std::int64_t)gridDim.x * blockDim.x)
        best[v] = labels[v];
}

// ------------------------------------------------------------ exchange
struct JMove {
    std::int32_t v[2 * kJointSide];
    std::int32_t size, a, b, id;
    std::int64_t gain, net;
};

__host__ __device__ inline JMove jmove_empty() {
    JMove m;
    for (int j = 0; j < 2 * kJointSide; ++j) m.v[j] = -1;
    m.size = 0;
    m.a = -1;
    m.b = -1;
    m.id = 0;
    m.gain = 0;
    m.net = 0;
    return m;
}

__device__ inline std::int64_t jgap(std::int64_t net, std::int64_t lo, std::int64_t hi) {
    return net < lo ? lo - net : net > hi ? net - hi : 0;
}

template <int W>
__global__ void k_dense_affinity(RefArgs a, unsigned long long* A) {
    extern __shared__ unsigned long long smem[];
    const int lg = threadIdx.x % W, gi = threadIdx.x / W;
    unsigned long long* hist = smem + gi * a.k;
    const std::int64_t gpb = blockDim.x / W;
    for (std::int64_t v = blockIdx.x * gpb + gi; v < a.n; v += (std::int64_t)gridDim.x * gpb) {
        team_histogram(GroupTeam<W>{lg}, a, v, hist);
        for (int p = lg; p < a.k; p += W) A[v * a.k + p] = hist[p];
        wave_sync();
    }
}

__global__ void k_quotient(RefArgs a, const unsigned long long* A, unsigned long long* Q) {
    for (std::int64_t v = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < a.n;
         v += (std::int64_t)gridDim.x * blockDim.x) {
        const int la = a.labels[v];
        for (int b = la + 1; b < a.k; ++b) {
            const unsigned long long x = A[v * a.k + b];
            if (x) atomicAdd(&Q[la * a.k + b], x);
        }
    }
}

// joint_match (exchange.cuh:55-83): greedy mutual-best pairing of parts in
// rounds, one block.  The pair scores Q / (1 + visits)^2 are computed once
// into LDS (a pair's visit count changes only when the pair is matched, and
// matched parts are not scored again); each part's best partner (largest
// score, then smallest part) is found by a group of W lanes over
// q = sub, sub + W, ...
constexpr int kMatchThreads = 1024;
// The block also resets the pass's seed slots (seed_words of ~0) for
// k_joint_seeds, which runs next.
__global__ void __launch_bounds__(kMatchThreads) k_joint_match(int k, const unsigned long long* Q,
                                                               std::int32_t* partner, std::int32_t* visits,
                                                               unsigned long long* seeds, int seed_words) {
    __shared__ double score_of[kMaxParts * kMaxParts];
    __shared__ int choice[kMaxParts];
    __shared__ int mate[kMaxParts];
    __shared__ int progress;
    for (int x = threadIdx.x; x < seed_words; x += blockDim.x) seeds[x] = ~0ULL;
    for (int x = threadIdx.x; x < k * k; x += blockDim.x) {
        const int p = x / k, q = x % k;
        double v = 0.0;
        if (p < q && Q[x]) {
            const double penalty = 1.0 + visits[x];
            v = (double)Q[x] / (penalty * penalty);
        }
        score_of[x] = v;
    }
    for (int p = threadIdx.x; p < k; p += blockDim.x) mate[p] = -1;
    __syncthreads();
    int W = kWave;
    while (W > 1 && W * k > kMatchThreads) W >>= 1;
    const int p = threadIdx.x / W, sub = threadIdx.x % W;
    for (int round = 0; round < k / 2; ++round) {
        if (threadIdx.x == 0) progress = 0;
        double score = -1;
        int best = -1;
        if (p < k && mate[p] < 0)
            for (int q = sub; q < k; q += W) {
                if (q == p || mate[q] >= 0) continue;
                const double v = score_of[p < q ? p * k + q : q * k + p];
                if (v > 0.0 && v > score) {
                    score = v;
                    best = q;
                }
            }
        for (int d = W / 2; d; d >>= 1) {
            const double os = __shfl_xor(score, d, W);
            const int ob = __shfl_xor(best, d, W);
            if (os > score || (os == score && ob < best)) {
                score = os;
                best = ob;
            }
        }
        if (p < k && sub == 0) choice[p] = best;
        __syncthreads();
        if (p < k && sub == 0 && best >= 0 && choice[best] == p) {
            mate[p] = best;
            if (p < best) {
                ++visits[p * k + best];
                atomicAdd(&progress, 1);
            }
        }
        __syncthreads();
        const int gained = progress;
        __syncthreads();
        if (!gained) break;
    }
    for (int q = threadIdx.x; q < k; q += blockDim.x) partner[q] = mate[q];
}

__global__ void k_joint_seeds(RefArgs a, const unsigned long long* A, const std::int32_t* partner,
                              unsigned long long* seeds, int sw, int pass) {
    for (std::int64_t v = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < a.n;
         v += (std::int64_t)gridDim.x * blockDim.x) {
        const int p = a.labels[v], q = partner[p];
        if (q < 0 || !A[v * a.k + q]) continue;
        const std::uint32_t h = mix32((std::uint32_t)v ^ mix32((std::uint32_t)pass + 17));
        atomicMin(&seeds[p * sw + h % (std::uint32_t)sw], ((unsigned long long)h << 32) | (std::uint32_t)v);
    }
}

// ------------------------------------------------ exchange: transaction growth
// Growth of capacity-complementary transactions (the semantics of
// exchange.cuh:96-204).  A slot is a (partner seed, policy) pair; its
// transaction starts at the seed vertex and adds, up to eight members and at
// most four per side, the admissible vertex that ranks first by (marginal
// gain, balance gap, id), or by (gap, gain, id) under policy 0 while the net
// weight lies outside the feasible window.  Candidates are the vertices of a
// member's first 128 row entries that share the member's part, and, while no
// member sits on the partner side, the partner part's seeds; vertices of
// degree above 1024 never join.  Each step records the transaction as an
// archive fragment (positive gain, at most four members) and as the slot's
// best feasible transaction.
//
// CDNA design: one wave per slot with a candidate pool in LDS.  When a
// member joins, its row is read once and the entries that pass the static
// tests are appended to the pool by ballot compaction, together with their
// static marginal gain A(u, other) - A(u, own) (+2w for a row entry) and
// weight.  A step then scans at most 1024 pool records in LDS instead of
// re-reading every member row and the affinity rows behind it; records of a
// vertex that joins are retired.  The step's winner comes from a wave
// butterfly whose in-row exchanges are DPP moves, and the joining vertex's
// correction term (its edges to the members) is a DPP sum over its row.
constexpr int kGrowNominate = 128;                          // row entries that nominate
constexpr int kGrowPool = 7 * kGrowNominate + kJointSeeds;  // members 1..7 nominate; seeds once
constexpr int kGrowWaves = 2;                               // slots per block
constexpr std::uint8_t kPoolPartner = 1, kPoolSeed = 2, kPoolRetired = 4;

struct GrowPool {
    std::int64_t marginal[kGrowPool];
    std::int32_t u[kGrowPool];
    std::uint32_t w[kGrowPool];
    std::uint8_t kind[kGrowPool];
    std::int32_t members[8];
    std::int32_t member_label[8];
    int count;
};

struct GrowPick {
    std::int64_t marginal, gap;
    std::int32_t u, pad;
};

// x ranks before y (the step order of exchange.cuh:166-176).
__device__ inline bool grow_before(const GrowPick& x, const GrowPick& y, bool gap_first) {
    if (gap_first) {
        if (x.gap != y.gap) return x.gap < y.gap;
        if (x.marginal != y.marginal) return x.marginal > y.marginal;
    } else {
        if (x.marginal != y.marginal) return x.marginal > y.marginal;
        if (x.gap != y.gap) return x.gap < y.gap;
    }
    return x.u < y.u;
}

struct GrowBest {
    bool gap_first;
    __device__ GrowPick operator()(const GrowPick& x, const GrowPick& y) const {
        return grow_before(y, x, gap_first) ? y : x;
    }
};

// Appends what one new member nominates (member >= 0: its first 128 row
// entries in its own part) or, with member < 0, the partner part's seeds.
// Wave-uniform; every lane takes part.
__device__ inline void grow_nominate(const RefArgs& a, const unsigned long long* A, const unsigned long long* seeds,
                                     int sw, int source, int target, std::int32_t member, int size, GrowPool& P,
                                     int lane) {
    const int k = a.k;
    std::int64_t begin = 0, end = sw;
    int own = -1;
    if (member >= 0) {
        begin = a.off[member];
        end = a.off[member + 1];
        if (end > begin + kGrowNominate) end = begin + kGrowNominate;
        own = a.labels[member];
    }
    for (std::int64_t base = begin; base < end; base += kWave) {
        const std::int64_t e = base + lane;
        bool keep = false;
        std::int32_t u = -1;
        int p = -1;
        if (e < end) {
            if (member < 0) {
                const unsigned long long val = seeds[(std::int64_t)target * sw + e];
                if (val != ~0ULL) u = (std::int32_t)(std::uint32_t)val;
            } else {
                u = a.nbr[e];
            }
            if (u >= 0) {
                p = a.labels[u];
                keep = (p == source || p == target) && (member < 0 || p == own) && a.off[u + 1] - a.off[u] <= 1024;
                for (int j = 0; j < size; ++j) keep &= u != P.members[j];
            }
        }
        const unsigned long long ballot = __ballot(keep);
        if (keep) {
            const int r = P.count + __popcll(ballot & ((1ULL << lane) - 1ULL));
            const int other = p == source ? target : source;
            std::int64_t marginal = (std::int64_t)A[(std::int64_t)u * k + other] - (std::int64_t)A[(std::int64_t)u * k + p];
            if (member >= 0) marginal += 2 * (std::int64_t)ew_at(a.ew, e);
            P.marginal[r] = marginal;
            P.u[r] = u;
            P.w[r] = a.vw[u];
            P.kind[r] = (std::uint8_t)((p == source ? 0 : kPoolPartner) | (member < 0 ? kPoolSeed : 0));
        }
        wave_sync();
        if (lane == 0) P.count += __popcll(ballot);
        wave_sync();
    }
}

__global__ void __launch_bounds__(kGrowWaves* kWave) k_joint_grow(RefArgs a, const unsigned long long* A, int slots,
                                                                   int sw, const unsigned long long* seeds,
                                                                   const std::int32_t* partner, JMove* moves,
                                                                   JMove* archive) {
    __shared__ GrowPool pools[kGrowWaves];
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const int slot = blockIdx.x * kGrowWaves + wave;
    if (slot >= slots) return;
    GrowPool& P = pools[wave];
    const int policy = slot % 2;
    const int k = a.k;
    JMove best = jmove_empty();
    best.id = slot;
    if (lane == 0) {  // the same lane writes these slots again below
        moves[slot] = best;
        for (int j = 0; j < kJointArchive; ++j) archive[slot * kJointArchive + j] = jmove_empty();
    }
    const unsigned long long enc = seeds[slot / 2];
    if (enc == ~0ULL) return;
    const std::int32_t root = (std::int32_t)(std::uint32_t)enc;
    const int source = a.labels[root], target = partner[source];
    if (target < 0) return;
    if (lane == 0) {
        P.count = 0;
        P.members[0] = root;
        P.member_label[0] = source;
    }
    wave_sync();
    int size = 1, c0 = 1, c1 = 0;
    std::int64_t net = a.vw[root];
    const std::int64_t lo = (std::int64_t)a.loads[source] - (std::int64_t)a.cap;
    const std::int64_t hi = (std::int64_t)a.cap - (std::int64_t)a.loads[target];
    std::int64_t gain = (std::int64_t)A[(std::int64_t)root * k + target] - (std::int64_t)A[(std::int64_t)root * k + source];
    const int pa = source < target ? source : target, pb = source < target ? target : source;
    grow_nominate(a, A, seeds, sw, source, target, -1, size, P, lane);
    grow_nominate(a, A, seeds, sw, source, target, root, size, P, lane);
    for (int step = 0;; ++step) {
        if (lane == 0 && gain > 0 && size <= kJointArchive) {
            JMove st = jmove_empty();
            st.size = size;
            st.a = pa;
            st.b = pb;
            st.gain = gain;
            st.net = source == pa ? net : -net;
            st.id = slot * kJointArchive + step;
            for (int j = 0; j < size; ++j) {  // members in ascending id order
                int pos = j;
                while (pos && st.v[pos - 1] > P.members[j]) {
                    st.v[pos] = st.v[pos - 1];
                    --pos;
                }
                st.v[pos] = P.members[j];
            }
            archive[slot * kJointArchive + step] = st;
        }
        if (gain > best.gain && !jgap(net, lo, hi)) {
            best.size = size;
            best.a = pa;
            best.b = pb;
            best.gain = gain;
            best.net = source == pa ? net : -net;
            for (int j = 0; j < 8; ++j) best.v[j] = j < size ? P.members[j] : -1;
        }
        if (size == 8) break;
        const bool gap_first = policy == 0 && jgap(net, lo, hi) != 0;
        GrowPick pick{LLONG_MIN, LLONG_MAX, INT_MAX, 0};
        for (int r = lane; r < P.count; r += kWave) {
            const int kind = P.kind[r];
            const int side = kind & kPoolPartner;
            if ((kind & kPoolRetired) || ((kind & kPoolSeed) && c1) || (side ? c1 : c0) >= kJointSide) continue;
            if ((net > hi && !side) || (net < lo && side)) continue;
            const std::int64_t cnet = net + (side ? -(std::int64_t)P.w[r] : (std::int64_t)P.w[r]);
            const GrowPick c{P.marginal[r], jgap(cnet, lo, hi), P.u[r], 0};
            if (grow_before(c, pick, gap_first)) pick = c;
        }
        pick = wave_allreduce(pick, GrowBest{gap_first});
        if (pick.u == INT_MAX) break;
        const std::int32_t chosen = pick.u;
        const int lc = a.labels[chosen];
        const int side = lc == source ? 0 : 1;
        std::int64_t corr = 0;
        for (std::int64_t e = a.off[chosen] + lane; e < a.off[chosen + 1]; e += kWave) {
            const std::int32_t nb = a.nbr[e];
            for (int j = 0; j < size; ++j)
                if (nb == P.members[j]) corr += (P.member_label[j] == lc ? 2 : -2) * (std::int64_t)ew_at(a.ew, e);
        }
        corr = wave_allreduce(corr, PlusI64{});
        gain += (std::int64_t)A[(std::int64_t)chosen * k + (side ? source : target)] -
                (std::int64_t)A[(std::int64_t)chosen * k + lc] + corr;
        net += side ? -(std::int64_t)a.vw[chosen] : (std::int64_t)a.vw[chosen];
        if (side) ++c1;
        else ++c0;
        // Retire the newcomer's records, then let it nominate.
        for (int r = lane; r < P.count; r += kWave)
            if (P.u[r] == chosen) P.kind[r] |= kPoolRetired;
        if (lane == 0) {
            P.members[size] = chosen;
            P.member_label[size] = lc;
        }
        wave_sync();
        ++size;
        if (size < 8) grow_nominate(a, A, seeds, sw, source, target, chosen, size, P, lane);
    }
    if (lane == 0) moves[slot] = best;
}

// Orders for the archive and the transaction pool (complementary_moves.cuh:5-14, exchange.cuh:33-40).
struct MoveKeys {
    std::int64_t first, second, third;
};
struct NetOrder {
    __device__ bool operator()(const JMove& x, const JMove& y) const {  // x before y
        if (x.a != y.a) return x.a < y.a;
        if (x.net != y.net) return x.net < y.net;
        if (x.gain != y.gain) return x.gain > y.gain;
        if (x.size != y.size) return x.size < y.size;
        for (int j = 0; j < x.size; ++j)
            if (x.v[j] != y.v[j]) return x.v[j] < y.v[j];
        return x.id < y.id;
    }
    // Within a part the order starts with these, ascending.
    __device__ static MoveKeys keys(const JMove& x) {
        return MoveKeys{x.net, ~x.gain, (std::int64_t)x.size << 32 | (std::uint32_t)x.v[0]};
    }
};
struct JointOrder {
    __device__ bool operator()(const JMove& x, const JMove& y) const {
        if ((x.size != 0) != (y.size != 0)) return x.size != 0;
        if (x.a != y.a) return x.a < y.a;
        if (x.gain != y.gain) return x.gain > y.gain;
        return x.id < y.id;
    }
    __device__ static MoveKeys keys(const JMove& x) { return MoveKeys{~x.gain, x.id, 0}; }
};

// Moves in order without a sorting network over 64-byte records.  Both orders
// go by the part first and start with three words (keys()); only full ties
// look at the rest of the records.  Four launches: the non-empty moves per part
// and block of the source, with the parts' starts from the last block; their
// indices grouped by part (any order inside); runs of 256 moves of a part
// sorted by merges in LDS; the runs of a part merged, all by binary searches
// for each move's place.  The moves of a pair of parts carry its lower part:
// up to k = 32 a pair has 512 grown moves and 4 archived ones for each of them,
// and two more moves for every archived one, so a part has at most 2,048 moves
// in the archive and 4,608 in the pool (fewer above: 1,024 and 2,304 at k = 64).
// The bitonic networks that this replaces ran 66 dependent stages over records
// 64 bytes apart in LDS, 16 lanes to a bank, 64 to 74 us for each chunk of
// 2,048 moves and several launches for more; comparing all pairs of a part took
// 96 us for the archive of R-MAT scale 18 (k = 64), runs and merges take 43.
constexpr int kOrderThreads = 1024;
__global__ void __launch_bounds__(kOrderThreads) k_moves_count(const JMove* src, int count, int k, int* block_at,
                                                               int* starts, unsigned int* ticket,
                                                               unsigned long long* host, unsigned long long* flag,
                                                               unsigned long long seq) {
    __shared__ int hist[kMaxParts];
    __shared__ int first[kMaxParts + 1];
    const int t = threadIdx.x;
    if (t < kMaxParts) hist[t] = 0;
    __syncthreads();
    const int i = blockIdx.x * kOrderThreads + t;
    if (i < count && src[i].size) atomicAdd(&hist[src[i].a], 1);
    __syncthreads();
    if (t < k) block_at[blockIdx.x * k + t] = hist[t];
    if (!block_is_last(ticket)) return;
    int total = 0;
    if (t < k)
        for (int b = 0; b < (int)gridDim.x; ++b) total += block_at[b * k + t];
    if (t < kMaxParts) hist[t] = t < k ? total : 0;
    __syncthreads();
    if (t < kWave) {
        int sum = 0;
        for (int p0 = 0; p0 < kMaxParts; p0 += kWave) {
            const int n = hist[p0 + t], inc = wave_inclusive_scan<PlusOp>(n);
            first[p0 + t] = sum + inc - n;
            sum += __shfl(inc, kWave - 1);
        }
        if (t == 0) first[kMaxParts] = sum;
    }
    __syncthreads();
    if (t < k) {
        int at = first[t];
        for (int b = 0; b < (int)gridDim.x; ++b) {
            const int n = block_at[b * k + t];
            block_at[b * k + t] = at;
            at += n;
        }
        starts[t] = first[t];
    }
    if (t == 0) {
        starts[k] = first[kMaxParts];
        if (host) host[0] = (unsigned long long)first[kMaxParts];
    }
    if (host) publish_to_host(flag, seq);
}

__global__ void __launch_bounds__(kOrderThreads) k_moves_group(const JMove* src, int count, int k, const int* block_at,
                                                               int* order) {
    __shared__ int at[kMaxParts];
    const int t = threadIdx.x;
    if (t < k) at[t] = block_at[blockIdx.x * k + t];
    __syncthreads();
    const int i = blockIdx.x * kOrderThreads + t;
    if (i < count && src[i].size) order[atomicAdd(&at[src[i].a], 1)] = i;
}

constexpr int kRankThreads = 256;
constexpr int kRankSplit = 8;  // blocks per part
__device__ inline bool keys_less(const MoveKeys& x, const MoveKeys& y) {
    return x.first < y.first ||
           (x.first == y.first && (x.second < y.second || (x.second == y.second && x.third < y.third)));
}
__device__ inline bool keys_equal(const MoveKeys& x, const MoveKeys& y) {
    return x.first == y.first && x.second == y.second && x.third == y.third;
}

// Sorts each run of kRankThreads moves of a part (indices in order[]) into
// runs[]: merges of doubling width in LDS, a move's new place in each found by
// a binary search in the neighbouring run (36 search steps in all).  Equal
// moves (nothing tells them apart) keep their order.
template <typename Cmp>
__global__ void __launch_bounds__(kRankThreads) k_moves_runs(const JMove* src, const int* starts, const int* order,
                                                             Cmp before, JMove* runs) {
    __shared__ JMove tile[kRankThreads];
    __shared__ std::int64_t first[kRankThreads], second[kRankThreads], third[kRankThreads];
    __shared__ short at[2][kRankThreads];  // slots of the moves, by place
    const int t = threadIdx.x, b0 = starts[blockIdx.x], n = starts[blockIdx.x + 1] - b0;
    for (int j0 = blockIdx.y * kRankThreads; j0 < n; j0 += kRankSplit * kRankThreads) {
        const int c = n - j0 < kRankThreads ? n - j0 : kRankThreads;
        __syncthreads();
        if (t < c) {
            tile[t] = src[order[b0 + j0 + t]];
            const MoveKeys k = Cmp::keys(tile[t]);
            first[t] = k.first;
            second[t] = k.second;
            third[t] = k.third;
            at[0][t] = (short)t;
        }
        __syncthreads();
        int from = 0;
        for (int width = 1; width < c; width <<= 1, from ^= 1) {
            if (t < c) {
                const int run = t / width, other = run ^ 1, r0 = other * width;
                const int slot = at[from][t];
                const MoveKeys mine{first[slot], second[slot], third[slot]};
                int lo = 0, hi = c - r0 < width ? c - r0 : width;
                while (lo < hi) {  // moves of the other run before this one
                    const int mid = (lo + hi) >> 1, y = at[from][r0 + mid];
                    const MoveKeys o{first[y], second[y], third[y]};
                    bool earlier = keys_less(o, mine);
                    if (!earlier && keys_equal(o, mine))
                        earlier = before(tile[y], tile[slot]) || (other < run && !before(tile[slot], tile[y]));
                    if (earlier) lo = mid + 1;
                    else hi = mid;
                }
                at[from ^ 1][(run & ~1) * width + (t & (width - 1)) + lo] = (short)slot;
            }
            __syncthreads();
        }
        if (t < c) runs[b0 + j0 + t] = tile[at[from][t]];
    }
}

// Merges a part's runs: a move's place is its place in its run plus, for every
// other run, the moves of that run before it, found by binary search over keys
// staged kMergeRuns runs at a time.  Of equal moves the earlier run's are first.
constexpr int kMergeRuns = 8;
template <typename Cmp>
__global__ void __launch_bounds__(kRankThreads) k_moves_merge(const JMove* runs, const int* starts, Cmp before,
                                                              JMove* out) {
    __shared__ MoveKeys key[kMergeRuns * kRankThreads];
    const int t = threadIdx.x, b0 = starts[blockIdx.x], n = starts[blockIdx.x + 1] - b0;
    for (int j0 = blockIdx.y * kRankThreads; j0 < n; j0 += kRankSplit * kRankThreads) {
        const bool have = j0 + t < n;
        const JMove own = have ? runs[b0 + j0 + t] : jmove_empty();
        const MoveKeys mine = Cmp::keys(own);
        int rank = t;
        for (int s0 = 0; s0 < n; s0 += kMergeRuns * kRankThreads) {
            __syncthreads();
            for (int x = t; x < kMergeRuns * kRankThreads && s0 + x < n; x += kRankThreads)
                key[x] = Cmp::keys(runs[b0 + s0 + x]);
            __syncthreads();
            for (int r = 0; r < kMergeRuns; ++r) {
                const int r0 = s0 + r * kRankThreads;
                if (r0 >= n) break;
                if (r0 == j0 || !have) continue;
                int lo = 0, hi = n - r0 < kRankThreads ? n - r0 : kRankThreads;
                while (lo < hi) {  // moves of the run before this one
                    const int mid = (lo + hi) >> 1;
                    const MoveKeys o = key[r * kRankThreads + mid];
                    bool earlier = keys_less(o, mine);
                    if (!earlier && keys_equal(o, mine)) {
                        const JMove m = runs[b0 + r0 + mid];
                        earlier = before(m, own) || (r0 < j0 && !before(own, m));
                    }
                    if (earlier) lo = mid + 1;
                    else hi = mid;
                }
                rank += lo;
            }
        }
        if (have) out[b0 + rank] = own;
    }
}

// exchange.cuh:19-32 equality of consecutive sorted archive entries: flags the
// moves that do not repeat the one before, and counts them per tile; the
// second launch places them in order and hands their number to the host.  The
// number of moves is read on the device; the grid covers the most there can be.
__global__ void __launch_bounds__(kSelectThreads) k_unique_flags(const JMove* m, const int* count_dev,
                                                                 std::uint8_t* flags, std::int32_t* counts) {
    __shared__ int total;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    const int count = *count_dev, i = blockIdx.x * kSelectThreads + threadIdx.x;
    bool keep = i < count;
    if (keep && i > 0) {
        const JMove x = m[i - 1], y = m[i];
        bool same = x.size && x.size == y.size && x.a == y.a && x.b == y.b && x.gain == y.gain && x.net == y.net;
        for (int j = 0; same && j < x.size; ++j) {
            bool found = false;
            for (int q = 0; q < y.size; ++q) found |= x.v[j] == y.v[q];
            same = found;
        }
        keep = !same;
    }
    if (i < count) flags[i] = keep;
    const int mine = __popcll(__ballot(keep));
    if (lane_id() == 0 && mine) atomicAdd(&total, mine);
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = total;
}
__global__ void __launch_bounds__(kSelectThreads) k_unique_place(const JMove* m, const int* count_dev,
                                                                 const std::uint8_t* flags, const std::int32_t* counts,
                                                                 JMove* out, unsigned long long* host,
                                                                 unsigned long long* flag, unsigned long long seq) {
    const std::int64_t at =
        select_tile(flags, *count_dev, 1, counts, [&](std::int64_t j, std::int64_t i) { out[j] = m[i]; });
    if (blockIdx.x != gridDim.x - 1) return;
    if (threadIdx.x == 0) host[0] = (unsigned long long)at;
    publish_to_host(flag, seq);
}

__device__ inline int jnet_bound(const JMove* r, int count, int pa, std::int64_t net, bool upper) {
    int lo = 0, hi = count;
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        const JMove& x = r[mid];
        if (x.a < pa || (x.a == pa && (x.net < net || (upper && x.net == net)))) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// joint_combine (complementary_moves.cuh:31-75): one wave per fragment.
__global__ void k_joint_combine(RefArgs a, int count, const JMove* archive, int id_base, JMove* out) {
    const int lane = lane_id();
    const int i = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (i >= count) return;
    // Member loops run to the constant bound 8 with a size test, so the
    // members stay in registers.
    const JMove x = archive[i];
    const std::int64_t lo = (std::int64_t)a.loads[x.a] - (std::int64_t)a.cap;
    const std::int64_t hi = (std::int64_t)a.cap - (std::int64_t)a.loads[x.b];
    if (lane == 0) {
        JMove o = x;
        o.id = id_base + i;
        if (jgap(x.net, lo, hi)) o.size = 0;
        out[i] = o;
        out[count + i] = jmove_empty();
    }
    const int begin = jnet_bound(archive, count, x.a, lo - x.net, false);
    const int end = jnet_bound(archive, count, x.a, hi - x.net, true);
    // Up to four candidates (quartiles of the feasible range), checked
    // first; the member rows of x are then scanned once for all of them.
    int cand[4] = {-1, -1, -1, -1};
    std::int32_t cv[4][8];
    int nc = 0, previous = -1;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int t = 0; t < 8; ++t) cv[r][t] = -1;
        if (begin >= end) continue;
        const int j = begin + (int)(((std::int64_t)(end - begin - 1) * r) / 3);
        if (j == previous) continue;
        previous = j;
        if (j == i) continue;
        const JMove y = archive[j];
        if (y.a != x.a || y.b != x.b || x.size + y.size > 8) continue;
        bool overlap = false;
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int t = 0; t < 8; ++t) overlap |= u < x.size && t < y.size && x.v[u] == y.v[t];
        if (overlap) continue;
        cand[r] = j;
#pragma unroll
        for (int t = 0; t < 8; ++t) cv[r][t] = t < y.size ? y.v[t] : -1;
        ++nc;
    }
    std::int64_t corr[4] = {0, 0, 0, 0};
    if (nc)
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (u >= x.size) break;
            const std::int32_t v = x.v[u];
            const int lv = a.labels[v];
            for (std::int64_t e = a.off[v] + lane; e < a.off[v + 1]; e += kWave) {
                const std::int32_t nb = a.nbr[e];
                bool seen = false;
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int t = 0; t < 8; ++t) seen |= nb == cv[c][t];
                if (!seen) continue;
                const std::int64_t w = (lv == a.labels[nb] ? 2 : -2) * (std::int64_t)ew_at(a.ew, e);
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int t = 0; t < 8; ++t)
                        if (nb == cv[c][t]) corr[c] += w;
            }
        }
    std::int64_t best_gain = 0;
    int best = -1;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (cand[c] < 0) continue;
        const std::int64_t gain = x.gain + archive[cand[c]].gain + wave_sum(corr[c]);
        if (gain > best_gain || (gain == best_gain && gain > 0 && cand[c] < best)) {
            best_gain = gain;
            best = cand[c];
        }
    }
    if (lane == 0 && best >= 0) {
        JMove res = x;
        const JMove y = archive[best];
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int t = 0; t < 8; ++t)
                if (t < y.size && q == x.size + t) res.v[q] = y.v[t];
        res.size = x.size + y.size;
        res.gain = best_gain;
        res.net += y.net;
        res.id = id_base + count + i;
        out[count + i] = res;
    }
}

__global__ void k_joint_claim(const JMove* m, int count, std::int32_t* owners) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count)
        for (int j = 0; j < m[i].size; ++j) atomicMin(&owners[m[i].v[j]], i);
}
__global__ void k_joint_resolve(JMove* m, int count, const std::int32_t* owners) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    for (int j = 0; j < m[i].size; ++j)
        if (owners[m[i].v[j]] != i) {
            m[i].size = 0;
            break;
        }
}
// Clears the owner of every vertex and its moving flag before the claimed
// transactions are marked and accepted (nothing in between reads the flag).
__global__ void k_exchange_reset(std::int64_t n, std::int32_t* owners, std::uint32_t* state) {
    const std::uint32_t keep = ~(0xffu << (8 * kStateFlag));
    for (std::int64_t v = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < n;
         v += (std::int64_t)gridDim.x * blockDim.x) {
        owners[v] = INT_MAX;
        state[v] &= keep;
    }
}

// Also clears each transaction's event total for k_joint_events.
__global__ void k_joint_mark(RefArgs a, const JMove* m, int count, std::int32_t* owners, unsigned long long* events) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    events[i] = 0;
    for (int j = 0; j < m[i].size; ++j) {
        const std::int32_t v = m[i].v[j];
        owners[v] = i;
        a.targets[v] = a.labels[v] == m[i].a ? m[i].b : m[i].a;
    }
}
// Cut events of the claimed transactions (the semantics of
// exchange.cuh:205-262).  Every undirected edge with an end in a transaction
// contributes the change of its cut state once, counted from its lower end
// when both ends move: an edge inside one transaction, or to a vertex that
// stays, is charged whole to that transaction; an edge between transactions
// i < j is split into the change when i applies (charged to i) and the rest
// when j applies (charged to j), so prefix sums in list order are exact.
// Edges to a vertex of another transaction on other parts do not change.
//
// CDNA design: a block takes 32 consecutive transactions, stages their
// member rows (start, length, transaction) in LDS and walks them as one
// flattened edge range, so lanes stay busy whatever the row lengths.  Each
// wave reduces its lanes' charges to their own transactions by masked DPP
// butterflies, one per distinct transaction among its lanes (found by
// ballot), into 64-bit LDS totals; a charge to another transaction goes to
// global memory at once.  The totals are flushed once per block.  All sums
// are modulo 2^64, as the signed contributions of the reference.
constexpr int kEventTx = 32;
constexpr int kEventRows = kEventTx * 8;
constexpr int kEventThreads = 256;

__global__ void __launch_bounds__(kEventThreads) k_joint_events(RefArgs a, const JMove* m, int count,
                                                                const std::int32_t* owners,
                                                                unsigned long long* events) {
    __shared__ std::int32_t row_start[kEventRows];
    __shared__ std::int32_t row_first[kEventRows + 1];  // exclusive prefix of row lengths
    __shared__ std::int32_t row_vertex[kEventRows];
    __shared__ std::int32_t tx_a[kEventTx], tx_b[kEventTx];
    __shared__ unsigned long long totals[kEventTx];
    __shared__ std::int32_t wave_sums[kEventThreads / kWave];
    const int t = threadIdx.x, lane = lane_id(), w = t / kWave;
    const int tx0 = blockIdx.x * kEventTx;
    // Row t is member t % 8 of transaction t / 8 (length 0 if absent).
    {
        const int tx = t / 8, j = t % 8, i = tx0 + tx;
        std::int32_t len = 0, v = -1, start = 0;
        if (i < count && j < m[i].size) {
            v = m[i].v[j];
            start = a.off[v];
            len = a.off[v + 1] - start;
        }
        row_start[t] = start;
        row_vertex[t] = v;
        if (j == 0) {
            tx_a[tx] = i < count ? m[i].a : -1;
            tx_b[tx] = i < count ? m[i].b : -1;
            totals[tx] = 0;
        }
        const std::int32_t inc = wave_inclusive_scan<PlusOp>(len);
        if (lane == kWave - 1) wave_sums[w] = inc;
        __syncthreads();
        std::int32_t before = 0;
        for (int x = 0; x < w; ++x) before += wave_sums[x];
        row_first[t] = before + inc - len;
        if (t == kEventThreads - 1) row_first[kEventRows] = before + inc;
    }
    __syncthreads();
    const std::int32_t total = row_first[kEventRows];
    for (std::int32_t base = 0; base < total; base += kEventThreads) {
        const std::int32_t f = base + t;
        int key = -1;
        unsigned long long own = 0;
        if (f < total) {
            int lo = 0, hi = kEventRows - 1;  // last row whose first entry is <= f
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (row_first[mid] <= f) lo = mid;
                else hi = mid - 1;
            }
            const int tx = lo / 8, i = tx0 + tx;
            const std::int32_t v = row_vertex[lo];
            const std::int64_t e = (std::int64_t)row_start[lo] + (f - row_first[lo]);
            const std::int32_t u = a.nbr[e];
            const std::int32_t other = owners[u];
            const int lu = a.labels[u], lv = a.labels[v];
            const bool counted = u != v && (other == INT_MAX || (v < u && (lu == tx_a[tx] || lu == tx_b[tx])));
            if (counted) {
                const std::int64_t we = (std::int64_t)ew_at(a.ew, e);
                const int tv = a.targets[v];
                const int before = lv != lu;
                if (other == i || other == INT_MAX) {
                    const int after = tv != (other == i ? (int)a.targets[u] : lu);
                    own = (unsigned long long)((before - after) * we);
                } else {
                    const int tu = a.targets[u];
                    const int middle = i < other ? tv != lu : lv != tu;
                    const int after = tv != tu;
                    const unsigned long long first = (unsigned long long)((before - middle) * we);
                    const unsigned long long last = (unsigned long long)((middle - after) * we);
                    own = i < other ? first : last;
                    const unsigned long long theirs = i < other ? last : first;
                    if (theirs) atomicAdd(&events[other], theirs);
                }
                if (own) key = tx;
            }
        }
        // Per distinct transaction among the lanes: one masked butterfly sum.
        unsigned long long pending = __ballot(key >= 0);
        while (pending) {
            const int leader = __ffsll(pending) - 1;
            const int lk = __shfl(key, leader);
            const bool mine = key == lk;
            const unsigned long long s = wave_allreduce(mine ? own : 0ULL, PlusU64{});
            if (lane == leader) atomicAdd(&totals[lk], s);
            pending &= ~__ballot(mine);
        }
    }
    __syncthreads();
    if (t < kEventTx && tx0 + t < count && totals[t]) atomicAdd(&events[tx0 + t], totals[t]);
}
// joint_prefix / joint_accept (exchange.cuh:263-289).  One wave per part
// pa over its moves (the list is sorted by part): gain and net prefixes by
// wave scans, 64 moves per step.  The serial rule (walk the moves, keep the
// move where a feasible prefix gain first exceeds the best so far, starting
// from 0) keeps the first move of the largest feasible positive prefix
// gain, which is what the per-step maximum and first-lane ballot take.
__global__ void k_joint_prefix(RefArgs a, const JMove* m, int count, const unsigned long long* events,
                               std::int32_t* stops) {
    const int lane = lane_id();
    const int pa = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (pa >= a.k) return;
    int low = 0, high = count;
    while (low < high) {
        const int mid = (low + high) / 2;
        if (m[mid].a < pa) low = mid + 1;
        else high = mid;
    }
    int end = low;
    high = count;
    while (end < high) {
        const int mid = (end + high) / 2;
        if (m[mid].a <= pa) end = mid + 1;
        else high = mid;
    }
    const std::int64_t lo = (std::int64_t)a.loads[pa] - (std::int64_t)a.cap;
    std::int64_t gain = 0, net = 0, best = 0;
    int stop = -1;
    for (int base = low; base < end; base += kWave) {
        const int i = base + lane;
        std::int64_t g = 0, d = 0;
        int b = 0;
        bool live = false;
        if (i < end) {
            live = m[i].size != 0;
            if (live) {
                g = (std::int64_t)events[i];
                d = m[i].net;
                b = m[i].b;
            }
        }
        const std::int64_t pg = gain + wave_inclusive_scan<PlusOp>(g);
        const std::int64_t pn = net + wave_inclusive_scan<PlusOp>(d);
        std::int64_t cand = LLONG_MIN;
        if (live && !jgap(pn, lo, (std::int64_t)a.cap - (std::int64_t)a.loads[b])) cand = pg;
        const std::int64_t top = wave_max(cand);
        if (top > best) {
            best = top;
            stop = base + __ffsll((unsigned long long)__ballot(cand == top)) - 1;
        }
        gain = __shfl(pg, kWave - 1);
        net = __shfl(pn, kWave - 1);
    }
    if (lane == 0) stops[pa] = stop;
}
// Block 0 also clears the counter words [first, last) for the compaction,
// update and commit of the accepted moves.
__global__ void k_joint_accept(RefArgs a, const JMove* m, int count, const std::int32_t* stops, int first, int last) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0)
        for (int x = first + (int)threadIdx.x; x < last; x += blockDim.x) a.ctr[x] = 0;
    if (i < count && m[i].size && i <= stops[m[i].a])
        for (int j = 0; j < m[i].size; ++j) a.flags[m[i].v[j]] = 1;
}

// ---------------------------------------------------------- basics
template <typename L>
__global__ void k_project(std::int64_t n, const std::int32_t* map, const L* coarse, L* fine) {
    for (std::int64_t v = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < n;
         v += (std::int64_t)gridDim.x * blockDim.x)
        fine[v] = coarse[map[v]];
}
template <typename A, typename B>
__global__ void k_convert(std::int64_t n, const A* in, B* out) {
    for (std::int64_t v = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < n;
         v += (std::int64_t)gridDim.x * blockDim.x)
        out[v] = (B)in[v];
}

inline int grid_for(std::int64_t n, int per_block = 256, int cap = 8192) {
    return static_cast<int>(std::max<std::int64_t>(1, std::min<std::int64_t>(ceil_div(n, per_block), cap)));
}

template <typename A, typename B>
void convert(Context& c, std::int64_t n, const A* in, B* out) {
    if (n <= 0) return;
    hipLaunchKernelGGL((k_convert<A, B>), dim3(grid_for(n, 256, 4096)), dim3(256), 0, c.stream(), n, in, out);
    GP_LAUNCH_CHECK();
}

// Cut of symmetric labels and, with loads, the part loads, in one pass.
template <typename L>
std::uint64_t cut_of(Context& c, const DGraph& g, const L* labels, int k, std::uint64_t* loads = nullptr) {
    const std::uint64_t d = recount(c, g, labels, k, loads);
    if (d & 1ULL) throw std::runtime_error("refinement cut is not symmetric");
    return d / 2;
}

}  // namespace

// ====================================================================== host

void project(Context& c, std::int64_t n, const std::int32_t* map, const std::int32_t* coarse, std::int32_t* fine) {
    if (n <= 0) return;
    hipLaunchKernelGGL((k_project<std::int32_t>), dim3(grid_for(n)), dim3(256), 0, c.stream(), n, map, coarse, fine);
    GP_LAUNCH_CHECK();
}

std::uint64_t device_edge_weight_sum(Context& c, const DGraph& g) {
    if (!g.ew) return static_cast<std::uint64_t>(g.m);
    DBuf<unsigned long long> out = c.buf<unsigned long long>(1);
    fill<unsigned long long>(c, out.get(), 1, 0ULL);
    if (g.m > 0) {
        hipLaunchKernelGGL((k_reduce_sum<std::uint32_t>), dim3(grid_for(g.m)), dim3(256), 0, c.stream(), g.ew.get(), g.m,
                           out.get());
        GP_LAUNCH_CHECK();
    }
    return c.read_scalar(out.get());
}

namespace {

class LevelRefiner {
public:
    LevelRefiner(Context& c, const DGraph& g, Label* labels, std::vector<std::uint64_t>& loads,
                 const RefineOptions& o, std::uint64_t cap, LevelStats& st)
        : c_(c), g_(g), loads_host_(loads), o_(o), st_(st) {
        const std::int64_t n = g.n;
        const int k = o.parts;
        std::memset(&a_, 0, sizeof a_);
        a_.n = n;
        a_.off = g.off.get();
        a_.nbr = g.nbr.get();
        a_.ew = g.ew_ptr();
        a_.vw = g.vw.get();
        a_.k = k;
        a_.cap = cap;
        a_.labels = labels;
        state_ = c.buf<std::uint32_t>(n);
        // Gains of at most the row weight: 32 bits below 2^31.
        if (row_weight_bound() < (1ULL << 31))
            gains32_ = c.buf<std::int32_t>(n);
        else
            gains_ = c.buf<std::int64_t>(n);
        frontier_ = c.buf<std::int32_t>(n);
        cand_ = c.buf<std::int32_t>(n);
        movers_ = c.buf<std::int32_t>(n);
        medium_ = c.buf<std::int32_t>(n);
        heavy_ = c.buf<std::int32_t>(n);
        // Counters and part loads share one allocation: one read returns both.
        // Counters, part loads, then the device loop words, the best loads and
        // the heavy-edge flag.
        ctr_ = c.buf<unsigned long long>(static_cast<std::size_t>(kCtrCount + k + kLoopWords + k + 1));
        loads0_ = c.buf<unsigned long long>(static_cast<std::size_t>(k));
        bucket_ = c.buf<std::int32_t>(n);
        counts_ = c.buf<unsigned long long>(static_cast<std::size_t>(k) * kBalanceWidth);
        std::uint8_t* lanes = reinterpret_cast<std::uint8_t*>(state_.get());
        a_.state = state_.get();
        a_.targets = StateLane<std::int8_t>{reinterpret_cast<std::int8_t*>(lanes + kStateTarget)};
        a_.flags = StateLane<std::uint8_t>{lanes + kStateFlag};
        a_.member = StateLane<std::uint8_t>{lanes + kStateMember};
        a_.own = StateLane<std::uint8_t>{lanes + kStateOwn};
        a_.gains = gains_.get();
        a_.gains32 = gains32_.get();
        a_.ctr = ctr_.get();
        a_.loads = ctr_.get() + kCtrCount;
        a_.loads0 = loads0_.get();
        a_.bucket = bucket_.get();
        a_.counts = counts_.get();
        unsigned long long* heavy_edge = ctr_.get() + kCtrCount + 2 * k + kLoopWords;
        std::uint64_t total = 0;
        for (auto x : loads) total += x;
        if (total > static_cast<std::uint64_t>(n)) {
            prices_ = c.buf<double>(static_cast<std::size_t>(k));
            samples_ = c.buf<RepairSample>(static_cast<std::size_t>(k));
            a_.prices = prices_.get();
            a_.samples = samples_.get();
        }
        hipLaunchKernelGGL(k_level_begin, dim3(1), dim3(256), 0, c.stream(), ctr_.get(), part_words(loads), a_.loads, k,
                           heavy_edge, prices_.get());
        GP_LAUNCH_CHECK();
        if (g.ew && g.m > 0) {
            hipLaunchKernelGGL(k_heavy_edge, dim3(grid_for(g.m, 256 * 16, 256)), dim3(256), 0, c.stream(), g.m,
                               g.ew.get(), heavy_edge);
            GP_LAUNCH_CHECK();
            a_.heavy_edge = heavy_edge;
        }
        // Boundary vertices seed the frontier; per-level resets (its tier
        // counters were cleared with the counter block above).
        tiers(BoundaryBody{{a_}}, nullptr, n, nullptr, nullptr, nullptr, nullptr, 0, kTier, true);
    }

    // The level's part loads after the host has put other labels in place.
    void set_loads(const std::vector<std::uint64_t>& loads) {
        hipLaunchKernelGGL(k_set_parts, dim3(1), dim3(kMaxParts), 0, c_.stream(), part_words(loads), a_.loads, a_.k);
        GP_LAUNCH_CHECK();
    }

    std::uint64_t max_load() const {
        std::uint64_t m = 0;
        for (auto x : loads_host_) m = std::max(m, x);
        return m;
    }

    // Clears the moving flag and the target (-1) of every vertex, the state
    // the exchange starts from.
    void clear_moves(Context& c) {
        hipLaunchKernelGGL(k_clear_moves, dim3(grid_for(a_.n, 256, 2048)), dim3(256), 0, c.stream(), state_.get(),
                           a_.labels, a_.n);
        GP_LAUNCH_CHECK();
    }

    // Short-row bins fit 32 bits when every row of the level weighs less
    // than 2^32 (the level's incident-weight bound).
    bool narrow_bins() const { return row_weight_bound() <= 0xffffffffULL; }
    // Rows of unit weights weigh their length, whose bound a changed graph
    // keeps when its weight bound is unknown.
    std::uint64_t row_weight_bound() const {
        return g_.ew ? g_.incident_bound : std::min(g_.incident_bound, g_.row_len_bound);
    }

    // slot: the two tier list counters; zeroed: they are known to be zero
    // (cleared with the counter block since their last use).
    template <class Body>
    void tiers(const Body& body, const std::int32_t* list, std::int64_t n, const unsigned long long* count,
               std::int32_t* out, unsigned long long* out_count, unsigned long long* acc, int scratch,
               int slot = kTier, bool zeroed = false, int entries_slot = -1, std::int64_t max_rows = -1) {
        run_tiers(c_, body, list, n, count, medium_.get(), heavy_.get(), ctr_.get() + slot, out, out_count, acc,
                  scratch, max_rows < 0 ? a_.n : max_rows, g_.row_len_bound, zeroed,
                  entries_slot >= 0 && c_.profiling() ? ctr_.get() + entries_slot : nullptr);
    }

    // One LP round over the frontier; returns the number of movers and the cut delta.
    std::int64_t lp_round(std::int64_t& delta) {
        const hipStream_t s = c_.stream();
        const std::int64_t n = a_.n;
        if (!ctr_clear_) fill<unsigned long long>(c_, ctr_.get(), kCtrCount, 0ULL);
        ctr_clear_ = false;
        hipLaunchKernelGGL(k_compact_flags<StateLane<std::uint8_t>>, dim3(grid_for(n, kCompactTile, 512)), dim3(kCompactThreads), 0, s, n,
                           a_.member,
                           frontier_.get(), ctr_.get() + kFrontier, nullptr);
        GP_LAUNCH_CHECK();
        // Algorithmic bytes per scanned row: offsets 8, label and weight 8,
        // target and gain 12, and per entry neighbour 4, neighbour label 4
        // and edge weight 4 when weighted; added once the row sums are read.
        propose_sweeps();
        return apply(true, false, delta, true);
    }

    // The launches of one LP round of a device-controlled loop: the frontier
    // compaction does nothing once the loop word kRun is zero, so every later
    // launch of the round finds empty lists; the commit's last block ends it.
    // Returns the number the round publishes in the mailbox flag.
    unsigned long long round_issue(const LoopParams& P, Label* best_labels, bool vec) {
        const hipStream_t s = c_.stream();
        const std::int64_t n = a_.n;
        unsigned long long* L = ctr_.get() + kCtrCount + a_.k;
        hipLaunchKernelGGL(k_compact_flags<StateLane<std::uint8_t>>, dim3(grid_for(n, kCompactTile, 512)), dim3(kCompactThreads), 0, s, n, a_.member, frontier_.get(), ctr_.get() + kFrontier, L + kRun);
        GP_LAUNCH_CHECK();
        propose_sweeps();
        // Levels of at most kKeepInline vertices checkpoint where the round is
        // decided; larger ones in a launch of their own.
        const bool inline_keep = n <= kKeepInline;
        const unsigned long long seq = c_.next_seq();
        RoundEnd end{};
        end.mode = kEndDecide;
        end.P = P;
        end.ticket = c_.ticket();
        end.host = c_.mailbox();
        end.flag = c_.mailbox_flag();
        end.seq = seq;
        end.keep = inline_keep ? best_labels : nullptr;
        end.vec = vec;
        apply_launch(true, false, true, end);
        if (!inline_keep) {
            hipLaunchKernelGGL(k_lp_keep, dim3(grid_for(ceil_div(n, 16), 256, 1024)), dim3(256), 0, s, L + kImproved,
                               a_.labels, best_labels, n, vec);
            GP_LAUNCH_CHECK();
        }
        return seq;
    }

    // The LP proposal and afterburner sweeps of a round (counter block clear).
    void propose_sweeps() {
        unsigned long long* row_sum = c_.profiling() ? ctr_.get() + kRowSum : nullptr;
        c_.timed("lp_propose", 0.0, [&] {
            if (narrow_bins())
                tiers(LpProposeBody<unsigned>{{a_}}, frontier_.get(), 0, ctr_.get() + kFrontier, cand_.get(),
                      ctr_.get() + kCand, row_sum, a_.k, kTier, true);
            else
                tiers(LpProposeBody<unsigned long long>{{a_}}, frontier_.get(), 0, ctr_.get() + kFrontier, cand_.get(),
                      ctr_.get() + kCand, row_sum, a_.k, kTier, true);
        });
        c_.timed("after", 0.0, [&] {
            if (a_.gains32)
                tiers(AfterBody<std::int32_t>{{a_}}, cand_.get(), 0, ctr_.get() + kCand, movers_.get(),
                      ctr_.get() + kMovers, nullptr, 0, kTierB, true, kEntAfter);
            else
                tiers(AfterBody<std::int64_t>{{a_}}, cand_.get(), 0, ctr_.get() + kCand, movers_.get(),
                      ctr_.get() + kMovers, nullptr, 0, kTierB, true, kEntAfter);
        });
    }

    // The LP round loop of the level with its control on the device
    // (lp_decide applies the host loop's rules after each round).  The
    // host issues each round before it has seen the previous one end
    // (ahead) or right after, watching only the mailbox; it takes over when
    // a round leaves a part over capacity, for the repair and the rest of
    // that round, and then re-arms the loop.  Same rounds, moves and
    // checkpoints as the host loop.
    void lp_loop(int rounds, bool graph_mode, std::uint64_t& cut, std::uint64_t& best_cut, Label* best_labels,
                 std::vector<std::uint64_t>& best_loads) {
        const hipStream_t s = c_.stream();
        const int k = a_.k;
        const bool vec = reinterpret_cast<std::uintptr_t>(a_.labels) % 16 == 0 &&
                         reinterpret_cast<std::uintptr_t>(best_labels) % 16 == 0;
        const LoopParams P{k,
                           rounds,
                           o_.stale_rounds,
                           graph_mode ? 1 : 0,
                           g_.row_len_bound <= static_cast<std::uint64_t>(kTierLight) ? 1 : 0,
                           c_.profiling() ? 1 : 0,
                           a_.cap,
                           significand_0999()};
        const int ahead = c_.loop_ahead();
        volatile unsigned long long* mail = c_.mailbox();
        std::uint64_t phase = 0, stale = 0, empty = 0, lp_moves = 0;
        bool copy_best = true;
        while (phase < static_cast<std::uint64_t>(rounds) && stale < static_cast<std::uint64_t>(o_.stale_rounds)) {
            reset_samples();
            const std::uint64_t phase0 = phase;
            hipLaunchKernelGGL(k_lp_arm, dim3(1), dim3(256), 0, s, ctr_.get(), k, 1ULL, phase, stale, empty, cut,
                               best_cut, lp_moves, copy_best ? 1 : 0);
            GP_LAUNCH_CHECK();
            mail[kRun] = 1;  // the stream is idle: no round of an earlier run is in flight
            std::vector<std::size_t> marks;
            unsigned long long seqs[2] = {0, 0};  // of the last two rounds issued
            auto issue = [&] {
                marks.push_back(c_.pending_mark());
                seqs[0] = seqs[1];
                seqs[1] = round_issue(P, best_labels, vec);
            };
            issue();
            for (;;) {
                if (ahead) issue();
                c_.wait_flag(c_.mailbox_flag(), seqs[ahead ? 0 : 1]);
                if (!mail[kRun]) break;
                if (!ahead) issue();
            }
            // Issuing ahead, the stop may come from the round still in
            // flight: wait for the stream before reading the full state.
            if (ahead) c_.sync();
            std::vector<unsigned long long> h(static_cast<std::size_t>(kLoopWords + 2 * k));
            for (std::size_t i = 0; i < h.size(); ++i) h[i] = mail[i];
            ctr_clear_ = true;
            phase = h[kPhase];
            stale = h[kStale];
            empty = h[kEmpty];
            cut = h[kCut];
            best_cut = h[kBestCut];
            lp_moves = h[kLpMoves];
            for (int p = 0; p < k; ++p) {
                loads_host_[static_cast<std::size_t>(p)] = h[static_cast<std::size_t>(kLoopWords + p)];
                best_loads[static_cast<std::size_t>(p)] = h[static_cast<std::size_t>(kLoopWords + k + p)];
            }
            // Rounds issued after the stop did nothing: drop their intervals.
            const std::size_t ran = static_cast<std::size_t>(phase - phase0);
            if (ran < marks.size()) c_.drop_pending(marks[ran]);
            if (c_.profiling()) {
                const double w = a_.ew ? 4.0 : 0.0;
                c_.add_bytes("lp_propose", 28.0 * (double)h[kAccFrontier] + (8.0 + w) * (double)h[kAccRowSum]);
                const double g = a_.gains32 ? 4.0 : 0.0;  // 32-bit gains: 4 B less per row and entry
                c_.add_bytes("after", (16.0 - g) * (double)h[kAccAfterR] + (16.0 - g + w) * (double)h[kAccAfterE]);
                c_.add_bytes("update", 24.0 * (double)h[kAccUpdateR] + (8.0 + w) * (double)h[kAccUpdateE]);
            }
            const int reason = static_cast<int>(h[kReason]);
            if (reason == kCutUnderflow) throw std::runtime_error("incremental cut underflow");
            if (reason == kDeferred)
                throw std::logic_error("rows longer than the level's row-length bound were deferred and not processed");
            if (reason != kNeedRepair) break;
            // The rest of the round as the host loop runs it.
            if (!rebalance(cut)) break;
            publish_prices();
            ++stale;
            copy_best = false;
            if (cut < best_cut) {
                if (graph_mode) {
                    if (best_cut - cut > best_cut / 1000) stale = 0;
                } else if ((long double)cut < 0.999L * (long double)best_cut)
                    stale = 0;
                best_cut = cut;
                c_.copy_d2d(best_labels, a_.labels, static_cast<std::size_t>(a_.n) * sizeof(Label));
                best_loads = loads_host_;
                copy_best = true;
            }
        }
        st_.rounds = static_cast<int>(phase);
        st_.lp_moves += lp_moves;
    }

    // Update + commit of the current mover list.  zeroed: the delta and
    // third-sweep tier counters are still zero from the counter block's
    // clear at the start of the round or repair iteration.
    // donors, settled: as k_commit takes them (null outside repair).
    void apply_launch(bool lp, bool samples, bool zeroed, const RoundEnd& end, const std::int32_t* donors = nullptr,
                      bool settled = true) {
        const hipStream_t s = c_.stream();
        if (!zeroed) fill<unsigned long long>(c_, ctr_.get() + kDelta, 1, 0ULL);
        if (!zeroed && c_.profiling()) fill<unsigned long long>(c_, ctr_.get() + kEntUpdate, 2, 0ULL);
        c_.timed("update", 0.0, [&] {
            tiers(UpdateBody{{a_}, samples && a_.samples}, movers_.get(), 0, ctr_.get() + kMovers, nullptr, nullptr,
                  ctr_.get() + kDelta, 0, kTierC, zeroed, kEntUpdate);
            hipLaunchKernelGGL(k_commit, dim3(grid_for(a_.n, kCommitThreads, kCommitBlocks)), dim3(kCommitThreads), 0,
                               s, a_, movers_.get(), ctr_.get() + kMovers, lp, samples && a_.samples, donors, ctr_.get() + kSelected,
                               settled, end);
            GP_LAUNCH_CHECK();
        });
        if (samples) samples_clear_ = false;
    }

    std::int64_t apply(bool lp, bool samples, std::int64_t& delta, bool zeroed = false,
                       const std::int32_t* donors = nullptr, bool settled = true) {
        std::vector<unsigned long long> h(static_cast<std::size_t>(kCtrCount + a_.k));
        // The read-back also clears the counters (not the part loads behind them).
        RoundEnd end{};
        end.mode = kEndRead;
        end.ticket = c_.ticket();
        end.host = c_.read_buffer();
        end.flag = c_.read_flag();
        end.seq = c_.next_seq();
        end.words = static_cast<int>(h.size());
        apply_launch(lp, samples, zeroed, end, donors, settled);
        c_.wait_flag(end.flag, end.seq);
        std::memcpy(h.data(), c_.read_buffer(), h.size() * sizeof(unsigned long long));
        ctr_clear_ = true;
        selected_ = (std::int64_t)h[kSelected];
        // With no row above kTierLight entries no medium launch was made; a
        // row the light launch deferred would have gone unprocessed.
        if (g_.row_len_bound <= static_cast<std::uint64_t>(kTierLight) && (h[kTier] || h[kTierB] || h[kTierC]))
            throw std::logic_error("rows longer than the level's row-length bound were deferred and not processed");
        for (int p = 0; p < a_.k; ++p) loads_host_[static_cast<std::size_t>(p)] = h[static_cast<std::size_t>(kCtrCount + p)];
        delta = (std::int64_t)h[kDelta];
        if (c_.profiling()) {
            // Algorithmic bytes per row and per entry of each sweep (weighted
            // graphs add 4 B of edge weight per entry): LP proposal 28 + 8;
            // afterburner 16 + 16 (neighbour, state word, gain; 4 B less each
            // with 32-bit gains); update and commit 24 + 8 (neighbour, state
            // word); repair proposal 24 + 8 (offsets, label, weight, bucket and
            // target out; neighbour and its label per entry).
            const double w = a_.ew ? 4.0 : 0.0;
            if (lp) {
                c_.add_bytes("lp_propose", 28.0 * (double)h[kFrontier] + (8.0 + w) * (double)h[kRowSum]);
                const double g = a_.gains32 ? 4.0 : 0.0;
                c_.add_bytes("after", (16.0 - g) * (double)h[kEntAfter + 1] + (16.0 - g + w) * (double)h[kEntAfter]);
            }
            c_.add_bytes("update", 24.0 * (double)h[kEntUpdate + 1] + (8.0 + w) * (double)h[kEntUpdate]);
            if (samples)
                c_.add_bytes("repair_propose", 24.0 * (double)h[kEntRepair + 1] + (8.0 + w) * (double)h[kEntRepair]);
        }
        return (std::int64_t)h[kMovers];
    }

    bool update_cut(std::uint64_t& cut, std::int64_t delta) {
        if (delta >= 0) {
            if ((std::uint64_t)delta > cut) throw std::runtime_error("incremental cut underflow");
            cut -= (std::uint64_t)delta;
        } else
            cut += (std::uint64_t)(-delta);
        if (o_.strict_verify) verify(cut);
        return true;
    }

    // Strict mode (incremental.cuh:846-853): after every committed batch the
    // incremental cut must equal a full CSR recount of the labels and the
    // part loads a full recount of the vertex weights.
    void verify(std::uint64_t cut) {
        std::vector<std::uint64_t> loads(static_cast<std::size_t>(a_.k));
        if (cut_of(c_, g_, a_.labels, a_.k, loads.data()) != cut)
            throw std::runtime_error("incremental cut differs from CSR scan");
        if (loads != loads_host_) throw std::runtime_error("incremental part weights differ from a recount");
        ++st_.strict_checks;
    }

    // Sparse connection rows of the eligible donors (ConnBody by the row
    // tiers over the positions [0, ne) of E): ne from the device when
    // count_dev is not null, then at most max_rows.
    void conn_rows(const std::int32_t* E, std::int64_t ne, const unsigned long long* count_dev, std::int64_t max_rows,
                   const std::uint8_t* skip, unsigned long long* vals, std::uint8_t* parts, std::uint8_t* nnz) {
        // Within a repair iteration the second sweep's tier counters are
        // still zero from the iteration's counter clear (k_repair_begin).
        if (narrow_bins())
            tiers(ConnBody<unsigned>{{a_}, E, skip, vals, parts, nnz}, nullptr, ne, count_dev, nullptr, nullptr, nullptr,
                  a_.k, kTierB, true, -1, max_rows);
        else
            tiers(ConnBody<unsigned long long>{{a_}, E, skip, vals, parts, nnz}, nullptr, ne, count_dev, nullptr,
                  nullptr, nullptr, a_.k, kTierB, true, -1, max_rows);
    }

    // Arrays of a level's repair iterations: the donor selection's, and the
    // state and connection rows of what one tail launch takes.
    struct RepairBuffers {
        DBuf<unsigned long long> prefix, excess, S, tried, slack, requests, conn;
        DBuf<std::int32_t> bstar, counts, E;
        DBuf<std::uint8_t> elig, done, conn_part, conn_nnz;
        DBuf<DonorInfo> live;
        int rounds = 0, tiles = 0;
    };

    RepairBuffers repair_buffers() {
        RepairBuffers b;
        const std::size_t n = static_cast<std::size_t>(a_.n), k = static_cast<std::size_t>(a_.k);
        b.rounds = select_rounds(a_.n);
        b.tiles = ceil_div(a_.n, (std::int64_t)b.rounds * kSelectThreads);
        b.prefix = c_.buf<unsigned long long>(k * kBalanceWidth);
        b.bstar = c_.buf<std::int32_t>(k);
        b.excess = c_.buf<unsigned long long>(k);
        b.S = c_.buf<unsigned long long>(static_cast<std::size_t>(b.tiles) * k);
        b.counts = c_.buf<std::int32_t>(static_cast<std::size_t>(b.tiles));
        b.elig = c_.buf<std::uint8_t>(n);
        b.E = c_.buf<std::int32_t>(n);
        const std::size_t tail = static_cast<std::size_t>(std::min<std::int64_t>(a_.n, kTailDonors));
        b.live = c_.buf<DonorInfo>(tail);
        b.done = c_.buf<std::uint8_t>(tail);
        b.tried = c_.buf<unsigned long long>(2 * tail);
        b.slack = c_.buf<unsigned long long>(k);
        b.requests = c_.buf<unsigned long long>(k);
        b.conn = c_.buf<unsigned long long>(tail * k);
        b.conn_part = c_.buf<std::uint8_t>(tail * k);
        b.conn_nnz = c_.buf<std::uint8_t>(tail);
        return b;
    }

    // Reservation of the selected donors when one tail launch takes them all:
    // their connection rows (those of donors admitted in attempt 0 go unused),
    // then all attempts.  The count stays on the device; with more donors
    // than that it is zero there and both launches do nothing.
    void reserve_tail(RepairBuffers& b) {
        const unsigned long long* count = ctr_.get() + kSelected + 1;
        const std::int64_t rows = std::min<std::int64_t>(a_.n, kTailDonors);
        conn_rows(b.E.get(), 0, count, rows, nullptr, b.conn.get(), b.conn_part.get(), b.conn_nnz.get());
        const ReserveState r{b.E.get(),        rows,           b.conn.get(),  b.conn_part.get(), b.conn_nnz.get(),
                             b.requests.get(), b.slack.get(),  b.done.get(),  b.tried.get(),     b.live.get(),
                             0,                count};
        hipLaunchKernelGGL(k_reserve_tail, dim3(1), dim3(kTailThreads), 0, c_.stream(), a_, r, 0, movers_.get(),
                           ctr_.get() + kMovers);
        GP_LAUNCH_CHECK();
    }

    // Reservation of ne selected donors, more than one tail launch takes.
    void reserve_groups(RepairBuffers& b, std::int64_t ne) {
        const hipStream_t s = c_.stream();
        const int k = a_.k;
        DBuf<std::int32_t> keys = c_.buf<std::int32_t>(static_cast<std::size_t>(ne));
        DBuf<unsigned long long> S =
            c_.buf<unsigned long long>(static_cast<std::size_t>(ceil_div(ne, kKeyTile)) * k);
        // Connection rows are read from the second attempt on, and only for
        // donors still waiting; they are built once attempt 0 is done.
        DBuf<unsigned long long> conn = c_.buf<unsigned long long>(static_cast<std::size_t>(ne) * k);
        DBuf<std::uint8_t> conn_part = c_.buf<std::uint8_t>(static_cast<std::size_t>(ne) * k);
        DBuf<std::uint8_t> conn_nnz = c_.buf<std::uint8_t>(static_cast<std::size_t>(ne));
        DBuf<DonorInfo> live = c_.buf<DonorInfo>(static_cast<std::size_t>(ne));  // later the waiting donors only
        DBuf<std::uint8_t> done_buf = c_.buf<std::uint8_t>(static_cast<std::size_t>(ne));
        DBuf<unsigned long long> tried = c_.buf<unsigned long long>(static_cast<std::size_t>(ne) * 2);
        const std::int32_t* E = b.E.get();
        std::uint8_t* done = done_buf.get();
        unsigned long long* requests = b.requests.get();
        hipLaunchKernelGGL(k_donor_start, dim3(grid_for(ne)), dim3(256), 0, s, a_, E, ne, live.get(), done,
                           tried.get());
        GP_LAUNCH_CHECK();
        ReserveState r{E,        ne,            conn.get(), conn_part.get(), conn_nnz.get(), requests,
                       b.slack.get(), done, tried.get(), live.get(), ne, nullptr};
        // Attempts run in groups between host checks: an attempt without a
        // chooser changes nothing (no tried bits, no requests, no admissions),
        // so the attempts after the last active one are no-ops.  Between
        // groups the live list drops donors that are admitted or have no
        // part left; it stays in ascending order, so ranks are unchanged.
        constexpr int kAttemptGroup = 4;
        constexpr std::int64_t kCompactMin = 4096;
        DBuf<unsigned long long> active = c_.buf<unsigned long long>(kAttemptGroup);
        for (int attempt = 0; attempt < k;) {
            const int group = std::min(kAttemptGroup, k - attempt);
            const std::int64_t nlv = r.nlive;
            const int nb = static_cast<int>(ceil_div(nlv, kKeyTile));
            fill<unsigned long long>(c_, active.get(), kAttemptGroup, 0ULL);
            for (int j = 0; j < group; ++j, ++attempt) {
                if (attempt == 1) {
                    conn_rows(E, ne, nullptr, -1, done, conn.get(), conn_part.get(), conn_nnz.get());
                }
                // Blocks stride over the donors: the per-block room table and
                // part order are set up once per block.
                hipLaunchKernelGGL(k_choose, dim3(grid_for(nlv, kTierThreads / kChooseLanes, 1024)), dim3(kTierThreads), 0, s, a_,
                                   r, attempt, keys.get(), active.get() + j);
                GP_LAUNCH_CHECK();
                hipLaunchKernelGGL((k_keyed_sums<DonorWeight>), dim3(nb), dim3(kTierThreads), 0, s, keys.get(), nlv, k,
                                   nb, DonorWeight{r.live}, S.get());
                GP_LAUNCH_CHECK();
                // Ranks start at the start-of-attempt totals; totals advance.
                hipLaunchKernelGGL(k_keyed_scan, dim3(ceil_div(k, kTierThreads / kWave)), dim3(kTierThreads), 0, s,
                                   S.get(), nb, k, requests);
                GP_LAUNCH_CHECK();
                hipLaunchKernelGGL((k_keyed_apply<AdmitFn>), dim3(nb), dim3(kTierThreads), 0, s, keys.get(), nlv,
                                   S.get(), nb, AdmitFn{a_, r}, movers_.get(), ctr_.get() + kMovers);
                GP_LAUNCH_CHECK();
            }
            if (!c_.read_scalar(active.get() + group - 1)) break;
            if (nlv >= kCompactMin && attempt < k) {
                DBuf<std::uint8_t> lf = c_.buf<std::uint8_t>(static_cast<std::size_t>(nlv));
                DBuf<std::int32_t> li = c_.buf<std::int32_t>(static_cast<std::size_t>(nlv));
                DBuf<std::int64_t> lc = c_.buf<std::int64_t>(1);
                hipLaunchKernelGGL(k_live_flags, dim3(grid_for(nlv)), dim3(256), 0, s, r.live, nlv, done, lf.get());
                GP_LAUNCH_CHECK();
                stable_select(c_, lf.get(), nlv, li.get(), lc.get());
                const std::int64_t next = c_.read_scalar(lc.get());
                if (next == 0) break;
                DBuf<DonorInfo> live2 = c_.buf<DonorInfo>(static_cast<std::size_t>(next));
                hipLaunchKernelGGL(k_gather_info, dim3(grid_for(next)), dim3(256), 0, s, r.live, li.get(), next,
                                   live2.get());
                GP_LAUNCH_CHECK();
                live.swap(live2);
                r.live = live.get();
                r.nlive = next;
            }
            // A donor list that fits one block finishes in one launch.
            if (r.nlive <= kTailDonors && attempt < k) {
                hipLaunchKernelGGL(k_reserve_tail, dim3(1), dim3(kTailThreads), 0, s, a_, r, attempt, movers_.get(),
                                   ctr_.get() + kMovers);
                GP_LAUNCH_CHECK();
                break;
            }
        }
    }

    // Capacity repair loop (rebalance_graph.cuh:160-280); returns feasibility.
    bool rebalance(std::uint64_t& cut) {
        const hipStream_t s = c_.stream();
        const std::int64_t n = a_.n;
        const int k = a_.k;
        int iterations = 0;
        bool feasible = false;
        std::int64_t count = 0;
        RepairBuffers b = repair_buffers();
        const SelectState q{b.bstar.get(), b.prefix.get(), b.excess.get(), b.S.get(),     b.counts.get(),
                            b.elig.get(),  b.E.get(),      b.live.get(),   b.done.get(),  b.tried.get(),
                            b.slack.get(), b.requests.get(), ctr_.get() + kSelected,
                            static_cast<unsigned long long>(kTailDonors)};
        // Whether the last iteration had more eligible donors than one tail
        // launch takes: then the host reads their number before it goes on.
        bool many = false;
        const std::int64_t ncounts = (std::int64_t)k * kBalanceWidth;
        do {
            static_assert(kCtrCount <= kBalanceWidth, "the counter block clears inside the bucket clear");
            // The counter block is zero after a read-back that cleared it
            // (every iteration's last); then one launch starts the iteration.
            const bool zeroed = ctr_clear_;
            ctr_clear_ = false;
            const int donor_grid = grid_for(n, kCompactTile, 512);
            if (zeroed) {
                hipLaunchKernelGGL(k_repair_donors, dim3(std::max(donor_grid, grid_for(ncounts, kCompactThreads))),
                                   dim3(kCompactThreads), 0, s, a_,
                                   cand_.get(), ctr_.get() + kDonors, loads0_.get(), counts_.get(), ncounts);
            } else {
                hipLaunchKernelGGL(k_repair_begin, dim3(grid_for(ncounts)), dim3(256), 0, s, a_, loads0_.get(),
                                   counts_.get(), ncounts, ctr_.get(), (int)kCtrCount);
                GP_LAUNCH_CHECK();
                hipLaunchKernelGGL(k_repair_donors, dim3(donor_grid), dim3(kCompactThreads), 0, s, a_, cand_.get(),
                                   ctr_.get() + kDonors, nullptr, nullptr, 0);
            }
            GP_LAUNCH_CHECK();
            c_.timed("repair_propose", 0.0, [&] {
                if (narrow_bins())
                    tiers(RepairProposeBody<unsigned>{{a_}}, cand_.get(), 0, ctr_.get() + kDonors, nullptr, nullptr,
                          nullptr, a_.k, kTier, true, kEntRepair);
                else
                    tiers(RepairProposeBody<unsigned long long>{{a_}}, cand_.get(), 0, ctr_.get() + kDonors, nullptr,
                          nullptr, nullptr, a_.k, kTier, true, kEntRepair);
            });
            hipLaunchKernelGGL(k_bucket_scan, dim3(k), dim3(kScanThreads), 0, s, a_, b.prefix.get(),
                               b.bstar.get(), b.excess.get());
            GP_LAUNCH_CHECK();
            if (n <= kSelectSmallMax) {
                hipLaunchKernelGGL(k_donors_small, dim3(1), dim3(kDonorThreads), 0, s, a_, q);
                GP_LAUNCH_CHECK();
            } else {
                hipLaunchKernelGGL(k_select_weights, dim3(b.tiles), dim3(kSelectThreads), 0, s, a_, q, b.rounds);
                GP_LAUNCH_CHECK();
                hipLaunchKernelGGL(k_select_eligible, dim3(b.tiles), dim3(kSelectThreads), 0, s, a_, q, b.rounds);
                GP_LAUNCH_CHECK();
                hipLaunchKernelGGL(k_select_place, dim3(b.tiles), dim3(kSelectThreads), 0, s, a_, q, b.rounds);
                GP_LAUNCH_CHECK();
            }
            // The number of eligible donors decides the form of the
            // reservation.  As long as one tail launch took the last
            // iteration's, the launches of this one go out without a look at
            // it: with more they move nothing, and the read-back at their end
            // says so.
            std::int64_t delta = 0;
            std::int64_t ne = many ? (std::int64_t)c_.read_scalar(ctr_.get() + kSelected) : 0;
            if (ne <= kTailDonors) {
                reserve_tail(b);
                count = apply(false, true, delta, true, cand_.get(), false);
                ne = selected_;
                many = false;
            }
            if (ne > kTailDonors) {
                reserve_groups(b, ne);
                count = apply(false, true, delta, true, cand_.get(), true);
                many = true;
            }
            ++iterations;
            if (count) {
                update_cut(cut, delta);
                st_.repair_moves += static_cast<std::uint64_t>(count);
            }
            feasible = max_load() <= a_.cap;
        } while (!feasible && count && iterations < 2 * k + 4);
        st_.repair_iterations += iterations;
        return feasible;
    }

    // Capacity-complementary exchange (incremental.cuh:974-1041).
    void exchange(int passes, std::uint64_t& cut, std::uint64_t& best_cut) {
        const hipStream_t s = c_.stream();
        ctr_clear_ = false;
        const std::int64_t n = a_.n;
        const int k = a_.k;
        int sw = std::min(kJointSeeds, std::max(32, 4096 / k));
        const int slots = k * sw * 2;
        DBuf<unsigned long long> A = c_.buf<unsigned long long>(static_cast<std::size_t>(n) * k);
        DBuf<unsigned long long> Q = c_.buf<unsigned long long>(static_cast<std::size_t>(k) * k);
        DBuf<std::int32_t> visits = c_.buf<std::int32_t>(static_cast<std::size_t>(k) * k);
        DBuf<std::int32_t> partner = c_.buf<std::int32_t>(static_cast<std::size_t>(k));
        DBuf<unsigned long long> seeds = c_.buf<unsigned long long>(static_cast<std::size_t>(k) * sw);
        DBuf<JMove> grown = c_.buf<JMove>(static_cast<std::size_t>(slots));
        DBuf<JMove> archive = c_.buf<JMove>(static_cast<std::size_t>(slots) * kJointArchive);
        DBuf<std::int32_t> owners = c_.buf<std::int32_t>(n);
        DBuf<std::int32_t> stops = c_.buf<std::int32_t>(static_cast<std::size_t>(k));
        auto dense = [&] {
            hipLaunchKernelGGL((k_dense_affinity<64>), dim3(grid_for(n, 4, 4096)), dim3(256), 4 * k * sizeof(unsigned long long), s, a_,
                               A.get());
            GP_LAUNCH_CHECK();
        };
        dense();
        fill<unsigned long long>(c_, Q.get(), (std::int64_t)k * k, 0ULL);
        fill<std::int32_t>(c_, visits.get(), (std::int64_t)k * k, 0);
        hipLaunchKernelGGL(k_quotient, dim3(grid_for(n)), dim3(256), 0, s, a_, A.get(), Q.get());
        GP_LAUNCH_CHECK();
        int empty = 0;
        for (int pass = 0; pass < passes; ++pass) {
            hipLaunchKernelGGL(k_joint_match, dim3(1), dim3(kMatchThreads), 0, s, k, Q.get(), partner.get(), visits.get(),
                               seeds.get(), k * sw);
            GP_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_joint_seeds, dim3(grid_for(n)), dim3(256), 0, s, a_, A.get(), partner.get(),
                               seeds.get(), sw, pass);
            GP_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_joint_grow, dim3(ceil_div(slots, kGrowWaves)), dim3(kGrowWaves * kWave), 0, s, a_,
                               A.get(), slots, sw,
                               seeds.get(), partner.get(), grown.get(), archive.get());
            GP_LAUNCH_CHECK();
            // Archive: non-empty, sorted by net order, unique.
            const int an = slots * kJointArchive;
            DBuf<JMove> frag;
            const int fragments = compact_sort(archive.get(), an, NetOrder{}, frag, true);
            const int pool_cap = slots + 2 * fragments;
            DBuf<JMove> pool = c_.buf<JMove>(static_cast<std::size_t>(std::max(pool_cap, 1)));
            c_.copy_d2d(pool.get(), grown.get(), static_cast<std::size_t>(slots) * sizeof(JMove));
            if (fragments) {
                hipLaunchKernelGGL(k_joint_combine, dim3(ceil_div(fragments, 4)), dim3(256), 0, s, a_, fragments,
                                   frag.get(), slots, pool.get() + slots);
                GP_LAUNCH_CHECK();
            }
            DBuf<JMove> moves;
            const int active = compact_sort(pool.get(), pool_cap, JointOrder{}, moves, false);
            if (!active) {
                if (++empty >= 2) break;
                continue;
            }
            fill<std::int32_t>(c_, owners.get(), n, INT_MAX);
            hipLaunchKernelGGL(k_joint_claim, dim3(ceil_div(active, 256)), dim3(256), 0, s, moves.get(), active,
                               owners.get());
            hipLaunchKernelGGL(k_joint_resolve, dim3(ceil_div(active, 256)), dim3(256), 0, s, moves.get(), active,
                               owners.get());
            hipLaunchKernelGGL(k_exchange_reset, dim3(grid_for(n)), dim3(256), 0, s, n, owners.get(), state_.get());
            DBuf<unsigned long long> events = c_.buf<unsigned long long>(static_cast<std::size_t>(active));
            hipLaunchKernelGGL(k_joint_mark, dim3(ceil_div(active, 256)), dim3(256), 0, s, a_, moves.get(), active,
                               owners.get(), events.get());
            GP_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_joint_events, dim3(ceil_div(active, kEventTx)), dim3(kEventThreads), 0, s, a_,
                               moves.get(), active,
                               owners.get(), events.get());
            hipLaunchKernelGGL(k_joint_prefix, dim3(ceil_div(k, 4)), dim3(256), 0, s, a_, moves.get(), active,
                               events.get(), stops.get());
            // The accept also clears the mover count and every counter the
            // update and commit of this batch use (delta, its tier lists,
            // profiled entries).
            hipLaunchKernelGGL(k_joint_accept, dim3(ceil_div(active, 256)), dim3(256), 0, s, a_, moves.get(), active,
                               stops.get(), (int)kMovers, (int)kCtrCount);
            hipLaunchKernelGGL(k_compact_flags<StateLane<std::uint8_t>>, dim3(grid_for(n, kCompactTile, 512)), dim3(kCompactThreads), 0, s,
                               n, a_.flags,
                               movers_.get(), ctr_.get() + kMovers, nullptr);
            GP_LAUNCH_CHECK();
            const unsigned long long cnt = c_.read_scalar(ctr_.get() + kMovers);
            if (!cnt) {
                if (++empty >= 2) break;
                continue;
            }
            empty = 0;
            std::int64_t delta = 0;
            apply(false, false, delta, true);
            if (delta <= 0) throw std::runtime_error("non-improving boundary group batch");
            update_cut(cut, delta);
            st_.group_moves += cnt;
            if (max_load() > a_.cap || cut >= best_cut) throw std::runtime_error("capacity exchange violated cut/capacity");
            best_cut = cut;
            dense();
        }
        // Later passes wrote the mover counter after the last read.
        ctr_clear_ = false;
    }

    // The non-empty moves of src in cmp order, repeats dropped when unique is
    // set; their number (out holds room for `count`).
    template <typename Cmp>
    int compact_sort(const JMove* src, int count, Cmp cmp, DBuf<JMove>& out, bool unique) {
        const hipStream_t s = c_.stream();
        if (count <= 0) return 0;
        const int k = a_.k, blocks = ceil_div(count, kOrderThreads);
        DBuf<std::int32_t> block_at = c_.buf<std::int32_t>(static_cast<std::size_t>(blocks) * k);
        DBuf<std::int32_t> starts = c_.buf<std::int32_t>(static_cast<std::size_t>(k) + 1);
        DBuf<std::int32_t> order = c_.buf<std::int32_t>(static_cast<std::size_t>(count));
        out = c_.buf<JMove>(static_cast<std::size_t>(count));
        const unsigned long long seq = c_.next_seq();
        hipLaunchKernelGGL(k_moves_count, dim3(blocks), dim3(kOrderThreads), 0, s, src, count, k, block_at.get(),
                           starts.get(), c_.ticket(), unique ? nullptr : c_.read_buffer(), c_.read_flag(), seq);
        GP_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_moves_group, dim3(blocks), dim3(kOrderThreads), 0, s, src, count, k, block_at.get(),
                           order.get());
        GP_LAUNCH_CHECK();
        DBuf<JMove> runs = c_.buf<JMove>(static_cast<std::size_t>(count));
        hipLaunchKernelGGL((k_moves_runs<Cmp>), dim3(k, kRankSplit), dim3(kRankThreads), 0, s, src, starts.get(),
                           order.get(), cmp, runs.get());
        GP_LAUNCH_CHECK();
        hipLaunchKernelGGL((k_moves_merge<Cmp>), dim3(k, kRankSplit), dim3(kRankThreads), 0, s, runs.get(),
                           starts.get(), cmp, out.get());
        GP_LAUNCH_CHECK();
        if (unique) {
            DBuf<JMove> left = c_.buf<JMove>(static_cast<std::size_t>(count));
            DBuf<std::uint8_t> flags = c_.buf<std::uint8_t>(static_cast<std::size_t>(count));
            const int tiles = ceil_div(count, kSelectThreads);
            DBuf<std::int32_t> counts = c_.buf<std::int32_t>(static_cast<std::size_t>(tiles));
            hipLaunchKernelGGL(k_unique_flags, dim3(tiles), dim3(kSelectThreads), 0, s, out.get(), starts.get() + k,
                               flags.get(), counts.get());
            GP_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_unique_place, dim3(tiles), dim3(kSelectThreads), 0, s, out.get(), starts.get() + k,
                               flags.get(), counts.get(), left.get(), c_.read_buffer(), c_.read_flag(), seq);
            GP_LAUNCH_CHECK();
            out.swap(left);
        }
        c_.wait_flag(c_.read_flag(), seq);
        return static_cast<int>(c_.read_buffer()[0]);
    }

    void publish_prices() {
        if (!prices_) return;
        hipLaunchKernelGGL(k_publish_prices, dim3(1), dim3(kMaxParts), 0, c_.stream(), samples_.get(), prices_.get(),
                           a_.k);
        GP_LAUNCH_CHECK();
        samples_clear_ = true;
    }

    void reset_samples() {
        if (samples_ && !samples_clear_)
            fill<unsigned long long>(c_, reinterpret_cast<unsigned long long*>(samples_.get()), 2 * a_.k, 0ULL);
        samples_clear_ = true;
    }

    Context& c_;
    const DGraph& g_;
    std::vector<std::uint64_t>& loads_host_;
    const RefineOptions& o_;
    LevelStats& st_;
    RefArgs a_;
    DBuf<std::uint32_t> state_;
    DBuf<std::int32_t> frontier_, cand_, movers_, medium_, heavy_, bucket_;
    DBuf<std::int64_t> gains_;
    DBuf<std::int32_t> gains32_;
    DBuf<unsigned long long> ctr_, loads0_, counts_;
    DBuf<double> prices_;
    DBuf<RepairSample> samples_;
    // Host knowledge that the counter block (first kCtrCount words) or the
    // repair samples are zero on the device, so their clear can be skipped.
    bool ctr_clear_ = false;
    bool samples_clear_ = false;
    std::int64_t selected_ = 0;  // eligible donors of the last repair iteration, as the last read-back had it
};

}  // namespace

namespace {

LevelStats refine_level_impl(Context& c, const DGraph& g, Label* labels, std::vector<std::uint64_t>& loads,
                             const RefineOptions& o, std::uint64_t cap, int rounds, bool has_known_cut,
                             std::uint64_t known_cut) {
    LevelStats st;
    st.n = g.n;
    st.m = g.m;
    st.refined = 1;
    const int k = o.parts;
    LevelRefiner R(c, g, labels, loads, o, cap, st);
    std::uint64_t cut = has_known_cut ? known_cut : cut_of(c, g, labels, k);
    if (o.strict_verify && has_known_cut) {
        // incremental.cuh:777-778: the carried cut must equal a recount.
        if (cut_of(c, g, labels, k) != known_cut) throw std::runtime_error("known projection cut differs from CSR scan");
        ++st.strict_checks;
    }
    st.initial_cut = cut;
    if (R.max_load() > cap) {
        R.reset_samples();
        if (!R.rebalance(cut)) {
            st.initial_repair_failed = 1;
            st.final_cut = cut;
            return st;
        }
    }
    const std::uint64_t feasible_start = cut;
    std::uint64_t best_cut = cut;
    DBuf<Label> best_labels = c.buf<Label>(static_cast<std::size_t>(g.n));
    std::vector<std::uint64_t> best_loads = loads;
    c.copy_d2d(best_labels.get(), labels, static_cast<std::size_t>(g.n) * sizeof(Label));
    const bool graph_mode = g.n >= o.graph_loop_threshold;
    int stale = 0, empty = 0;
    // Strict mode recounts on the host after every batch: host loop.
    const bool device_loop = o.device_loop && c.device_loop() && !o.strict_verify;
    if (device_loop) R.lp_loop(rounds, graph_mode, cut, best_cut, best_labels.get(), best_loads);
    const int host_rounds = device_loop ? 0 : rounds;
    for (int phase = 0; phase < host_rounds && stale < o.stale_rounds; ++phase) {
        st.rounds = phase + 1;
        R.reset_samples();
        std::int64_t delta = 0;
        const std::int64_t count = R.lp_round(delta);
        if (!count) {
            if (++empty >= 2) break;
            ++stale;
            continue;
        }
        empty = 0;
        R.update_cut(cut, delta);
        st.lp_moves += static_cast<std::uint64_t>(count);
        if (R.max_load() > cap && !R.rebalance(cut)) break;
        R.publish_prices();
        ++stale;
        if (cut < best_cut) {
            if (graph_mode) {
                if (best_cut - cut > best_cut / 1000) stale = 0;
            } else if ((long double)cut < 0.999L * (long double)best_cut)
                stale = 0;
            best_cut = cut;
            c.copy_d2d(best_labels.get(), labels, static_cast<std::size_t>(g.n) * sizeof(Label));
            best_loads = loads;
        }
    }
    c.copy_d2d(labels, best_labels.get(), static_cast<std::size_t>(g.n) * sizeof(Label));
    loads = best_loads;
    R.set_loads(loads);
    cut = best_cut;
    if (rounds > 0 && o.exchange_rounds > 0 && g.n <= o.exchange_max_n) {
        R.clear_moves(c);
        R.exchange(o.exchange_rounds, cut, best_cut);
    }
    st.final_cut = cut;
    std::uint64_t mx = 0;
    for (auto x : loads) mx = std::max(mx, x);
    if (cut != best_cut || cut > feasible_start || mx > cap)
        throw std::runtime_error("incremental refinement postcondition failed");
    if (o.strict_verify) {
        // The restored checkpoint: its cut and loads against recounts.
        R.verify(cut);
    }
    return st;
}

}  // namespace

bool debug_below_0999(std::uint64_t cut, std::uint64_t best) { return below_0999(cut, best, significand_0999()); }

LevelStats refine_level(Context& c, const DGraph& g, std::int32_t* labels, std::vector<std::uint64_t>& loads,
                        const RefineOptions& o, std::uint64_t cap, int rounds, bool has_known_cut,
                        std::uint64_t known_cut) {
    DBuf<Label> lab = c.buf<Label>(static_cast<std::size_t>(g.n));
    convert(c, g.n, labels, lab.get());
    LevelStats st = refine_level_impl(c, g, lab.get(), loads, o, cap, rounds, has_known_cut, known_cut);
    convert(c, g.n, lab.get(), labels);
    return st;
}

UncoarsenResult uncoarsen(Context& c, const Hierarchy& h, const std::int32_t* coarsest_labels, const RefineOptions& o) {
    const int k = o.parts;
    UncoarsenResult res;
    const DGraph& cg = h.level(h.levels() - 1);
    DBuf<Label> labels = c.buf<Label>(static_cast<std::size_t>(cg.n));
    convert(c, cg.n, coarsest_labels, labels.get());
    std::vector<std::uint64_t> loads(static_cast<std::size_t>(k), 0);
    const std::uint64_t directed = recount(c, cg, labels.get(), k, loads.data());
    std::uint64_t total = 0;
    for (auto x : loads) total += x;
    const long double raw = (long double)total * o.imbalance / k;
    const std::uint64_t cap = (std::uint64_t)std::floor(raw);
    if (cap < total / (unsigned)k + (total % (unsigned)k != 0))
        throw std::invalid_argument("integer partition capacity cannot hold total weight");
    if (directed & 1ULL) throw std::runtime_error("refinement cut is not symmetric");
    LevelStats st =
        refine_level_impl(c, cg, labels.get(), loads, o, cap, o.max_rounds, !o.strict_verify, directed / 2);
    res.levels.push_back(st);
    std::uint64_t last_cut = st.final_cut;
    std::int64_t last_refined = cg.n;
    for (int lvl = h.levels() - 2; lvl >= 0; --lvl) {
        const DGraph& fg = h.level(lvl);
        DBuf<Label> fl = c.buf<Label>(static_cast<std::size_t>(fg.n));
        if (fg.n > 0) {
            hipLaunchKernelGGL((k_project<Label>), dim3(grid_for(fg.n)), dim3(256), 0, c.stream(), fg.n,
                               h.maps[static_cast<std::size_t>(lvl)].get(), labels.get(), fl.get());
            GP_LAUNCH_CHECK();
        }
        labels = std::move(fl);
        LevelStats ls;
        ls.n = fg.n;
        ls.m = fg.m;
        if (o.strict_verify) {
            // refine.cu:641-659: projection preserves the cut and the part loads.
            std::vector<std::uint64_t> projected(static_cast<std::size_t>(k));
            if (cut_of(c, fg, labels.get(), k, projected.data()) != last_cut || projected != loads)
                throw std::runtime_error("GPU projection failed cut or part-weight preservation");
            ++ls.strict_checks;
        }
        std::uint64_t maxload = 0;
        for (auto x : loads) maxload = std::max(maxload, x);
        const bool refine = lvl == 0 || maxload > cap || (double)fg.n >= o.growth_ratio * (double)last_refined;
        if (refine) {
            const std::uint64_t projection_checks = ls.strict_checks;
            ls = refine_level_impl(c, fg, labels.get(), loads, o, cap, o.max_rounds, true, last_cut);
            ls.strict_checks += projection_checks;
            if (!ls.initial_repair_failed) last_refined = fg.n;
        } else {
            ls.initial_cut = ls.final_cut = last_cut;
        }
        last_cut = ls.final_cut;
        res.levels.push_back(ls);
    }
    std::uint64_t maxload = 0;
    for (auto x : loads) maxload = std::max(maxload, x);
    if (maxload > cap) throw std::runtime_error("final original partition violates capacity");
    const DGraph& g0 = h.level(0);
    res.labels = c.buf<std::int32_t>(static_cast<std::size_t>(g0.n));
    convert(c, g0.n, labels.get(), res.labels.get());
    res.loads = loads;
    res.cut = last_cut;
    return res;
}

}  // namespace gp
