// Device update of a resident CSR by a batch of undirected edge deletions
// and insertions (repartition requests of a server's resident graphs; no
// counterpart in the reference, whose graphs are read from disk once).
//
// Semantics: deletions apply first, then insertions; deleting an absent
// edge changes nothing, and an insertion of an edge present after the
// deletions, or given twice, is dropped (the first weight is kept).  Each
// row keeps its surviving entries in their old order, followed by its new
// neighbours in ascending order.  Inserted edges carry the given weights (1
// when none are given); a graph with implicit unit weights gets an explicit
// weight array when an inserted weight is not 1.
//
// Layout on the device: the directed delta records (both directions) sorted
// by (source, kind, neighbour), with one record range per changed row.  Rows
// without a record move by an entry-parallel copy (each entry finds its row
// by a binary search over the old offsets); a changed row is scanned and
// rebuilt by one wave, each entry looked up by binary search among the row's
// sorted deletions and insertions (hub rows carry many records).  Bound:
// HBM, one read and one write of the CSR.
#include "gp_update.hpp"

#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <vector>

namespace gp {

namespace {

struct DeltaRows {
    const std::int32_t* row;      // changed rows, ascending
    const std::int32_t* first;    // records of row i: [first[i], first[i + 1])
    const std::int32_t* mid;      // deletions [first[i], mid[i]), insertions [mid[i], first[i + 1])
    const std::int32_t* dst;      // record neighbour, ascending within each kind
    const std::uint32_t* weight;  // insert weight
    std::uint8_t* present;        // per insertion: its edge is in the row after the deletions
    std::int64_t count;           // changed rows
};

// Position of u in the ascending range [lo, hi) of a, or -1.
__device__ inline std::int32_t find_sorted(const std::int32_t* a, std::int32_t lo, std::int32_t hi, std::int32_t u) {
    const std::int32_t end = hi;
    while (lo < hi) {
        const std::int32_t mid = lo + ((hi - lo) >> 1);
        if (a[mid] < u) lo = mid + 1;
        else hi = mid;
    }
    return lo < end && a[lo] == u ? lo : -1;
}

__global__ void k_delta_degree(std::int64_t n, const std::int32_t* off, std::int32_t* deg) {
    for (std::int64_t v = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < n;
         v += (std::int64_t)gridDim.x * blockDim.x)
        deg[v] = off[v + 1] - off[v];
}

// One wave per changed row: the entries that survive the row's deletions
// (a binary search over the sorted deletions each), and the insertions whose
// edge is among them (flagged present).  deg[v] receives the survivors.
__global__ void k_delta_scan_rows(const std::int32_t* off, const std::int32_t* nbr, DeltaRows d, std::int32_t* deg) {
    const int lane = lane_id();
    const std::int64_t waves = (std::int64_t)gridDim.x * blockDim.x / kWave;
    for (std::int64_t i = (blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x) / kWave; i < d.count; i += waves) {
        const std::int32_t v = d.row[i];
        const std::int64_t b = off[v], e = off[v + 1];
        const std::int32_t f0 = d.first[i], fm = d.mid[i], f1 = d.first[i + 1];
        std::int64_t kept = 0;
        for (std::int64_t x = b + lane; x < e; x += kWave) {
            const std::int32_t u = nbr[x];
            if (fm > f0 && find_sorted(d.dst, f0, fm, u) >= 0) continue;
            ++kept;
            const std::int32_t r = f1 > fm ? find_sorted(d.dst, fm, f1, u) : -1;
            if (r >= 0) d.present[r] = 1;
        }
        kept = wave_sum(kept);
        if (lane == 0) deg[v] = (std::int32_t)kept;
    }
}

// One thread per changed row: survivors plus the insertions not present.
__global__ void k_delta_row_degree(DeltaRows d, std::int32_t* deg, std::uint8_t* changed) {
    for (std::int64_t i = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; i < d.count;
         i += (std::int64_t)gridDim.x * blockDim.x) {
        const std::int32_t v = d.row[i];
        std::int32_t added = 0;
        for (std::int32_t r = d.mid[i]; r < d.first[i + 1]; ++r) added += !d.present[r];
        deg[v] += added;
        changed[v] = 1;
    }
}

// Entries of unchanged rows, one thread per old entry.
__global__ void k_delta_copy(std::int64_t n, std::int64_t m, const std::int32_t* off, const std::int32_t* nbr,
                             const std::uint32_t* ew, const std::uint8_t* changed, const std::int32_t* noff,
                             std::int32_t* nnbr, std::uint32_t* new_ew) {
    for (std::int64_t x = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; x < m;
         x += (std::int64_t)gridDim.x * blockDim.x) {
        std::int64_t lo = 0, hi = n - 1;  // last row whose first entry is <= x
        while (lo < hi) {
            const std::int64_t mid = (lo + hi + 1) >> 1;
            if (off[mid] <= x) lo = mid;
            else hi = mid - 1;
        }
        if (changed[lo]) continue;
        const std::int64_t y = noff[lo] + (x - off[lo]);
        nnbr[y] = nbr[x];
        if (new_ew) new_ew[y] = ew ? ew[x] : 1u;
    }
}

// One wave per changed row: the survivors in their old order (ballot
// compaction), then the insertions not present, ascending.
__global__ void k_delta_rows(const std::int32_t* off, const std::int32_t* nbr, const std::uint32_t* ew, DeltaRows d,
                             const std::int32_t* noff, std::int32_t* nnbr, std::uint32_t* new_ew) {
    const int lane = lane_id();
    const unsigned long long below = (1ULL << lane) - 1ULL;
    const std::int64_t waves = (std::int64_t)gridDim.x * blockDim.x / kWave;
    for (std::int64_t i = (blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x) / kWave; i < d.count; i += waves) {
        const std::int32_t v = d.row[i];
        const std::int64_t b = off[v], e = off[v + 1];
        const std::int32_t f0 = d.first[i], fm = d.mid[i], f1 = d.first[i + 1];
        std::int64_t y = noff[v];
        for (std::int64_t x0 = b; x0 < e; x0 += kWave) {
            const std::int64_t x = x0 + lane;
            std::int32_t u = 0;
            bool keep = false;
            if (x < e) {
                u = nbr[x];
                keep = fm == f0 || find_sorted(d.dst, f0, fm, u) < 0;
            }
            const unsigned long long mask = __ballot(keep);
            if (keep) {
                const std::int64_t at = y + __popcll(mask & below);
                nnbr[at] = u;
                if (new_ew) new_ew[at] = ew ? ew[x] : 1u;
            }
            y += __popcll(mask);
        }
        for (std::int32_t r0 = fm; r0 < f1; r0 += kWave) {
            const std::int32_t r = r0 + lane;
            const bool add = r < f1 && !d.present[r];
            const unsigned long long mask = __ballot(add);
            if (add) {
                const std::int64_t at = y + __popcll(mask & below);
                nnbr[at] = d.dst[r];
                if (new_ew) new_ew[at] = d.weight[r];
            }
            y += __popcll(mask);
        }
    }
}

// ---- the delta's records, ordered on the device
// Both directions of every change as (source, insertion, neighbour) in one
// key, `bits` bits per vertex; the value is the record's number, so that a
// stable sort keeps repeats in the caller's order.
__global__ void k_delta_records(std::int64_t count, const std::int32_t* u, const std::int32_t* v,
                                const std::uint8_t* insert, int bits, std::uint64_t* keys, std::uint32_t* vals) {
    for (std::int64_t i = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; i < 2 * count;
         i += (std::int64_t)gridDim.x * blockDim.x) {
        const std::int64_t e = i / 2;
        const std::uint64_t a = (std::uint32_t)((i & 1) ? v[e] : u[e]), b = (std::uint32_t)((i & 1) ? u[e] : v[e]);
        keys[i] = a << (bits + 1) | (std::uint64_t)(insert[e] != 0) << bits | b;
        vals[i] = (std::uint32_t)i;
    }
}
__global__ void k_delta_first(std::int64_t total, const std::uint64_t* keys, std::uint8_t* flags) {
    for (std::int64_t i = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; i < total;
         i += (std::int64_t)gridDim.x * blockDim.x)
        flags[i] = i == 0 || keys[i] != keys[i - 1];
}
// The distinct records and which of them start a row (none past their number).
__global__ void k_delta_gather(std::int64_t total, const std::int64_t* distinct, const std::int32_t* idx,
                               const std::uint64_t* keys, const std::uint32_t* vals, const std::uint32_t* w, int bits,
                               std::uint64_t* ukeys, std::int32_t* dst, std::uint32_t* weight, std::uint8_t* heads) {
    const std::int64_t nu = *distinct;
    for (std::int64_t j = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; j < total;
         j += (std::int64_t)gridDim.x * blockDim.x) {
        if (j >= nu) {
            heads[j] = 0;
            continue;
        }
        const std::uint64_t key = keys[idx[j]];
        ukeys[j] = key;
        dst[j] = (std::int32_t)(key & ((1ULL << bits) - 1));
        weight[j] = w && (key >> bits & 1) ? w[vals[idx[j]] / 2] : 1u;
        heads[j] = j == 0 || keys[idx[j - 1]] >> (bits + 1) != key >> (bits + 1);
    }
}
// Rows and, within each, the first insertion (deletions come first).
__global__ void k_delta_heads(std::int64_t nrows, std::int64_t nu, const std::uint64_t* ukeys, int bits,
                              std::int32_t* rows, std::int32_t* first, std::int32_t* mid) {
    for (std::int64_t r = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; r < nrows;
         r += (std::int64_t)gridDim.x * blockDim.x) {
        const std::int32_t b = first[r], e = r + 1 < nrows ? first[r + 1] : (std::int32_t)nu;
        rows[r] = (std::int32_t)(ukeys[b] >> (bits + 1));
        std::int32_t lo = b, hi = e;
        while (lo < hi) {
            const std::int32_t m = lo + (hi - lo) / 2;
            if (ukeys[m] >> bits & 1) hi = m;
            else lo = m + 1;
        }
        mid[r] = lo;
        if (r + 1 == nrows) first[nrows] = (std::int32_t)nu;
    }
}
// Longest row.
__global__ void __launch_bounds__(kResultThreads) k_longest_row(std::int64_t n, const std::int32_t* deg,
                                                                unsigned long long* out) {
    __shared__ unsigned long long part[kResultThreads / kWave];
    std::uint64_t m = 0;
    for (std::int64_t v = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < n;
         v += (std::int64_t)gridDim.x * blockDim.x)
        m = m > (std::uint64_t)deg[v] ? m : (std::uint64_t)deg[v];
    m = wave_max(m);
    if (lane_id() == 0) part[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kResultThreads / kWave; ++w) m = m > part[w] ? m : part[w];
        if (m) atomicMax(out, (unsigned long long)m);
    }
}

inline int blocks_for(std::int64_t n) {
    return static_cast<int>(std::max<std::int64_t>(1, std::min<std::int64_t>((n + 255) / 256, 4096)));
}

}  // namespace

std::int64_t apply_delta(Context& c, DGraph& g, std::int64_t count, const std::int32_t* u, const std::int32_t* v,
                         const std::uint32_t* w, const std::uint8_t* insert) {
    if (count < 0 || (count > 0 && (!u || !v || !insert))) throw std::invalid_argument("invalid edge delta");
    bool unit = true;
    for (std::int64_t i = 0; i < count; ++i) {
        if (u[i] < 0 || u[i] >= g.n || v[i] < 0 || v[i] >= g.n || u[i] == v[i])
            throw std::invalid_argument("edge delta names an invalid vertex or a self loop");
        if (!insert[i] || !w) continue;
        if (!w[i]) throw std::invalid_argument("inserted edge weights must be positive");
        unit &= w[i] == 1u;
    }
    if (!count) return g.m;
    if (count > 0x3fffffffLL) throw std::invalid_argument("edge delta exceeds 32-bit record numbers");
    // Directed records sorted by (source, kind, neighbour), repeats dropped (the
    // first insertion's weight is kept), on the device: on the host the sort
    // and five copies, each with its own wait, were two thirds of a
    // repartition (mesh of 262,001 points: 2.9 -> 1.05 ms in all; the longest
    // row, now known, also spares the refinement its long-row launches and
    // 64-bit gains).  The changes go up in one copy.
    Arena* home = g.off.arena();  // the new arrays belong where the graph's do
    const hipStream_t s = c.stream();
    const std::size_t cnt = static_cast<std::size_t>(count), flag_words = (cnt + 3) / 4;
    std::vector<std::uint32_t> pack((w ? 3 : 2) * cnt + flag_words);
    std::memcpy(pack.data(), u, cnt * 4);
    std::memcpy(pack.data() + cnt, v, cnt * 4);
    std::memcpy(pack.data() + 2 * cnt, insert, cnt);
    if (w) std::memcpy(pack.data() + 2 * cnt + flag_words, w, cnt * 4);
    DBuf<std::uint32_t> d_pack = c.buf<std::uint32_t>(pack.size());
    c.upload(d_pack.get(), pack.data(), pack.size() * 4);
    const std::int32_t* d_u = reinterpret_cast<const std::int32_t*>(d_pack.get());
    const std::uint8_t* d_insert = reinterpret_cast<const std::uint8_t*>(d_pack.get() + 2 * cnt);
    const std::uint32_t* d_w = w ? d_pack.get() + 2 * cnt + flag_words : nullptr;
    const std::int64_t total_recs = 2 * count;
    const std::size_t recs = static_cast<std::size_t>(total_recs);
    const int bits = std::max(1, bit_width_u64(static_cast<std::uint64_t>(g.n - 1)));
    DBuf<std::uint64_t> keys = c.buf<std::uint64_t>(recs), ukeys = c.buf<std::uint64_t>(recs);
    DBuf<std::uint32_t> vals = c.buf<std::uint32_t>(recs);
    const int rec_blocks = blocks_for(total_recs);
    hipLaunchKernelGGL(k_delta_records, dim3(rec_blocks), dim3(256), 0, s, count, d_u, d_u + cnt, d_insert, bits,
                       keys.get(), vals.get());
    GP_LAUNCH_CHECK();
    radix_sort_pairs(c, keys, vals, total_recs, 0, 2 * bits + 1);
    DBuf<std::uint8_t> flags = c.buf<std::uint8_t>(recs);
    DBuf<std::int32_t> idx = c.buf<std::int32_t>(recs);
    DBuf<std::int64_t> counts = c.buf<std::int64_t>(2);  // distinct records, rows
    hipLaunchKernelGGL(k_delta_first, dim3(rec_blocks), dim3(256), 0, s, total_recs, keys.get(), flags.get());
    GP_LAUNCH_CHECK();
    stable_select(c, flags.get(), total_recs, idx.get(), counts.get());
    DBuf<std::int32_t> d_rows = c.buf<std::int32_t>(recs), d_first = c.buf<std::int32_t>(recs + 1),
                       d_mid = c.buf<std::int32_t>(recs), d_dst = c.buf<std::int32_t>(recs);
    DBuf<std::uint8_t> d_present = c.buf<std::uint8_t>(recs);
    DBuf<std::uint32_t> d_weight = c.buf<std::uint32_t>(recs);
    hipLaunchKernelGGL(k_delta_gather, dim3(rec_blocks), dim3(256), 0, s, total_recs, counts.get(), idx.get(),
                       keys.get(), vals.get(), d_w, bits, ukeys.get(), d_dst.get(), d_weight.get(), flags.get());
    GP_LAUNCH_CHECK();
    stable_select(c, flags.get(), total_recs, d_first.get(), counts.get() + 1);
    std::int64_t made[2];
    c.read(made, counts.get(), sizeof made);
    const std::int64_t nrows = made[1];
    hipLaunchKernelGGL(k_delta_heads, dim3(blocks_for(nrows)), dim3(256), 0, s, nrows, made[0], ukeys.get(), bits,
                       d_rows.get(), d_first.get(), d_mid.get());
    GP_LAUNCH_CHECK();
    fill<std::uint8_t>(c, d_present.get(), made[0], 0);
    const DeltaRows d{d_rows.get(), d_first.get(), d_mid.get(), d_dst.get(), d_weight.get(), d_present.get(), nrows};

    DBuf<std::int32_t> deg(home, static_cast<std::size_t>(g.n) + 1);
    DBuf<std::uint8_t> changed(home, static_cast<std::size_t>(g.n));
    fill<std::uint8_t>(c, changed.get(), g.n, 0);
    hipLaunchKernelGGL(k_delta_degree, dim3(blocks_for(g.n)), dim3(256), 0, s, g.n, g.off.get(), deg.get());
    GP_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_delta_scan_rows, dim3(blocks_for(nrows * kWave)), dim3(256), 0, s, g.off.get(), g.nbr.get(),
                       d, deg.get());
    GP_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_delta_row_degree, dim3(blocks_for(nrows)), dim3(256), 0, s, d, deg.get(), changed.get());
    GP_LAUNCH_CHECK();
    fill<std::int32_t>(c, deg.get() + g.n, 1, 0);
    // Entries of the new graph and its longest row.
    DBuf<unsigned long long> total = c.buf<unsigned long long>(2);
    fill<unsigned long long>(c, total.get(), 2, 0ULL);
    hipLaunchKernelGGL(k_longest_row, dim3(result_grid(g.n)), dim3(kResultThreads), 0, s, g.n, deg.get(),
                       total.get() + 1);
    GP_LAUNCH_CHECK();
    DBuf<std::int32_t> noff(home, static_cast<std::size_t>(g.n) + 1);
    exclusive_sum<unsigned long long>(c, deg.get(), noff.get(), g.n + 1, total.get());
    unsigned long long sizes[2];
    c.read(sizes, total.get(), sizeof sizes);
    const unsigned long long m2 = sizes[0];
    if (m2 > 0x7fffffffULL) throw std::invalid_argument("updated graph exceeds 32-bit CSR limits");
    DBuf<std::int32_t> nnbr(home, static_cast<std::size_t>(std::max<unsigned long long>(m2, 1)));
    const bool weighted = g.ew || !unit;
    DBuf<std::uint32_t> new_ew;
    if (weighted) new_ew = DBuf<std::uint32_t>(home, static_cast<std::size_t>(std::max<unsigned long long>(m2, 1)));
    if (g.m > 0) {
        hipLaunchKernelGGL(k_delta_copy, dim3(blocks_for(g.m)), dim3(256), 0, s, g.n, g.m, g.off.get(), g.nbr.get(),
                           g.ew_ptr(), changed.get(), noff.get(), nnbr.get(), weighted ? new_ew.get() : nullptr);
        GP_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_delta_rows, dim3(blocks_for(nrows * kWave)), dim3(256), 0, s, g.off.get(), g.nbr.get(), g.ew_ptr(),
                       d, noff.get(), nnbr.get(), weighted ? new_ew.get() : nullptr);
    GP_LAUNCH_CHECK();
    c.sync();
    g.off = std::move(noff);
    g.nbr = std::move(nnbr);
    g.ew = std::move(new_ew);
    g.m = static_cast<std::int64_t>(m2);
    // Bounds carried by coarsening are unknown for the new rows, but for their
    // length.
    g.max_degree = std::numeric_limits<std::uint64_t>::max();
    g.has_heavy = true;
    g.incident_bound = std::numeric_limits<std::uint64_t>::max();
    g.row_len_bound = sizes[1];
    return g.m;
}

}  // namespace gp
