// Edge cut and part loads of device-resident labels: the verification
// counts of the reference (host_cut, include/graph.hpp:67-69; the device cut
// and load recounts of src/refine.cu:63-98 and the final check of
// src/uncoarsen.cu:90-100), in one launch.
//
// Rows and entries together are split evenly over the waves, whatever the row
// lengths: a wave finds its first row and entry with a 64-way search (each
// step, 64 lanes probe 64 offsets) and walks its entries in windows of
// kCutRows rows, whose ends and labels it stages in LDS.  The row of a given
// entry is the number of row ends at or below it, so ballots tell the rows of
// a batch's first and last entry: a batch in one row (hubs) broadcasts its
// label, otherwise each lane finds its row by a binary search between the two.
// kCutBatch neighbours per lane are loaded before their labels are gathered.
// Part loads are summed per block in LDS over an even split of the vertices.
// Each block writes one row of partials: [directed cut weight, labels outside
// [0, k), load_0 .. load_{k-1}]; the last block to finish adds the rows up and
// writes the totals straight to the host's read-back buffer.
//
// R-MAT scale 20 (31 M entries, k = 64), counted again and again: 141 us (168
// when graph and labels change from call to call); 64 vertices per wave, the
// earlier split, took 14.5 ms, one wave walking all the hubs, and an even
// split of the entries alone 360 us, where a wave meets hundreds of rows with
// an entry or none.  kCutBatch 8 instead of 4: 196 us.
//
// Bound: the gather of a label per entry (L2 serves most of it).  Bytes per
// call: 4(n+1) offsets + 4n labels + 4n vertex weights + m (4 neighbour
// [+ 4 edge weight]).
#include "gp_metrics.hpp"

#include <algorithm>
#include <mutex>
#include <stdexcept>
#include <unordered_map>

// Scratch of the allocation-free evaluation (edge_cut_noalloc): room for the
// partial rows of the largest evaluation, 512 rows of 130 words (cut,
// out-of-range count, 128 loads), 532,480 bytes.  Every GPU holds its own copy
// until the process ends.
// Host code never passes this name to a kernel: it is a host-side stand-in,
// and the device address comes from hipGetSymbolAddress per device.
static __device__ __align__(256) unsigned long long scratch[gp::kNoAllocScratchWords];

namespace gp {

namespace {

constexpr int kCutThreads = 1024;
constexpr int kCutWaves = kCutThreads / kWave;
constexpr int kCutPer = 4;                  // staged rows per lane
constexpr int kCutRows = kCutPer * kWave;   // rows of a window

// Where the walk over rows and their entries stands after `d` steps, a row
// counting one step before its entries: the row reached, the last r in [0, n)
// with off[r] + r <= d.  The whole wave takes part.
__device__ inline std::int64_t wave_row_at(const std::int32_t* off, std::int64_t n, std::int64_t d) {
    std::int64_t lo = 0, len = n;  // the answer lies in [lo, lo + len)
    while (len > 1) {
        const std::int64_t step = (len + kWave - 1) / kWave;
        const std::int64_t at = lo + step * lane_id();
        const bool below = step * lane_id() < len && off[at] + at <= d;
        const int hits = __popcll(__ballot(below));  // ascending: the first hits lanes
        const std::int64_t first = step * (hits > 0 ? hits - 1 : 0);
        lo += first;
        len = len - first < step ? len - first : step;
    }
    return lo;
}

template <bool Weighted, class L>
__global__ void __launch_bounds__(kCutThreads) k_edge_cut(std::int64_t n, const std::int32_t* off,
                                                          const std::int32_t* nbr, const std::uint32_t* ew,
                                                          const std::uint32_t* vw, const L* labels, int k,
                                                          unsigned long long* partials, unsigned int* ticket,
                                                          unsigned long long* host, unsigned long long* flag,
                                                          unsigned long long seq) {
    __shared__ unsigned long long loads[kMaxParts];
    __shared__ std::int32_t send[kCutWaves][kCutRows];
    __shared__ L slab[kCutWaves][kCutRows];
    __shared__ unsigned long long red[kCutWaves][2];
    const int lane = lane_id(), w = threadIdx.x / kWave;
    for (int p = threadIdx.x; p < k; p += kCutThreads) loads[p] = 0;
    __syncthreads();
    unsigned long long cut = 0, bad = 0;

    for (std::int64_t v = blockIdx.x * (std::int64_t)kCutThreads + threadIdx.x; v < n;
         v += (std::int64_t)gridDim.x * kCutThreads) {
        const int lab = (int)labels[v];
        if (static_cast<unsigned>(lab) < static_cast<unsigned>(k))
            atomicAdd(&loads[lab], static_cast<unsigned long long>(vw[v]));
        else
            ++bad;
    }

    // This wave's entries [pos, stop): an even share of rows and entries.
    const std::int64_t m = n > 0 ? (std::int64_t)off[n] : 0;
    const std::int64_t waves = (std::int64_t)gridDim.x * kCutWaves;
    const std::int64_t share = (n + m + waves - 1) / waves;
    const std::int64_t d0 = (blockIdx.x * (std::int64_t)kCutWaves + w) * share;
    std::int64_t row = 0, pos = 0, stop = 0;
    if (d0 < n + m) {
        row = wave_row_at(off, n, d0);
        const std::int64_t d1 = d0 + share, row1 = d1 < n + m ? wave_row_at(off, n, d1) : 0;
        const std::int64_t e0 = off[row + 1], e1 = off[row1 + 1];
        pos = d0 - row < e0 ? d0 - row : e0;
        stop = d1 >= n + m ? m : d1 - row1 < e1 ? d1 - row1 : e1;
    }
    while (pos < stop) {
        std::int32_t end[kCutPer];
#pragma unroll
        for (int i = 0; i < kCutPer; ++i) {
            const std::int64_t r = row + i * kWave + lane;
            end[i] = off[r < n ? r + 1 : n];
            send[w][i * kWave + lane] = end[i];
            slab[w][i * kWave + lane] = labels[r < n ? r : n - 1];
        }
        wave_sync();
        const std::int64_t last_end = __shfl(end[kCutPer - 1], kWave - 1);
        const std::int64_t window = last_end < stop ? last_end : stop;
        while (pos < window) {
            const std::int64_t batch = pos + kCutBatch * kWave < window ? pos + kCutBatch * kWave : window;
            std::int32_t u[kCutBatch];
            std::uint32_t wt[kCutBatch];
#pragma unroll
            for (int j = 0; j < kCutBatch; ++j) {
                const std::int64_t e = pos + j * kWave + lane;
                const std::int64_t x = e < batch ? e : batch - 1;
                u[j] = nbr[x];
                wt[j] = Weighted ? ew[x] : 1u;
            }
            // Rows of the batch's first and last entry.
            int r0 = 0, r1 = 0;
#pragma unroll
            for (int i = 0; i < kCutPer; ++i) {
                r0 += __popcll(__ballot(end[i] <= pos));
                r1 += __popcll(__ballot(end[i] < batch));
            }
            L lu[kCutBatch];
#pragma unroll
            for (int j = 0; j < kCutBatch; ++j) lu[j] = labels[u[j]];
            cut += batch_cut(send[w], slab[w], r0, r1, pos, (int)(batch - pos), lane, lu, wt);
            pos = batch;
        }
        row += kCutRows;
        wave_sync();
    }

    cut = wave_sum(cut);
    bad = wave_sum(bad);
    if (lane == 0) {
        red[w][0] = cut;
        red[w][1] = bad;
    }
    __syncthreads();
    const int cols = k + 2;
    unsigned long long* own = partials + static_cast<std::size_t>(blockIdx.x) * cols;
    if (threadIdx.x < 2) {
        unsigned long long s = 0;
        for (int x = 0; x < kCutWaves; ++x) s += red[x][threadIdx.x];
        own[threadIdx.x] = s;
    }
    for (int p = threadIdx.x; p < k; p += kCutThreads) own[2 + p] = loads[p];
    if (!block_is_last(ticket)) return;

    // Column sums: groups of threads take every groups-th row, then a tree in
    // LDS (the staging arrays are done with).
    __shared__ unsigned long long sums[kMaxParts + 2];
    for (int c = threadIdx.x; c < cols; c += kCutThreads) sums[c] = 0;
    __syncthreads();
    const int groups = kCutThreads / cols;
    const int g = threadIdx.x / cols, c = threadIdx.x % cols;
    if (g < groups) {
        unsigned long long s = 0;
        for (unsigned b = g; b < gridDim.x; b += groups) s += partials[static_cast<std::size_t>(b) * cols + c];
        if (s) atomicAdd(&sums[c], s);
    }
    __syncthreads();
    for (int x = threadIdx.x; x < cols; x += kCutThreads) host[x] = sums[x];
    publish_to_host(flag, seq);
}

// Labels as bytes, 255 for one outside [0, k).
__global__ void __launch_bounds__(256) k_byte_labels(std::int64_t n, const std::int32_t* labels, int k,
                                                     std::uint8_t* out) {
    for (std::int64_t v = blockIdx.x * (std::int64_t)blockDim.x + threadIdx.x; v < n;
         v += (std::int64_t)gridDim.x * blockDim.x) {
        const std::int32_t lab = labels[v];
        out[v] = static_cast<unsigned>(lab) < static_cast<unsigned>(k) ? static_cast<std::uint8_t>(lab) : 255;
    }
}

// From this many vertices on (1 MiB of int32 labels, a quarter of an XCD's L2),
// int32 labels are narrowed to bytes before the entries gather them, where
// scratch can be allocated.  Whole calls with and without, counting again and
// again: R-MAT scale 18 63 and 64 us, scale 20 141 and 169, a mesh of 2 M
// points 117 and 191, a grid of 4 M cells (its gathers are local) 81 and 77.
constexpr std::int64_t kByteLabelsMin = 1 << 18;

// Launch and read-back: `totals` gets the directed cut, the number of labels
// outside [0, k) and the k part loads.
template <class L>
void count_into(Context& c, const DGraph& g, const L* labels, int k, unsigned long long* partials,
                unsigned long long* totals) {
    const int blocks = edge_cut_blocks(g.n, g.m);
    const unsigned long long seq = c.next_seq();
    if (g.ew)
        hipLaunchKernelGGL((k_edge_cut<true, L>), dim3(blocks), dim3(kCutThreads), 0, c.stream(), g.n, g.off.get(),
                           g.nbr.get(), g.ew.get(), g.vw.get(), labels, k, partials, c.ticket(), c.read_buffer(),
                           c.read_flag(), seq);
    else
        hipLaunchKernelGGL((k_edge_cut<false, L>), dim3(blocks), dim3(kCutThreads), 0, c.stream(), g.n, g.off.get(),
                           g.nbr.get(), nullptr, g.vw.get(), labels, k, partials, c.ticket(), c.read_buffer(),
                           c.read_flag(), seq);
    GP_LAUNCH_CHECK();
    c.wait_flag(c.read_flag(), seq);
    std::memcpy(totals, c.read_buffer(), static_cast<std::size_t>(k + 2) * sizeof(unsigned long long));
}

}  // namespace

// One batch per thread on small graphs; on large ones two blocks per CU, all
// resident.
int edge_cut_blocks(std::int64_t n, std::int64_t m) {
    const std::int64_t b = (n + m + kCutBatch * kCutThreads - 1) / (kCutBatch * kCutThreads);
    return static_cast<int>(b < 1 ? 1 : (b > kEdgeCutMaxBlocks ? kEdgeCutMaxBlocks : b));
}

std::size_t edge_cut_scratch_words(std::int64_t n, std::int64_t m, int k) {
    return static_cast<std::size_t>(edge_cut_blocks(n, m)) * static_cast<std::size_t>(k + 2);
}

void edge_cut_into(Context& c, const DGraph& g, const std::int32_t* labels, int k, unsigned long long* scratch,
                   std::uint8_t* byte_labels, std::uint64_t* cut, std::uint64_t* loads) {
    if (k < 2 || k > kMaxParts) throw std::invalid_argument("parts must be in [2, 128]");
    if (!labels && g.n > 0) throw std::invalid_argument("labels must be a device pointer");
    unsigned long long host[kMaxParts + 2];
    if (byte_labels) {
        hipLaunchKernelGGL(k_byte_labels, dim3(static_cast<unsigned>(std::min<std::int64_t>(ceil_div(g.n, 256), 2048))),
                           dim3(256), 0, c.stream(), g.n, labels, k, byte_labels);
        GP_LAUNCH_CHECK();
        count_into(c, g, byte_labels, k, scratch, host);
    } else {
        count_into(c, g, labels, k, scratch, host);
    }
    if (host[1]) throw std::invalid_argument("labels outside [0, parts)");
    if (host[0] & 1ULL) throw std::runtime_error("directed cut is odd: the graph is not symmetric");
    *cut = host[0] / 2;
    for (int p = 0; p < k; ++p) loads[p] = host[2 + p];
}

template <class L>
std::uint64_t recount(Context& c, const DGraph& g, const L* labels, int k, std::uint64_t* loads) {
    DBuf<unsigned long long> partials = c.buf<unsigned long long>(edge_cut_scratch_words(g.n, g.m, k));
    unsigned long long host[kMaxParts + 2];
    count_into(c, g, labels, k, partials.get(), host);
    if (loads)
        for (int p = 0; p < k; ++p) loads[p] = host[2 + p];
    return host[0];
}
template std::uint64_t recount(Context&, const DGraph&, const std::uint8_t*, int, std::uint64_t*);
template std::uint64_t recount(Context&, const DGraph&, const std::int32_t*, int, std::uint64_t*);

std::uint64_t debug_batch_cut(const std::int32_t* ends, const std::int32_t* labels, int rows, std::int64_t pos,
                              int len, const std::int32_t* lu) {
    if (rows < 1 || rows > kCutRows || len < 1 || len > kCutBatch * kWave || pos < 0 ||
        pos > (std::int64_t)ends[rows - 1] - len)
        throw std::invalid_argument("the batch lies outside the staged rows");
    // The kernel's ballots: row ends at or below the first, and below the last.
    int r0 = 0, r1 = 0;
    for (int r = 0; r < rows; ++r) {
        r0 += ends[r] <= pos;
        r1 += ends[r] < pos + len;
    }
    std::uint64_t cut = 0;
    for (int lane = 0; lane < kWave; ++lane) {
        std::int32_t own[kCutBatch];
        std::uint32_t wt[kCutBatch];
        for (int j = 0; j < kCutBatch; ++j) {
            own[j] = lu[std::min(j * kWave + lane, len - 1)];
            wt[j] = 1;
        }
        cut += batch_cut(ends, labels, r0, r1, pos, len, lane, own, wt);
    }
    return cut;
}

void edge_cut(Context& c, const DGraph& g, const std::int32_t* labels, int k, std::uint64_t* cut,
              std::uint64_t* loads) {
    DBuf<unsigned long long> buf = c.buf<unsigned long long>(edge_cut_scratch_words(g.n, g.m, k));
    DBuf<std::uint8_t> bytes;
    if (g.n >= kByteLabelsMin && labels) bytes = c.buf<std::uint8_t>(static_cast<std::size_t>(g.n));
    edge_cut_into(c, g, labels, k, buf.get(), bytes.get(), cut, loads);
}

namespace {

std::mutex g_scratch_mutex;
std::unordered_map<int, unsigned long long*> g_scratch_address;  // device -> address of `scratch`

}  // namespace

unsigned long long* resolve_noalloc_scratch(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    auto it = g_scratch_address.find(device);
    if (it != g_scratch_address.end()) return it->second;
    int current = -1;
    GP_HIP(hipGetDevice(&current));
    if (current != device) throw std::logic_error("resolve_noalloc_scratch: device is not current");
    void* ptr = nullptr;
    GP_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) throw HipError("hipGetSymbolAddress returned no address for the evaluation scratch");
    auto* p = static_cast<unsigned long long*>(ptr);
    g_scratch_address.emplace(device, p);
    return p;
}

void edge_cut_noalloc(Context& c, const DGraph& g, const std::int32_t* labels, int k, std::uint64_t* cut,
                      std::uint64_t* loads) {
    if (k < 2 || k > kMaxParts) throw std::invalid_argument("parts must be in [2, 128]");
    const std::size_t words = edge_cut_scratch_words(g.n, g.m, k);
    if (words > kNoAllocScratchWords)
        throw std::invalid_argument("evaluation needs " + std::to_string(words) + " scratch words, above the " +
                                    std::to_string(kNoAllocScratchWords) + " of the static scratch");
    unsigned long long* p = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        auto it = g_scratch_address.find(c.device());
        if (it != g_scratch_address.end()) p = it->second;
    }
    if (!p) throw std::logic_error("evaluation scratch of this device was not resolved at context creation");
    // No word of the scratch has to start at zero: every block writes the
    // whole partial row that the last one reads.
    edge_cut_into(c, g, labels, k, p, nullptr, cut, loads);
}

}  // namespace gp
