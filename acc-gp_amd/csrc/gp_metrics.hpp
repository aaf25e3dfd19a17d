// Edge cut and part loads of device-resident labels (host_cut,
// include/graph.hpp:67-69; refine.cu:63-98).
#pragma once
#include "gp_graph.hpp"

namespace gp {

// Blocks of an evaluation, at most two per CU.
constexpr int kEdgeCutMaxBlocks = 512;
int edge_cut_blocks(std::int64_t n, std::int64_t m);
// Scratch words of one evaluation: one row of k + 2 partials per block.
std::size_t edge_cut_scratch_words(std::int64_t n, std::int64_t m, int k);

// What one lane of the cut kernel adds for a batch of `len` entries (at most
// kCutBatch * kWave) from entry `pos` on: entry j * kWave + lane of it for each
// j, of weight wt[j], when its neighbour's label lu[j] differs from its row's.
// ends, labels: ends and labels of the staged rows; the batch's first entry lies
// in row r0 of them, its last in r1.  Lanes are told apart by their place in the
// batch: pos + kCutBatch * kWave passes 2^31 at the end of the largest graphs.
constexpr int kCutBatch = 4;  // entries per lane in flight
template <class L>
__host__ __device__ inline unsigned long long batch_cut(const std::int32_t* ends, const L* labels, int r0, int r1,
                                                        std::int64_t pos, int len, int lane,
                                                        const L (&lu)[kCutBatch], const std::uint32_t (&wt)[kCutBatch]) {
    unsigned long long cut = 0;
    const L lab0 = labels[r0];
#pragma unroll
    for (int j = 0; j < kCutBatch; ++j) {
        const int at = j * kWave + lane;
        const std::int32_t e = (std::int32_t)pos + (at < len ? at : len - 1);
        L lab = lab0;
        if (r0 != r1) {
            int lo = r0, hi = r1;  // first staged row whose end lies after e
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (ends[mid] <= e) lo = mid + 1;
                else hi = mid;
            }
            lab = labels[lo];
        }
        if (at < len && lab != lu[j]) cut += wt[j];
    }
    return cut;
}
// All lanes' sum for one batch with entries of weight 1, on the host: `rows`
// staged rows, lu[i] the label of the batch's i-th neighbour.  For tests.
std::uint64_t debug_batch_cut(const std::int32_t* ends, const std::int32_t* labels, int rows, std::int64_t pos,
                              int len, const std::int32_t* lu);

// Cut and loads of `labels` (device, n entries in [0, k)) with the partials
// in caller scratch of edge_cut_scratch_words(n, m, k) words; byte_labels: null,
// or room for n bytes, which the labels are narrowed to first; loads_host gets
// k words.  Synchronizes the context stream.
void edge_cut_into(Context& c, const DGraph& g, const std::int32_t* labels, int k, unsigned long long* scratch,
                   std::uint8_t* byte_labels, std::uint64_t* cut, std::uint64_t* loads_host);
// The same with the scratch from the context arena.
void edge_cut(Context& c, const DGraph& g, const std::int32_t* labels, int k, std::uint64_t* cut,
              std::uint64_t* loads_host);

// Words of the static device scratch of edge_cut_noalloc: what the largest
// evaluation takes.
constexpr std::size_t kNoAllocScratchWords =
    static_cast<std::size_t>(kEdgeCutMaxBlocks) * static_cast<std::size_t>(kMaxParts + 2);
// Resolves (once per device, that device current) and caches the device
// address of the static scratch; called at context creation.
unsigned long long* resolve_noalloc_scratch(int device);
// edge_cut with its partials in the static scratch of the context's device:
// allocates nothing (no arena, no hipMalloc).  Calls that overlap on one GPU
// share the scratch and race.
void edge_cut_noalloc(Context& c, const DGraph& g, const std::int32_t* labels, int k, std::uint64_t* cut,
                      std::uint64_t* loads_host);

// Directed cut weight of in-range labels (byte or int32), not halved, and
// with loads the k part loads; partials from the context arena.
template <class L>
std::uint64_t recount(Context& c, const DGraph& g, const L* labels, int k, std::uint64_t* loads);

}  // namespace gp
