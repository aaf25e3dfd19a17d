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

// Cut and loads of `labels` (device, n entries in [0, k)) with the partials
// in caller scratch of edge_cut_scratch_words(n, m, k) words; byte_labels: null,
// or room for n bytes, which the labels are narrowed to first; loads_host gets
// k words.  Synchronizes the context stream.
void edge_cut_into(Context& c, const DGraph& g, const std::int32_t* labels, int k, unsigned long long* scratch,
                   std::uint8_t* byte_labels, std::uint64_t* cut, std::uint64_t* loads_host);
// The same with the scratch from the context arena.
void edge_cut(Context& c, const DGraph& g, const std::int32_t* labels, int k, std::uint64_t* cut,
              std::uint64_t* loads_host);

// Words of the static device scratch of edge_cut_noalloc: more than the
// largest evaluation takes (kEdgeCutMaxBlocks partial rows).
constexpr std::size_t kNoAllocScratchWords = 1025 * static_cast<std::size_t>(kMaxParts + 2);
static_assert(kEdgeCutMaxBlocks <= 1025, "the static scratch holds every partial row");
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
