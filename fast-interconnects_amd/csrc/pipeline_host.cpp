// Host helpers shared by the execution-method plan (plan.cpp) and the join
// server (server.cpp): one side's buffers and its pass-1 launches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "internal.hpp"
#include "pipeline.hpp"

namespace fij {

void place_pipeline_side(PipelineSide& s, KeyType t, uint64_t n, uint32_t F1, uint32_t F2, uint32_t G1, bool two_pass,
                         uint32_t tiles, Placer& a) {
  const uint32_t tb = tuple_bytes(t);
  s.n = n;
  s.padded_len1 = n + static_cast<uint64_t>(F1) * pad_tuples(t);
  s.g1 = G1;
  s.scan1_len = scan_state_words(F1);
  a.take(&s.off1, F1);
  a.take(&s.local1, static_cast<uint64_t>(G1) * F1);
  a.take(&s.counts1, static_cast<uint64_t>(F1) * G1);
  a.take(&s.scan1, s.scan1_len);
  uint8_t *rel1 = nullptr, *rel2 = nullptr;
  // one spare tuple after the end: pass 2 reads 8-byte tuples in aligned
  // pairs, and the last pair may end one tuple past the relation
  a.take(&rel1, (s.padded_len1 + 1) * tb);
  a.take(&s.plen, F1);
  a.take(&s.pstart, F1 + 1);
  a.take(&s.tile_start, F1 + 1);
  s.meta = nullptr;
  if (two_pass) {
    a.take(&rel2, n * tb);
    a.take(&s.meta, (static_cast<uint64_t>(tiles) + 1) * F2);
  }
  s.rel1 = rel1;
  s.rel2 = rel2;
}

hipError_t alloc_pipeline_side(PipelineSide& s, KeyType t, uint64_t n, uint32_t F1, uint32_t F2, uint32_t G1,
                               bool two_pass, uint32_t tiles, std::vector<void*>& allocs) {
  Placer a;
  a.allocs = &allocs;
  place_pipeline_side(s, t, n, F1, F2, G1, two_pass, tiles, a);
  return a.error;
}

uint32_t pass1_chunks(KeyType t, uint64_t n, uint32_t most) {
  // at least one step of the scatter's loaders per chunk
  const uint64_t step = t == KeyType::I32 ? 2048 : 1024;
  return static_cast<uint32_t>(std::max<uint64_t>(1, std::min<uint64_t>(most, (n + step - 1) / step)));
}

void split_chunks(KeyType t, uint64_t n_b, uint64_t n_p, uint32_t total, uint32_t* g_b, uint32_t* g_p) {
  uint32_t b = 1;
  if (total > 2 && n_b + n_p) {
    const double share = static_cast<double>(n_b) / static_cast<double>(n_b + n_p);
    b = static_cast<uint32_t>(share * total + 0.5);
    b = b < 1 ? 1 : (b > total - 1 ? total - 1 : b);
  }
  *g_b = pass1_chunks(t, n_b, b);
  *g_p = pass1_chunks(t, n_p, total > b ? total - b : 1);
}

namespace {

const PipelineSide* side_of(const PipelineDevice& d, uint32_t i) {
  return (d.sides >> i) & 1u ? (i ? &d.probe : &d.build) : nullptr;
}

OffsetsScan scan_of(const PipelineDevice& d, const PipelineSide& s) {
  return OffsetsScan{s.counts1, s.local1, s.off1, s.scan1, 0, d.F1, s.g1, d.pad, 0};
}

PartitionLaunch scatter_of(const PipelineDevice& d, const PipelineSide& s, KeyType t, uint32_t block,
                           uint32_t lds_total) {
  PartitionLaunch a{};
  a.type = t;
  a.keys = s.keys;
  a.pays = s.pays;
  a.n = s.n;
  a.chunks = s.g1;
  a.chunk_len = balanced_chunk_len(t, s.n, s.g1);
  a.radix_bits = d.bits1;
  a.ignore_bits = 0;
  a.chunk_offsets = s.local1;
  a.relation = s.rel1;
  a.block = block;
  a.lds_bytes = lds_total;
  a.buffered = true;
  a.hashed = d.hashed;
  return a;
}

}  // namespace

hipError_t enqueue_pass1_prefix_sum(const PipelineDevice& d, KeyType t, uint32_t block, hipStream_t stream,
                                    void* const* key_copies) {
  const PipelineSide* a = side_of(d, 0) ? side_of(d, 0) : side_of(d, 1);
  const PipelineSide* b = d.sides == 3 ? &d.probe : nullptr;
  HistParams ha = hist_params(t, a->keys, a->n, a->g1, d.bits1, block, a->counts1, a->scan1);
  ha.stamp = d.stamps;
  HistParams hb = b ? hist_params(t, b->keys, b->n, b->g1, d.bits1, block, b->counts1, b->scan1) : ha;
  if (d.hashed) {
    const uint64_t n = d.sides & 1 ? d.build.n : 0;  // a server has looked at its build sides before
    sample_build_keys(ha, d.build.keys, n, d.hashed);
    sample_build_keys(hb, d.build.keys, n, d.hashed);
  }
  if (key_copies) {
    ha.dst_keys = key_copies[a == &d.build ? 0 : 1];
    hb.dst_keys = key_copies[1];
  }
  const hipError_t e = launch_hist_pair(t, ha, hb, a->g1, b ? b->g1 : 0, d.hashed != nullptr, block, stream);
  if (e != hipSuccess) return e;
  const OffsetsScan sa = scan_of(d, *a), sb = b ? scan_of(d, *b) : sa;
  return launch_offsets_scan(sa, b ? &sb : nullptr, stream);
}

hipError_t enqueue_pass1_scatter(const PipelineDevice& d, KeyType t, uint32_t block, uint32_t lds_total,
                                 hipStream_t stream) {
  PartitionLaunch a = scatter_of(d, d.sides & 1 ? d.build : d.probe, t, block, lds_total);
  a.stamp = d.stamps ? d.stamps + 1 : nullptr;
  if (d.sides == 3) return launch_partition_pair(a, scatter_of(d, d.probe, t, block, lds_total), stream);
  return launch_partition(a, stream);
}

}  // namespace fij
