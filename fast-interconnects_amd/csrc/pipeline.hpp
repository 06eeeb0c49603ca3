// Device-visible state of the batched radix-join pipeline (pipeline.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "internal.hpp"
#include "one_pass_rules.hpp"

namespace fij {

// One relation's buffers.  rel1 is the pass-1 partitioned relation in the
// contiguous layout (each partition one range, 128 bytes of padding in front
// of it): chunk c writes partition p from local1[c][p] on, partition p starts
// at off1[p].  rel2 holds the pass-2 output: the concatenation of all pass-1
// partitions, each cut into tiles of tile2 tuples that are sorted by the
// pass-2 digit.
struct PipelineSide {
  const void* keys;           // input columns
  const void* pays;
  uint64_t n;
  uint32_t g1;                // pass-1 chunks of this side (at most PipelineDevice::G1)
  uint64_t* off1;             // [F1] partition starts in rel1
  uint64_t* local1;           // [g1][F1] per-chunk write offsets
  uint32_t* counts1;          // [g1][F1] per-chunk histograms
  uint64_t* scan1;            // look-back scan state of the offsets scan
  uint64_t scan1_len;
  void* rel1;                 // Tuple[padded_len1]
  uint64_t padded_len1;       // n + F1 * pad
  uint32_t* plen;             // [F1]
  uint64_t* pstart;           // [F1 + 1] start of partition p in rel2
  uint32_t* tile_start;       // [F1 + 1] first pass-2 tile of partition p
  void* rel2;                 // Tuple[n]
  uint32_t* meta;             // [tiles + 1][F2] per tile and pass-2 digit: run start | run end << 16
};

// Join work counters, each on its own 128-byte line: one per XCD (work
// groups are dispatched to the 8 XCDs round-robin), then the ticket counter
// over the deferred-item flags, a word that is non-zero when any item was
// deferred, the number of block-table work units made of them (stored from
// the front of `units`), the ticket counter of the wave-table units, that of
// the block-table units, and the number of wave-table units (stored from the
// back of `units`); then the HBM-table counters: slots reserved in the HBM
// table arena (a 64-bit word), items given an HBM table, their build and
// probe work units, the tickets over those, and their finished units (which
// only the single-pass join counts).
constexpr uint32_t kJoinCounters = 8;
constexpr uint32_t kJoinCounterStride = 32;
constexpr uint32_t kOverflowTicket = kJoinCounters * kJoinCounterStride;
constexpr uint32_t kOverflowAny = (kJoinCounters + 1) * kJoinCounterStride;
constexpr uint32_t kUnitCount = (kJoinCounters + 2) * kJoinCounterStride;
constexpr uint32_t kUnitTicket = (kJoinCounters + 3) * kJoinCounterStride;
constexpr uint32_t kBlockTicket = (kJoinCounters + 4) * kJoinCounterStride;
constexpr uint32_t kWaveUnitCount = (kJoinCounters + 5) * kJoinCounterStride;
constexpr uint32_t kHbmSlots = (kJoinCounters + 6) * kJoinCounterStride;
constexpr uint32_t kBigCount = (kJoinCounters + 7) * kJoinCounterStride;
constexpr uint32_t kHbmBuildUnits = (kJoinCounters + 8) * kJoinCounterStride;
constexpr uint32_t kHbmProbeUnits = (kJoinCounters + 9) * kJoinCounterStride;
constexpr uint32_t kHbmBuildTicket = (kJoinCounters + 10) * kJoinCounterStride;
constexpr uint32_t kHbmProbeTicket = (kJoinCounters + 11) * kJoinCounterStride;
constexpr uint32_t kHbmBuildDone = (kJoinCounters + 12) * kJoinCounterStride;
constexpr uint32_t kHbmProbeDone = (kJoinCounters + 13) * kJoinCounterStride;
constexpr uint32_t kJoinCounterWords = (kJoinCounters + 14) * kJoinCounterStride;

// Counters of a join's finished blocks (finish_join), each on a line of its own.
constexpr uint32_t kDoneGroups = 16, kDoneStride = 32;
constexpr uint32_t kDoneWords = (kDoneGroups + 1) * kDoneStride;

// Phase stamps of a timed join (the device's constant-rate clock, written to
// pinned host memory by the first block of a phase as it starts; the last
// one as the result is written): histograms, scatter, pass 2, join, deferred
// joins, end.  Events between the phases cost 5.5 us of device time each.
constexpr uint32_t kStamps = 6;
__device__ __forceinline__ void stamp_phase(uint64_t* stamps, uint32_t phase) {
  if (stamps && blockIdx.x == 0 && threadIdx.x == 0) stamps[phase] = wall_clock64();
}

// One work unit of a single-pass join: a whole pass-1 build partition against
// a range of its probe partition (tuple indices in rel1).
struct PartUnit {
  uint64_t build_at, probe_at;
  uint32_t build_n, probe_n;
  uint32_t part, reserved;
};
struct PipelineDevice {
  PipelineSide build;
  PipelineSide probe;
  uint32_t F1, F2, G1;
  uint32_t bits1, bits2;
  uint32_t pad;
  uint32_t tile2;
  uint32_t sides;             // bit 0: build, bit 1: probe -- the sides the plan and pass-2 kernels process
  uint32_t* work_counter;     // [kJoinCounterWords]
  uint8_t* overflow;          // [F1 * F2] 1 = item deferred to the general join (zero between joins)
  uint4* units;               // [unit_cap] {item, first probe run, end probe run, 1 = wave table}
  uint32_t unit_cap;          // at least the items plus one per 65,536 probe tuples
  PartUnit* part_units;       // single-pass plans: [part_unit_cap(F1, probe tuples)]
  JoinAggregate* aggregates;  // [agg_len]
  uint32_t agg_len;
  JoinAggregate* result;      // single-pass joins of one plan or request: where the join's sums go, and
  uint32_t* done;             // [kDoneWords] the finished blocks (zero between joins)
  uint64_t* stamps;           // [kStamps] or nullptr: not timed
  // Many joins in one plan (batched joins): pass-1 partition p belongs to
  // join p >> job_shift, whose count and sums are added to
  // job_results[job_slot[join]] instead of the per-block aggregates.
  // job_results == nullptr: one join.
  JoinAggregate* job_results;
  const uint32_t* job_slot;
  uint32_t job_shift;
  // HBM hash tables of deferred items whose build side exceeds a block's
  // LDS table.  hbm_cap == 0: none; such items refill wave LDS tables.
  void* hbm_table;            // Tuple[hbm_cap], every word all ones between joins
  uint32_t hbm_cap;           // slots (power of two)
  uint32_t big_cap;           // entries of `big`
  uint4* big;                 // [big_cap] {item, first slot, log2 slots, 0}
  uint4* hbm_units;           // [hbm_unit_cap] {big index, first run, end run, 0}: build units from the front,
                              // probe units from the back
  uint32_t hbm_unit_cap;
  // single pass: 128 KiB block tables (one block per CU) instead of 64 KiB ones
  uint32_t big_block_tables;
  uint32_t* hashed;           // adaptive digits (single pass): the decision of each join, or nullptr: radix digits
};

// One join side of a batched plan: its pass-1 region and where its
// partitions start in the batched plan's arrays (plan_batched_kernel).
struct BatchSide {
  uint64_t rel1_end;    // one past the side's pass-1 region in rel1 (tuples)
  uint64_t rel2_base;   // first tuple of the side's pass-2 output in rel2
  uint32_t part_base;   // first pass-1 partition (join * F1)
  uint32_t reserved;
};

// Arrays placed in one allocation, 256-byte aligned (a first round without base
// adds up their sizes, a second one sets the pointers), or each allocated by
// itself and recorded in `allocs`.
struct Placer {
  uint8_t* base = nullptr;
  uint64_t used = 0;
  std::vector<void*>* allocs = nullptr;
  hipError_t error = hipSuccess;  // of the allocations
  template <typename T>
  void take(T** p, uint64_t count) {
    const uint64_t bytes = (count ? count : 1) * sizeof(T);
    void* v = base ? base + used : nullptr;
    if (allocs && error == hipSuccess && (error = hipMalloc(&v, bytes)) == hipSuccess) allocs->push_back(v);
    used += (bytes + 255) / 256 * 256;
    *p = static_cast<T*>(v);
  }
};
// Places arrays with place(Placer&) in one new device allocation, recorded in
// `allocs`.
template <typename Place>
hipError_t place_on_device(std::vector<void*>& allocs, Place place) {
  Placer sizes, at;
  place(sizes);
  const hipError_t e = hipMalloc(reinterpret_cast<void**>(&at.base), sizes.used);
  if (e != hipSuccess) return e;
  allocs.push_back(at.base);
  place(at);
  return hipSuccess;
}

// One side's buffers (capacity n tuples, F1 x F2 partitions, G1 chunks; rel2
// and meta only for two passes, meta with `tiles` + 1 rows), placed by `a` or
// allocated and recorded in `allocs`.  rel1 holds n + F1 * pad_tuples(t)
// tuples: the plan using it must set its pad to pad_tuples(t).
void place_pipeline_side(PipelineSide& s, KeyType t, uint64_t n, uint32_t F1, uint32_t F2, uint32_t G1, bool two_pass,
                         uint32_t tiles, Placer& a);
hipError_t alloc_pipeline_side(PipelineSide& s, KeyType t, uint64_t n, uint32_t F1, uint32_t F2, uint32_t G1,
                               bool two_pass, uint32_t tiles, std::vector<void*>& allocs);
// Pass 1 of the sides in d.sides (each in its g1 chunks): contiguous
// histograms + offsets scans, then the scatters, one launch each.
// The histograms copy the keys to key_copies[side] (device columns) if given.
hipError_t enqueue_pass1_prefix_sum(const PipelineDevice& d, KeyType t, uint32_t block, hipStream_t stream,
                                    void* const* key_copies = nullptr);
hipError_t enqueue_pass1_scatter(const PipelineDevice& d, KeyType t, uint32_t block, uint32_t lds_total,
                                 hipStream_t stream);
// Chunks of n tuples: at most `most`, none shorter than a step of the
// scatter (but for the last ones).
uint32_t pass1_chunks(KeyType t, uint64_t n, uint32_t most);
// Chunks of the two sides of one join when a launch covers both: `total`
// blocks shared in proportion to the sides' lengths (at least one each), so
// that every block has the same work and no launch waits for the tail of
// another.  With one block per compute unit for each side in turn, the
// histogram, scan and scatter of 2^20 + 2^24 int32 tuples at 9 bits took 26 +
// 22 + 77 us, in one launch each 20 + 6 + 74 us; 2^27 + 2^27 int64 tuples 343 +
// 22 + 1,760 us and 331 + 5 + 1,735 us (the scatter's time differs by more than
// that from process to process).
void split_chunks(KeyType t, uint64_t n_b, uint64_t n_p, uint32_t total, uint32_t* g_b, uint32_t* g_p);

uint32_t pipeline_tile2(KeyType t);
size_t pipeline_sort2_lds(KeyType t, uint32_t F2);
hipError_t launch_pipeline_plan(const PipelineDevice& d, hipStream_t stream);
// Partition lengths, pass-2 starts and tile maps of every join side of a
// batched plan (sides[2 * join + side]; the tiles of all joins of a side
// form one range, side_tiles[2 * joins] is scratch); resets the join
// counters and the joins' results.  pstart / tile_start [F1] hold the
// totals.
hipError_t launch_pipeline_plan_batched(const PipelineDevice& d, const BatchSide* sides, uint32_t joins,
                                        uint32_t* side_tiles, uint64_t rel2_total_b, uint64_t rel2_total_p,
                                        hipStream_t stream);
// Pass 2 of both relations in one persistent launch of `grid` blocks.
hipError_t launch_pipeline_sort2(const PipelineDevice& d, KeyType t, uint32_t grid, hipStream_t stream);
// dst = the sum of the n per-block aggregates src (one block); the end stamp of
// a timed join.
hipError_t launch_sum_aggregates(const JoinAggregate* src, uint32_t n, JoinAggregate* dst, uint64_t* stamps,
                                 hipStream_t stream);
// One join whose build side fits a block's LDS table (table_join_tuples): one
// launch without partitioning.  partial: at least max_grid entries; done:
// [kDoneWords], zero between joins.
struct TableJoin {
  const void *build_keys, *build_pays, *probe_keys, *probe_pays;
  uint64_t n_b, n_p;
  JoinAggregate* partial;
  uint32_t* done;
  JoinAggregate* result;
  uint64_t* stamps;  // or nullptr
};
uint64_t table_join_tuples(KeyType t);
hipError_t launch_table_join(KeyType t, const TableJoin& j, uint32_t cus, uint32_t max_grid, hipStream_t stream);
// Two passes: the register-resident join of every work item (deferred =
// false), then the join of the items it deferred (deferred = true).
hipError_t launch_pipeline_join(const PipelineDevice& d, KeyType t, bool deferred, uint32_t grid, hipStream_t stream);
// Single pass, instead of the plan and join launches of two: partition
// lengths and work units of the joins in d (sides of join j in sides[2 j],
// sides[2 j + 1]; one join and sides == nullptr for a plan of its own), reset
// of the join counters (and of the joins' results).
hipError_t launch_one_pass_plan(const PipelineDevice& d, KeyType t, const BatchSide* sides, uint32_t joins,
                                hipStream_t stream);
// ... the join of every unit and of the partitions with HBM hash tables, and
// the sum in *d.result (d.job_results: in the joins' results).
hipError_t launch_one_pass_join(const PipelineDevice& d, KeyType t, uint32_t grid, hipStream_t stream);

}  // namespace fij
