// Sizes and limits of the single-pass joins, for the host and the kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "internal.hpp"

namespace fij {

// n tuples cut into ranges of `per` tuples: how many, and where range r ends.
// A partition may hold nearly 2^32 tuples, so neither rounds up by adding.
__host__ __device__ constexpr uint32_t range_count(uint32_t n, uint32_t per) {
  return n / per + (n % per != 0 ? 1u : 0u);
}
__host__ __device__ constexpr uint32_t range_end(uint32_t n, uint32_t per, uint32_t r) {
  return n - r * per < per ? n : (r + 1) * per;
}

// Probe tuples of a unit: at least kPartUnitMin (or the whole partition), so
// that at most one unit per partition and one per kPartUnitMin tuples exist.
constexpr uint32_t kPartUnitMin = 8192, kPartUnitMax = 65536;
constexpr uint64_t part_unit_cap(uint64_t partitions, uint64_t probe_len) {
  return partitions + probe_len / kPartUnitMin + 1;
}

// Units of a partition pair, each of `per` probe tuples but for the last:
// about 16 times the build tuples (a unit's build work is paid once per unit:
// 20 batched joins of 2^18..2^20 int32 build tuples took 349 us with 8 times,
// 283 us with 16), evenly.  A unit streams them once per fill of the table, of
// `fill` build tuples: those of a partition that stands out by more than two
// fills are shorter, as the others will be done before them (one of 64
// partitions of 10,000 int32 tuples, in 32 KiB tables: 490 -> 260 us; where all
// partitions are of four fills more units only build more, 282 -> 328 us).
struct PartUnits {
  uint32_t units, per;
};
__host__ __device__ constexpr PartUnits part_units_of(uint32_t build_n, uint32_t probe_n, uint32_t fill = ~0u) {
  if (build_n == 0 || probe_n == 0) return {0, kPartUnitMin};
  const uint32_t fills = range_count(build_n, fill), most = fills > 2 ? 2 * kPartUnitMax / fills : kPartUnitMax;
  const uint32_t want = build_n < most / 16 ? 16 * build_n : most;
  const uint32_t units = range_count(probe_n, want < kPartUnitMin ? kPartUnitMin : want);
  return {units, range_count(probe_n, units)};
}

// Build tuples a deferred item may have to be joined from one block-shared
// LDS table (3/4 of its slots): the 64 KiB table, or the 128 KiB one of
// single-pass plans with big_block_tables.
constexpr uint32_t pipeline_block_table_tuples(KeyType t, bool big = false) {
  return (big ? 131072u : 65536u) / (t == KeyType::I32 ? 8u : 16u) * 3 / 4;
}

// Slots of the block-shared table of the single-pass joins: 64 KiB of keys and
// values, 128 KiB (big_block_tables), or 32 KiB for partitions that fill those
// half on average (20 batched joins of 2^18..2^20 int32 build tuples: 283 us
// with 64 KiB tables, 240 us).
constexpr uint32_t block_table_slots(KeyType t) { return t == KeyType::I32 ? 8192 : 4096; }
inline uint32_t one_pass_slots(KeyType t, uint64_t build_len, uint64_t partitions, bool big) {
  const uint32_t slots = block_table_slots(t);
  return big ? 2 * slots : build_len <= partitions * (slots / 4) ? slots / 2 : slots;
}
// Build tuples of one fill of a table: 5/8 of the slots at int64, 9/16 at int32.
// Fuller buckets overflow, and probes that leave theirs (in a table with
// duplicate keys every one whose bucket is full) made fills of 70 % 0.7 to 0.9
// times as fast as two passes, at int32 fills of 60 % 0.94 to 1.5 times.
constexpr uint32_t block_table_fill(KeyType t, uint32_t slots) { return slots / 16 * (t == KeyType::I32 ? 9 : 10); }
// Tuples of a work unit of a partition with an HBM table.  A thread has one
// random access in flight, so a unit takes as long as a thread has tuples, and
// with blocks to wait for: a 128th of the range, but kTableUnitMin at least and
// kTableUnitMax at most.  One of 64 partitions of 12,000 int64 tuples, in 32 KiB
// tables, and 4 M probe tuples, 6 and 60 % of them in that partition: 743 and
// 617 us with units of 65,536, 238 and 428 with a 64th, 182 and 305 so, 200 and
// 468 with a 512th.
constexpr uint32_t kTableUnitMin = 4096, kTableUnitMax = 65536;
__host__ __device__ constexpr uint32_t table_unit_tuples(uint32_t n) {
  return n / 128 < kTableUnitMin ? kTableUnitMin : n / 128 < kTableUnitMax ? n / 128 : kTableUnitMax;
}
// Build tuples up to which a partition fills the table several times although
// the arena would have room for an HBM table: three times the slots of the 64 or
// 128 KiB table, up to 6 fills (5 at int64), of 32 KiB tables up to 11 (10).
// Each fill streams the probe tuples again, an HBM table costs a random access
// per probe tuple and a chain per repeated key.  Among 64 partitions one of
// 10,000 int32 tuples, in 32 KiB tables: 260 us in LDS, 145 to 255 us in HBM, of
// 20,000 306 and 130 to 205 us; of 14,000 with 500 copies of every key 0.2 and 7
// ms.  In larger tables LDS wins up to there.
constexpr uint32_t one_pass_lds_tuples(KeyType t, bool big) { return 3 * block_table_slots(t) * (big ? 2 : 1); }

// Single-pass plans (fij_join_plan_bits, single-pass batched classes): 9
// bits, the widest pass-1 fanout whose line rings fit LDS.
constexpr uint32_t kOnePassBits = 9;
// Whether a build side's single-pass partitions hold on average at most 2/3
// of a (big) block table (half again of headroom for uneven ones).
inline bool block_tables_hold(KeyType t, uint64_t build_len, uint64_t partitions, bool big) {
  return build_len * 3 <= static_cast<uint64_t>(pipeline_block_table_tuples(t, big)) * partitions * 2;
}
// Single pass of kOnePassBits: with 128 KiB tables where 64 KiB ones do not
// hold the partitions (the big ones run one block per CU and are slower for
// build sides the small ones hold).
inline bool one_pass_fits(KeyType t, uint64_t build_len) {
  return block_tables_hold(t, build_len, 1ull << kOnePassBits, true);
}
// Build tuples of one fill of a 128 KiB table.
inline uint64_t one_pass_fill(KeyType t) { return block_table_fill(t, 2 * block_table_slots(t)); }
// Whether the scatter's 32-bit offsets reach the end of a relation of `len`
// tuples in this many partitions, each behind its padding.
inline bool pass1_offsets_fit(KeyType t, uint64_t len, uint64_t partitions) {
  return len + partitions * pad_tuples(t) * 2 < 0xFFFFFFFFull;
}
// Build tuples up to which a two-pass plan runs in a single pass of
// kOnePassBits instead, whatever the probe side: two fills of 9/16 of the slots
// on average at int64, one at int32 (1/32 of headroom for uneven partitions).
// Per probe tuple of t bytes a second fill reads t again, a second pass reads
// and writes t and gathers short runs: 3 M x 2^28 int64 tuples take 3.4 ms in a
// single pass and 4.5 ms in two, 4.56 M x 2^29 int32 tuples 3.0 and 5.0 ms
// (with three copies of every build key 6.0 and 6.5 ms).
inline uint64_t one_pass_limit(KeyType t) {
  return (static_cast<uint64_t>(pipeline_block_table_tuples(t, true)) * (t == KeyType::I32 ? 3 : 6) / 4 << kOnePassBits) *
         31 / 32;
}
// Whether it does for these lengths: beyond, two fills pay for probe sides that
// are not too long: int32 tuples are moved in half the time and probed in the
// same (7,300,000 x 10 M tuples: 167 against 323 us; 7 M x 220 M 1.7 to 2.8
// against 2.1 to 2.8 ms, by keys; x 2^29 4.0 to 6.9 against 4.7 to 6.4 ms); at
// int64 the tables fill up (5,000,011 x 20,000,003 tuples: 390 against 590 us,
// with copies 560 against 660; 5,070,000 x 150 M 2.2 to 3.6 against 2.6 to 3.3
// ms).
inline bool one_pass_join(KeyType t, uint64_t build_len, uint64_t probe_len) {
  if (!pass1_offsets_fit(t, probe_len, 1u << kOnePassBits)) return false;
  if (build_len <= one_pass_limit(t)) return true;
  const uint64_t fill = one_pass_fill(t) << kOnePassBits;
  return t == KeyType::I32 ? build_len <= fill * 3 / 2 && probe_len / 32 <= build_len
                           : build_len <= 2 * fill * 31 / 32 && probe_len / 16 <= build_len;
}
// Whether every join of at most these lengths runs in a single pass: a plan for
// them needs no pass-2 buffers.
inline bool one_pass_always(KeyType t, uint64_t build_len, uint64_t probe_len) {
  return build_len <= one_pass_limit(t) && pass1_offsets_fit(t, probe_len, 1u << kOnePassBits);
}
// Pass-2 bits of a two-pass plan of 9 + b2 bits whose items hold about a
// third of a 64 KiB block table's build tuples (1,024 int64, 2,048 int32):
// for probe sides far longer than the build side, whose items go to the
// block join anyway, fewer pass-2 digits give longer runs.
inline uint32_t probe_heavy_bits2(KeyType t, uint64_t build_len) {
  const uint64_t per_item = pipeline_block_table_tuples(t, false) / 3;
  const uint64_t items = (build_len >> kOnePassBits) / per_item;
  uint32_t b2 = 1;
  while (b2 < 12 && (1ull << b2) < items) ++b2;
  return b2;
}
// The class of a batch's single-pass join: its bits, the longest build side of
// the class and whether its tables are the 128 KiB ones.  A factor of four each
// from 2^14 (int64: 2^13) tuples on: 5, 7 and 9 bits leave 512 to 2,048 (256 to
// 1,024) tuples in a partition, for 32 KiB tables; beyond, 9 bits and 128 KiB
// tables (64 KiB ones up to twice that: 3 joins of 550,000 x 2.2 M int64 tuples
// 145 -> 160 us, of 2 M x 8 M int32 tuples 269 -> 273 us), in two classes that
// overlap (in one, 6 joins of 1.2 to 3.4 M x 12 times as many int32 tuples
// 1,108 -> 1,224 us).
struct OnePassClass {
  uint32_t bits, build;
  bool big_tables;
};
inline OnePassClass one_pass_class(KeyType t, uint64_t build_len) {
  uint32_t bits = 5;
  uint64_t most = t == KeyType::I32 ? 1u << 16 : 1u << 15;
  for (; build_len > most && bits < kOnePassBits; bits += 2) most <<= 2;
  const bool big = build_len > most;
  if (big) most <<= 1;
  if (build_len > most) most = 2 * one_pass_fill(t) << kOnePassBits;
  return {bits, static_cast<uint32_t>(most), big};
}
// big_block_tables of a single-pass plan of `partitions` partitions.
inline uint32_t big_block_tables_for(KeyType t, uint64_t build_len, uint64_t partitions) {
  return block_tables_hold(t, build_len, partitions, false) ? 0u : 1u;
}

}  // namespace fij
