// Sizes and limits of the single-pass joins, for the host and the kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

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
// 283 us with 16), evenly.
struct PartUnits {
  uint32_t units, per;
};
__host__ __device__ constexpr PartUnits part_units_of(uint32_t build_n, uint32_t probe_n) {
  if (build_n == 0 || probe_n == 0) return {0, kPartUnitMin};
  const uint32_t want = build_n < kPartUnitMax / 16 ? 16 * build_n : kPartUnitMax;
  const uint32_t units = range_count(probe_n, want < kPartUnitMin ? kPartUnitMin : want);
  return {units, range_count(probe_n, units)};
}

}  // namespace fij
