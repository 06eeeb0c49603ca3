// Single-pass joins: pass 1 leaves every partition of both relations as one
// contiguous range, and a build partition that fits a block's LDS table is
// joined by streaming its probe partition against it.
//
//   one_pass_plan_kernel  partition lengths, and work units {build range, probe
//                         range} of every partition pair; a build partition
//                         beyond the LDS table fills it several times, a much
//                         longer one (one_pass_lds_tuples) gets a hash table in
//                         the HBM arena when the arena has room
//   part_join_kernel      one block per unit: the build range goes into a
//                         block-shared table, the probe range is streamed
//                         against it; then the HBM tables, and the sum
//
// Semantics as in the other joins: every pair of equal keys counts, null keys
// never join, count and sums wrap at 64 bits.
#include "bucket_table.hpp"
#include "common.hpp"
#include "hbm_table.hpp"
#include "internal.hpp"
#include "join_result.hpp"
#include "one_pass_rules.hpp"
#include "pipeline.hpp"

#include <algorithm>

namespace fij {
namespace {

template <typename U>
__device__ __forceinline__ U uniform_load(const U* ptr) {
  return *(const __attribute__((address_space(4))) U*)(ptr);
}

template <typename K>
constexpr KeyType kKeyType = sizeof(K) == 4 ? KeyType::I32 : KeyType::I64;

// One block per join.  `sides` == nullptr: one join, whose sides end at their
// padded_len1; that block sets the counters.  In batches (which have no HBM
// arena) the counters were reset by an earlier launch.
__global__ __launch_bounds__(1024) void one_pass_plan_kernel(PipelineDevice d, const BatchSide* sides, uint32_t F1j,
                                                             uint32_t fill, uint32_t long_tuples,
                                                             uint32_t lds_tuples) {
  extern __shared__ uint32_t lds[];
  __shared__ uint32_t wave_tmp[1024 / kWave + 1];
  __shared__ uint32_t s_base, s_slots, s_big, s_build_units, s_probe_units;
  uint32_t* first = lds;           // [F1j] units of a partition, then their exclusive scan
  uint32_t* probe_n = lds + F1j;   // [F1j]
  uint32_t* per = lds + 2 * F1j;   // [F1j] probe tuples per unit
  stamp_phase(d.stamps, 2);
  const uint32_t tid = threadIdx.x, j = blockIdx.x;
  const uint64_t end_b = sides ? sides[2 * j].rel1_end : d.build.padded_len1;
  const uint64_t end_p = sides ? sides[2 * j + 1].rel1_end : d.probe.padded_len1;
  if (tid == 0) s_slots = s_big = s_build_units = s_probe_units = 0;
  if (sides && tid == 0) d.job_results[d.job_slot[j]] = JoinAggregate{0, 0, 0};
  __syncthreads();
  auto range = [&](const PipelineSide& s, uint64_t end, uint32_t p, uint64_t& at) -> uint32_t {
    const uint32_t vp = j * F1j + p;
    at = s.off1[vp];
    return static_cast<uint32_t>((p + 1 < F1j ? s.off1[vp + 1] - d.pad : end) - at);
  };
  for (uint32_t p = tid; p < F1j; p += blockDim.x) {
    uint64_t at;
    const uint32_t nb = range(d.build, end_b, p, at), np = range(d.probe, end_p, p, at);
    PartUnits cut = part_units_of(nb, np, nb > long_tuples ? fill : ~0u);
    if (cut.units) {
      if (nb > lds_tuples && d.hbm_cap && nb <= (d.hbm_cap >> 1)) {
        // an HBM table of at least twice the build tuples, if the arena (at
        // most 2^26 slots) has room.  A partition that finds none takes no
        // slots; the sum of the others' stays below 2^32.
        const uint32_t lg = max(8u, 64u - static_cast<uint32_t>(__builtin_clzll(2ull * nb - 1)));
        uint32_t slot = s_slots;
        for (;;) {
          const uint32_t seen = slot + (1u << lg) <= d.hbm_cap ? atomicCAS(&s_slots, slot, slot + (1u << lg)) : slot;
          if (seen == slot) break;
          slot = seen;
        }
        const uint32_t big = slot + (1u << lg) <= d.hbm_cap ? atomicAdd(&s_big, 1u) : d.big_cap;
        if (big < d.big_cap) {
          cut.units = 0;
          d.big[big] = make_uint4(j * F1j + p, slot, lg, 0u);
          const uint32_t b_per = table_unit_tuples(nb), p_per = table_unit_tuples(np);
          const uint32_t bu = range_count(nb, b_per), pu = range_count(np, p_per);
          const uint32_t b0 = atomicAdd(&s_build_units, bu), p0 = atomicAdd(&s_probe_units, pu);
          for (uint32_t u = 0; u < bu; ++u) d.hbm_units[b0 + u] = make_uint4(big, u * b_per, range_end(nb, b_per, u), 0u);
          for (uint32_t u = 0; u < pu; ++u)
            d.hbm_units[d.hbm_unit_cap - 1 - (p0 + u)] = make_uint4(big, u * p_per, range_end(np, p_per, u), 0u);
        }
      }
    }
    first[p] = cut.units;
    probe_n[p] = np;
    per[p] = cut.per;
    if (d.sides & 1) d.build.plen[j * F1j + p] = nb;
    if (d.sides & 2) d.probe.plen[j * F1j + p] = np;
  }
  __syncthreads();
  const uint32_t total = block_exclusive_scan<uint32_t>(first, F1j, wave_tmp);
  if (tid == 0) {
    if (sides) {
      s_base = total ? atomicAdd(d.work_counter + kUnitCount, total) : 0u;
    } else {
      s_base = 0;
      d.work_counter[kUnitCount] = total;
      d.work_counter[kBlockTicket] = 0;
      d.work_counter[kHbmSlots] = s_slots;
      d.work_counter[kHbmSlots + 1] = 0;
      d.work_counter[kHbmBuildUnits] = s_build_units;
      d.work_counter[kHbmProbeUnits] = s_probe_units;
      for (uint32_t c : {kHbmBuildTicket, kHbmBuildDone, kHbmProbeTicket, kHbmProbeDone}) d.work_counter[c] = 0;
    }
  }
  __syncthreads();
  for (uint32_t u = tid; u < total; u += blockDim.x) {
    uint32_t lo = 0, hi = F1j;  // the last partition whose first unit is at or before u
    while (hi - lo > 1) {
      const uint32_t m = (lo + hi) / 2;
      if (first[m] <= u) lo = m; else hi = m;
    }
    PartUnit w;
    uint64_t build_at, probe_at;
    w.build_n = range(d.build, end_b, lo, build_at);
    range(d.probe, end_p, lo, probe_at);
    const uint32_t from = (u - first[lo]) * per[lo];
    w.build_at = build_at;
    w.probe_at = probe_at + from;
    w.probe_n = min(per[lo], probe_n[lo] - from);
    w.part = j * F1j + lo;
    w.reserved = 0;
    d.part_units[s_base + u] = w;
  }
}

__global__ void reset_counters_kernel(uint32_t* counters) {
  for (uint32_t i = threadIdx.x; i < kJoinCounterWords; i += blockDim.x) counters[i] = 0;
}

// Adds the block's sums to the result of join `job` of a batch and clears them.
template <uint32_t BLOCK>
__device__ __forceinline__ void add_result(const PipelineDevice& d, uint64_t (*red)[BLOCK / kWave], uint32_t job,
                                           uint64_t& cnt, uint64_t& sb, uint64_t& sp) {
  block_sums<BLOCK>(red, cnt, sb, sp);
  if (threadIdx.x == 0 && cnt) {
    JoinAggregate* r = d.job_results + d.job_slot[job];
    atomicAdd(reinterpret_cast<unsigned long long*>(&r->count), static_cast<unsigned long long>(cnt));
    atomicAdd(reinterpret_cast<unsigned long long*>(&r->sum_build), static_cast<unsigned long long>(sb));
    atomicAdd(reinterpret_cast<unsigned long long*>(&r->sum_probe), static_cast<unsigned long long>(sp));
  }
  cnt = sb = sp = 0;
}

// The HBM tables of a join (plans of one join only: batches and served joins
// have no arena): build, probe and clear, for blocks that have run out of work
// units.  Units are taken by ticket and a block waits only once every unit of
// the phase is taken, so it waits for blocks that are running and never for
// one that has yet to start.  As launches of their own, which nearly every
// join leaves without work, the probes and the clearing took 9 us of each.
// No more blocks than units take part, so that few wait.
template <typename K, uint32_t BLOCK>
__device__ __forceinline__ void table_phases(const PipelineDevice& d, uint32_t n_build, uint32_t* s_next,
                                             uint64_t& cnt, uint64_t& sb, uint64_t& sp) {
  const uint32_t n_probe = uniform_load(d.work_counter + kHbmProbeUnits);
  const uint32_t blocks = min(gridDim.x, max(n_build, n_probe));
  if (blockIdx.x >= blocks) return;
  const uint32_t tid = threadIdx.x;
  auto take = [&](uint32_t ticket) {
    if (tid == 0) *s_next = atomicAdd(d.work_counter + ticket, 1u);
    __syncthreads();
    const uint32_t u = __builtin_amdgcn_readfirstlane(*s_next);
    __syncthreads();  // every thread has read it
    return u;
  };
  // counts the block's finished units and waits for all n of the phase
  auto finish = [&](uint32_t counter, uint32_t mine, uint32_t n) {
    __threadfence();  // the thread's stores are visible before its units count
    __syncthreads();
    if (tid == 0) {
      if (mine) atomicAdd(d.work_counter + counter, mine);
      // relaxed: an acquire would drop the L2's lines at every look, while the
      // chains of the blocks that work run through it
      while (__hip_atomic_load(d.work_counter + counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < n)
        __builtin_amdgcn_s_sleep(127);
    }
    __syncthreads();
    __threadfence();  // what was read before is read again
  };
  uint32_t mine = 0;
  for (uint32_t u; (u = take(kHbmBuildTicket)) < n_build; ++mine) {
    const uint4 unit = scalar_load(d.hbm_units + u);
    const uint4 big = scalar_load(d.big + unit.x);
    Tuple<K>* const table = static_cast<Tuple<K>*>(d.hbm_table) + big.y;
    const Tuple<K>* rel = static_cast<const Tuple<K>*>(d.build.rel1) + uniform_load(d.build.off1 + big.x);
    for (uint32_t i = unit.y + tid; i < unit.z; i += BLOCK) {
      const Tuple<K> t = load_tuple<K>(rel + i);
      if (t.key != null_key<K>()) hbm_insert<K>(table, big.z, t.key, t.value);
    }
  }
  finish(kHbmBuildDone, mine, n_build);
  mine = 0;
  for (uint32_t u; (u = take(kHbmProbeTicket)) < n_probe; ++mine) {
    const uint4 unit = scalar_load(d.hbm_units + (d.hbm_unit_cap - 1 - u));
    const uint4 big = scalar_load(d.big + unit.x);
    const Tuple<K>* const table = static_cast<const Tuple<K>*>(d.hbm_table) + big.y;
    const Tuple<K>* rel = static_cast<const Tuple<K>*>(d.probe.rel1) + uniform_load(d.probe.off1 + big.x);
    for (uint32_t i = unit.y + tid; i < unit.z; i += BLOCK) {
      const Tuple<K> t = load_tuple_nt<K>(rel + i);
      if (t.key != null_key<K>()) hbm_probe<K>(table, big.z, t.key, t.value, cnt, sb, sp);
    }
  }
  finish(kHbmProbeDone, mine, n_probe);
  uint4* const words = static_cast<uint4*>(d.hbm_table);
  const uint64_t n = static_cast<uint64_t>(uniform_load(d.work_counter + kHbmSlots)) * sizeof(Tuple<K>) / 16;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * BLOCK + tid; i < n; i += static_cast<uint64_t>(blocks) * BLOCK)
    words[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
}

// 16 bytes of tuples from 16-byte aligned memory.
template <typename K>
struct TupleVec {
  static constexpr uint32_t N = 16 / sizeof(Tuple<K>);  // 2 of 8 bytes, 1 of 16
  typedef K type __attribute__((ext_vector_type(16 / sizeof(K))));
};

// Joins the work units, one block per unit (the first by block index, the rest
// by ticket, taken while the current unit runs).
//
// Bound by the read of the probe partitions (with inserts and probes left out
// of a copy: 36 of 46 us, 126 of 174 us, 230 of 240 us for the shapes below),
// plus what the phases of a block do not overlap.  2^20 + 2^24 int32 tuples in
// 512 partitions: 46 us, where the two-pass plans' register join (23 us, every
// item only put off), unit counting (8 us) and block join (48 us, every
// tuple's run looked up although a partition is one run) ran before; 20 batched
// joins of 2^18..2^20 int32 build tuples 1,053 -> 240 us; 5,000,011 +
// 20,000,003 int64 tuples (two fills) 174 us.  Two and four vectors per buffer,
// two or four probes together and build tuples loaded a fill ahead all lay
// within 3 % of each other; the smallest register need was taken.
template <typename K, uint32_t CAP, uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK, CAP * 2 * sizeof(K) <= 32768 ? 6 : 4) void part_join_kernel(PipelineDevice d) {
  using V = TupleVec<K>;
  using VT = typename V::type;
  constexpr uint32_t FILL = block_table_fill(kKeyType<K>, CAP);
  constexpr uint32_t NV = 2;                  // vectors in flight per buffer
  constexpr uint32_t NT = NV * V::N;          // their tuples
  constexpr uint32_t PROBES = 2;              // probed together
  extern __shared__ __attribute__((aligned(16))) uint64_t lds_u64[];
  __shared__ uint32_t s_next, s_dup;
  __shared__ uint64_t red[3][BLOCK / kWave];
  const uint32_t tid = threadIdx.x;
  uint64_t cnt = 0, sb = 0, sp = 0;
  stamp_phase(d.stamps, 3);
  const uint32_t n_units = uniform_load(d.work_counter + kUnitCount);
  uint32_t job = 0;
  bool hashed = d.hashed && uniform_load(d.hashed) != 0;  // the digits of the job's partitions
  for (uint32_t u = blockIdx.x; u < n_units;) {
    uint32_t ticket = 0;
    if (tid == 0) ticket = atomicAdd(d.work_counter + kBlockTicket, 1u);
    const PartUnit unit = scalar_load(d.part_units + u);
    if (d.job_results && (unit.part >> d.job_shift) != job) {
      add_result<BLOCK>(d, red, job, cnt, sb, sp);
      job = unit.part >> d.job_shift;
      hashed = uniform_load(d.hashed + job) != 0;
    }
    const uint32_t nb = unit.build_n;
    // a range as aligned 16-byte vectors: the first one may begin a tuple
    // before the range (the padding in front of a partition, or the range
    // before it) and the last end one after it (the next range, or the spare
    // tuple behind the relation); those tuples are skipped
    const uint32_t off_b = unit.build_at % V::N, off_p = unit.probe_at % V::N;
    const auto vb = as_global(static_cast<const VT*>(d.build.rel1) + unit.build_at / V::N);
    const auto vp = as_global(static_cast<const VT*>(d.probe.rel1) + unit.probe_at / V::N);
    const uint32_t nvp = (unit.probe_n + off_p + V::N - 1) / V::N;
    auto load = [&](VT (&x)[NV], uint32_t v0) {
#pragma unroll
      for (uint32_t k = 0; k < NV; ++k) x[k] = __builtin_nontemporal_load(vp + min(v0 + k * BLOCK + tid, nvp - 1));
    };
    const uint32_t digit = unit.part & ((1u << d.bits1) - 1u);
    const uint32_t other = hashed ? (digit ^ 1u) << (32u - d.bits1) : digit ^ 1u;
    const K free_key = static_cast<K>(hashed ? other * kDigitMulInverse : other);
    const K no_key = static_cast<K>(hashed ? (other + 1u) * kDigitMulInverse : other | (1u << d.bits1));
    uint32_t wave_cnt = 0;
    VT xa[NV], xb[NV];
    load(xa, 0);  // in flight while the table is built
    // equal fills
    const uint32_t fills = range_count(nb, FILL), fill = range_count(nb, fills);
    for (uint32_t f = 0; f < fills; ++f) {
      const uint32_t f0 = f * fill, nf = range_end(nb, fill, f) - f0;
      const BucketTable<K> tab(lds_u64, CAP, BucketTable<K>::lg_buckets(CAP, nf), free_key, hashed, d.bits1);
      tab.clear();
      if (tid == 0) s_dup = 0;
      __syncthreads();
      {
        const uint32_t lo = off_b + f0, hi = off_b + f0 + nf;  // tuples of the range, counted from vb
        const uint32_t v_end = (hi + V::N - 1) / V::N;
        bool dup = false;
        for (uint32_t v0 = lo / V::N; v0 < v_end; v0 += 2 * BLOCK) {
          VT x[2];
#pragma unroll
          for (uint32_t k = 0; k < 2; ++k) x[k] = vb[min(v0 + k * BLOCK + tid, v_end - 1)];
#pragma unroll
          for (uint32_t k = 0; k < 2; ++k) {
            const uint32_t v = v0 + k * BLOCK + tid;
#pragma unroll
            for (uint32_t e = 0; e < V::N; ++e) {
              const uint32_t at = v * V::N + e;
              const K key = x[k][2 * e];
              if (v < v_end && at >= lo && at < hi && key != null_key<K>()) dup |= tab.insert(key, x[k][2 * e + 1]);
            }
          }
        }
        if (dup) s_dup = 1;
      }
      __syncthreads();
      const bool unique = __builtin_amdgcn_readfirstlane(s_dup) == 0;
      auto probe = [&](const VT (&x)[NV], uint32_t v0) {
        // batches inside the range need no test per tuple
        const bool inside = v0 >= off_p && (v0 + NV * BLOCK) * V::N <= off_p + unit.probe_n;
#pragma unroll
        for (uint32_t g = 0; g < NT; g += PROBES) {
          K key[PROBES], pay[PROBES];
#pragma unroll
          for (uint32_t i = 0; i < PROBES; ++i) {
            key[i] = x[(g + i) / V::N][2 * ((g + i) % V::N)];
            pay[i] = x[(g + i) / V::N][2 * ((g + i) % V::N) + 1];
          }
          if (!inside) {
#pragma unroll
            for (uint32_t i = 0; i < PROBES; ++i) {
              // counted from the range's start (wraps below it)
              const uint32_t at = (v0 + (g + i) / V::N * BLOCK + tid) * V::N + (g + i) % V::N - off_p;
              if (at >= unit.probe_n) key[i] = no_key;
            }
          }
          tab.probe(unique, key, pay, wave_cnt, cnt, sb, sp);
        }
      };
      if (f0) load(xa, 0);
      constexpr uint32_t STEP = NV * BLOCK;
      for (uint32_t v0 = 0;; v0 += 2 * STEP) {
        load(xb, v0 + STEP);
        probe(xa, v0);
        if (v0 + STEP >= nvp) break;
        load(xa, v0 + 2 * STEP);
        probe(xb, v0 + STEP);
        if (v0 + 2 * STEP >= nvp) break;
      }
      if (f + 1 < fills) __syncthreads();  // probes done before the table is cleared
    }
    if (lane_id() == 0) cnt += wave_cnt;
    if (tid == 0) s_next = gridDim.x + ticket;
    __syncthreads();  // probes done; the table may be cleared
    u = __builtin_amdgcn_readfirstlane(s_next);
    __syncthreads();  // every thread has read s_next
  }
  if (d.job_results) {
    add_result<BLOCK>(d, red, job, cnt, sb, sp);
    return;
  }
  const uint32_t n_build = d.hbm_cap ? uniform_load(d.work_counter + kHbmBuildUnits) : 0u;
  if (n_build) {
    stamp_phase(d.stamps, 4);
    table_phases<K, BLOCK>(d, n_build, &s_next, cnt, sb, sp);
  }
  if (finish_join<BLOCK>(d.aggregates, d.done, d.result, red, &s_next, cnt, sb, sp) && d.stamps && tid == 0) {
    d.stamps[5] = wall_clock64();
    if (!n_build) d.stamps[4] = d.stamps[5];
  }
}

template <typename K, uint32_t CAP, uint32_t BLOCK>
hipError_t launch_part_join(const PipelineDevice& d, uint32_t grid, hipStream_t stream) {
  auto kern = part_join_kernel<K, CAP, BLOCK>;
  const size_t lds = bucket_table_bytes<K>(CAP);
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                            static_cast<int>(lds));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(BLOCK), lds, stream, d);
  return hipGetLastError();
}

template <typename K>
hipError_t launch_one_pass_join_t(const PipelineDevice& d, uint32_t grid, hipStream_t stream) {
  // one block of 1,024 threads per CU with a 128 KiB table, two of 512 with 64
  // KiB, three with 32 KiB
  constexpr uint32_t SLOTS = block_table_slots(kKeyType<K>);
  auto blocks = [&](uint32_t n) { return d.job_results ? n : std::min(n, d.agg_len); };
  switch (one_pass_slots(kKeyType<K>, d.build.n, d.F1, d.big_block_tables != 0)) {
    case 2 * SLOTS: return launch_part_join<K, 2 * SLOTS, 1024>(d, blocks((grid + 1) / 2), stream);
    case SLOTS: return launch_part_join<K, SLOTS, 512>(d, blocks(grid), stream);
    default: return launch_part_join<K, SLOTS / 2, 512>(d, blocks(grid + grid / 2), stream);
  }
}

}  // namespace

hipError_t launch_one_pass_plan(const PipelineDevice& d, KeyType t, const BatchSide* sides, uint32_t joins,
                                hipStream_t stream) {
  if (joins == 0) return hipSuccess;
  const uint32_t F1j = d.F1 / joins;
  if (sides) {
    hipLaunchKernelGGL(reset_counters_kernel, dim3(1), dim3(1024), 0, stream, d.work_counter);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(one_pass_plan_kernel, dim3(joins), dim3(1024), 3 * F1j * 4, stream, d, sides, F1j,
                     block_table_fill(t, one_pass_slots(t, d.build.n, d.F1, d.big_block_tables != 0)),
                     static_cast<uint32_t>(std::min<uint64_t>(~0u, 2 * (d.build.n / d.F1))),
                     one_pass_lds_tuples(t, d.big_block_tables != 0));
  return hipGetLastError();
}

hipError_t launch_one_pass_join(const PipelineDevice& d, KeyType t, uint32_t grid, hipStream_t stream) {
  if (t == KeyType::I32) return launch_one_pass_join_t<int32_t>(d, grid, stream);
  return launch_one_pass_join_t<int64_t>(d, grid, stream);
}

}  // namespace fij
