// Radix join: per-partition LDS hash build and probe with aggregation.
//
// Semantics follow sql-ops/cudautils/radix_join.cu: partitions are assigned
// to blocks by the reference's greedy rule (:58-98); each block builds an LDS
// table for each of its partitions and probes it (:103-194 perfect hashing,
// :199-311 bucket chaining).  The reference aggregates SUM(probe.value) into
// per-thread partials; this library writes those partials unchanged (when
// asked) and additionally a per-block {match count, SUM(build.value),
// SUM(probe.value)} as wrapping 64-bit integers.
#include "bucket_table.hpp"
#include "common.hpp"
#include "internal.hpp"

namespace fij {
namespace {

constexpr uint32_t kChainBuckets = 2048;  // sql-ops/build.rs:72
constexpr uint32_t kChainTail = 0xFFFFu;

struct JoinParams {
  const void* build_rel;
  const uint64_t* build_offsets;
  uint64_t build_len;
  const void* probe_rel;
  const uint64_t* probe_offsets;
  uint64_t probe_len;
  uint32_t radix_bits;
  uint32_t ignore_bits;
  uint32_t ht_entries;
  int64_t* result_set;
  JoinAggregate* aggregates;
  const uint32_t* task_assignments;
  uint32_t* status;
  uint32_t table_slots;  // of the largest bucket table (a power of two)
};

// Largest fanout whose task assignment runs by pointer doubling (its LDS:
// prefix sums and two jump arrays of F + 1 entries).
constexpr uint32_t kAssignDoublingMax = 8192;

// radix_join.cu:58-98.  One block: partition sizes are staged in LDS in
// parallel, then the reference's greedy cut is computed in parallel, with
// the same result.
__global__ __launch_bounds__(1024) void assign_tasks_kernel(const uint64_t* probe_offsets,
                                                            uint32_t probe_len, uint32_t pad,
                                                            uint32_t radix_bits, uint32_t grid,
                                                            uint32_t* ta) {
  extern __shared__ uint32_t sizes[];
  const uint32_t F = 1u << radix_bits;
  for (uint32_t p = threadIdx.x; p < F; p += blockDim.x) {
    const uint32_t upper = (p + 1 < F) ? static_cast<uint32_t>(probe_offsets[p + 1] - pad) : probe_len;
    sizes[p] = static_cast<uint32_t>(upper - probe_offsets[p]);
  }
  __syncthreads();
  // The greedy rule: a task ends at the first partition whose size brings
  // the task to at least avg probe tuples.
  if (F <= kAssignDoublingMax) {
    // With P the exclusive prefix sums of the sizes, the task starting at
    // partition s ends before J(s) = the first j > s with P[j] >= P[s] + avg
    // (F if none), so ta[k] = J^k(0): J by binary searches, then J^m
    // squared and applied to ta[0 .. m) in log2(grid) rounds.
    __shared__ uint32_t wave_tmp[1024 / kWave + 1];
    const uint32_t avg = (probe_len - pad * F + grid - 1u) / grid;
    uint32_t* P = sizes;                                       // [F + 1]
    uint16_t* cur = reinterpret_cast<uint16_t*>(sizes + F + 1);  // [F + 1]
    uint16_t* nxt = cur + F + 1;                               // [F + 1]
    const uint32_t total = block_exclusive_scan<uint32_t>(P, F, wave_tmp);
    if (threadIdx.x == 0) P[F] = total;
    __syncthreads();
    for (uint32_t s0 = threadIdx.x; s0 <= F; s0 += blockDim.x) {
      uint32_t lo = s0 + 1, hi = F + 1;
      if (s0 < F) {
        const uint64_t target = static_cast<uint64_t>(P[s0]) + avg;
        while (lo < hi) {
          const uint32_t mid = (lo + hi) / 2;
          if (P[mid] >= target) hi = mid; else lo = mid + 1;
        }
      }
      cur[s0] = static_cast<uint16_t>(min(lo, F));
    }
    if (threadIdx.x == 0) {
      ta[0] = 0;
      ta[grid] = F;
    }
    __syncthreads();
    for (uint64_t m = 1; m < grid; m *= 2) {
      for (uint64_t i = threadIdx.x; i < m && m + i < grid; i += blockDim.x) ta[m + i] = cur[ta[i]];
      for (uint32_t s0 = threadIdx.x; s0 <= F; s0 += blockDim.x) nxt[s0] = cur[cur[s0]];
      __syncthreads();
      uint16_t* t = cur;
      cur = nxt;
      nxt = t;
    }
    return;
  }
  // Larger fanouts: taken 64 partitions at a time by wave 0: an inclusive
  // scan of the sizes gives every lane the running sum since the last cut,
  // a ballot finds the next cut; one step per cut.
  if (threadIdx.x < kWave) {
    const uint32_t lane = threadIdx.x;
    const uint32_t probe_tuples = probe_len - pad * F;
    const uint32_t avg = (probe_tuples + grid - 1u) / grid;
    if (lane == 0) ta[0] = 0;
    uint32_t task_id = 1, task_size = 0;  // wave-uniform
    for (uint32_t base = 0; base < F && task_id < grid; base += kWave) {
      const bool valid = base + lane < F;
      const uint32_t incl = wave_inclusive_scan(valid ? sizes[base + lane] : 0u);
      uint32_t carry = task_size, before = 0, from = 0;  // running sum at lane l: carry + incl[l] - before
      while (task_id < grid) {
        const uint64_t hit = ballot(lane >= from && valid && carry + incl - before >= avg);
        if (hit == 0) break;
        const uint32_t l = static_cast<uint32_t>(__builtin_ctzll(hit));
        if (lane == 0) ta[task_id] = base + l + 1;
        task_id += 1;
        carry = 0;
        before = __builtin_amdgcn_readlane(incl, l);
        from = l + 1;
      }
      task_size = carry + __builtin_amdgcn_readlane(incl, kWave - 1) - before;
    }
    for (uint32_t t = task_id + lane; t <= grid; t += kWave) ta[t] = F;
  }
}

// The partitions part .. end - 1 of a block, whose results are task `owner`'s.
struct TaskPart {
  uint32_t part, end, owner;
};

// A task takes partitions up to the average number of probe tuples, so tasks
// of about two partitions alternate with tasks of one and as many blocks are
// left without any.  With at least as many blocks as partitions those blocks
// take the second and later partitions of the others' tasks, and a launch
// lasts one partition instead of two: with N tasks the i-th block behind them
// takes the i-th such partition, partition i + k + 1 of the task k with
// ta[k] - k <= i < ta[k + 1] - (k + 1).  Blocks with a task start on it and
// those that no partition is left for end without a look at the others (each
// block has a compute unit's LDS: 13.4 us for the launches of 64 partitions of
// 1,000 + 4,000 tuples became 15 with that look).
__device__ __forceinline__ TaskPart block_task(const JoinParams& p) {
  const uint32_t* const ta = p.task_assignments;
  const uint32_t F = 1u << p.radix_bits, b = blockIdx.x;
  if (F > gridDim.x) return {ta[b], ta[b + 1], b};
  if (ta[b] < F) return {ta[b], ta[b] + 1, b};
  if (ta[F - 1] < F) return {F, F, b};  // a task per partition
  __shared__ uint32_t s_tasks, s_owner;
  if (threadIdx.x == 0) s_tasks = s_owner = 0;
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < gridDim.x; k += blockDim.x)
    if (ta[k] < F) atomicMax(&s_tasks, k + 1);
  __syncthreads();
  const uint32_t n = s_tasks, i = b - n;
  if (i >= F - n) return {F, F, b};  // uniform
  for (uint32_t k = threadIdx.x; k < n; k += blockDim.x)
    if (ta[k] - k <= i && i < ta[k + 1] - (k + 1)) s_owner = k;
  __syncthreads();
  const uint32_t k = s_owner;
  return {i + k + 1, i + k + 2, k};
}

// Probe tuples q0 .. q1 - 1 (at least one) of a block, streamed through two
// buffers of N tuples per thread: thread i takes tuples q0 + i, q0 + i +
// blockDim, ... (lanes past the end repeat the last tuple).
template <typename K>
struct ProbeStream {
  static constexpr uint32_t N = 4;
  const Tuple<K>* probe;
  uint64_t q0, q1;
  Tuple<K> a[N], b[N];

  __device__ __forceinline__ void load(Tuple<K> (&t)[N], uint64_t i0) {
#pragma unroll
    for (uint32_t k = 0; k < N; ++k)
      t[k] = load_tuple<K>(probe + min<uint64_t>(i0 + k * blockDim.x + threadIdx.x, q1 - 1));
  }
  __device__ __forceinline__ void start() {
    if (q0 < q1) load(a, q0);
  }
  // f(tuples, live): bit k of live = tuple k is in the range.
  template <typename Fn>
  __device__ __forceinline__ void run(Fn f) {
    const uint64_t step = static_cast<uint64_t>(N) * blockDim.x;
    auto live = [&](uint64_t i0) {
      uint32_t m = 0;
#pragma unroll
      for (uint32_t k = 0; k < N; ++k) m |= i0 + k * blockDim.x + threadIdx.x < q1 ? 1u << k : 0u;
      return m;
    };
    for (uint64_t i0 = q0; i0 < q1; i0 += 2 * step) {
      load(b, i0 + step);
      f(a, live(i0));
      if (i0 + step >= q1) break;
      load(a, i0 + 2 * step);
      f(b, live(i0 + step));
    }
  }
};

__device__ __forceinline__ void partition_range(const uint64_t* offsets, uint64_t padded_len, uint32_t F,
                                                uint32_t p, uint32_t pad, uint64_t& begin, uint64_t& end) {
  begin = offsets[p];
  end = (p + 1 < F) ? offsets[p + 1] - pad : padded_len;
}

template <typename K>
__device__ __forceinline__ uint32_t perfect_index(K key, uint32_t ignore_bits) {
  return static_cast<uint32_t>(static_cast<uint64_t>(static_cast<int64_t>(key)) >> ignore_bits);
}

// Bucket of the chaining table: the key's index above the ignored bits (a
// u32, as key_to_partition returns it) widened to the key type, then the
// key type's multiply-shift hash -- 64-bit for i64 keys
// (radix_join.cu:283-284,296-297: hash<K>(key_to_partition(...))).
template <typename K>
__device__ __forceinline__ uint32_t chain_bucket(K key, uint32_t ignore_bits, uint32_t log2_buckets) {
  return mult_shift_hash<K>(static_cast<K>(perfect_index<K>(key, ignore_bits)), log2_buckets);
}

template <typename U>
__device__ __forceinline__ void add_u64(U* at, uint64_t v) {
  static_assert(sizeof(U) == 8, "64-bit words");
  atomicAdd(reinterpret_cast<unsigned long long*>(at), static_cast<unsigned long long>(v));
}

// Block-wide sum of three u64 values into *out (+=), which other blocks of its
// task may add to.
__device__ void block_aggregate(JoinAggregate* out, uint64_t c, uint64_t sb, uint64_t sp) {
  __shared__ uint64_t red[3][16];
  const uint32_t w = threadIdx.x / kWave;
  const uint64_t wc = wave_broadcast_last(wave_inclusive_scan(c));
  const uint64_t wb = wave_broadcast_last(wave_inclusive_scan(sb));
  const uint64_t wp = wave_broadcast_last(wave_inclusive_scan(sp));
  if (lane_id() == 0) {
    red[0][w] = wc;
    red[1][w] = wb;
    red[2][w] = wp;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t a = 0, b = 0, d = 0;
    for (uint32_t i = 0; i < blockDim.x / kWave; ++i) {
      a += red[0][i];
      b += red[1][i];
      d += red[2][i];
    }
    add_u64(&out->count, a);
    add_u64(&out->sum_build, b);
    add_u64(&out->sum_probe, d);
  }
}

template <typename K>
__global__ __launch_bounds__(1024) void join_perfect_kernel(JoinParams p) {
  extern __shared__ uint64_t lds_u64[];
  Tuple<K>* ht = reinterpret_cast<Tuple<K>*>(lds_u64);
  const uint32_t F = 1u << p.radix_bits;
  const uint32_t pad = padding_len<K>();
  const uint32_t E = p.ht_entries;
  const Tuple<K>* build = static_cast<const Tuple<K>*>(p.build_rel);
  const Tuple<K>* probe = static_cast<const Tuple<K>*>(p.probe_rel);
  uint64_t cnt = 0, sb = 0, sp = 0;
  int64_t ref_sum = 0;
  bool overflow = false;
  const TaskPart task = block_task(p);
  if (task.part == task.end) return;  // uniform: adds nothing
  for (uint32_t part = task.part; part < task.end; ++part) {
    ProbeStream<K> stream;
    stream.probe = probe;
    uint64_t b0, b1;
    partition_range(p.build_offsets, p.build_len, F, part, pad, b0, b1);
    partition_range(p.probe_offsets, p.probe_len, F, part, pad, stream.q0, stream.q1);
    stream.start();  // in flight while the table is built
    for (uint32_t i = threadIdx.x; i < E; i += blockDim.x) {
      ht[i].key = null_key<K>();
      ht[i].value = 0;
    }
    __syncthreads();
    for (uint64_t i = b0 + threadIdx.x; i < b1; i += blockDim.x) {
      const Tuple<K> t = load_tuple<K>(build + i);
      if (t.key == null_key<K>()) continue;  // null keys never join
      const uint32_t idx = perfect_index<K>(t.key, p.ignore_bits);
      if (idx < E) ht[idx] = t;
      else overflow = true;
    }
    __syncthreads();
    stream.run([&](const Tuple<K>(&t)[ProbeStream<K>::N], uint32_t live) {
#pragma unroll
      for (uint32_t k = 0; k < ProbeStream<K>::N; ++k) {
        const uint32_t idx = perfect_index<K>(t[k].key, p.ignore_bits);
        if (((live >> k) & 1u) && t[k].key != null_key<K>() && idx < E && ht[idx].key == t[k].key) {
          cnt += 1;
          sb += static_cast<uint64_t>(static_cast<int64_t>(ht[idx].value));
          sp += static_cast<uint64_t>(static_cast<int64_t>(t[k].value));
          ref_sum += static_cast<int64_t>(t[k].value);
        }
      }
    });
    __syncthreads();
  }
  if (overflow && p.status) atomicOr(p.status, kStatusHashTableFull);
  if (p.result_set)
    add_u64(p.result_set + static_cast<uint64_t>(blockDim.x) * task.owner + threadIdx.x, static_cast<uint64_t>(ref_sum));
  if (p.aggregates) block_aggregate(p.aggregates + task.owner, cnt, sb, sp);
}

// Whether a bucket table answers a partition's probes faster than chains, whose
// build costs half as much and for which copies of a key are cheaper.  64
// partitions of n build tuples and r * n probe tuples, chains and tables, us:
// int32, different keys: n = 1,500 r = 8 16.5 16.5, r = 32 31 28; 4,096 r = 4 21
// 20, r = 8 31 25; 12,000 r = 4 68 67, r = 16 225 174; int64: 2,048 r = 16 27 27;
// 4,096 r = 8 31 29, r = 16 49 41; 5,000 r = 16 65 67.  Keys of two copies: int32
// 4,096 r = 8 35 36, 12,000 r = 16 250 308; int64 4,096 r = 16 57 69.
template <typename K>
__device__ __forceinline__ bool table_pays(uint32_t slots, uint32_t nbuild, uint64_t nprobe) {
  const bool few = sizeof(K) == 4 && nbuild <= slots / 8 * 3;  // level also where keys repeat
  return nbuild > kChainBuckets / 2 && nbuild <= slots / 16 * (sizeof(K) == 4 ? 12 : 9) && nprobe >= 32768 &&
         nprobe >= static_cast<uint64_t>(few ? 8 : 16) * nbuild;
}

// One partition's build tuples (at most 3/4 of p.table_slots) in a bucket table
// and its probe tuples against it; false, with nothing joined, if keys repeat
// and chains are better then.
template <typename K>
__device__ __forceinline__ bool bucket_join(const JoinParams& p, uint64_t* lds, uint32_t* s_dup,
                                            const Tuple<K>* build, uint32_t nbuild, ProbeStream<K>& stream,
                                            uint64_t& cnt, uint64_t& sb, uint64_t& sp) {
  using Table = BucketTable<K, true>;
  const Table tab(lds, p.table_slots, Table::lg_buckets(p.table_slots, nbuild), null_key<K>());
  tab.clear();
  if (threadIdx.x == 0) *s_dup = 0;
  __syncthreads();
  bool dup = false;
  for (uint32_t i = threadIdx.x; i < nbuild; i += blockDim.x) {
    const Tuple<K> t = load_tuple<K>(build + i);
    if (t.key != null_key<K>()) dup |= tab.insert(t.key, t.value);  // null keys never join
  }
  if (dup) *s_dup = 1;
  __syncthreads();
  const bool unique = __builtin_amdgcn_readfirstlane(*s_dup) == 0;
  if (!unique && (sizeof(K) == 8 || nbuild > p.table_slots / 8 * 3)) return false;
  uint32_t wave_cnt = 0;
  stream.run([&](const Tuple<K>(&t)[ProbeStream<K>::N], uint32_t live) {
#pragma unroll
    for (uint32_t g = 0; g < ProbeStream<K>::N; g += 2) {
      K key[2], pay[2];
#pragma unroll
      for (uint32_t i = 0; i < 2; ++i) {
        key[i] = (live >> (g + i)) & 1u ? t[g + i].key : null_key<K>();
        pay[i] = t[g + i].value;
      }
      tab.probe(unique, key, pay, wave_cnt, cnt, sb, sp);
    }
  });
  if (lane_id() == 0) cnt += wave_cnt;
  return true;
}

// Build partitions go into chains (radix_join.cu:208-392's layout), or, where
// table_pays, into a bucket table.  Chains cost two reads per entry, and the
// value of a match (reading it with each key: 85 instead of 82 us for the probes
// of 64 partitions of 6,000 + 96,000 int64 tuples); as long as they are short,
// that is less than clearing and filling a table.
template <typename K>
__global__ __launch_bounds__(1024) void join_chaining_kernel(JoinParams p) {
  extern __shared__ __attribute__((aligned(16))) uint64_t lds_u64[];
  __shared__ uint32_t s_dup;
  const uint32_t E = p.ht_entries;  // entries (<= 0xFFFF)
  K* keys = reinterpret_cast<K*>(lds_u64);
  K* vals = keys + E;
  uint32_t* heads = reinterpret_cast<uint32_t*>(vals + E);
  uint16_t* links = reinterpret_cast<uint16_t*>(heads + kChainBuckets);
  const uint32_t log2_buckets = 31u - __builtin_clz(kChainBuckets);
  const uint32_t F = 1u << p.radix_bits;
  const uint32_t pad = padding_len<K>();
  const Tuple<K>* build = static_cast<const Tuple<K>*>(p.build_rel);
  const Tuple<K>* probe = static_cast<const Tuple<K>*>(p.probe_rel);
  uint64_t cnt = 0, sb = 0, sp = 0;
  bool overflow = false;
  const TaskPart task = block_task(p);
  if (task.part == task.end) return;  // uniform: adds nothing
  for (uint32_t part = task.part; part < task.end; ++part) {
    ProbeStream<K> stream;
    stream.probe = probe;
    uint64_t b0, b1;
    partition_range(p.build_offsets, p.build_len, F, part, pad, b0, b1);
    partition_range(p.probe_offsets, p.probe_len, F, part, pad, stream.q0, stream.q1);
    stream.start();  // in flight while the table is built
    const uint64_t nb = b1 - b0;
    if (nb > E) overflow = true;
    const uint32_t nbuild = nb > E ? E : static_cast<uint32_t>(nb);
    if (table_pays<K>(p.table_slots, nbuild, stream.q1 - stream.q0) &&
        bucket_join<K>(p, lds_u64, &s_dup, build + b0, nbuild, stream, cnt, sb, sp)) {
      __syncthreads();
      continue;
    }
    for (uint32_t i = threadIdx.x; i < kChainBuckets; i += blockDim.x) heads[i] = kChainTail;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < nbuild; i += blockDim.x) {
      const Tuple<K> t = load_tuple<K>(build + b0 + i);
      keys[i] = t.key;
      vals[i] = t.value;
      if (t.key == null_key<K>()) continue;  // stored but never linked: null keys never join
      const uint32_t bucket = chain_bucket<K>(t.key, p.ignore_bits, log2_buckets);
      links[i] = static_cast<uint16_t>(atomicExch(&heads[bucket], i));
    }
    __syncthreads();
    // the chains of a buffer's tuples are walked together: a step's LDS reads
    // are in flight at once (entry 0 is read where a chain has ended)
    stream.run([&](const Tuple<K>(&t)[ProbeStream<K>::N], uint32_t live) {
      constexpr uint32_t N = ProbeStream<K>::N;
      uint32_t e[N];
#pragma unroll
      for (uint32_t k = 0; k < N; ++k) {
        const uint32_t head = heads[chain_bucket<K>(t[k].key, p.ignore_bits, log2_buckets)];
        e[k] = ((live >> k) & 1u) && t[k].key != null_key<K>() ? head : kChainTail;
      }
      for (;;) {
        bool any = false;
#pragma unroll
        for (uint32_t k = 0; k < N; ++k) any |= e[k] != kChainTail;
        if (!ballot(any)) break;
        K key[N];
        uint32_t next[N];
#pragma unroll
        for (uint32_t k = 0; k < N; ++k) {
          const uint32_t at = e[k] != kChainTail ? e[k] : 0u;
          key[k] = keys[at];
          next[k] = links[at];
        }
#pragma unroll
        for (uint32_t k = 0; k < N; ++k) {
          if (e[k] == kChainTail) continue;
          if (key[k] == t[k].key) {
            cnt += 1;
            sb += static_cast<uint64_t>(static_cast<int64_t>(vals[e[k]]));
            sp += static_cast<uint64_t>(static_cast<int64_t>(t[k].value));
          }
          e[k] = next[k];
        }
      }
    });
    __syncthreads();
  }
  if (overflow && p.status) atomicOr(p.status, kStatusHashTableFull);
  if (p.result_set) add_u64(p.result_set + static_cast<uint64_t>(blockDim.x) * task.owner + threadIdx.x, sp);
  if (p.aggregates) block_aggregate(p.aggregates + task.owner, cnt, sb, sp);
}

template <typename K>
hipError_t launch_join_t(const JoinLaunch& a, hipStream_t stream) {
  JoinParams p{};
  p.build_rel = a.build_rel;
  p.build_offsets = a.build_offsets;
  p.build_len = a.build_len;
  p.probe_rel = a.probe_rel;
  p.probe_offsets = a.probe_offsets;
  p.probe_len = a.probe_len;
  p.radix_bits = a.radix_bits;
  p.ignore_bits = a.ignore_bits;
  p.result_set = a.result_set;
  p.aggregates = a.aggregates;
  p.task_assignments = a.task_assignments;
  p.status = a.status;
  if (a.scheme == JoinScheme::Perfect) {
    auto kern = join_perfect_kernel<K>;
    const uint32_t lds = dynamic_lds_budget(reinterpret_cast<const void*>(kern), a.lds_bytes);
    if (lds < 2 * sizeof(Tuple<K>)) return hipErrorInvalidConfiguration;
    // cuda_radix_join.rs:234-237: entries = LDS / sizeof(entry) - 1.
    p.ht_entries = lds / sizeof(Tuple<K>) - 1;
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(lds));
    hipLaunchKernelGGL(kern, dim3(a.grid), dim3(a.block), lds, stream, p);
  } else {
    auto kern = join_chaining_kernel<K>;
    const uint32_t lds = dynamic_lds_budget(reinterpret_cast<const void*>(kern), a.lds_bytes);
    if (lds < kChainBuckets * 4 + 64) return hipErrorInvalidConfiguration;
    // radix_join.cu:213-221: entries = (LDS - buckets*4) / (2 + k + v), u16 links.
    uint32_t entries = (lds - kChainBuckets * 4) / (2 + 2 * sizeof(K));
    if (entries > kChainTail) entries = kChainTail;
    p.ht_entries = entries;
    p.table_slots = 256;
    while (bucket_table_bytes<K>(2 * p.table_slots) <= lds) p.table_slots *= 2;
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(lds));
    hipLaunchKernelGGL(kern, dim3(a.grid), dim3(a.block), lds, stream, p);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_assign_tasks(const uint64_t* probe_offsets, uint64_t probe_len, uint32_t pad,
                               uint32_t radix_bits, uint32_t grid, uint32_t* task_assignments,
                               hipStream_t stream) {
  const uint32_t F = 1u << radix_bits;
  const size_t lds = F <= kAssignDoublingMax ? (F + 1) * 4 + 2 * (F + 1) * 2 : F * 4;
  hipLaunchKernelGGL(assign_tasks_kernel, dim3(1), dim3(1024), lds, stream, probe_offsets,
                     static_cast<uint32_t>(probe_len), pad, radix_bits, grid, task_assignments);
  return hipGetLastError();
}

hipError_t launch_join(const JoinLaunch& a, hipStream_t stream) {
  if (a.type == KeyType::I32) return launch_join_t<int32_t>(a, stream);
  return launch_join_t<int64_t>(a, stream);
}

}  // namespace fij
