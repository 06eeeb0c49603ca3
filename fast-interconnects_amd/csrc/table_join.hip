// Joins whose build side fits one block's LDS table: one launch, no
// partitioning.  Every block builds the whole build side into its table and
// streams its share of the probe side against it; the last block to finish
// sums the blocks' results.
#include "bucket_table.hpp"
#include "common.hpp"
#include "internal.hpp"
#include "join_result.hpp"
#include "pipeline.hpp"

namespace fij {
namespace {

// 16 bytes of a column, only as aligned as its elements.
template <typename K>
struct ColumnVec {
  static constexpr uint32_t N = 16 / sizeof(K);
  typedef K type __attribute__((ext_vector_type(16 / sizeof(K)), aligned(sizeof(K))));
};

// The build side (n tuples, at most 3/4 of CAP) into the block's table.
// Returns the table; `unique`: no build key occurs twice.  Begins and ends with a barrier.
template <typename K, uint32_t CAP, uint32_t BLOCK>
__device__ __forceinline__ BucketTable<K, true> build_table(uint64_t* lds, const K* keys, const K* pays, uint32_t n,
                                                            uint32_t* s_dup, bool& unique) {
  using Table = BucketTable<K, true>;
  constexpr uint32_t U = 4;  // build tuples in flight per thread
  const uint32_t tid = threadIdx.x;
  const Table tab(lds, CAP, Table::lg_buckets(CAP, n), null_key<K>());
  __syncthreads();  // the table may still be probed
  tab.clear();
  if (tid == 0) *s_dup = 0;
  __syncthreads();
  bool dup = false;
  for (uint32_t i0 = 0; i0 < n; i0 += U * BLOCK) {
    K k[U], v[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const uint32_t i = min(i0 + u * BLOCK + tid, n - 1);
      k[u] = as_global(keys)[i];
      v[u] = as_global(pays)[i];
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u)
      if (i0 + u * BLOCK + tid < n && k[u] != null_key<K>()) dup |= tab.insert(k[u], v[u]);
  }
  if (dup) *s_dup = 1;
  __syncthreads();
  unique = __builtin_amdgcn_readfirstlane(*s_dup) == 0;
  return tab;
}

// Streams columns [0, n) against the table: vectors first + k * stride of
// BLOCK vectors each (first: the block's place among the blocks that share
// the range), and, for the first block, the last n % V tuples one by one.
template <typename K, uint32_t BLOCK>
struct ColumnStream {
  using VT = typename ColumnVec<K>::type;
  static constexpr uint32_t V = ColumnVec<K>::N;
  static constexpr uint32_t NV = 2;  // vectors of each column in flight per buffer
  const K *keys, *pays;
  uint64_t n, nv, first, stride;
  VT ka[NV], pa[NV], kb[NV], pb[NV];

  __device__ __forceinline__ ColumnStream(const K* k, const K* p, uint64_t tuples, uint32_t block, uint32_t blocks)
      : keys(k), pays(p), n(tuples), nv(tuples / V), first(static_cast<uint64_t>(block) * BLOCK),
        stride(static_cast<uint64_t>(blocks) * BLOCK) {}
  __device__ __forceinline__ void load(VT (&k)[NV], VT (&p)[NV], uint64_t v0) {
#pragma unroll
    for (uint32_t u = 0; u < NV; ++u) {
      const uint64_t v = min(v0 + u * stride + threadIdx.x, nv - 1);
      k[u] = __builtin_nontemporal_load(as_global(reinterpret_cast<const VT*>(keys)) + v);
      p[u] = __builtin_nontemporal_load(as_global(reinterpret_cast<const VT*>(pays)) + v);
    }
  }
  // The first vectors' loads, before the table is built.
  __device__ __forceinline__ void start() {
    if (nv) load(ka, pa, first);
  }
  template <typename Table>
  __device__ __forceinline__ void probe(const Table& tab, bool unique, const VT (&k)[NV], const VT (&p)[NV],
                                        uint64_t v0, uint32_t& wave_cnt, uint64_t& cnt, uint64_t& sb, uint64_t& sp) {
#pragma unroll
    for (uint32_t u = 0; u < NV; ++u) {
      const bool live = v0 + u * stride + threadIdx.x < nv;
#pragma unroll
      for (uint32_t g = 0; g < V; g += 2) {
        const K key[2] = {live ? k[u][g] : null_key<K>(), live ? k[u][g + 1] : null_key<K>()};
        const K pay[2] = {p[u][g], p[u][g + 1]};
        tab.probe(unique, key, pay, wave_cnt, cnt, sb, sp);
      }
    }
  }
  template <typename Table>
  __device__ __forceinline__ void run(const Table& tab, bool unique, uint64_t& cnt, uint64_t& sb, uint64_t& sp) {
    uint32_t wave_cnt = 0;
    const uint64_t step = NV * stride;
    for (uint64_t v0 = first; v0 < nv; v0 += 2 * step) {  // uniform
      load(kb, pb, v0 + step);
      probe(tab, unique, ka, pa, v0, wave_cnt, cnt, sb, sp);
      if (v0 + step >= nv) break;
      load(ka, pa, v0 + 2 * step);
      probe(tab, unique, kb, pb, v0 + step, wave_cnt, cnt, sb, sp);
    }
    if (lane_id() == 0) cnt += wave_cnt;
    const uint64_t i = nv * V + threadIdx.x;
    if (first == 0 && i < n && keys[i] != null_key<K>()) {
      const K key = keys[i];
      tab.template probe_from<false>(tab.bucket(key), key, pays[i], cnt, sb, sp);
    }
  }
};

// One join; the last block writes the sums of all to *result (finish_join).
//
// Bound by the chain launch -> build -> probe for short probe sides and by the
// read of the probe columns for long ones.  1,500 x 6,007 int32 tuples: one
// launch of 7 us where 11 launches partitioned both sides in 9 bits (86 us);
// the whole call 140 -> 19 us.  Every block pays the build, so a block gets at
// least 4 steps of probe tuples.
template <typename K, uint32_t CAP, uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK, CAP * 2 * sizeof(K) <= 32768 ? 6 : 4) void table_join_kernel(TableJoin j) {
  extern __shared__ __attribute__((aligned(16))) uint64_t lds_u64[];
  __shared__ uint32_t s_dup, s_last;
  __shared__ uint64_t red[3][BLOCK / kWave];
  if (j.stamps && blockIdx.x == 0 && threadIdx.x == 0) j.stamps[0] = wall_clock64();
  uint64_t cnt = 0, sb = 0, sp = 0;
  if (j.n_b) {
    ColumnStream<K, BLOCK> s(static_cast<const K*>(j.probe_keys), static_cast<const K*>(j.probe_pays), j.n_p,
                             blockIdx.x, gridDim.x);
    s.start();
    bool unique;
    const auto tab = build_table<K, CAP, BLOCK>(lds_u64, static_cast<const K*>(j.build_keys),
                                                static_cast<const K*>(j.build_pays), static_cast<uint32_t>(j.n_b),
                                                &s_dup, unique);
    s.run(tab, unique, cnt, sb, sp);
  }
  if (finish_join<BLOCK>(j.partial, j.done, j.result, red, &s_last, cnt, sb, sp) && j.stamps && threadIdx.x == 0)
    j.stamps[5] = wall_clock64();
}

template <typename K, uint32_t CAP, uint32_t BLOCK>
hipError_t launch_table_join_t(const TableJoin& j, uint32_t grid, hipStream_t stream) {
  auto kern = table_join_kernel<K, CAP, BLOCK>;
  const size_t lds = bucket_table_bytes<K>(CAP);
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                            static_cast<int>(lds));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(BLOCK), lds, stream, j);
  return hipGetLastError();
}

template <typename K>
hipError_t launch_table_join_k(const TableJoin& j, uint32_t cus, uint32_t max_grid, hipStream_t stream) {
  // 128 KiB tables (one block of 1,024 threads per CU) for build sides beyond
  // half of a 32 KiB one (four blocks of 512)
  constexpr uint32_t BIG = 131072 / (2 * sizeof(K)), SMALL = BIG / 4;
  const bool big = j.n_b > SMALL / 2;
  const uint64_t per_block = static_cast<uint64_t>(big ? 1024 : 512) * ColumnVec<K>::N * 4;
  const uint64_t want = (j.n_p + per_block - 1) / per_block;
  const uint64_t cap = std::min<uint64_t>(big ? cus : 4 * cus, max_grid);
  const uint32_t grid = static_cast<uint32_t>(std::max<uint64_t>(1, std::min<uint64_t>(want, cap)));
  if (big) return launch_table_join_t<K, BIG, 1024>(j, grid, stream);
  return launch_table_join_t<K, SMALL, 512>(j, grid, stream);
}

}  // namespace

uint64_t table_join_tuples(KeyType t) { return 131072u / tuple_bytes(t) * 3 / 4; }

hipError_t launch_table_join(KeyType t, const TableJoin& j, uint32_t cus, uint32_t max_grid, hipStream_t stream) {
  if (t == KeyType::I32) return launch_table_join_k<int32_t>(j, cus, max_grid, stream);
  return launch_table_join_k<int64_t>(j, cus, max_grid, stream);
}

}  // namespace fij
