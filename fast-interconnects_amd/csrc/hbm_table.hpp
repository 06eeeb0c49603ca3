// Linear-probing hash tables in the plan's HBM arena, shared by the two-pass
// and the single-pass joins: a build side that no block's LDS table holds gets
// 2^lg slots (at least twice its build tuples), every word all ones when free.
// Hashing and probing follow the no-partitioning join
// (no_partitioning_join.cu:39-249): multiply-shift from the key, linear
// probing, every match counted; i32 entries are installed by one 64-bit CAS of
// key and payload against an all-ones entry, i64 by a CAS on the key and then
// the payload store.
#pragma once

#include "common.hpp"

namespace fij {

template <typename K>
__device__ __forceinline__ void hbm_insert(Tuple<K>* tab, uint32_t lg, K key, K val) {
  const uint64_t mask = (1ull << lg) - 1;
  uint64_t h = mult_shift_hash<K>(key, lg);
  for (uint64_t a = 0; a <= mask; ++a, h = (h + 1) & mask) {
    if constexpr (sizeof(K) == 4) {
      const unsigned long long want = static_cast<unsigned long long>(static_cast<uint32_t>(key)) |
                                      (static_cast<unsigned long long>(static_cast<uint32_t>(val)) << 32);
      if (atomicCAS(reinterpret_cast<unsigned long long*>(tab + h), ~0ull, want) == ~0ull) return;
    } else {
      if (atomicCAS(reinterpret_cast<unsigned long long*>(&tab[h].key), ~0ull, static_cast<unsigned long long>(key)) ==
          ~0ull) {
        tab[h].value = val;
        return;
      }
    }
  }
}

// Every build tuple with this key matches; probing ends at the first free
// slot.  (The i64 payload of a slot whose key was just installed may still be
// in flight while tables are built: probes run in a later launch, or behind the
// wait for all build units.)
template <typename K>
__device__ __forceinline__ void hbm_probe(const Tuple<K>* tab, uint32_t lg, K key, K pay, uint64_t& cnt, uint64_t& sb,
                                          uint64_t& sp) {
  const uint64_t mask = (1ull << lg) - 1;
  uint64_t h = mult_shift_hash<K>(key, lg);
  for (uint64_t a = 0; a <= mask; ++a, h = (h + 1) & mask) {
    const Tuple<K> e = load_tuple<K>(tab + h);
    if (e.key == null_key<K>()) return;
    if (e.key == key) {
      cnt += 1;
      sb += static_cast<uint64_t>(static_cast<int64_t>(e.value));
      sp += static_cast<uint64_t>(static_cast<int64_t>(pay));
    }
  }
}

}  // namespace fij
