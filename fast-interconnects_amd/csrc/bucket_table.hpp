// Block-shared LDS hash table of the joins that stream a probe range against one
// build range (single-pass partitions, build sides of one table).
#pragma once

#include "common.hpp"

namespace fij {

// Block-shared table of buckets of four slots, filled in order and probed
// linearly from the key's bucket: LDS reads of a bucket's keys (16 bytes at i32)
// and of one value answer a probe unless the key's bucket was full.  (Reading
// all four values with the keys instead of the one of the slot behind them:
// 187 instead of 174 us for 5,000,011 + 20,000,003 int64 tuples, int32 level.)
// Probing is bound by instructions (a wave of 64 takes 4 cycles for each), so
// the common case is straight-line code: buckets are at most 1/4 full on
// average where the table allows it, which leaves 0.4 % of the keys outside
// their bucket, and a table without duplicate keys (the insert finds out: the
// later of two equal keys passes the earlier one) stops at a match.
//
// free_key marks free slots; no build tuple may have it.  The keys of a
// partition share their low digit, so the single-pass joins take a key of
// another digit: a null key (-1) then needs no test of its own when it is
// probed, and lanes past a range's end carry a second key of another digit.
// NULLS: free_key is the null key itself, and null keys are kept from probing.
template <typename K, bool NULLS = false>
struct BucketTable {
  typedef K Quad __attribute__((ext_vector_type(4)));
  Quad* keys;      // [buckets]
  Quad* vals;      // [buckets]
  uint32_t shift;  // hash bits below the bucket index
  uint32_t mask;   // buckets - 1
  K free_key;

  __device__ __forceinline__ uint32_t bucket(K key) const {
    uint32_t h = static_cast<uint32_t>(key) * 2654435769u;
    if constexpr (sizeof(K) == 8) h += static_cast<uint32_t>(static_cast<uint64_t>(key) >> 32) * 2246822519u;
    return h >> shift;
  }
  // Returns whether an equal key was passed.
  __device__ __forceinline__ bool insert(K key, K val) const {
    bool dup = false;
    uint32_t s = 4 * bucket(key);
    K* const k = reinterpret_cast<K*>(keys);
    for (;; s = (s + 1) & (4 * mask + 3)) {
      K prev;
      if constexpr (sizeof(K) == 8)
        prev = static_cast<K>(atomicCAS(reinterpret_cast<unsigned long long*>(&k[s]),
                                        static_cast<unsigned long long>(free_key),
                                        static_cast<unsigned long long>(key)));
      else
        prev = static_cast<K>(atomicCAS(reinterpret_cast<unsigned int*>(&k[s]), static_cast<unsigned int>(free_key),
                                        static_cast<unsigned int>(key)));
      if (prev == free_key) {
        reinterpret_cast<K*>(vals)[s] = val;
        return dup;
      }
      dup |= prev == key;
    }
  }
  static __device__ __forceinline__ void add(K v, K pay, uint64_t& sb, uint64_t& sp) {
    sb += static_cast<uint64_t>(static_cast<int64_t>(v));
    sp += static_cast<uint64_t>(static_cast<int64_t>(pay));
  }
  // Probes N tuples of a lane together in a table without duplicate keys; the
  // matches in first buckets are counted by the scalar unit (wave_cnt).
  template <uint32_t N>
  __device__ __forceinline__ void probe_unique(const K (&key)[N], const K (&pay)[N], uint32_t& wave_cnt, uint64_t& cnt,
                                               uint64_t& sb, uint64_t& sp) const {
    uint32_t at[N];
    Quad k[N];
    K v[N];
    bool more[N];
#pragma unroll
    for (uint32_t i = 0; i < N; ++i) {
      at[i] = bucket(key[i]);
      k[i] = keys[at[i]];
    }
#pragma unroll
    for (uint32_t i = 0; i < N; ++i) {
      const uint32_t s = k[i].y == key[i] ? 1u : k[i].z == key[i] ? 2u : k[i].w == key[i] ? 3u : 0u;
      v[i] = reinterpret_cast<const K*>(vals)[4 * at[i] + s];
    }
    bool any = false;
#pragma unroll
    for (uint32_t i = 0; i < N; ++i) {
      const bool m0 = k[i].x == key[i], m1 = k[i].y == key[i], m2 = k[i].z == key[i], m3 = k[i].w == key[i];
      const bool ok = !NULLS || key[i] != free_key;
      const uint64_t m = ballot(m0) | ballot(m1) | ballot(m2) | ballot(m3);
      wave_cnt += static_cast<uint32_t>(__popcll(NULLS ? m & ballot(ok) : m));
      if (ok && (m0 || m1 || m2 || m3)) add(v[i], pay[i], sb, sp);
      more[i] = ok && !(m0 || m1 || m2 || m3) && k[i].w != free_key;
      any |= more[i];
    }
    if (ballot(any)) {
#pragma unroll
      for (uint32_t i = 0; i < N; ++i)
        if (more[i]) probe_from((at[i] + 1) & mask, key[i], pay[i], cnt, sb, sp);
    }
  }
  // Probes from bucket b to the first bucket with a free slot: every match
  // counts (not for a null key when NULLS).
  __device__ __forceinline__ void probe_from(uint32_t b, K key, K pay, uint64_t& cnt, uint64_t& sb,
                                             uint64_t& sp) const {
    for (;; b = (b + 1) & mask) {
      const Quad k = keys[b];
      const uint32_t m = (k.x == key ? 1u : 0u) | (k.y == key ? 2u : 0u) | (k.z == key ? 4u : 0u) |
                         (k.w == key ? 8u : 0u);
      if (m) {
        const Quad v = vals[b];
        cnt += __popc(m);
        if (m & 1u) add(v.x, pay, sb, sp);
        if (m & 2u) add(v.y, pay, sb, sp);
        if (m & 4u) add(v.z, pay, sb, sp);
        if (m & 8u) add(v.w, pay, sb, sp);
      }
      if (k.w == free_key) return;
    }
  }
};

}  // namespace fij
