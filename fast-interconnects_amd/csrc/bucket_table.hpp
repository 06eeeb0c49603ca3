// Block-shared LDS hash table of the joins that stream a probe range against one
// build range (single-pass partitions, build sides of one table).
#pragma once

#include "common.hpp"

namespace fij {

// A key's first kTableCopies tuples (and some more where they spread over two
// buckets) take slots; the others are added up in a side table, one entry {key,
// count, sum} per key, within kCopyEntries entries from the key's place, or take
// slots after all if other keys hold those.  A probe that matches kTableCopies
// slots looks there too.  With every copy in a slot of its own, c copies of a
// key take c^2 / 2 compare-and-swaps in series, and the probes of all keys whose
// bucket lies in the run walk it: 12,000 int32 tuples, 3,000 of one key, against
// 2^20 took 15.2 ms, 39 us now (24 us if all keys differ); 12,000 with 1 to 7
// copies at random against 2^24 356 us, 215 us now.  Three copies made those 163
// us, but keys of four each 157 instead of 134 us (and 20 % more shared by all
// inserts where buckets are 3/4 full); eight left them at 310.
constexpr uint32_t kTableCopies = 4, kCopyEntries = 8;

// LDS of a table of `slots` slots: keys and values, and a side table of
// slots / 8 entries.
template <typename K>
constexpr uint32_t bucket_table_bytes(uint32_t slots) {
  return slots * 2 * sizeof(K) + slots / 8 * (sizeof(K) == 4 ? 12 : 20);
}

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
// partition share their digit, so the single-pass joins take a key of another
// digit: a null key (-1) then needs no test of its own when it is probed, and
// lanes past a range's end carry a second key of another digit.
// NULLS: free_key is the null key itself, and null keys are kept from probing.
template <typename K, bool NULLS = false>
struct BucketTable {
  typedef K Quad __attribute__((ext_vector_type(4)));
  Quad* keys;      // [buckets]
  Quad* vals;      // [buckets]
  uint32_t shift;  // bits of the key's word below the bucket index
  uint32_t mask;   // buckets - 1
  KeyMul mul;      // of the word (kBucketMul when NULLS)
  K free_key;
  // the side table, [buckets / 2]: sums of values (int32: at most 2^14 values of
  // 32 bits below bit 46 and their count above it), keys, counts (int64)
  uint64_t* copy_sums;
  K* copy_keys;
  uint32_t* copy_counts;

  // A table of at most `slots` slots (a power of two, at least 256) in `lds`,
  // of 2^lg buckets; hashed: for keys that share the top `bits` bits of their
  // word as digit (not when NULLS).
  __device__ __forceinline__ BucketTable(uint64_t* lds, uint32_t slots, uint32_t lg, K free, bool hashed = false,
                                         uint32_t bits = 0)
      : keys(reinterpret_cast<Quad*>(lds)), vals(keys + slots / 4), shift(32u - lg),
        mask((1u << lg) - 1u), mul(hashed ? KeyMul{kDigitMul.lo << bits, kDigitMul.hi << bits} : kBucketMul),
        free_key(free),
        copy_sums(reinterpret_cast<uint64_t*>(vals + slots / 4)), copy_keys(reinterpret_cast<K*>(copy_sums + slots / 8)),
        copy_counts(reinterpret_cast<uint32_t*>(copy_keys + slots / 8)) {}
  // log2 of the buckets for n tuples: at most 1/4 full where `slots` allow it.
  static __device__ __forceinline__ uint32_t lg_buckets(uint32_t slots, uint32_t n) {
    return min(29u - static_cast<uint32_t>(__builtin_clz(slots)), max(6u, 32u - static_cast<uint32_t>(__builtin_clz(n | 1u))));
  }
  // Frees every slot (all threads; a barrier follows).
  __device__ __forceinline__ void clear() const {
    const Quad free{free_key, free_key, free_key, free_key};
    for (uint32_t i = threadIdx.x; i <= mask; i += blockDim.x) keys[i] = free;
    for (uint32_t i = threadIdx.x; i <= mask / 4; i += blockDim.x) reinterpret_cast<uint4*>(copy_sums)[i] = make_uint4(0, 0, 0, 0);
    for (uint32_t i = threadIdx.x; i <= mask / 8; i += blockDim.x) {
      reinterpret_cast<Quad*>(copy_keys)[i] = free;
      if constexpr (sizeof(K) == 8) reinterpret_cast<uint4*>(copy_counts)[i] = make_uint4(0, 0, 0, 0);
    }
  }
  __device__ __forceinline__ uint32_t bucket(K key) const {
    return key_word<K>(key, NULLS ? kBucketMul : mul) >> shift;
  }
  // Puts the key into a slot if it is free; returns what the slot held.
  __device__ __forceinline__ K take(K* slot, K key) const {
    if constexpr (sizeof(K) == 8)
      return static_cast<K>(atomicCAS(reinterpret_cast<unsigned long long*>(slot), static_cast<unsigned long long>(free_key),
                                      static_cast<unsigned long long>(key)));
    else
      return static_cast<K>(atomicCAS(reinterpret_cast<unsigned int*>(slot), static_cast<unsigned int>(free_key),
                                      static_cast<unsigned int>(key)));
  }
  // Returns whether an equal key was passed.  The first bucket's slots are
  // tried one by one; beyond, buckets are read before a slot is tried.
  __device__ __forceinline__ bool insert(K key, K val) const {
    const uint32_t b = bucket(key);
    uint32_t same = 0;
    for (uint32_t i = 0; i < 4; ++i) {
      const K prev = take(reinterpret_cast<K*>(keys + b) + i, key);
      if (prev == free_key) {
        reinterpret_cast<K*>(vals + b)[i] = val;
        return same != 0;
      }
      same += prev == key ? 1u : 0u;
    }
    return insert_far((b + 1) & mask, same, key, val);
  }
  // ... from bucket b on, behind `same` copies of the key.
  __device__ __forceinline__ bool insert_far(uint32_t b, uint32_t same, K key, K val) const {
    bool room = true;  // in the key's part of the side table
    for (;;) {
      if (same >= kTableCopies && room) {
        if (insert_copy(key, val)) return true;
        room = false;
      }
      const Quad k = keys[b];
      if (k.w == free_key) {
        const uint32_t s = k.x == free_key ? 0u : k.y == free_key ? 1u : k.z == free_key ? 2u : 3u;
        if (take(reinterpret_cast<K*>(keys + b) + s, key) != free_key) continue;  // the bucket is read again
        reinterpret_cast<K*>(vals + b)[s] = val;
        return same != 0 || k.x == key || k.y == key || k.z == key;
      }
      same += (k.x == key ? 1u : 0u) + (k.y == key ? 1u : 0u) + (k.z == key ? 1u : 0u) + (k.w == key ? 1u : 0u);
      b = (b + 1) & mask;
    }
  }
  // False if other keys hold all entries where this one may be.
  __device__ __forceinline__ bool insert_copy(K key, K val) const {
    uint32_t s = bucket(key) / 2;
    for (uint32_t i = 0; i < kCopyEntries; ++i, s = (s + 1) & (mask / 2)) {
      const K prev = take(copy_keys + s, key);
      if (prev != free_key && prev != key) continue;
      const uint64_t v = static_cast<uint64_t>(static_cast<int64_t>(val));
      atomicAdd(reinterpret_cast<unsigned long long*>(copy_sums + s),
                static_cast<unsigned long long>(sizeof(K) == 4 ? v + (1ull << 46) : v));
      if constexpr (sizeof(K) == 8) atomicAdd(copy_counts + s, 1u);
      return true;
    }
    return false;
  }
  // The matches of a key with kTableCopies tuples in slots beyond those.
  __device__ __forceinline__ void probe_copies(K key, K pay, uint64_t& cnt, uint64_t& sb, uint64_t& sp) const {
    uint32_t s = bucket(key) / 2;
    for (uint32_t i = 0; i < kCopyEntries; ++i, s = (s + 1) & (mask / 2)) {
      const K k = copy_keys[s];
      if (k == free_key) return;
      if (k != key) continue;
      uint64_t sum = copy_sums[s], n;
      if constexpr (sizeof(K) == 4) {
        const uint64_t low = static_cast<uint64_t>(static_cast<int64_t>(sum << 18) >> 18);
        n = (sum - low) >> 46;
        sum = low;
      } else {
        n = copy_counts[s];
      }
      cnt += n;
      sb += sum;
      sp += n * static_cast<uint64_t>(static_cast<int64_t>(pay));
      return;
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
        if (more[i]) probe_from<true>((at[i] + 1) & mask, key[i], pay[i], cnt, sb, sp);
    }
  }
  // Probes from bucket b to the first bucket with a free slot: every match
  // counts (not for a null key when NULLS).  UNIQUE: a key occurs once.
  template <bool UNIQUE>
  __device__ __forceinline__ void probe_from(uint32_t b, K key, K pay, uint64_t& cnt, uint64_t& sb,
                                             uint64_t& sp) const {
    const uint32_t before = static_cast<uint32_t>(cnt);
    for (;; b = (b + 1) & mask) {
      const Quad k = keys[b];
      const uint32_t m = (k.x == key ? 1u : 0u) | (k.y == key ? 2u : 0u) | (k.z == key ? 4u : 0u) |
                         (k.w == key ? 8u : 0u);
      if (m) {
        if constexpr (UNIQUE) {
          cnt += 1;
          return add(reinterpret_cast<const K*>(vals)[4 * b + (m >> 1) - (m >> 3)], pay, sb, sp);
        }
        const Quad v = vals[b];
        cnt += __popc(m);
        if (m & 1u) add(v.x, pay, sb, sp);
        if (m & 2u) add(v.y, pay, sb, sp);
        if (m & 4u) add(v.z, pay, sb, sp);
        if (m & 8u) add(v.w, pay, sb, sp);
      }
      if (k.w == free_key) break;
    }
    if (!UNIQUE && static_cast<uint32_t>(cnt) - before >= kTableCopies) probe_copies(key, pay, cnt, sb, sp);
  }
  // Probes N tuples of a lane; unique (uniform): no build key occurs twice.
  template <uint32_t N>
  __device__ __forceinline__ void probe(bool unique, const K (&key)[N], const K (&pay)[N], uint32_t& wave_cnt,
                                        uint64_t& cnt, uint64_t& sb, uint64_t& sp) const {
    if (unique) return probe_unique(key, pay, wave_cnt, cnt, sb, sp);
#pragma unroll
    for (uint32_t i = 0; i < N; ++i)
      if (!NULLS || key[i] != free_key) probe_from<false>(bucket(key[i]), key[i], pay[i], cnt, sb, sp);
  }
};

}  // namespace fij
