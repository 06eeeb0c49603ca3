// Host side of the batched radix-join execution method (fij_join_plan_*).
//
// A plan owns every intermediate buffer of one join shape (allocated once,
// as the reference allocates its partitions and stream states before the
// timed phases: radix-join/src/execution_methods/gpu_radix_join.rs:153-205,
// :307-396), so that executing it launches kernels only.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/fij.h"
#include "internal.hpp"
#include "pipeline.hpp"

namespace fij {
fij_status set_error(fij_status s, const char* msg);
}

using namespace fij;

struct fij_join_plan {
  fij_join_plan_config cfg;
  KeyType kt;
  PipelineDevice d;
  PipelineDevice one;  // two-pass plans: the same buffers as a single pass of kOnePassBits
  bool two_pass;       // the plan has pass-2 buffers
  uint32_t max_tiles[2];
  uint32_t sort2_grid;
  uint32_t join_grid;
  uint32_t g1_cap;
  uint32_t block1;
  uint32_t lds_total;
  std::vector<void*> allocs;
  uint32_t cus;
  uint32_t clock_khz;  // rate of the device clock the phases are stamped with
  uint32_t* done;      // [kDoneWords] finished blocks, zero between joins
  uint32_t* hashed;    // single-pass joins: whether the last one's digits were hashed
  // what the last enqueued join wrote or did not launch
  struct Host {
    JoinAggregate result;
    uint64_t stamps[kStamps];
  };
  Host* host;
  enum class Timed { None, Phases, OneLaunch } timed;
};

namespace {

fij_status plan_fail(fij_status s, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  return set_error(s, buf);
}

fij_status hip_fail(hipError_t e, const char* what) {
  return plan_fail(e == hipErrorOutOfMemory ? FIJ_OUT_OF_MEMORY : FIJ_DEVICE_ERROR, "%s: %s", what,
                   hipGetErrorString(e));
}

#define PLAN_HIP(expr)                                \
  do {                                                \
    hipError_t e_ = (expr);                           \
    if (e_ != hipSuccess) return hip_fail(e_, #expr); \
  } while (0)

template <typename T>
fij_status alloc(fij_join_plan* p, T** out, uint64_t count) {
  void* ptr = nullptr;
  hipError_t e = hipMalloc(&ptr, std::max<uint64_t>(count, 1) * sizeof(T));
  if (e != hipSuccess) return hip_fail(e, "hipMalloc");
  p->allocs.push_back(ptr);
  *out = static_cast<T*>(ptr);
  return FIJ_OK;
}

void release(fij_join_plan* p) {
  for (void* a : p->allocs) (void)hipFree(a);
  p->allocs.clear();
  if (p->host) (void)hipHostFree(p->host);
}

// Partitions the pass-1 buffers are sized for: the plan's own, or those of
// the single pass that a two-pass plan may take.
uint32_t pass1_fanout(const fij_join_plan* p) {
  return p->d.bits2 ? std::max(p->d.F1, 1u << kOnePassBits) : p->d.F1;
}

fij_status alloc_side(fij_join_plan* p, PipelineSide& s, uint64_t n, uint32_t tiles) {
  const hipError_t e =
      alloc_pipeline_side(s, p->kt, n, pass1_fanout(p), p->d.F2, p->d.G1, p->two_pass, tiles, p->allocs);
  return e == hipSuccess ? FIJ_OK : hip_fail(e, "hipMalloc");
}

}  // namespace

extern "C" {

fij_status fij_join_plan_bits(fij_type type, uint64_t build_len, uint64_t probe_len, uint32_t* radix_bits_1,
                              uint32_t* radix_bits_2) {
  if (!radix_bits_1 || !radix_bits_2) return plan_fail(FIJ_INVALID_ARGUMENT, "invalid argument");
  if (type != FIJ_TYPE_I32 && type != FIJ_TYPE_I64) return plan_fail(FIJ_INVALID_ARGUMENT, "unknown type");
  const KeyType kt = type == FIJ_TYPE_I32 ? KeyType::I32 : KeyType::I64;
  if (one_pass_fits(kt, build_len)) {
    *radix_bits_1 = kOnePassBits;
    *radix_bits_2 = 0;
    return FIJ_OK;
  }
  // a probe side 16 times the build side or longer: items of about a third
  // of a block table, joined from block tables over long runs
  if (probe_len >= 16 * build_len) {
    *radix_bits_1 = kOnePassBits;
    *radix_bits_2 = probe_heavy_bits2(kt, build_len);
    return FIJ_OK;
  }
  uint32_t small = 0;
  return fij_join_autotune(type, build_len, probe_len, &small, radix_bits_1, radix_bits_2);
}

fij_status fij_join_plan_create(const fij_join_plan_config* cfg, fij_join_plan** out) {
  if (!cfg || !out) return plan_fail(FIJ_INVALID_ARGUMENT, "NULL argument");
  if (cfg->type != FIJ_TYPE_I32 && cfg->type != FIJ_TYPE_I64) return plan_fail(FIJ_INVALID_ARGUMENT, "unknown type");
  if (cfg->radix_bits_1 < 1 || cfg->radix_bits_1 > 12)
    return plan_fail(FIJ_UNSUPPORTED, "pass-1 radix bits must be in [1, 12]");
  if (cfg->radix_bits_2 > 12) return plan_fail(FIJ_UNSUPPORTED, "pass-2 radix bits must be in [0, 12]");
  const KeyType kt = cfg->type == FIJ_TYPE_I32 ? KeyType::I32 : KeyType::I64;
  if (cfg->radix_bits_1 + cfg->radix_bits_2 > 8 * key_bytes(kt))
    return plan_fail(FIJ_INVALID_ARGUMENT, "more radix bits than key bits");
  int dev = 0;
  PLAN_HIP(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  PLAN_HIP(hipGetDeviceProperties(&prop, dev));
  int optin = 0;
  uint32_t lds_total = static_cast<uint32_t>(prop.sharedMemPerBlock);
  if (hipDeviceGetAttribute(&optin, hipDeviceAttributeSharedMemPerBlockOptin, dev) == hipSuccess && optin > 0)
    lds_total = std::max<uint32_t>(lds_total, static_cast<uint32_t>(optin));
  const uint32_t cus = static_cast<uint32_t>(prop.multiProcessorCount);

  int clock_khz = 0;
  PLAN_HIP(hipDeviceGetAttribute(&clock_khz, hipDeviceAttributeWallClockRate, dev));

  fij_join_plan* p = new fij_join_plan();
  p->clock_khz = static_cast<uint32_t>(std::max(clock_khz, 1));
  p->host = nullptr;
  p->timed = fij_join_plan::Timed::None;
  p->cus = cus;
  p->cfg = *cfg;
  p->kt = kt;
  p->lds_total = lds_total;
  std::memset(&p->d, 0, sizeof(p->d));
  p->d.bits1 = cfg->radix_bits_1;
  p->d.bits2 = cfg->radix_bits_2;
  p->d.F1 = 1u << cfg->radix_bits_1;
  p->d.F2 = 1u << cfg->radix_bits_2;
  p->d.G1 = cfg->pass1_chunks ? cfg->pass1_chunks : cus;
  p->g1_cap = p->d.G1;
  p->d.pad = pad_tuples(kt);
  p->d.tile2 = pipeline_tile2(kt);
  p->d.sides = 3;
  p->block1 = cfg->pass1_block ? std::min<uint32_t>(cfg->pass1_block, 1024) : 1024;
  p->join_grid = cfg->join_blocks ? cfg->join_blocks : cus * 2;
  // aggregates: the joins with small tables keep more than two blocks per CU
  p->d.agg_len = cfg->join_blocks ? cfg->join_blocks : cus * 4;
  p->two_pass = p->d.bits2 && !one_pass_always(kt, cfg->build_len, cfg->probe_len);
  fij_status st = FIJ_OK;
  const uint64_t lens[2] = {cfg->build_len, cfg->probe_len};
  for (int rel = 0; rel < 2 && st == FIJ_OK; ++rel) {
    uint64_t chunk = 0;
    if (cfg->pass1_chunks) st = fij_input_chunk_size(static_cast<fij_type>(cfg->type), lens[rel], p->d.G1, &chunk);
    if (st == FIJ_OK && cfg->pass1_chunks && chunk * (p->d.G1 - 1) > lens[rel])
      st = plan_fail(FIJ_INVALID_ARGUMENT, "relation of %llu tuples is too short for %u chunks",
                     static_cast<unsigned long long>(lens[rel]), p->d.G1);
    // the scatter addresses a chunk's writes relative to its first partition
    // with 32-bit offsets; in the contiguous layout they span the relation
    if (st == FIJ_OK && !pass1_offsets_fit(kt, lens[rel], p->d.F1))
      st = plan_fail(FIJ_INTEGER_OVERFLOW, "relation of %llu tuples exceeds the 32-bit pass-1 offsets",
                     static_cast<unsigned long long>(lens[rel]));
    p->max_tiles[rel] = p->d.bits2 ? static_cast<uint32_t>((lens[rel] + p->d.tile2 - 1) / p->d.tile2 + p->d.F1) : 0;
  }
  if (st == FIJ_OK && p->d.bits2 && pipeline_sort2_lds(kt, p->d.F2) > lds_total)
    st = plan_fail(FIJ_UNSUPPORTED, "pass-2 tile does not fit LDS for this fanout / chunk count");
  // pass 2: one persistent block per compute unit (its LDS tile fills the CU)
  p->sort2_grid = p->d.bits2 ? std::min<uint32_t>(cus, p->max_tiles[0] + p->max_tiles[1]) : 0;
  if (st == FIJ_OK) st = alloc_side(p, p->d.build, cfg->build_len, p->max_tiles[0]);
  if (st == FIJ_OK) st = alloc_side(p, p->d.probe, cfg->probe_len, p->max_tiles[1]);
  if (st == FIJ_OK) st = alloc(p, &p->d.work_counter, kJoinCounterWords);
  const uint64_t items = static_cast<uint64_t>(p->d.F1) * (p->d.bits2 ? p->d.F2 : 1);
  // work units of deferred items: at most one per item plus one per 65536
  // probe tuples
  p->d.unit_cap = static_cast<uint32_t>(items + cfg->probe_len / 65536 + 1);
  if (st == FIJ_OK && p->two_pass) st = alloc(p, &p->d.overflow, items);
  if (st == FIJ_OK && p->two_pass) st = alloc(p, &p->d.units, p->d.unit_cap);
  if (st == FIJ_OK) st = alloc(p, &p->d.part_units, part_unit_cap(pass1_fanout(p), cfg->probe_len));
  // the deferred-item flags start at zero (complete before any stream uses
  // them); every join leaves them at zero
  if (st == FIJ_OK && p->two_pass &&
      (hipMemset(p->d.overflow, 0, items) != hipSuccess || hipDeviceSynchronize() != hipSuccess))
    st = plan_fail(FIJ_DEVICE_ERROR, "clearing the deferred-item flags failed");
  // HBM hash tables of deferred items with large build sides: an arena of
  // 2^k slots, twice the build relation (at most 2^26 slots), every word all
  // ones; one table per item at most, each at least 256 slots
  {
    uint64_t slots = 1024;
    while (slots < 2 * cfg->build_len && slots < (1ull << 26)) slots <<= 1;
    p->d.hbm_cap = static_cast<uint32_t>(slots);
    p->d.big_cap = static_cast<uint32_t>(std::min<uint64_t>(items, slots / 256));
    p->d.hbm_unit_cap =
        static_cast<uint32_t>(2ull * p->d.big_cap + (cfg->build_len + cfg->probe_len) / kTableUnitMin + 2);
    // (the block counters are cleared with the arena)
    if (st == FIJ_OK) st = alloc(p, &p->done, kDoneWords);
    if (st == FIJ_OK) st = alloc(p, &p->hashed, 1);
    if (st == FIJ_OK && hipMemset(p->done, 0, kDoneWords * sizeof(uint32_t)) != hipSuccess)
      st = plan_fail(FIJ_DEVICE_ERROR, "clearing the block counters failed");
    void* arena = nullptr;
    if (st == FIJ_OK && hipMalloc(&arena, slots * tuple_bytes(kt)) != hipSuccess)
      st = plan_fail(FIJ_OUT_OF_MEMORY, "cannot allocate the HBM hash-table arena");
    if (arena) p->allocs.push_back(arena);
    p->d.hbm_table = arena;
    if (st == FIJ_OK) st = alloc(p, &p->d.big, p->d.big_cap);
    if (st == FIJ_OK) st = alloc(p, &p->d.hbm_units, p->d.hbm_unit_cap);
    if (st == FIJ_OK && (hipMemset(arena, 0xFF, slots * tuple_bytes(kt)) != hipSuccess ||
                         hipDeviceSynchronize() != hipSuccess))
      st = plan_fail(FIJ_DEVICE_ERROR, "initialising the HBM hash-table arena failed");
  }
  if (st == FIJ_OK) st = alloc(p, &p->d.aggregates, p->d.agg_len);
  if (st == FIJ_OK && hipHostMalloc(reinterpret_cast<void**>(&p->host), sizeof(fij_join_plan::Host),
                                    hipHostMallocDefault) != hipSuccess)
    st = plan_fail(FIJ_OUT_OF_MEMORY, "cannot allocate the pinned result");
  if (st == FIJ_OK) std::memset(p->host, 0, sizeof(fij_join_plan::Host));
  if (st != FIJ_OK) {
    release(p);
    delete p;
    return st;
  }
  p->one = p->d;
  p->one.bits1 = kOnePassBits;
  p->one.bits2 = 0;
  p->one.F1 = 1u << kOnePassBits;
  p->one.F2 = 1;
  // (wider fanouts have no line rings)
  p->one.hashed = p->hashed;
  p->d.hashed = p->d.bits2 || p->d.bits1 > kOnePassBits ? nullptr : p->hashed;
  *out = p;
  return FIJ_OK;
}

fij_status fij_join_plan_destroy(fij_join_plan* plan) {
  if (!plan) return FIJ_OK;
  release(plan);
  delete plan;
  return FIJ_OK;
}

}  // extern "C"

namespace {

// Enqueues one join of the plan's shape over columns of n_b and n_p tuples
// (at most the plan's lengths): launches only, so it can be captured.  The
// result goes to *device_result or, timed, with the phases' stamps to the
// plan's pinned memory (device_result == nullptr).
fij_status enqueue_join(fij_join_plan* p, const void* build_keys, const void* build_pays, uint64_t n_b,
                        const void* probe_keys, const void* probe_pays, uint64_t n_p,
                        fij_join_aggregate* device_result, hipStream_t st) {
  if (n_b > p->cfg.build_len || n_p > p->cfg.probe_len)
    return plan_fail(FIJ_INVALID_ARGUMENT, "join of %llu x %llu tuples exceeds the plan's %llu x %llu",
                     static_cast<unsigned long long>(n_b), static_cast<unsigned long long>(n_p),
                     static_cast<unsigned long long>(p->cfg.build_len),
                     static_cast<unsigned long long>(p->cfg.probe_len));
  if ((n_b && (!build_keys || !build_pays)) || (n_p && (!probe_keys || !probe_pays)))
    return plan_fail(FIJ_INVALID_ARGUMENT, "NULL input column");
  const size_t kb = key_bytes(p->kt);
  for (const void* c : {build_keys, build_pays, probe_keys, probe_pays})
    if (c && reinterpret_cast<uintptr_t>(c) % kb)
      return plan_fail(FIJ_INVALID_ARGUMENT, "input columns must be aligned to their element size");
  using Timed = fij_join_plan::Timed;
  JoinAggregate* result = device_result ? reinterpret_cast<JoinAggregate*>(device_result) : &p->host->result;
  uint64_t* stamps = device_result ? nullptr : p->host->stamps;
  if (n_b <= table_join_tuples(p->kt)) {
    // the whole build side fits a block's LDS table: no partitioning
    const TableJoin j{build_keys, build_pays, probe_keys, probe_pays, n_b, n_p, p->d.aggregates, p->done, result, stamps};
    PLAN_HIP(launch_table_join(p->kt, j, p->cus, p->d.agg_len, st));
    if (!device_result) p->timed = Timed::OneLaunch;
    return FIJ_OK;
  }
  // A two-pass plan's join of a build side that a single pass leaves in
  // partitions of at most two table fills is run in one: the probe tuples are
  // read once more instead of partitioned once more.
  PipelineDevice& d = p->d.bits2 && one_pass_join(p->kt, n_b, n_p) ? p->one : p->d;
  d.stamps = stamps;
  d.build.keys = build_keys;
  d.build.pays = build_pays;
  d.probe.keys = probe_keys;
  d.probe.pays = probe_pays;
  d.build.n = n_b;
  d.probe.n = n_p;
  d.build.padded_len1 = n_b + static_cast<uint64_t>(d.F1) * d.pad;
  d.probe.padded_len1 = n_p + static_cast<uint64_t>(d.F1) * d.pad;
  // pass-1 chunks: one block per compute unit, shared by the sides; a chunk
  // count that the caller chose holds for each side
  if (p->cfg.pass1_chunks) {
    d.build.g1 = pass1_chunks(p->kt, n_b, p->g1_cap);
    d.probe.g1 = pass1_chunks(p->kt, n_p, p->g1_cap);
  } else {
    split_chunks(p->kt, n_b, n_p, p->g1_cap, &d.build.g1, &d.probe.g1);
  }
  d.big_block_tables = d.bits2 ? 0u : big_block_tables_for(p->kt, n_b, d.F1);
  PLAN_HIP(enqueue_pass1_prefix_sum(d, p->kt, p->block1, st));
  PLAN_HIP(enqueue_pass1_scatter(d, p->kt, p->block1, p->lds_total, st));
  if (d.bits2) {
    PLAN_HIP(launch_pipeline_plan(d, st));
    PLAN_HIP(launch_pipeline_sort2(d, p->kt, p->sort2_grid, st));
    PLAN_HIP(launch_pipeline_join(d, p->kt, false, p->join_grid, st));
    PLAN_HIP(launch_pipeline_join(d, p->kt, true, p->join_grid, st));
    PLAN_HIP(launch_sum_aggregates(d.aggregates, d.agg_len, result, stamps, st));
  } else {
    d.result = result;
    d.done = p->done;
    PLAN_HIP(launch_one_pass_plan(d, p->kt, nullptr, 1, st));
    PLAN_HIP(launch_one_pass_join(d, p->kt, p->join_grid, st));
  }
  if (!device_result) p->timed = Timed::Phases;
  return FIJ_OK;
}

}  // namespace

extern "C" {

fij_status fij_join_plan_enqueue(fij_join_plan* p, const void* build_keys, const void* build_pays,
                                 const void* probe_keys, const void* probe_pays, void* stream) {
  if (!p) return plan_fail(FIJ_INVALID_ARGUMENT, "plan is NULL");
  return enqueue_join(p, build_keys, build_pays, p->cfg.build_len, probe_keys, probe_pays, p->cfg.probe_len,
                      nullptr, static_cast<hipStream_t>(stream));
}

fij_status fij_join_plan_enqueue_sized(fij_join_plan* p, const void* build_keys, const void* build_pays,
                                       uint64_t build_len, const void* probe_keys, const void* probe_pays,
                                       uint64_t probe_len, fij_join_aggregate* device_result, void* stream) {
  if (!p || !device_result) return plan_fail(FIJ_INVALID_ARGUMENT, "plan or result is NULL");
  return enqueue_join(p, build_keys, build_pays, build_len, probe_keys, probe_pays, probe_len, device_result,
                      static_cast<hipStream_t>(stream));
}

fij_status fij_join_plan_result(fij_join_plan* p, void* stream, fij_join_aggregate* result, fij_join_timing* timing) {
  if (!p) return plan_fail(FIJ_INVALID_ARGUMENT, "plan is NULL");
  PLAN_HIP(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
  const fij_join_plan::Host& h = *p->host;
  if (result) *result = fij_join_aggregate{h.result.count, h.result.sum_build, h.result.sum_probe};
  if (timing) {
    using Timed = fij_join_plan::Timed;
    if (p->timed == Timed::None) return plan_fail(FIJ_DEVICE_ERROR, "no join of this plan has been enqueued");
    auto ms = [&](uint32_t from, uint32_t to) {
      return static_cast<float>(static_cast<double>(h.stamps[to] - h.stamps[from]) / p->clock_khz);
    };
    *timing = fij_join_timing{};
    timing->total_ms = ms(0, 5);
    if (p->timed == Timed::OneLaunch) {
      timing->join_ms = timing->build_probe_ms = timing->total_ms;
    } else {
      timing->prefix_sum_ms = ms(0, 1);
      timing->partition_ms = ms(1, 2);
      timing->join_ms = ms(2, 5);
      timing->pass2_ms = ms(2, 3);
      timing->build_probe_ms = ms(3, 4);
      timing->deferred_ms = ms(4, 5);
    }
  }
  return FIJ_OK;
}

fij_status fij_join_plan_execute(fij_join_plan* p, const void* build_keys, const void* build_pays,
                                 const void* probe_keys, const void* probe_pays, fij_join_aggregate* result,
                                 fij_join_timing* timing, void* stream) {
  fij_status s = fij_join_plan_enqueue(p, build_keys, build_pays, probe_keys, probe_pays, stream);
  if (s != FIJ_OK) return s;
  return fij_join_plan_result(p, stream, result, timing);
}

fij_status fij_join_plan_device_bytes(const fij_join_plan* p, uint64_t* bytes) {
  if (!p || !bytes) return plan_fail(FIJ_INVALID_ARGUMENT, "NULL argument");
  const uint64_t tb = tuple_bytes(p->kt), F1 = pass1_fanout(p);
  const uint64_t lens[2] = {p->cfg.build_len, p->cfg.probe_len};
  uint64_t total = 0;
  for (uint64_t n : lens) {
    total += (n + F1 * p->d.pad) * tb + F1 * (p->d.G1 + 1ull) * 8;
    total += F1 * p->d.G1 * 4 + scan_state_words(F1) * 8 + F1 * 4 + (F1 + 1) * 12;
    if (p->two_pass) total += n * tb;
  }
  total += part_unit_cap(F1, p->cfg.probe_len) * sizeof(PartUnit);
  if (p->two_pass) total += (static_cast<uint64_t>(p->max_tiles[0]) + p->max_tiles[1] + 2) * p->d.F2 * 4;
  total += static_cast<uint64_t>(p->d.hbm_cap) * tb + (static_cast<uint64_t>(p->d.big_cap) + p->d.hbm_unit_cap) * 16;
  *bytes = total;
  return FIJ_OK;
}

}  // extern "C"
