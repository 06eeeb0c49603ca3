"""Out-of-core joins whose keys are in host memory take no more device memory
than those whose keys are on the device already: their key copies give way."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "fast-interconnects_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# fij_ooc_join on tests/hip_stand_in.cpp with kernels that only leave even
# partitions: whether it succeeds within each limit of device memory, and its peak
PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "internal.hpp"
#include "pipeline.hpp"
extern uint64_t memory_limit, memory_used, memory_peak;
extern hipMemoryType column_type;
namespace fij {
fij_status set_error(fij_status s, const char*) { return s; }
void cpu_partition_contiguous(KeyType, const void*, const void*, uint64_t, uint32_t, uint32_t, uint32_t, void*, uint64_t*) {}
HistParams hist_params(KeyType, const void*, uint64_t n, uint32_t, uint32_t, uint32_t, uint32_t*, uint64_t*) {
  HistParams p{};
  p.n = n;
  return p;
}
void sample_build_keys(HistParams&, const void*, uint64_t, uint32_t*) {}
static uint64_t lengths[2];
hipError_t launch_hist_pair(KeyType, const HistParams& a, const HistParams& b, uint32_t, uint32_t, bool, uint32_t, hipStream_t) {
  lengths[0] = a.n, lengths[1] = b.n;
  return hipSuccess;
}
hipError_t launch_offsets_scan(const OffsetsScan& a, const OffsetsScan* b, hipStream_t) {
  for (int r = 0; r < 2; ++r) {
    const OffsetsScan& s = r ? *b : a;
    for (uint64_t p = 0; p < s.fanout; ++p) s.offsets[p] = lengths[r] * p / s.fanout + (p + 1) * s.pad;
  }
  return hipSuccess;
}
hipError_t launch_partition(const PartitionLaunch&, hipStream_t) { return hipSuccess; }
hipError_t launch_partition_pair(const PartitionLaunch&, const PartitionLaunch&, hipStream_t) { return hipSuccess; }
hipError_t launch_pipeline_join(const PipelineDevice&, KeyType, bool, uint32_t, hipStream_t) { return hipSuccess; }
hipError_t launch_pipeline_plan(const PipelineDevice&, hipStream_t) { return hipSuccess; }
hipError_t launch_pipeline_sort2(const PipelineDevice&, KeyType, uint32_t, hipStream_t) { return hipSuccess; }
hipError_t launch_sum_aggregates(const JoinAggregate*, uint32_t, JoinAggregate*, uint64_t*, hipStream_t) { return hipSuccess; }
size_t pipeline_sort2_lds(KeyType, uint32_t) { return 1024; }
uint32_t pipeline_tile2(KeyType) { return 8192; }
}  // namespace fij
int main(int argc, char** argv) {
  const uint64_t nb = strtoull(argv[1], nullptr, 10), np = strtoull(argv[2], nullptr, 10);
  fij_ooc_config c{};
  c.type = FIJ_TYPE_I64;
  c.radix_bits_1 = 5, c.radix_bits_2 = 6;
  c.cache_bytes = strtoull(argv[3], nullptr, 10);
  c.staging_tuples = strtoull(argv[4], nullptr, 10);
  std::vector<int64_t> column(np);
  auto join = [&](hipMemoryType t, uint64_t limit) {
    column_type = t, memory_limit = limit, memory_peak = 0;
    fij_join_aggregate r;
    const int s = fij_ooc_join(&c, column.data(), column.data(), nb, column.data(), column.data(), np, &r, nullptr);
    if (memory_used != 0) abort();
    return s;
  };
  if (join(hipMemoryTypeDevice, ~0ull) != FIJ_OK) abort();
  const uint64_t most = memory_peak;
  for (int i = 1; i <= 40; ++i) {
    const uint64_t limit = most * i / 32;
    const int dev = join(hipMemoryTypeDevice, limit), host = join(hipMemoryTypeHost, limit);
    printf("%d %d\\n", dev, host);
  }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("ooc")
    (d / "main.cpp").write_text(PROGRAM)
    flags = ["-x", "hip", "--cuda-host-only", "-fPIC", "-std=c++17", "-I", os.path.join(REPO, "include"), "-I", CSRC, "-w"]
    sources = [str(d / "main.cpp"), os.path.join(REPO, "tests", "hip_stand_in.cpp")] + \
        [os.path.join(CSRC, f) for f in ("ooc.cpp", "pipeline_host.cpp")]
    objects = []
    for s in sources:
        objects.append(str(d / os.path.basename(s)) + ".o")
        subprocess.run([HIPCC] + flags + ["-c", s, "-o", objects[-1]], check=True)
    subprocess.run(["g++"] + objects + ["-o", str(d / "ooc"), "-lpthread"], check=True)
    return str(d / "ooc")


@pytest.mark.parametrize("cache", [0, 20_000_000, 1 << 40])
def test_host_keys_need_no_more_memory(program, cache):
    out = subprocess.run([program, "500000", "1500000", str(cache), "1000000"], check=True, capture_output=True, text=True)
    lines = [line.split() for line in out.stdout.splitlines()]
    assert len(lines) == 40 and lines[-1] == ["0", "0"] and lines[0][0] != "0"
    assert all(dev == host for dev, host in lines)
