"""The rules that cut single-pass joins into work units, compiled for the host:
up to the longest partitions that a plan accepts (nearly 2^32 tuples)."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include "one_pass_rules.hpp"
using namespace fij;
int main(int argc, char** argv) {
  if (argc == 2) {  // tuples of a partition with an HBM table: units, tuples of a unit, end of the last
    const uint32_t n = strtoul(argv[1], nullptr, 10), per = table_unit_tuples(n), r = range_count(n, per);
    printf("%u %u %u\\n", r, per, r ? range_end(n, per, r - 1) : 0u);
    return 0;
  }
  if (argc == 6) {  // tuples of a fill, build and probe tuples: units, tuples of a unit
    const uint32_t fill = strtoul(argv[1], nullptr, 10);
    const PartUnits u = part_units_of(strtoul(argv[2], nullptr, 10), strtoul(argv[3], nullptr, 10), fill);
    printf("%u %u\\n", u.units, u.per);
    return 0;
  }
  if (argc == 5) {  // type, build tuples, partitions, big tables: slots, a fill, build tuples joined in LDS
    const KeyType t = argv[1][0] == '0' ? KeyType::I32 : KeyType::I64;
    const bool big = argv[4][0] == '1';
    const uint32_t slots = one_pass_slots(t, strtoull(argv[2], nullptr, 10), strtoull(argv[3], nullptr, 10), big);
    printf("%u %u %u\\n", slots, block_table_fill(t, slots), one_pass_lds_tuples(t, big));
    return 0;
  }
  if (argc == 4) {  // type, build and probe tuples: one pass, always one pass
    const KeyType t = argv[1][0] == '0' ? KeyType::I32 : KeyType::I64;
    const uint64_t b = strtoull(argv[2], nullptr, 10), p = strtoull(argv[3], nullptr, 10);
    printf("%d %d\\n", one_pass_join(t, b, p), one_pass_always(t, b, p));
    return 0;
  }
  for (int i = 1; i + 1 < argc; i += 2) {
    const uint32_t nb = strtoul(argv[i], nullptr, 10), np = strtoul(argv[i + 1], nullptr, 10);
    const PartUnits u = part_units_of(nb, np);
    const uint32_t r = range_count(np, 65536);
    printf("%u %u %u %u\\n", u.units, u.per, r, r ? range_end(np, 65536, r - 1) : 0u);
  }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", os.path.join(REPO, "include"),
                    "-I", os.path.join(REPO, "fast-interconnects_amd", "csrc"), "rules.cpp", "-o", "rules"], cwd=d, check=True)

    def ask(pairs):
        args = [str(x) for p in pairs for x in p]
        out = subprocess.run([str(d / "rules")] + args, check=True, capture_output=True, text=True)
        return [tuple(int(x) for x in line.split()) for line in out.stdout.splitlines()]
    return ask


def test_units_cover_partitions_of_every_length(rules):
    builds = [0, 1, 511, 512, 513, 2048, 4095, 4096, 5000, (1 << 32) - 20_000]
    probes = [0, 1, 8191, 8192, 8193, 65_536, 65_537, 1 << 24, (1 << 32) - 65_536, (1 << 32) - 65_535, (1 << 32) - 20_000,
              (1 << 32) - 514, (1 << 32) - 1]
    pairs = [(b, p) for b in builds for p in probes]
    for (nb, np_), (units, per, ranges, end) in zip(pairs, rules(pairs)):
        assert ranges == -(-np_ // 65_536) and end == np_
        if nb == 0 or np_ == 0:
            assert units == 0
            continue
        assert 1 <= per <= max(8192, min(16 * nb, 65_536))
        assert (units - 1) * per < np_ <= units * per  # no tuple left out, no empty unit
        assert units <= np_ // 8192 + 1


@pytest.mark.parametrize("type,pad", [(0, 16), (1, 8)])
def test_single_pass_offsets_stay_below_2_32(rules, type, pad):
    """A plan of few pass-1 bits accepts relations that 512 padded partitions
    would carry past 2^32: those take two passes."""
    last = (1 << 32) - 2 - 512 * pad * 2
    for build in (20_000, 4_571_136):
        assert rules([(type, build, last)]) == [(1, 1)]
        assert rules([(type, build, last + 1)]) == [(0, 0)]
        assert rules([(type, build, (1 << 32) - 600)]) == [(0, 0)]
    assert rules([(type, 4_571_137, 5_000_000)]) == [(1, 0)]  # by its lengths, not always


@pytest.mark.parametrize("type,fills", [(0, (2304, 4608, 9216)), (1, (1280, 2560, 5120))])
def test_tables_and_their_fills(rules, type, fills):
    """32 KiB tables up to half their slots on average, then 64 KiB ones; and how
    often a partition may fill them before it takes an HBM table."""
    half = 2048 >> type
    for build, big, at, most in ((half << 9, 0, 0, (11, 10)), ((half << 9) + 1, 0, 1, (6, 5)), (1, 1, 2, (6, 5))):
        [(slots, fill, lds)] = rules([(type, build, 512, big)])
        assert slots == half << at + 1 and fill == fills[at]
        assert -(-lds // fill) == most[type]


def test_units_of_partitions_with_hbm_tables(rules):
    """At most as many as a plan has room for (one per 4,096 tuples and one), and
    at least 32 of a long range: one block probed 65,536 tuples in 0.3 ms."""
    for n in (1, 4095, 4096, 4097, 128 * 4096 - 1, 128 * 4096 + 127, 240_000, 128 * 65_536, 128 * 65_536 + 1, (1 << 32) - 20_000,
              (1 << 32) - 1):
        [(units, per, end)] = rules([(n,)])
        assert end == n and (units - 1) * per < n <= units * per
        assert units <= n // 4096 + 1
        assert units >= min(32, n // 4096)


def test_units_of_partitions_of_many_fills_are_shorter(rules):
    """... down to 8,192 probe tuples; those of one or two fills are not."""
    for fill in (1280, 9216):
        for fills in (1, 2, 3, 5, 11, 400):
            nb = fill * fills
            for np_ in (1, 8193, 240_000, 1 << 24, (1 << 32) - 20_000):
                [(units, per)] = rules([(fill, nb, np_, "", "")])
                longest = max(8192, min(16 * nb, 65_536 if fills <= 2 else 131_072 // fills))
                assert longest // 2 < per <= longest or np_ <= longest
                assert (units - 1) * per < np_ <= units * per and units <= np_ // 8192 + 1
