"""The classes of a batch's single-pass joins, compiled for the host: the tables
that a class's joins are joined in hold what it promises."""
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
  const KeyType t = argv[1][0] == '0' ? KeyType::I32 : KeyType::I64;
  for (int i = 2; i < argc; ++i) {
    const OnePassClass c = one_pass_class(t, strtoull(argv[i], nullptr, 10));
    const OnePassClass longest = one_pass_class(t, c.build);
    printf("%u %u %d %d\\n", c.bits, c.build, c.big_tables,
           longest.bits == c.bits && longest.build == c.build && longest.big_tables == c.big_tables);
  }
}
"""


@pytest.mark.parametrize("type", [0, 1])
def test_classes(type, tmp_path):
    (tmp_path / "classes.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", os.path.join(REPO, "include"),
                    "-I", os.path.join(REPO, "fast-interconnects_amd", "csrc"), "classes.cpp", "-o", "classes"],
                   cwd=tmp_path, check=True)
    last = (7_077_888, 5_079_040)[type]  # the longest build side that takes a single pass
    edges = [m >> type for m in (1 << 16, 1 << 18, 1 << 20, 1 << 21)]
    sizes = [1, 1000] + [e + k for e in edges for k in (0, 1)] + [3_145_728 >> type, last]
    out = subprocess.run([str(tmp_path / "classes"), str(type)] + [str(n) for n in sizes], check=True, capture_output=True,
                         text=True).stdout.splitlines()
    half_small = (2048, 1024)[type]  # tuples that fill a 32 KiB table half
    two_fills = 2 * (9216, 5120)[type]
    for n, line in zip(sizes, out):
        bits, build, big, closed = (int(x) for x in line.split())
        assert closed and n <= build
        assert bits == (5 if n <= edges[0] else 7 if n <= edges[1] else 9)
        assert big == (n > edges[2])
        if big:
            assert build == (edges[3] if n <= edges[3] else two_fills << 9)
        else:
            assert build == half_small << bits
