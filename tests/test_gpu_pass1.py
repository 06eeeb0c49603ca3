"""Pass 1 of the joins and the offsets scan at the edges of their tiles:
fanouts below and above one scan tile, chunk counts below and above the
scan's groups, sides of very different lengths in one launch, sides shorter
than one step of the scatter."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import sync, to_dev

pytestmark = pytest.mark.gpu

CONTIG = fij.HistogramAlgorithm.Contiguous


@pytest.mark.parametrize("bits,grid", [(1, 1), (3, 63), (4, 64), (5, 65), (7, 300), (11, 257)])
def test_contiguous_offsets_at_tile_edges(bits, grid):
    n = 200_003
    keys = orc.gen_uniform(n, 7, 1, 0, 1 << 30, np.int32)
    part = fij.GpuRadixPartitioner(CONTIG, fij.RadixPartitionAlgorithm.SSWWCv2, fij.RadixBits(bits), grid, 1024)
    offs = fij.PartitionOffsets(CONTIG, grid, bits, fij.KeyType.I32)
    for _ in range(2):  # the scan state is cleared by every call
        part.prefix_sum(fij.RadixPass.First, to_dev(keys), offs)
        sync()
        want, want_local = orc.contiguous_prefix_sum(keys, grid, bits, 0)
        np.testing.assert_array_equal(offs.host_offsets(), want)
        np.testing.assert_array_equal(offs.host_local_offsets(), want_local)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n_r,n_s", [(1, 1), (1, 300_001), (40_001, 3), (20_001, 2_500_007), (700_001, 20_011)])
@pytest.mark.parametrize("bits", [(9, 3), (3, 1), (6, 0), (10, 2)])
def test_sides_of_unequal_lengths(dtype, n_r, n_s, bits):
    rk = orc.gen_uniform(n_r, 3, 1, 1, max(1, n_r // 2), dtype)
    rp = orc.gen_uniform(n_r, 3, 2, -(1 << 20), 1 << 21, dtype)
    sk = orc.gen_uniform(n_s, 3, 3, 1, n_r, dtype)
    sp = orc.gen_uniform(n_s, 3, 4, -(1 << 20), 1 << 21, dtype)
    plan = fij.JoinPlan(dtype, n_r, n_s, *bits)
    got, _ = plan.execute(to_dev(rk), to_dev(rp), to_dev(sk), to_dev(sp))
    assert got == orc.sort_merge_join(rk, rp, sk, sp)
