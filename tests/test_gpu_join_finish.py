"""Joins that end in their last block: grids of one block, of one counter and
of grouped counters (more than 64 blocks, not a multiple of 16), and single-pass
joins with hash tables of several partitions, built, probed and cleared by the
blocks that have run out of work units, several times in a row."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev

pytestmark = pytest.mark.gpu


def columns(dtype, n_r, n_s, seed):
    return (orc.gen_perm(n_r, seed, dtype, 1), orc.gen_uniform(n_r, seed, 2, -99, 1 << 18, dtype),
            orc.gen_uniform(n_s, seed, 3, 1, n_r + n_r // 3 + 2, dtype), orc.gen_uniform(n_s, seed, 4, -99, 1 << 18, dtype))


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("blocks", [1, 2, 64, 65, 77, 0])
def test_grids(dtype, blocks):
    n_r, n_s = 30_000, 400_001
    plan = fij.JoinPlan(dtype, n_r, n_s, 7, 0, join_blocks=blocks)
    for seed, r in ((50, n_r), (51, 900), (52, n_r)):  # partitioned, one table, partitioned
        cols = columns(dtype, r, n_s, seed)
        dev = [to_dev(c) for c in cols]
        out = fij.aggregates_array(1)
        for _ in range(2):
            plan.enqueue_sized(*dev, out)
            fij.synchronize()
            assert fij.sum_aggregates(out) == orc.sort_merge_join(*cols)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_tables_of_several_partitions(dtype):
    bits, n_r, n_s = 2, 400_000, 1_500_003
    plan = fij.JoinPlan(dtype, n_r, n_s, bits, 0)
    for seed in (60, 61, 62):
        cols = columns(dtype, n_r, n_s, seed)
        assert plan.execute(*[to_dev(c) for c in cols])[0] == orc.sort_merge_join(*cols)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n_s", [1, 1023, 1025, 66_000, 500_001])
def test_served_probe_grids(dtype, n_s):
    cols = columns(dtype, 3000, n_s, 70)
    srv = fij.JoinServer(dtype, [(1, 1 << 19)], max_probe_len=1 << 19, table_build_max=1 << 16)
    b = srv.add_build(to_dev(cols[0]), to_dev(cols[1]))
    for _ in range(2):
        assert srv.wait(srv.submit(b, to_dev(cols[2]), to_dev(cols[3])))[0] == orc.sort_merge_join(*cols)
