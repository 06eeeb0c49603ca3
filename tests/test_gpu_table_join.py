"""Plans whose build side fits one block's LDS table (one launch without
partitioning): sizes around a table, an odd number of probe tuples, unaligned
columns, null and duplicate keys, a long probe side over many blocks."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev

pytestmark = pytest.mark.gpu

FULL = {np.int32: 12_288, np.int64: 6_144}  # build tuples a table holds


def both_ways(dtype, cols, bits=(3, 2), offset=0):
    """The join through execute and through a sized join into device memory,
    columns `offset` elements into their buffers."""
    dev = []
    for c in cols:
        d = to_dev(np.concatenate([np.zeros(offset, dtype), c]))
        dev.append(d.view(offset, offset + len(c)))
    plan = fij.JoinPlan(dtype, len(cols[0]), len(cols[2]), *bits)
    res = fij.DeviceArray(3, np.uint64)
    got = []
    for _ in range(2):
        got.append(plan.execute(*dev)[0])
        plan.enqueue_sized(*dev, res)
        got.append(tuple(int(x) for x in res.to_host()))
    assert len(set(got)) == 1
    return got[0]


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n_r", [1, 63, 1025, 2049, "full", "over"])
@pytest.mark.parametrize("n_s", [1, 4099, 1_000_003])
def test_build_and_probe_sizes(dtype, n_r, n_s):
    n_r = {"full": FULL[dtype], "over": FULL[dtype] + 1}.get(n_r, n_r)
    rk = orc.gen_perm(n_r, 5, dtype, 1)
    rp = orc.gen_uniform(n_r, 5, 2, -(1 << 20), 1 << 21, dtype)
    sk = orc.gen_uniform(n_s, 5, 3, 1, n_r + n_r // 3 + 1, dtype)
    sp = orc.gen_uniform(n_s, 5, 4, -(1 << 20), 1 << 21, dtype)
    assert both_ways(dtype, (rk, rp, sk, sp)) == orc.sort_merge_join(rk, rp, sk, sp)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_nulls_duplicates_and_alignment(dtype, offset):
    rk = orc.gen_uniform(3_001, 6, 1, -5, 700, dtype)
    sk = orc.gen_uniform(50_003, 6, 2, -5, 900, dtype)
    rp, sp = orc.gen_iota(len(rk), 1, dtype), orc.gen_iota(len(sk), 1, dtype)
    assert (rk == -1).any() and (sk == -1).any()
    assert both_ways(dtype, (rk, rp, sk, sp), offset=offset) == orc.sort_merge_join(rk, rp, sk, sp)


def test_timing_of_one_launch():
    """A join without partitioning reports its time as the join's."""
    n = 5_000
    k = orc.gen_perm(n, 3, np.int64, 1)
    plan = fij.JoinPlan(np.int64, n, n, 4, 0)
    d = to_dev(k)
    with pytest.raises(fij.FijError):
        plan.result()  # nothing enqueued yet
    got, t = plan.execute(d, d, d, d)
    assert got[0] == n
    assert t["total_ms"] > 0 and t["join_ms"] == t["total_ms"] and t["prefix_sum_ms"] == 0
