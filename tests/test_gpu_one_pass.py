"""Single-pass joins at the edges of their block tables and work units: build
partitions of one tuple, of a table fill and beyond it (several fills without
an arena, HBM tables with one), duplicate and null keys in the last partition,
probe ranges that begin and end at every alignment."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev

pytestmark = pytest.mark.gpu


def plan_join(dtype, bits, cols):
    plan = fij.JoinPlan(dtype, len(cols[0]), len(cols[2]), bits, 0)
    dev = [to_dev(c) for c in cols]
    got = [plan.execute(*dev)[0] for _ in range(2)]  # the second join finds the first one's tables cleared
    assert got[0] == got[1]
    return got[0]


# build tuples per partition around a fill of the 64 KiB table (6,144 int32,
# 3,072 int64 tuples) and of the 128 KiB one
@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("per_part", [1, 3071, 3073, 6143, 6145, 12_289])
def test_build_partition_sizes(dtype, per_part):
    bits, n_s = 2, 70_001
    n_r = per_part << bits
    rk = orc.gen_perm(n_r, 5, dtype, 1)
    rp = orc.gen_uniform(n_r, 5, 2, -(1 << 20), 1 << 21, dtype)
    sk = orc.gen_uniform(n_s, 5, 3, 1, n_r + n_r // 3 + 1, dtype)
    sp = orc.gen_uniform(n_s, 5, 4, -(1 << 20), 1 << 21, dtype)
    assert plan_join(dtype, bits, (rk, rp, sk, sp)) == orc.sort_merge_join(rk, rp, sk, sp)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_duplicates_and_nulls_in_the_last_partition(dtype):
    bits = 3
    rk = orc.gen_uniform(20_011, 6, 1, -9, 900, dtype)  # many copies of a key, -1 among them
    sk = orc.gen_uniform(90_007, 6, 2, -9, 1200, dtype)
    rp, sp = orc.gen_iota(len(rk), 1, dtype), orc.gen_iota(len(sk), 1, dtype)
    assert (rk == -1).any() and (sk == -1).any()
    assert plan_join(dtype, bits, (rk, rp, sk, sp)) == orc.sort_merge_join(rk, rp, sk, sp)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_one_partition_holds_everything(dtype):
    """Keys of one digit: the other partitions are empty, the one build
    partition exceeds every LDS table."""
    bits, n_r, n_s = 6, 40_000, 300_001
    rk = (orc.gen_perm(n_r, 7, np.int64, 1) * 64 + 5).astype(dtype)
    sk = (orc.gen_uniform(n_s, 7, 2, 1, n_r + 999, np.int64) * 64 + 5).astype(dtype)
    rp, sp = orc.gen_iota(n_r, 1, dtype), orc.gen_iota(n_s, 1, dtype)
    want = orc.sort_merge_join(rk, rp, sk, sp)
    assert plan_join(dtype, bits, (rk, rp, sk, sp)) == want
    # a served build side has no arena: several table fills
    srv = fij.JoinServer(dtype, [(1, 1 << 19)], max_probe_len=1 << 19)
    b = srv.add_build(to_dev(rk), to_dev(rp))
    assert srv.wait(srv.submit(b, to_dev(sk), to_dev(sp)))[0] == want
    srv.close()


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n_s", [1, 2, 3, 511, 8191, 8192, 8193, 16_385])
def test_probe_range_lengths(dtype, n_s):
    n_r = 14_003
    rk = orc.gen_perm(n_r, 8, dtype, 1)
    rp = orc.gen_iota(n_r, 3, dtype)
    sk = orc.gen_uniform(n_s, 8, 2, 1, n_r, dtype)
    sp = orc.gen_iota(n_s, 1, dtype)
    assert plan_join(dtype, 1, (rk, rp, sk, sp)) == orc.sort_merge_join(rk, rp, sk, sp)


@pytest.mark.parametrize("dtype,n_r", [(np.int32, 12_000_001), (np.int64, 6_000_001)])
def test_two_pass_plan_beyond_two_fills(dtype, n_r):
    """Build sides just beyond what a two-pass plan joins in a single pass,
    and, sized, just within it: the same joins through both."""
    n_s = 3_000_017
    limit = {np.int32: 11_796_480, np.int64: 5_898_240}[dtype]
    rk = orc.gen_perm(n_r, 11, dtype, 1)
    rp = orc.gen_iota(n_r, 5, dtype)
    sk = orc.gen_uniform(n_s, 11, 2, 1, n_r + n_r // 5, dtype)
    sp = orc.gen_iota(n_s, 0, dtype)
    plan = fij.JoinPlan(dtype, n_r, n_s, 9, 7)
    d = [to_dev(c) for c in (rk, rp, sk, sp)]
    res = fij.DeviceArray(3, np.uint64)
    for n in (n_r, limit + 1, limit, n_r):
        plan.enqueue_sized(d[0].view(0, n), d[1].view(0, n), d[2], d[3], res)
        got = tuple(int(x) for x in res.to_host())
        at = np.empty(n_r + 1, np.int64)
        at.fill(-1)
        at[rk[:n].astype(np.int64)] = np.arange(n)
        hit = sk <= n_r
        hit[hit] = at[sk[hit].astype(np.int64)] >= 0
        rows = at[sk[hit].astype(np.int64)]
        want = (int(hit.sum()), int(rp[rows].astype(np.int64).sum()), int(sp[hit].astype(np.int64).sum()))
        assert got == want


@pytest.mark.parametrize("dtype,limits", [(np.int32, (4_571_136, 7_077_888)), (np.int64, (4_571_136, 5_079_040))])
def test_two_pass_plan_at_the_single_pass_limits(dtype, limits):
    """Sized joins of a two-pass plan around the build sides up to which it
    takes a single pass, for every probe side and for short ones."""
    n_r, n_s = limits[1] + 1, 2_000_003
    rk = orc.gen_perm(n_r, 12, dtype, 1)
    rk[: n_r // 3] = rk[n_r // 3 : 2 * (n_r // 3)]  # a third of the keys twice
    rp = orc.gen_iota(n_r, 5, dtype)
    sk = orc.gen_uniform(n_s, 12, 2, 1, n_r + n_r // 5, dtype)
    sp = orc.gen_iota(n_s, 0, dtype)
    plan = fij.JoinPlan(dtype, n_r, n_s, 9, 7)
    d = [to_dev(c) for c in (rk, rp, sk, sp)]
    res = fij.DeviceArray(3, np.uint64)
    for n in (limits[0], limits[0] + 1, limits[1], limits[1] + 1):
        plan.enqueue_sized(d[0].view(0, n), d[1].view(0, n), d[2], d[3], res)
        assert tuple(int(x) for x in res.to_host()) == orc.sort_merge_join(rk[:n], rp[:n], sk, sp)
