"""Build keys that repeat: few and many copies of every key, one key among
others, more heavy keys than a block table's side entries take, values at the
ends of their type; in every join that builds block tables.  And what a heavy
key may cost."""
import time

import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev
from test_gpu_join import partition_one_pass
from test_gpu_operator_join import join_case

pytestmark = pytest.mark.gpu

COPIES = [3, 4, 5, 8, 13, 100, "heavy", "one"]


def build_side(dtype, n, copies, seed):
    if copies == "one":
        keys = np.full(n, 7, np.int64)
    elif copies == "heavy":
        keys = orc.gen_perm(n, seed, np.int64, 1)
        keys[: min(n // 3, 6000)] = 7
    else:
        keys = orc.gen_perm(n, seed, np.int64, 0) // copies + 1
    info = np.iinfo(dtype)
    pays = orc.gen_uniform(n, seed, 2, -(1 << 20), 1 << 21, dtype)
    pays[::3], pays[1::5] = info.min, info.max
    return keys.astype(dtype), pays


def columns(dtype, n, n_s, copies, seed=21):
    rk, rp = build_side(dtype, n, copies, seed)
    sk = orc.gen_uniform(n_s, seed, 3, -1, int(rk.max()) + int(rk.max()) // 4 + 2, dtype)
    sk[: 50] = 7
    return rk, rp, sk, orc.gen_uniform(n_s, seed, 4, -(1 << 20), 1 << 21, dtype)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("copies", COPIES)
@pytest.mark.parametrize("n", [300, 2048, 6144, 12_288])
def test_table_joins(dtype, n, copies):
    cols = columns(dtype, n, 5003, copies)
    plan = fij.JoinPlan(dtype, n, len(cols[2]), 5, 0)
    assert plan.execute(*[to_dev(c) for c in cols])[0] == orc.sort_merge_join(*cols)


# 32 KiB, 64 KiB and 128 KiB tables, and two fills
@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("copies", COPIES)
@pytest.mark.parametrize("per_part", [900, 2700, 4300, 8800])
def test_single_pass_joins(dtype, per_part, copies):
    bits = 4
    n = (per_part << bits) // (1 if dtype == np.int32 else 2) + 1
    cols = columns(dtype, 13_001 if copies == "one" else n, 30_011, copies)
    plan = fij.JoinPlan(dtype, len(cols[0]), len(cols[2]), bits, 0)
    assert plan.execute(*[to_dev(c) for c in cols])[0] == orc.sort_merge_join(*cols)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("copies", COPIES)
def test_operators(dtype, copies):
    for n in (1500, 6000):
        join_case(dtype, *columns(dtype, n, 9001, copies), 0, 1, 256)


# build partitions around the lengths that go into bucket tables (chains below,
# beyond, and, for some, where a key repeats) against probe partitions around
# the length from which they do
@pytest.mark.parametrize("dtype,n", [(np.int32, n) for n in (1024, 1025, 4097, 6144, 6145, 12_288, 12_289)] +
                         [(np.int64, n) for n in (1024, 1025, 4608, 4609)])
@pytest.mark.parametrize("copies", [1, 3, "heavy"])
def test_operator_tables_and_chains(dtype, n, copies):
    few = dtype == np.int32 and n <= 6144
    least = max(32_768, n * (8 if few else 16))
    for n_s in (least - 1, least):
        join_case(dtype, *columns(dtype, n, n_s, copies), 0, 1, 1024)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_batches_and_served_joins(dtype):
    cols = [columns(dtype, 20_000 + 9000 * i, 40_001, c, 30 + i) for i, c in enumerate(COPIES[:-1])]
    dev = [tuple(to_dev(c) for c in x) for x in cols]
    want = [orc.sort_merge_join(*c) for c in cols]
    assert fij.JoinBatch(dtype, len(cols)).execute(dev)[0] == want
    srv = fij.JoinServer(dtype, [(2, 1 << 17)], max_probe_len=1 << 17)
    for d, w in zip(dev, want):
        assert srv.wait(srv.submit(srv.add_build(d[0], d[1]), d[2], d[3]))[0] == w
    srv.close()


def test_a_heavy_key_costs_an_operator_little():
    """... where the partition goes into a bucket table."""
    dtype, n, n_s = np.int32, 6000, 100_000
    pays = orc.gen_iota(n, 1, dtype), orc.gen_iota(n_s, 1, dtype)
    rk = orc.gen_perm(n, 9, np.int64, 1).astype(dtype)
    sk = orc.gen_uniform(n_s, 9, 3, 8, n, dtype)
    heavy = rk.copy()
    heavy[:2000] = 7

    def best(keys):
        build, probe = (partition_one_pass(k, p, 0, fij.KeyType.I32) for k, p in ((keys, pays[0]), (sk, pays[1])))
        tasks, agg = fij.DeviceArray.zeros(2, np.uint32), fij.aggregates_array(1)
        join = fij.HipRadixJoin(fij.RadixPass.First, fij.RadixBits(0), fij.HashingScheme.BucketChaining, 1, 1024)
        times = []
        for _ in range(6):
            fij.synchronize()
            t = time.perf_counter()
            join.join(build, probe, None, tasks, agg)
            fij.synchronize()
            times.append(time.perf_counter() - t)
        return min(times)
    assert best(heavy) < 4 * best(rk)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n", [6000, 300_007])
def test_a_heavy_key_costs_little(dtype, n):
    """A key with 2,000 copies that few probes ask for: 0.02 ms of work, where
    a compare-and-swap per pair of copies takes milliseconds."""
    n_s = 1 << 20
    rk = orc.gen_perm(n, 9, np.int64, 1).astype(dtype)
    sk = orc.gen_uniform(n_s, 9, 3, 1, n, dtype)
    pays = to_dev(orc.gen_iota(n, 1, dtype)), to_dev(orc.gen_iota(n_s, 1, dtype))
    heavy = rk.copy()
    heavy[:2000] = 7
    plan = fij.JoinPlan(dtype, n, n_s, 9, 0)

    def best(keys):
        dev = to_dev(keys), pays[0], to_dev(sk), pays[1]
        return min(plan.execute(*dev)[1]["total_ms"] for _ in range(6))
    assert best(heavy) < 6 * best(rk)
