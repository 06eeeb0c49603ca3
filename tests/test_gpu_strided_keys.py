"""Joins in one pass of keys whose low bits say little (multiples of powers of
two): results, and what they may cost."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev

pytestmark = pytest.mark.gpu

TYPES = [np.int32, np.int64]


def keys_of(numbers, stride, dtype):
    """numbers * stride, wrapped into the type; stride "pairs": two of every 64."""
    i = numbers.astype(np.uint64)
    k = (i >> np.uint64(1)) * np.uint64(64) + (i & np.uint64(1)) if stride == "pairs" else i * np.uint64(stride)
    return k.astype(np.uint32).view(np.int32) if dtype == np.int32 else k.view(np.int64)


def columns(dtype, n, n_s, stride, seed=5, order=None):
    rk = keys_of(np.arange(1, n + 1) if order else orc.gen_perm(n, seed, np.int64, 1), stride, dtype)
    sk = keys_of(orc.gen_uniform(n_s, seed, 3, 1, n + n // 4, np.int64), stride, dtype)
    rk[:: n // 3], sk[:: n_s // 7] = -1, -1  # some null keys
    return (rk, orc.gen_uniform(n, seed, 2, -(1 << 20), 1 << 21, dtype), sk,
            orc.gen_uniform(n_s, seed, 4, -(1 << 20), 1 << 21, dtype))


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("stride", [1, 2, 32, 512, 4096, 1 << 16, 3 << 9, 1 << 33, "pairs"])
@pytest.mark.parametrize("bits", [(9, 0), (8, 8), (4, 0), (1, 0)])
def test_plans(dtype, stride, bits):
    """Of one pass, and of two that run in one."""
    if stride == 1 << 33 and dtype == np.int32:
        stride = 1 << 13
    n, n_s = (65_537, 200_003) if bits[0] > 4 else (20_011, 50_003)
    cols = columns(dtype, n, n_s, stride, order=stride == 512)
    plan = fij.JoinPlan(dtype, n, n_s, *bits)
    assert plan.execute(*[to_dev(c) for c in cols])[0] == orc.sort_merge_join(*cols)


@pytest.mark.parametrize("dtype", TYPES)
def test_one_plan_with_either_digits(dtype):
    n, n_s = 70_001, 150_007
    plan, out = fij.JoinPlan(dtype, n, n_s, 9, 0), fij.DeviceArray.zeros(3, np.uint64)
    for k, stride in enumerate([1, 1024, 1, 512, "pairs"]):
        cols = columns(dtype, n - 20_000 * (k % 3), n_s - 1000 * k, stride, k + 1)
        dev = [to_dev(c) for c in cols]
        plan.enqueue_sized(*dev, out)
        assert tuple(int(x) for x in out.to_host()) == orc.sort_merge_join(*cols)


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("graph", [True, False])
def test_batches(dtype, graph):
    """Classes of 5, 7 and 9 bits, with joins of either digits in each."""
    cols = [columns(dtype, n, 4 * n + 13, stride, n) for n in (13_001, 40_003, 150_007, 600_011)
            for stride in (1, 32, 4096)]
    got = fij.JoinBatch(dtype, len(cols), use_graph=graph).execute([tuple(to_dev(c) for c in x) for x in cols])[0]
    assert got == [orc.sort_merge_join(*x) for x in cols]


@pytest.mark.parametrize("dtype", TYPES)
def test_served_joins(dtype):
    cols = [columns(dtype, 30_011 + 9000 * k, 50_001, stride, k + 1) for k, stride in enumerate([1, 512, 4096, "pairs"])]
    dev = [[to_dev(c) for c in x] for x in cols]
    srv = fij.JoinServer(dtype, [(3, 1 << 17)], max_probe_len=1 << 17)
    ids = [srv.add_build(d[0], d[1]) for d in dev]
    asked = [srv.submit(i, d[2], d[3]) for _ in range(3) for i, d in zip(ids, dev)]
    assert [srv.wait(a)[0] for a in asked] == 3 * [orc.sort_merge_join(*x) for x in cols]
    srv.close()


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("bits", [(9, 0), (8, 8)])
def test_strides_cost_little(dtype, bits):
    """Multiples of 64 took 11 times as long as consecutive keys (1,634 for 153
    us at these sizes of int32) with all of them in 8 of 512 partitions."""
    n, n_s = 1 << 20, 1 << 24
    plan = fij.JoinPlan(dtype, n, n_s, *bits)

    def best(stride):
        dev = [to_dev(c) for c in columns(dtype, n, n_s, stride)]
        return min(plan.execute(*dev)[1]["total_ms"] for _ in range(6))

    assert best(64) < 2 * best(1)
