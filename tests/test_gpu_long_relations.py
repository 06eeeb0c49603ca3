"""Probe sides of nearly 2^32 tuples, the longest that a plan accepts."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev

pytestmark = pytest.mark.gpu


def columns(n, lo, count):
    """n int32 keys drawn from [lo, lo + count) and payloads of 1 on the device."""
    keys, pays = fij.DeviceArray(n, np.int32), fij.DeviceArray(n, np.int32)
    fij.gen_uniform(keys, 3, 1, lo, count)
    fij.gen_uniform(pays, 3, 2, 1, 1)
    return keys, pays


@pytest.mark.parametrize("n_r,stride", [(2048 * 512, 1), (60_000, 512)])
def test_one_probe_partition(n_r, stride):
    """Every probe tuple has the same key: one partition's units hold them all,
    against a block table, and against a table in device memory (its digit holds
    the whole build side)."""
    n_s = (1 << 32) - 20_000
    rk = (orc.gen_perm(n_r, 5, np.int64, 0) * stride + 3).astype(np.int32)
    rp = orc.gen_iota(n_r, 1, np.int32)
    key = int(rk[77])
    sk, sp = columns(n_s, key, 1)
    plan = fij.JoinPlan(np.int32, n_r, n_s, 9, 0)
    got = plan.execute(to_dev(rk), to_dev(rp), sk, sp)[0]
    assert got == (n_s, int(rp[77]) * n_s, n_s)


@pytest.mark.parametrize("keys", [20_000, 1])
def test_few_pass_1_bits(keys):
    """16 partitions fit the 32-bit offsets of pass 1, the 512 of a single pass
    would not; with one key, one partition has nearly 2^32 tuples to cut into
    tiles."""
    n_r, n_s = 20_000, (1 << 32) - 1000
    rk, rp = orc.gen_perm(n_r, 6, np.int32, 1), np.full(n_r, 7, np.int32)
    sk, sp = columns(n_s, 1, keys)  # every probe key matches
    plan = fij.JoinPlan(np.int32, n_r, n_s, 4, 4)
    got = plan.execute(to_dev(rk), to_dev(rp), sk, sp)[0]
    assert got == (n_s, 7 * n_s, n_s)
