"""The partition join's blocks and tables: as many blocks as partitions (blocks
without a task of their own take the later partitions of the others' tasks),
more and fewer of them; build partitions of no tuple, about half an entry per
chain bucket (1,024), the largest bucket table (12,288 int32, 6,144 int64
tuples) and beyond it; duplicate and null keys.  Sums per task and per thread
against the partitions that the assignment gives the task."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import sync, to_dev
from test_gpu_join import partition_one_pass

pytestmark = pytest.mark.gpu


def join_case(dtype, rk, rp, sk, sp, bits, grid, block, scheme=fij.HashingScheme.BucketChaining):
    kt = fij.KeyType.I32 if dtype == np.int32 else fij.KeyType.I64
    brel, prel = partition_one_pass(rk, rp, bits, kt), partition_one_pass(sk, sp, bits, kt)
    result = fij.DeviceArray.zeros(grid * block, np.int64)
    tasks = fij.DeviceArray.zeros(grid + 1, np.uint32)
    agg = fij.aggregates_array(grid)
    j = fij.HipRadixJoin(fij.RadixPass.First, fij.RadixBits(bits), scheme, grid, block)
    for _ in range(2):  # the sums are added to
        j.join(brel, prel, result, tasks, agg)
    sync()
    assert fij.device_status() == 0
    ta = tasks.to_host()
    got = agg.to_host().view(np.uint64).reshape(grid, 3)
    threads = result.to_host().reshape(grid, block)
    mask = (1 << bits) - 1
    for b in range(grid):
        def share(k):
            part = k.astype(np.int64) & mask
            return (part >= ta[b]) & (part < ta[b + 1]) & (k != -1)
        r, s = share(rk), share(sk)
        want = orc.sort_merge_join(rk[r], rp[r], sk[s], sp[s])
        assert tuple(int(x) for x in got[b]) == tuple((2 * w) % 2 ** 64 for w in want), b
        assert int(threads[b].sum()) % 2 ** 64 == 2 * want[2] % 2 ** 64, b


def columns(dtype, n_r, n_s, seed, copies=1):
    rk = (orc.gen_perm(n_r, seed, np.int64, 0) // copies).astype(dtype)
    rk[:: max(7, n_r // 3)] = -1
    sk = orc.gen_uniform(n_s, seed, 3, -2, n_r // copies + n_r // 5 + 4, dtype)
    return rk, orc.gen_uniform(n_r, seed, 2, -99, 1 << 18, dtype), sk, orc.gen_uniform(n_s, seed, 4, -99, 1 << 18, dtype)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("bits,grid", [(4, 16), (4, 17), (4, 40), (4, 15), (4, 3), (0, 1), (0, 5)])
@pytest.mark.parametrize("scheme", [fij.HashingScheme.BucketChaining, fij.HashingScheme.Perfect])
def test_blocks(dtype, bits, grid, scheme):
    cols = columns(dtype, 6000, 50_003, 80) if scheme == fij.HashingScheme.BucketChaining else (
        orc.gen_perm(6000, 81, dtype, 0), orc.gen_iota(6000, 1, dtype),
        orc.gen_uniform(50_003, 81, 3, 0, 7000, dtype), orc.gen_iota(50_003, 1, dtype))
    join_case(dtype, *cols, bits, grid, 128, scheme)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n_r", [1, 1023, 1026, 6144, 6150, 8600, 12_288, 12_295, 15_000])
@pytest.mark.parametrize("copies", [1, 3])
def test_tables(dtype, n_r, copies):
    if dtype == np.int64 and n_r > 8600:
        pytest.skip("beyond the table's entries at int64")
    join_case(dtype, *columns(dtype, n_r, 20_011, 82, copies), 0, 1, 1024)
