"""Single-pass joins with build partitions of no tuple, of one, and around one
and two fills of each of the three block tables."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev

pytestmark = pytest.mark.gpu

BITS = 5
# tuples of a fill, and of the partitions that make the mean choose the table
FILLS = {(np.int32, 32): (2304, 1500), (np.int32, 64): (4608, 2000), (np.int32, 128): (9216, 3000),
         (np.int64, 32): (1280, 800), (np.int64, 64): (2560, 1000), (np.int64, 128): (5120, 1400)}


@pytest.mark.parametrize("dtype,kib", FILLS)
@pytest.mark.parametrize("copies", [1, 2, 9])
def test_partitions_around_a_fill(dtype, kib, copies):
    fill, other = FILLS[dtype, kib]
    F = 1 << BITS
    sizes = np.full(F, other)
    sizes[[3, 30, 11, 7, 20, 0, 31]] = 0, 1, fill - 1, fill, fill + 1, 2 * fill, 2 * fill + 1
    mean = sizes.sum() / F
    quarter = 65_536 // (8 * np.dtype(dtype).itemsize)  # half the slots of a 32 KiB table
    assert (32 if mean <= quarter else 64 if mean <= 2 * quarter else 128) == kib and sizes.sum() > 12_288
    # `copies` of the keys p, p + F, ... in partition p
    rk = np.concatenate([p + F * (1 + np.arange(n) // copies) for p, n in enumerate(sizes)])
    rk = rk[orc.gen_perm(len(rk), 8, np.int64, 0)].astype(dtype)
    n_s = 90_001
    sk = orc.gen_uniform(n_s, 8, 3, 0, F * (2 * fill // copies + 40), dtype)
    cols = (rk, orc.gen_uniform(len(rk), 8, 2, -(1 << 20), 1 << 21, dtype), sk,
            orc.gen_uniform(n_s, 8, 4, -(1 << 20), 1 << 21, dtype))
    plan = fij.JoinPlan(dtype, len(rk), n_s, BITS, 0)
    assert plan.execute(*[to_dev(c) for c in cols])[0] == orc.sort_merge_join(*cols)
