"""Work units of the items that the two-pass join defers: every item (sides far
beyond the registers, the register join left out) or only those of heavy keys,
items without build or probe tuples, and items of many units (written by a
whole wave) with block tables and with hash tables of the arena."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,n_r", [(np.int32, 7_300_003), (np.int64, 5_300_003)])
@pytest.mark.parametrize("bits", [(9, 2), (4, 4), (8, 6)])  # all deferred in block tables, in the arena's; few deferred
@pytest.mark.parametrize("spread", [1, 4])  # 4: three quarters of the pass-1 partitions are empty
def test_deferred_units(dtype, n_r, bits, spread):
    n_s = 2_000_009
    rk = orc.gen_perm(n_r, 91, dtype, 1)
    rk[:9000] = 77  # a build side beyond a block's table
    sk = orc.gen_uniform(n_s, 91, 2, 1, n_r + n_r // 9, dtype)
    sk[: n_s // 3] = 4242  # about ten units of one item
    sk[n_s // 3 : n_s // 3 + 40] = 77
    rk, sk = (rk * spread).astype(dtype), (sk * spread).astype(dtype)
    rp, sp = orc.gen_iota(n_r, 1, dtype), orc.gen_iota(n_s, 1, dtype)
    want = orc.sort_merge_join(rk, rp, sk, sp)
    plan = fij.JoinPlan(dtype, n_r, n_s, *bits)
    dev = [to_dev(c) for c in (rk, rp, sk, sp)]
    for _ in range(2):
        got, times = plan.execute(*dev)
        assert got == want
        assert all(0 <= t <= times["total_ms"] for t in times.values()), times
