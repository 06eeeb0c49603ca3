"""Batched joins at the edges of the single-pass size classes (2^14, 2^16, 2^18,
2^20 int32 build tuples and half as many int64, block-table limits) and beyond
them, in one submission with small joins, over one and several lanes."""
import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev

pytestmark = pytest.mark.gpu

EDGES = [12_289, 65_536, 65_537, 262_144, 262_145, 1 << 20, (1 << 20) + 1, (1 << 21) + 1]


def relations(dtype, n_r, n_s, seed):
    rk = orc.gen_perm(n_r, seed, dtype, 1)
    rk[:: max(3, n_r // 5)] = -1  # some null keys
    rk[1 : n_r : max(5, n_r // 3)] = 7  # and a key several times
    sk = orc.gen_uniform(n_s, seed, 3, -2, n_r + n_r // 4 + 3, dtype)
    return rk, orc.gen_uniform(n_r, seed, 2, -99, 1 << 18, dtype), sk, orc.gen_uniform(n_s, seed, 4, -99, 1 << 18, dtype)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("lanes,graph", [(1, False), (4, True)])
def test_class_edges(dtype, lanes, graph):
    half = 1 if dtype == np.int32 else 2
    sizes = [(n // half, n // half * 2 + 13) for n in EDGES] + [(1, 5), (700, 9000), (13_000, 1), (20_000, 0), (0, 900)]
    host = [relations(dtype, r, s, 40 + i) for i, (r, s) in enumerate(sizes)]
    batch = fij.JoinBatch(dtype, len(sizes), use_graph=graph, lanes=lanes)
    dev = [tuple(to_dev(c) for c in h) for h in host]
    want = [orc.sort_merge_join(*[c[h[k] != -1] for k, c in ((0, h[0]), (0, h[1]), (2, h[2]), (2, h[3]))]) for h in host]
    for _ in range(2):
        assert batch.execute(dev)[0] == want


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_long_chunks(dtype):
    """A class of more tuples than four chunks of 32,768 per compute unit: longer
    chunks, of which a short probe side beside the long ones is less than one."""
    sizes = [(600_011, 12_000_007), (530_000, 12_000_001), (524_289, 12_500_000), (700_001, 50_021), (640_000, 7)]
    host = [relations(dtype, r, s, 60 + i) for i, (r, s) in enumerate(sizes)]
    batch = fij.JoinBatch(dtype, len(sizes))
    dev = [tuple(to_dev(c) for c in h) for h in host]
    want = [orc.sort_merge_join(*[c[h[k] != -1] for k, c in ((0, h[0]), (0, h[1]), (2, h[2]), (2, h[3]))]) for h in host]
    assert batch.execute(dev)[0] == want
