"""Out-of-core joins whose histograms leave the keys on the device: lengths
around 16-byte vectors and steps, host columns at element offsets, build or
probe columns in device memory (no copy), and the length up to which keys are
copied (twice the staging size) and beyond it."""
import ctypes as C

import numpy as np
import pytest

import fij
import oracle_lib as orc
from gpu_helpers import to_dev

pytestmark = pytest.mark.gpu


def columns(dtype, n_r, n_s, seed):
    rk = orc.gen_perm(n_r, seed, dtype, 1)
    rk[:: max(5, n_r // 3)] = -1
    sk = orc.gen_uniform(n_s, seed, 3, -2, n_r + n_r // 3 + 3, dtype)
    return (rk, orc.gen_uniform(n_r, seed, 2, -99, 1 << 18, dtype), sk, orc.gen_uniform(n_s, seed, 4, -99, 1 << 18, dtype))


def want_of(h):
    r, s = h[0] != -1, h[2] != -1
    return orc.sort_merge_join(h[0][r], h[1][r], h[2][s], h[3][s])


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n_r,n_s", [(1, 1), (3, 2), (5, 4099), (4097, 131_072), (70_001, 131_073), (131_072, 70_003)])
@pytest.mark.parametrize("cache_frac", [0.0, 0.5])
def test_lengths(dtype, n_r, n_s, cache_frac):
    h = columns(dtype, n_r, n_s, 7)
    cols = [fij.HostArray.from_numpy(a) for a in h]
    cache = int(cache_frac * (n_r + n_s) * 2 * np.dtype(dtype).itemsize)
    got, _ = fij.ooc_join(dtype, *cols, 5, 4, cache_bytes=cache, staging_tuples=1 << 16)  # keys copied up to 2^17
    assert got == want_of(h)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("shift", [1, 3])
def test_columns_at_element_offsets(dtype, shift):
    h = columns(dtype, 30_011, 90_017, 8)
    size = np.dtype(dtype).itemsize
    cols = [fij.HostArray(len(a) + shift, dtype) for a in h]
    for c, a in zip(cols, h):
        c.a[shift:] = a
    ptr = [C.c_void_p(c.ptr + shift * size) for c in cols]
    kt = fij.KeyType.I32 if dtype == np.int32 else fij.KeyType.I64
    cfg = fij.OocConfig(int(kt), 5, 4, 0, 0, 0, 1 << 18, 0)
    res, t = fij.JoinAggregate(), fij.OocTiming()
    fij.check(fij.lib.fij_ooc_join(C.byref(cfg), ptr[0], ptr[1], len(h[0]), ptr[2], ptr[3], len(h[2]), C.byref(res),
                                   C.byref(t)))
    assert (res.count, res.sum_build, res.sum_probe) == want_of(h)


@pytest.mark.parametrize("on_device", [(0, 1), (2, 3), (0,), (3,)])
def test_columns_in_device_memory(on_device):
    h = columns(np.int64, 30_011, 90_017, 9)
    cols = [to_dev(a) if i in on_device else fij.HostArray.from_numpy(a) for i, a in enumerate(h)]
    assert fij.ooc_join(np.int64, *cols, 5, 4, cache_bytes=1 << 20)[0] == want_of(h)
