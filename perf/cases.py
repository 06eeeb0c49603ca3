"""The work that programs have this library do, as cases that can be timed.

Every case goes through the library's public Python entry points (JoinPlan, the
partitioner / radix-join operators, HipHashJoin, JoinBatch, JoinServer,
ooc_join).  A case is a dict of plain values:

  kind     which entry points: "plan", "operator", "two_pass", "np", "batch", "served", "ooc"
  type     "i32" or "i64" (keys and payloads)
  build, probe   tuples of the two relations (batch, served: their range as log2, with `shape`)
  keys     "dense": keys 1..build in a random order (primary keys); "wide": the same keys spread over
           the whole key type by an odd multiplier; "dups": build keys drawn with repetitions
  match    share of the probe keys that lie in the build side's key range
  zipf     exponent of the probe keys' skew (0: uniform)

Payloads: random on the build side, the row number on the probe side.  Results
are match counts and wrapping 64-bit sums, so they are whole numbers and the
same on every run.
"""
import math
import os
import random
import sys

import numpy as np
import torch  # before the library, so that both use one HIP runtime

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fast-interconnects_amd"))
import fij  # noqa: E402

DEV = "cuda" if torch.cuda.is_available() else "cpu"
CHUNK = 1 << 26


def listed():
    def plan(name, type, build, probe, keys="dense", match=1.0, zipf=0.0, bits=(0, 0), sized=False):
        return {"name": name, "kind": "plan", "type": type, "build": build, "probe": probe, "keys": keys, "match": match,
                "zipf": zipf, "bits1": bits[0], "bits2": bits[1], "sized": sized}

    return [
        # A lookup join of a dimension table of a few thousand rows: one call, its latency is what counts.
        plan("plan_tiny_i32", "i32", 1500, 6007),
        # A join inside a larger device program: sized, its result left in device memory, not waited for.
        plan("plan_short_i64", "i64", 65539, 1000003, keys="wide", match=0.8, sized=True),
        # The CPU-runnable configuration of the radix join: 2^20 with 2^24 int32 tuples; one pass.
        plan("plan_one_pass_i32", "i32", 1 << 20, 1 << 24),
        # An ordinary fact / dimension join of ragged sizes with 64-bit keys from all over their range; two passes.
        plan("plan_odd_i64", "i64", 5000011, 20000003, keys="wide", match=0.9),
        # The headline join: 2^27 with 2^27 int64 tuples, 9 + 9 bits.
        plan("plan_large_i64", "i64", 1 << 27, 1 << 27, bits=(9, 9)),
        # The skewed configuration: 2^27 with 2^30 int32 tuples, Zipf-distributed foreign keys, 8 + 8 bits.
        plan("plan_skew_i32", "i32", 1 << 27, 1 << 30, zipf=1.0, bits=(8, 8)),
        # The partition and join operators called one by one, as the radix-join program does for one pass.
        {"name": "operator_one_pass_i32", "kind": "operator", "type": "i32", "build": 1 << 20, "probe": 1 << 24, "keys": "dense",
         "match": 1.0, "zipf": 0.0, "bits1": 8},
        # The operators in the radix-join program's two-pass loop: transform, partition and join of every partition.
        {"name": "operator_two_pass_i64", "kind": "two_pass", "type": "i64", "build": 300007, "probe": 4000037, "keys": "dense",
         "match": 1.0, "zipf": 0.0, "bits1": 4, "bits2": 5},
        # The hashjoin program: a linear-probing table in device memory, built and probed.
        {"name": "np_join_i64", "kind": "np", "type": "i64", "build": 1 << 23, "probe": 1 << 26, "keys": "dense", "match": 1.0,
         "zipf": 0.0, "perfect": False},
        # Many independent joins of uneven sizes in one submission (sizes of the batched configuration, up to 2^20).
        {"name": "batch_i32", "kind": "batch", "type": "i32", "joins": 96, "lo": 10.0, "hi": 20.0, "shape": 7},
        # A burst of requests against resident build sides (the served configuration, up to 2^22 and 2^23 tuples).
        {"name": "served_i64", "kind": "served", "type": "i64", "builds": 10, "build_lo": 12.0, "build_hi": 22.0, "requests": 24,
         "probe_lo": 14.0, "probe_hi": 23.0, "shape": 3},
        # Relations in pinned host memory, half of the partitions spilled.
        {"name": "ooc_i64", "kind": "ooc", "type": "i64", "build": 1000003, "probe": 4000037, "keys": "dense", "match": 1.0, "zipf": 0.0,
         "bits1": 6, "bits2": 6, "cache": 0.5},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, even over its logarithm, mostly odd."""
    n = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    return max(lo, n | 1 if rng.random() < 0.8 else n)


def draw(rng):
    kind = rng.choice(["plan"] * 6 + ["operator", "two_pass", "np", "batch", "served", "ooc"])
    type = rng.choice(["i32", "i64"])
    k = 1 if type == "i32" else 2
    c = {"kind": kind, "type": type}
    if kind == "batch":
        lo = rng.uniform(9.0, 13.0)
        return dict(c, joins=rng.randint(16, 160), lo=lo, hi=rng.uniform(lo + 3, 20.5 - k / 2), shape=rng.randrange(1 << 20))
    if kind == "served":
        return dict(c, builds=rng.randint(2, 12), build_lo=rng.uniform(10, 14), build_hi=rng.uniform(18, 22.5),
                    requests=rng.randint(4, 32), probe_lo=rng.uniform(12, 15), probe_hi=rng.uniform(20, 23), shape=rng.randrange(1 << 20))
    if kind == "plan":
        build = _size(rng, 1 << 10, (1 << 28) // k // 2)
        probe = max(build, min(_size(rng, build, 64 * build), (1 << 30) // k // 2))
        c.update(build=build, probe=probe, keys=rng.choice(["dense", "wide", "dups"]), match=round(rng.uniform(0.2, 1.0), 2),
                 zipf=rng.choice([0.0, 0.0, 0.0, 0.5, 1.0]), bits1=0, bits2=0, sized=rng.random() < 0.5)
        return c
    c.update(keys=rng.choice(["dense", "wide"]), match=round(rng.uniform(0.3, 1.0), 2), zipf=rng.choice([0.0, 0.0, 0.75]))
    if kind == "operator":
        bits = rng.randint(6, 9)
        build = _size(rng, 1 << 12, (1 << bits) * 2500)
        return dict(c, build=build, probe=_size(rng, max(build, 1 << 16), 1 << 25), bits1=bits)
    if kind == "two_pass":
        b1, b2 = rng.randint(2, 5), rng.randint(3, 6)
        build = _size(rng, 1 << 14, (1 << (b1 + b2)) * 1500)
        return dict(c, build=build, probe=_size(rng, max(build, 1 << 17), 1 << 23), bits1=b1, bits2=b2, zipf=0.0)
    if kind == "np":
        build = _size(rng, 1 << 12, 1 << 24)
        perfect = rng.random() < 0.3
        return dict(c, build=build, probe=max(build, _size(rng, 1 << 16, 1 << 26)), perfect=perfect,
                    keys="dense" if perfect else c["keys"])
    build = _size(rng, 1 << 16, 1 << 21)
    return dict(c, build=build, probe=_size(rng, build, 1 << 23), bits1=rng.randint(4, 7), bits2=rng.randint(4, 7), zipf=0.0,
                cache=rng.choice([0.0, 0.3, 0.7, 2.0]))


# ------------------------------------------------------------------ inputs


def _dtype(case):
    return (torch.int32, np.int32, 4) if case["type"] == "i32" else (torch.int64, np.int64, 8)


def _keys(idx, case, dt):
    """Key of each key number (from 1 on)."""
    if case.get("keys") == "wide":
        if dt == torch.int32:
            return (idx * 0x9E3779B1).bitwise_and(0xFFFFFFFF).to(torch.int32)
        return idx * -7046029254386353131  # 0x9E3779B97F4A7C15
    return idx.to(dt)


def _relations(case, seed, build, probe):
    """(build keys, build payloads, probe keys, probe payloads) as torch tensors."""
    dt = _dtype(case)[0]
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    if case.get("keys") == "dups":
        order = torch.randint(0, max(1, build // 2), (build,), device=DEV, generator=g)
    else:
        order = torch.randperm(build, device=DEV, generator=g)
    bk = _keys(order + 1, case, dt)
    bp = torch.randint(0, 1 << 30, (build,), device=DEV, generator=g, dtype=dt)
    n, s = max(1, int(build / case.get("match", 1.0))), case.get("zipf", 0.0)
    sk = torch.empty(probe, device=DEV, dtype=dt)
    for a in range(0, probe, CHUNK):
        m = min(CHUNK, probe - a)
        if not s:
            idx = torch.randint(1, n + 1, (m,), device=DEV, generator=g)
        else:
            # ranks by the inverse of the continuous power law over [1, n + 1); a rank's key is `order`'s
            u = torch.rand(m, device=DEV, generator=g, dtype=torch.float64)
            x = torch.exp(u * math.log(n + 1.0)) if s == 1.0 else (u * ((n + 1.0) ** (1 - s) - 1) + 1) ** (1 / (1 - s))
            idx = x.to(torch.int64).clamp_(1, n)
            inside = idx <= build
            idx = torch.where(inside, order[(idx - 1).clamp_(max=build - 1)] + 1, idx)
        sk[a:a + m] = _keys(idx, case, dt)
    sp = torch.arange(probe, device=DEV, dtype=dt)
    return bk, bp, sk, sp


def _column(t, dtype):
    """The library's device column of a tensor's values."""
    a = fij.DeviceArray(t.numel(), dtype)
    fij.check(fij.lib.fij_memcpy(fij.C.c_void_p(a.ptr), fij.C.c_void_p(t.data_ptr()), a.nbytes(), None))
    return a


def _columns(case, seed, build, probe):
    return [_column(t, _dtype(case)[1]) for t in _relations(case, seed, build, probe)]


def _sizes(case):
    """Sizes of a batch's joins / a server's builds and requests: the case's, the same for every seed."""
    r = random.Random(case["shape"])
    if case["kind"] == "batch":
        got = []
        for _ in range(case["joins"]):
            b = int(2 ** r.uniform(case["lo"], case["hi"]))
            got.append((b, int(b * r.uniform(4, 16))))
        return got
    builds = [int(2 ** r.uniform(case["build_lo"], case["build_hi"])) for _ in range(case["builds"])]
    return builds, [(r.randrange(len(builds)), int(2 ** r.uniform(case["probe_lo"], case["probe_hi"]))) for _ in range(case["requests"])]


def _served_inputs(case, seed):
    """Build sides, and for every request its build side and probe columns, as tensors."""
    builds, requests = _sizes(case)
    sides = [_relations(case, seed * 1000 + i, b, 1)[:2] for i, b in enumerate(builds)]
    asked = []
    for i, (b, n) in enumerate(requests):
        c = dict(case, match=0.8)
        asked.append((b, _relations(c, seed * 1000 + 500 + i, builds[b], n)[2:]))
    return sides, asked


# ----------------------------------------------------------------- prepare


def prepare(case, seed):
    kind = case["kind"]
    npt = _dtype(case)[1]
    kt = fij.KeyType.I32 if case["type"] == "i32" else fij.KeyType.I64
    s = {"kind": kind, "type": npt, "kt": kt}
    cus = fij.device_limits()["compute_units"]
    if kind == "batch":
        s["joins"] = [_columns(case, seed * 1000 + i, b, p) for i, (b, p) in enumerate(_sizes(case))]
        s["batch"] = fij.JoinBatch(npt, len(s["joins"]))
    elif kind == "served":
        sides, asked = _served_inputs(case, seed)
        s["server"] = fij.JoinServer(npt, [(8, 1 << 20), (4, 1 << 23)], max_probe_len=1 << 23, table_build_max=1 << 18)
        ids = []
        for bk, bp in sides:
            bk, bp = _column(bk, npt), _column(bp, npt)
            fij.synchronize()
            ids.append(s["server"].add_build(bk, bp))
        s["requests"] = [(ids[b], _column(k, npt), _column(p, npt)) for b, (k, p) in asked]
    elif kind == "ooc":
        s["cols"] = [fij.HostArray.from_numpy(t.cpu().numpy()) for t in _relations(case, seed, case["build"], case["probe"])]
        s["bits"] = (case["bits1"], case["bits2"])
        s["cache"] = int(case["cache"] * (case["build"] + case["probe"]) * 2 * np.dtype(npt).itemsize)
    else:
        s["cols"] = _columns(case, seed, case["build"], case["probe"])
    if kind == "plan":
        bits = (case["bits1"], case["bits2"]) if case["bits1"] else fij.plan_bits(npt, case["build"], case["probe"])
        s["plan"] = fij.JoinPlan(kt, case["build"], case["probe"], *bits)
        s["result"] = torch.zeros(3, dtype=torch.int64, device=DEV) if case["sized"] else None
    elif kind == "operator":
        F, b = fij.HistogramAlgorithm.Contiguous, case["bits1"]
        s["sides"] = []
        for n in (case["build"], case["probe"]):
            part = fij.GpuRadixPartitioner(F, fij.RadixPartitionAlgorithm.SSWWCv2, fij.RadixBits(b), _grid(cus, n, npt), 1024)
            s["sides"].append((part, fij.PartitionOffsets(F, part.grid_size, b, kt), fij.PartitionedRelation(n, F, b, part.grid_size, kt)))
        s["join"] = fij.HipRadixJoin(fij.RadixPass.First, fij.RadixBits(b), fij.HashingScheme.BucketChaining, 2 * cus, 1024)
        s["tasks"] = fij.DeviceArray.zeros(2 * cus + 1, np.uint32)
        s["agg"] = fij.aggregates_array(2 * cus)
    elif kind == "two_pass":
        _prepare_two_pass(s, case, cus)
    elif kind == "np":
        entries = 2
        while entries < 2 * case["build"]:
            entries *= 2
        scheme = fij.HashingScheme.Perfect if case["perfect"] else fij.HashingScheme.LinearProbing
        s["table"] = fij.HashTable(entries, kt)
        s["join"] = fij.HipHashJoin(scheme, s["table"], (2 * cus, 256), (2 * cus, 256))
        s["agg"] = fij.aggregates_array(2 * cus)
    return s


def _grid(cap, n, npt):
    """Chunks of a relation: at most cap, each of at least 128 bytes of keys, the last one not empty."""
    per = 128 // np.dtype(npt).itemsize
    g = max(1, min(cap, n // per))
    while g > 1 and -(-n // g) // per * per * (g - 1) > n:
        g -= 1
    return g


def _prepare_two_pass(s, case, cus):
    kt, npt, (b1, b2) = s["kt"], s["type"], (case["bits1"], case["bits2"])
    bits = fij.RadixBits(b1, b2)
    CH, CO, alg = fij.HistogramAlgorithm.Chunked, fij.HistogramAlgorithm.Contiguous, fij.RadixPartitionAlgorithm.SSWWCv2
    s["F1"], s["sides"] = 1 << b1, []
    for n in (case["build"], case["probe"]):
        g1 = _grid(cus, n, npt)
        most = n  # room for a partition of any length
        g2 = _grid(32, n >> (b1 + 3), npt)
        s["sides"].append({
            "p1": fij.GpuRadixPartitioner(CH, alg, bits, g1, 1024), "p2": fij.GpuRadixPartitioner(CO, alg, bits, g2, 1024),
            "off1": fij.PartitionOffsets(CH, g1, b1, kt), "rel1": fij.PartitionedRelation(n, CH, b1, g1, kt),
            "off2": fij.PartitionOffsets(CO, g2, b2, kt), "rel2": fij.PartitionedRelation(most, CO, b2, g2, kt),
            "keys": fij.DeviceArray(most, npt), "pays": fij.DeviceArray(most, npt)})
    s["join"] = fij.HipRadixJoin(fij.RadixPass.Second, bits, fij.HashingScheme.BucketChaining, 1 << b2, 512)
    s["tasks"] = fij.DeviceArray.zeros((1 << b2) + 1, np.uint32)
    s["agg"] = fij.aggregates_array(1 << b2)


# --------------------------------------------------------------------- run


def run(s):
    kind = s["kind"]
    if kind == "plan":
        if s["result"] is not None:
            s["plan"].enqueue_sized(*s["cols"], s["result"].data_ptr())
            return s["result"]
        return _whole(s["plan"].execute(*s["cols"])[0])
    if kind == "batch":
        return _whole(s["batch"].execute(s["joins"])[0])
    if kind == "served":
        ids = [s["server"].submit(*r) for r in s["requests"]]
        return _whole([s["server"].wait(i)[0] for i in ids])
    if kind == "ooc":
        return _whole(fij.ooc_join(s["type"], *s["cols"], *s["bits"], cache_bytes=s["cache"])[0])
    bk, bp, sk, sp = s["cols"]
    s["agg"].fill(0)
    if kind == "np":
        t = s["table"]
        fij.check(fij.lib.fij_np_table_init(int(t.ktype), fij.C.c_void_p(t.mem.ptr), t.entries, None))
        s["join"].build(bk, bp)
        s["join"].probe_sum(sk, sp, None, s["agg"])
        return _whole(fij.sum_aggregates(s["agg"]))
    if kind == "operator":
        first = fij.RadixPass.First
        for (part, offs, rel), (k, p) in zip(s["sides"], ((bk, bp), (sk, sp))):
            part.prefix_sum(first, k, offs)
            part.partition(first, k, p, offs, rel)
        s["join"].join(s["sides"][0][2], s["sides"][1][2], None, s["tasks"], s["agg"])
        return _whole(fij.sum_aggregates(s["agg"]))
    # two passes: the second one for each partition of the first
    offsets = []
    for side, (k, p) in zip(s["sides"], ((bk, bp), (sk, sp))):
        side["p1"].prefix_sum(fij.RadixPass.First, k, side["off1"])
        side["p1"].partition(fij.RadixPass.First, k, p, side["off1"], side["rel1"])
    for side in s["sides"]:
        offsets.append(side["rel1"].host_offsets())
    for part in range(s["F1"]):
        for side, host in zip(s["sides"], offsets):
            n = side["rel1"].partition_len(part, host)
            keys, pays = side["keys"].view(0, n), side["pays"].view(0, n)
            side["rel2"].resize(n)
            side["p2"].prefix_sum_and_transform(fij.RadixPass.Second, part, side["rel1"], keys, pays, side["off2"])
            side["p2"].partition(fij.RadixPass.Second, keys, pays, side["off2"], side["rel2"])
        s["join"].join(s["sides"][0]["rel2"], s["sides"][1]["rel2"], None, s["tasks"], s["agg"])
    return {"joined": _whole(fij.sum_aggregates(s["agg"])), "offsets": [o.astype(np.int64) for o in offsets]}


def _whole(v):
    """(count, sum of build payloads, sum of probe payloads) of one join or of several, as 64-bit whole numbers."""
    return np.array(v, dtype=np.uint64).view(np.int64)


# -------------------------------------------------------------------- work


def work(case):
    """Every key and payload read once; the operators also write the partitioned relations that they return."""
    t = 2 * _dtype(case)[2]
    if case["kind"] == "batch":
        n = sum(b + p for b, p in _sizes(case))
        return {"bytes": n * t + 24 * case["joins"], "flops": 0}
    if case["kind"] == "served":
        builds, requests = _sizes(case)
        return {"bytes": sum(builds[b] + n for b, n in requests) * t + 24 * len(requests), "flops": 0}
    n = case["build"] + case["probe"]
    return {"bytes": n * t * (2 if case["kind"] in ("operator", "two_pass") else 1) + 24, "flops": 0}


# ------------------------------------------------------------------- exact


def _join(bk, bp, sk, sp):
    """Count and wrapping sums of the equi-join, by sorting the build side; the null key (-1) joins nothing."""
    bk, bp = bk[bk != -1], bp[bk != -1]
    key, at = torch.sort(bk)
    total = torch.zeros(bk.numel() + 1, dtype=torch.int64, device=bk.device)
    torch.cumsum(bp[at].to(torch.int64), 0, out=total[1:])
    got = torch.zeros(3, dtype=torch.int64, device=bk.device)
    for a in range(0, sk.numel(), CHUNK):
        k = sk[a:a + CHUNK]
        lo, hi = torch.searchsorted(key, k), torch.searchsorted(key, k, right=True)
        n = hi - lo
        got += torch.stack([n.sum(), (total[hi] - total[lo]).sum(), (n * sp[a:a + CHUNK].to(torch.int64)).sum()])
    return got.cpu().numpy()


def _chunked_offsets(keys, bits, grid, itemsize):
    """Partition starts of every chunk, each partition behind 128 bytes of padding."""
    F, pad, per = 1 << bits, 128 // (2 * itemsize), 128 // itemsize
    n = keys.numel()
    length = -(-n // grid) // per * per
    out = []
    for c in range(grid):
        end = n if c + 1 == grid else (c + 1) * length
        counts = torch.bincount(keys[c * length:end].to(torch.int64) & (F - 1), minlength=F).cpu().numpy()
        out.append((length + F * pad) * c + np.cumsum(counts) - counts + (np.arange(F) + 1) * pad)
    return np.concatenate(out).astype(np.int64)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return np.stack([_join(*_relations(case, seed * 1000 + i, b, p)) for i, (b, p) in enumerate(_sizes(case))])
    if kind == "served":
        sides, asked = _served_inputs(case, seed)
        return np.stack([_join(*sides[b], *cols) for b, cols in asked])
    rel = _relations(case, seed, case["build"], case["probe"])
    if kind != "two_pass":
        return _join(*rel)
    npt = _dtype(case)[1]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    offsets = [_chunked_offsets(k, case["bits1"], _grid(cus, k.numel(), npt), np.dtype(npt).itemsize) for k in (rel[0], rel[2])]
    return {"joined": _join(*rel), "offsets": offsets}
