"""GPU tests of the one-pass form (up to 11 radix bits in one pass, atomically
reserved runs) and of the chained LDS tables: sizes around the tile, group and
table edges, against the numpy join and against the two-pass form of the same
plan (the standard tile shape asks for it)."""
import numpy as np
import pytest

import vjoin
import workloads
from joinref import np_join, sorted_pairs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = vjoin.Context(0)
    yield c
    c.close()


def _keys(rng, nr, ns, kw, nc, dup):
    """Build keys (each `dup` times), probe keys of which a third miss."""
    dt = np.uint32 if kw == 4 else np.uint64
    nd = max(1, nr // dup)
    distinct = workloads.mix64(np.arange(1, nd * nc + 1, dtype=np.uint64)).reshape(nd, nc).astype(dt)
    r = distinct[rng.permutation(nr) % nd]
    s = distinct[rng.integers(0, nd, ns)]
    if ns:
        s[::3, 0] ^= dt(1 << 30)
    return [r[:, c].copy() for c in range(nc)], [s[:, c].copy() for c in range(nc)]


def _pairs(ctx, dr, ds, opts, m, rid=None, sid=None):
    import torch
    o = [torch.full((max(m, 1),), -1, dtype=torch.int32, device="cuda") for _ in range(2)]
    rc, n = ctx.join_into(vjoin.table(dr, rid), vjoin.table(ds, sid), opts, o[0], o[1])
    assert rc == 0 and n == m, (rc, n, m, ctx.last_error())
    return sorted_pairs(o[0][:n].cpu().numpy().view(np.uint32), o[1][:n].cpu().numpy().view(np.uint32))


# (key bytes, columns, build rows, probe rows, rows per key, hash kind, plan): tiles are 4096 rows (12288, 8192 or
# 6144 by key bytes at 11 bits), nine tiles make cursor groups, a group's last tile may be one row
EDGES = [
    (4, 1, 1, 1, 1, "fnv", dict(passes=1, bits1=1)),
    (8, 1, 4096, 4097, 1, "fnv", dict(passes=1, bits1=8)),
    (4, 1, 8 * 4096, 8 * 4096 + 1, 1, "fnv", dict(passes=2, bits1=5, bits2=5)),
    (8, 1, 12288, 9 * 12288 + 1, 2, "fnv", dict(passes=2, bits1=6, bits2=5)),
    (8, 1, 8 * 12288 + 1, 8 * 12288, 1, "custom_xor_hw", dict(passes=2, bits1=3, bits2=8)),
    (4, 3, 8192, 9 * 8192 - 1, 3, "fnv", dict(passes=2, bits1=8, bits2=3)),
    (4, 4, 40000, 8 * 8192 + 1, 4, "custom_xor_hw", dict(passes=2, bits1=6, bits2=5)),
    (8, 4, 6144, 9 * 6144 + 1, 1, "fnv", dict(passes=2, bits1=6, bits2=5)),
    (8, 3, 30000, 8 * 4096 + 5, 2, "custom_mult", dict(passes=1, bits1=5)),
    (8, 2, 50000, 70001, 1, "fnv", dict(passes=2, bits1=4, bits2=3, table=vjoin.TABLE_WIDE)),
    # several walks per task and several tasks per partition, one build chunk more than a table holds
    (8, 1, 8193, 200003, 1, "fnv", dict(passes=0, table=vjoin.TABLE_WIDE)),
    (8, 1, 60000, 400003, 5, "fnv", dict(passes=1, bits1=2, table=vjoin.TABLE_WIDE)),
    (4, 1, 2049, 40000, 1, "fnv", dict(passes=0, table=vjoin.TABLE_STANDARD)),
]


@pytest.mark.parametrize("case", EDGES)
def test_edges_match_numpy_and_two_passes(ctx, case):
    kw, nc, nr, ns, dup, kind, plan = case
    rng = np.random.default_rng(nr * 31 + ns)
    r, s = _keys(rng, nr, ns, kw, nc, dup)
    want = np_join(workloads.reference_rows(r), workloads.reference_rows(s))
    dr, ds = workloads.to_device(r), workloads.to_device(s)
    one = _pairs(ctx, dr, ds, vjoin.join_opts(kind, **plan), len(want[0]))
    sm = ctx.summary()
    assert sm["bytes_pass2"] == 0  # at most one pass over the rows
    two = _pairs(ctx, dr, ds, vjoin.join_opts(kind, tile=vjoin.TILE_STANDARD, **plan), len(want[0]))
    for got in (one, two):
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), case


def test_one_key_only(ctx):
    """Every row in one partition and one chain: runs as long as a tile, build chunks of one key."""
    r = np.full(9001, 5, dtype=np.uint32)
    s = np.full(40, 5, dtype=np.uint32)
    s[::2] = 6
    want = np_join(r.reshape(-1, 1).astype(np.uint64), s.reshape(-1, 1).astype(np.uint64))
    dr, ds = workloads.to_device([r]), workloads.to_device([s])
    for plan in (dict(passes=2, bits1=6, bits2=5), dict(passes=1, bits1=4, table=vjoin.TABLE_WIDE), dict()):
        got = _pairs(ctx, dr, ds, vjoin.join_opts(**plan), len(want[0]))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), plan


@pytest.mark.parametrize("budget", [0, 1 << 40])
def test_kept_and_resident_tables_use_their_own_bits(budget):
    """Sizes where the one-pass and the two-pass form take different radix bits: what is admitted under a budget
    is the latter's need, what is kept and probed later is partitioned as the former says."""
    import torch
    rng = np.random.default_rng(5)
    nr, ns = 200_003, 300_001
    r, s = _keys(rng, nr, ns, 4, 1, 1)
    want = np_join(workloads.reference_rows(r), workloads.reference_rows(s))
    dr, ds = workloads.to_device(r), workloads.to_device(s)
    o = [torch.empty(ns, dtype=torch.int32, device="cuda") for _ in range(2)]
    srv = vjoin.Server(0, budget=budget, max_batch=4)
    try:
        first = srv.wait(srv.submit(vjoin.table(ds), o[0], o[1], build=vjoin.table(dr), keep_build=True))
        assert first["status"] == 0 and first["count"] == len(want[0]) and first["table"] > 0, first
        again = srv.wait(srv.submit(vjoin.table(ds), o[0], o[1], table=first["table"]))
        assert again["status"] == 0 and again["count"] == len(want[0])
        got = sorted_pairs(*(x[:len(want[0])].cpu().numpy().view(np.uint32) for x in o))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    finally:
        srv.close()
    c = vjoin.Context(0)
    try:
        c.set_budget(budget)
        built = c.build(vjoin.table(dr), vjoin.join_opts())
        rc, n = c.probe_into(built, vjoin.table(ds), vjoin.join_opts(), o[0], o[1])
        assert rc == 0 and n == len(want[0])
        got = sorted_pairs(*(x[:n].cpu().numpy().view(np.uint32) for x in o))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        built.free()
    finally:
        c.close()


@pytest.mark.parametrize("kw,nc,kind", [(4, 1, "fnv"), (8, 1, "custom_xor_hw"), (4, 3, "custom_add"), (8, 4, "fnv")])
@pytest.mark.parametrize("nr,ns,dup", [(1, 1, 1), (1, 5000, 1), (1536, 1025, 3), (1537, 40000, 1), (700, 200001, 700)])
def test_one_launch_form(ctx, kw, nc, kind, nr, ns, dup):
    """A build side that fits one table: row ids, 1-based output, an output too small and then regrown, calls in a
    row (its counters start from zero each time); per-stage timing takes the pipeline instead."""
    import torch
    rng = np.random.default_rng(nr + ns)
    r, s = _keys(rng, nr, ns, kw, nc, dup)
    rid, sid = rng.permutation(nr).astype(np.uint32) + 7, rng.permutation(ns).astype(np.uint32) + 9
    want = np_join(workloads.reference_rows(r), workloads.reference_rows(s), rid, sid)
    want = (want[0] + 1, want[1] + 1)
    m = len(want[0])
    dr, ds = workloads.to_device(r), workloads.to_device(s)
    drid, dsid = workloads.to_device([rid])[0], workloads.to_device([sid])[0]
    opts = vjoin.join_opts(kind, one_based=True)
    for timed in (False, False, True, False):
        ctx.set_profiling(timed)
        got = _pairs(ctx, dr, ds, opts, m, drid, dsid)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    if m > 1:
        o = [torch.full((m,), -1, dtype=torch.int32, device="cuda") for _ in range(2)]
        rc, n = ctx.join_into(vjoin.table(dr, drid), vjoin.table(ds, dsid), opts, o[0], o[1], capacity=m - 1)
        assert vjoin.STATUS[rc] == "VJ_ERR_CAPACITY" and n == m and int(o[0][m - 1]) == -1 == int(o[1][m - 1])
    a, b = ctx.join(vjoin.table(dr, drid), vjoin.table(ds, dsid), vjoin.join_opts(kind, one_based=True, out_capacity_hint=1))
    got = sorted_pairs(a.cpu().numpy().view(np.uint32), b.cpu().numpy().view(np.uint32))
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
