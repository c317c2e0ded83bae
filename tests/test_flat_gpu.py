"""GPU tests of the flat form (one open-addressed table in memory for build
sides past an LDS table that an XCD's L2 holds): against the numpy join and
against the partitioned pipeline of the same join, at the edges of its range,
with equal keys up to and past the links it follows, with row ids, 1-based
output, outputs too small, and calls in a row."""
import numpy as np
import pytest

import vjoin
import workloads
from joinref import np_join, sorted_pairs

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ctx():
    c = vjoin.Context(0)
    yield c
    c.close()


def _run(ctx, dr, ds, opts, m, rid=None, sid=None):
    import torch
    o = [torch.full((max(m, 1),), -1, dtype=torch.int32, device="cuda") for _ in range(2)]
    rc, n = ctx.join_into(vjoin.table(dr, rid), vjoin.table(ds, sid), opts, o[0], o[1])
    assert rc == 0 and n == m, (rc, n, m, ctx.last_error())
    return sorted_pairs(o[0][:n].cpu().numpy().view(np.uint32), o[1][:n].cpu().numpy().view(np.uint32))


def _same(a, b):
    return np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


# the largest build side of the form (2^18 rows of 4-byte keys, 2^16 of wider ones) and one row more (the pipeline),
# one row more than the one-launch form takes, probe sides around its thread and block steps
@pytest.mark.parametrize("kw,nc,kind,nr,ns", [
    (4, 1, "fnv", 1537, 1), (4, 1, "fnv", 1 << 18, 1024 * 3 + 1), (4, 1, "custom_xor_hw", (1 << 18) + 1, 4097),
    (4, 1, "fnv", 100_000, (1 << 20) + 1), (8, 1, "fnv", 1 << 16, 65537), (8, 1, "custom_mult", (1 << 16) + 1, 1023),
    (4, 2, "fnv", 40_000, (1 << 20) + 4095), (4, 4, "custom_xor_hw", 1 << 16, 100_001), (8, 3, "fnv", 769, 30_000),
    (8, 4, "custom_add", 5000, (1 << 20) + 7)])
def test_range_edges(ctx, kw, nc, kind, nr, ns):
    rng = np.random.default_rng(nr + ns + nc)
    dt = np.uint32 if kw == 4 else np.uint64
    keys = workloads.mix64(np.arange(2 * nr * nc, dtype=np.uint64)).astype(dt)
    if kw == 4 and nc == 1:
        keys = np.unique(keys)
        keys = keys[rng.permutation(len(keys))]
    keys = keys[:len(keys) // nc * nc].reshape(-1, nc)
    r, s = keys[:nr], keys[rng.integers(0, len(keys), ns)]
    r, s = [r[:, c].copy() for c in range(nc)], [s[:, c].copy() for c in range(nc)]
    want = np_join(workloads.reference_rows(r), workloads.reference_rows(s))
    dr, ds = workloads.to_device(r), workloads.to_device(s)
    for rep in range(2):
        assert _same(_run(ctx, dr, ds, vjoin.join_opts(kind), len(want[0])), want), rep
    flat = nr <= (1 << 18 if kw * nc == 4 else 1 << 16)
    assert (ctx.summary()["partitions"] == 1) == flat
    assert _same(_run(ctx, dr, ds, vjoin.join_opts(kind, tile=vjoin.TILE_LARGE), len(want[0])), want)
    assert ctx.summary()["partitions"] > 1


@pytest.mark.parametrize("kw,nc", [(4, 1), (8, 1), (4, 3)])
@pytest.mark.parametrize("dup", [2, 64, 65, 5000])
def test_equal_keys(ctx, kw, nc, dup):
    """Up to 64 rows of a key are followed link by link; a longer chain hands the join to the pipeline."""
    import torch
    rng = np.random.default_rng(dup + kw)
    dt = np.uint32 if kw == 4 else np.uint64
    nd = max(2, 5000 // dup)
    distinct = workloads.mix64(np.arange(1, nd * nc + 1, dtype=np.uint64)).reshape(nd, nc).astype(dt)
    r = np.repeat(distinct, dup, axis=0)[rng.permutation(nd * dup)]
    s = distinct[rng.integers(0, nd, 300)]
    s[::5, 0] ^= dt(1 << 29)
    r, s = [r[:, c].copy() for c in range(nc)], [s[:, c].copy() for c in range(nc)]
    rid, sid = rng.permutation(len(r[0])).astype(np.uint32) + 3, rng.permutation(300).astype(np.uint32) + 5
    want = np_join(workloads.reference_rows(r), workloads.reference_rows(s), rid, sid)
    want = (want[0] + 1, want[1] + 1)
    m = len(want[0])
    dr, ds = workloads.to_device(r), workloads.to_device(s)
    drid, dsid = workloads.to_device([rid])[0], workloads.to_device([sid])[0]
    opts = vjoin.join_opts(one_based=True)
    for rep in range(3):
        assert _same(_run(ctx, dr, ds, opts, m, drid, dsid), want), rep
    o = [torch.full((m,), -1, dtype=torch.int32, device="cuda") for _ in range(2)]
    rc, n = ctx.join_into(vjoin.table(dr, drid), vjoin.table(ds, dsid), opts, o[0], o[1], capacity=m // 2)
    assert vjoin.STATUS[rc] == "VJ_ERR_CAPACITY" and n == m
    assert (o[0][m // 2:] == -1).all() and (o[1][m // 2:] == -1).all()
    a, b = ctx.join(vjoin.table(dr, drid), vjoin.table(ds, dsid), vjoin.join_opts(one_based=True, out_capacity_hint=3))
    assert _same(sorted_pairs(a.cpu().numpy().view(np.uint32), b.cpu().numpy().view(np.uint32)), want)


def test_no_matches_signed_keys_and_empty_sides(ctx):
    r = np.arange(-3000, 0, dtype=np.int32)
    s = np.arange(-10, 4000, dtype=np.int32)
    dr, ds = workloads.to_device([r]), workloads.to_device([s])
    import torch
    o = [torch.empty(len(s), dtype=torch.int32, device="cuda") for _ in range(2)]
    for signed in (False, True):
        rc, n = ctx.join_into(vjoin.table(dr, key_signed=signed), vjoin.table(ds, key_signed=signed), vjoin.join_opts(), *o)
        assert rc == 0 and n == 10
    rc, n = ctx.join_into(vjoin.table(dr), vjoin.table([ds[0][10:]]), vjoin.join_opts(), *o)
    assert rc == 0 and n == 0
    rc, n = ctx.join_into(vjoin.table(dr), vjoin.table([ds[0][:0]]), vjoin.join_opts(), *o)
    assert rc == 0 and n == 0
