"""GPU tests of batches in the flat form (a table in memory per join, one grid
over all of a batch's blocks): against the numpy join, and the same batch in the
pipeline, with empty sides among the joins, sizes around the block steps, equal
keys up to and past the links it follows, and outputs too small."""
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


def _batch(ctx, joins, opts, wants, cut=None):
    """joins: (build columns, probe columns, build ids or None, probe ids or None), on the device."""
    import torch
    builds = [vjoin.table(r, a) for r, _, a, _ in joins]
    probes = [vjoin.table(s, b) for _, s, _, b in joins]
    caps = [len(w[0]) for w in wants]
    if cut is not None:
        caps[cut] //= 2
    outs = [[torch.full((len(w[0]) + 1,), -1, dtype=torch.int32, device="cuda") for w in wants] for _ in range(2)]
    rc, counts = ctx.join_batch(builds, probes, opts, outs[0], outs[1], caps)
    assert vjoin.STATUS[rc] == ("VJ_OK" if cut is None else "VJ_ERR_CAPACITY"), ctx.last_error()
    assert counts == [len(w[0]) for w in wants]
    for i, w in enumerate(wants):
        a, b = (o[i].cpu().numpy() for o in outs)
        assert (a[caps[i]:] == -1).all() and (b[caps[i]:] == -1).all(), i
        if i != cut:
            got = sorted_pairs(a[:caps[i]].view(np.uint32), b[:caps[i]].view(np.uint32))
            assert np.array_equal(got[0], w[0]) and np.array_equal(got[1], w[1]), i


def _make(rng, kw, nc, sizes, dup, ids):
    joins, wants = [], []
    for nr, ns in sizes:
        dt = np.uint32 if kw == 4 else np.uint64
        nd = max(1, nr // dup)
        keys = workloads.mix64(np.arange(1, 2 * nd * nc + 1, dtype=np.uint64) + np.uint64(nr)).astype(dt).reshape(-1, nc)
        r, s = keys[rng.permutation(nr) % nd], keys[rng.integers(0, len(keys), ns)]
        r, s = [r[:, c].copy() for c in range(nc)], [s[:, c].copy() for c in range(nc)]
        rid = rng.permutation(nr).astype(np.uint32) + 3 if ids else None
        sid = rng.permutation(ns).astype(np.uint32) + 5 if ids else None
        wants.append(np_join(workloads.reference_rows(r), workloads.reference_rows(s), rid, sid))
        dev = [workloads.to_device([x])[0] if ids else None for x in (rid, sid)]
        joins.append((workloads.to_device(r), workloads.to_device(s), *dev))
    return joins, wants


@pytest.mark.parametrize("kw,nc,kind,most", [(4, 1, "fnv", 1 << 18), (4, 1, "custom_mult", 3000), (8, 1, "fnv", 1 << 16),
                                             (4, 2, "custom_xor_hw", 50_000), (4, 3, "fnv", 70_000), (8, 4, "fnv", 20_000)])
@pytest.mark.parametrize("ids", [False, True])
def test_uneven_batches(ctx, kw, nc, kind, most, ids):
    """The largest build side of the form is among them; one more row takes the whole batch to the pipeline."""
    rng = np.random.default_rng(kw * 100 + nc)
    sizes = [(1, 1), (700, 4096), (0, 50), (512, 4097), (513, 2047), (60, 0), (most, 3 * most + 1), (2, 20_000), (0, 0),
             (1537, 8191)]
    joins, wants = _make(rng, kw, nc, sizes, 1, ids)
    for rep in range(2):
        _batch(ctx, joins, vjoin.join_opts(kind), wants)
    _batch(ctx, joins, vjoin.join_opts(kind, tile=vjoin.TILE_LARGE), wants)
    _batch(ctx, joins, vjoin.join_opts(kind), wants, cut=6)


def test_one_row_past_the_range(ctx):
    joins, wants = _make(np.random.default_rng(1), 8, 1, [(100, 300), ((1 << 16) + 1, 70_000), (5000, 5000)], 1, False)
    _batch(ctx, joins, vjoin.join_opts("fnv"), wants)


@pytest.mark.parametrize("kw,nc", [(4, 1), (8, 2)])
@pytest.mark.parametrize("dup", [3, 64, 65, 400])
def test_equal_keys(ctx, kw, nc, dup):
    """A chain past 64 rows in one join of the batch hands all of it to the pipeline."""
    rng = np.random.default_rng(dup)
    joins, wants = _make(rng, kw, nc, [(300, 300), (dup * 9, 700), (40, 9000)], dup, True)
    for rep in range(3):
        _batch(ctx, joins, vjoin.join_opts("fnv"), wants)
