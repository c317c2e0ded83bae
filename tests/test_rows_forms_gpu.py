"""GPU tests of the reference-layout join where the row-major keys become columns
on different ways: in the histogram of the one-pass form (sizes around its tiles
and steps), and in front of every other form. The numpy join of the rows,
mapped to primary keys, is the reference."""
import numpy as np
import pytest

import vjoin
import workloads
from joinref import np_join

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,nr,ns,kind,opts,budget", [
    (2, 70_001, 4096 * 9 + 1, "fnv", {}, 0),  # one-pass, tiles of 4096 rows
    (2, 200_000, 300_007, "custom_xor_hw", {}, 0),
    (3, 65_537, 131_071, "fnv", {}, 0),
    (4, 90_001, 70_003, "custom_add", {}, 0),
    (2, 300_001, 400_003, "fnv", {"passes": 2, "bits1": 5, "bits2": 6}, 0),  # 2^11 partitions: large tiles
    (3, 100_000, 90_001, "fnv", {"tile": vjoin.TILE_LARGE}, 1 << 30),
    (2, 100_000, 90_001, "fnv", {"passes": 2, "tile": 1}, 0),  # two-pass form
    (2, 40_000, 50_001, "fnv", {}, 0),  # flat form
    (4, 500, 20_001, "fnv", {}, 0),  # one launch
    (2, 0, 100_000, "fnv", {}, 0), (2, 100_000, 0, "fnv", {}, 0)])
def test_rows(nc, nr, ns, kind, opts, budget):
    import torch
    rng = np.random.default_rng(nr + ns)
    keys = workloads.mix64(np.arange(1, 2 * max(nr, 1) * nc + 1, dtype=np.uint64)).reshape(-1, nc)
    r, s = keys[rng.permutation(nr)], keys[rng.integers(0, len(keys), ns)]
    rp, sp = (workloads.mix64(np.arange(n, dtype=np.uint64) + np.uint64(7 * k)) for k, n in ((1, nr), (2, ns)))
    ri, si = np_join(r, s)
    want = np.stack([rp[ri.astype(np.int64)], sp[si.astype(np.int64)]], 1)
    want = want[np.lexsort((want[:, 1], want[:, 0]))]
    ctx = vjoin.Context(0)
    if budget:
        ctx.set_budget(budget)
    dev = [torch.from_numpy(np.ascontiguousarray(x).view(np.int64)).cuda() for x in (r, rp, s, sp)]
    for rep in range(2):
        before = [x.clone() for x in dev]
        v, k = ctx.join_rows(*dev, vjoin.join_opts(kind, **opts))
        got = v.cpu().numpy().view(np.uint64)
        assert np.array_equal(got[np.lexsort((got[:, 1], got[:, 0]))], want), rep
        assert np.array_equal(k.cpu().numpy(), np.arange(1, len(want) + 1))
        assert all(torch.equal(a, b) for a, b in zip(dev, before))
    ctx.close()
