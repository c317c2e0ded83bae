"""GPU test of the flat form past one L2's size (up to 2^17 build rows of keys over
4 bytes, probe sides of the build side's size up to 2^21 rows): the edges of that
range against the numpy join and against the pipeline."""
import numpy as np
import pytest

import vjoin
import workloads
from joinref import np_join, sorted_pairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw,nc,nr,ns,flat", [
    (8, 1, (1 << 16) + 1, (1 << 16) + 1, True), (8, 1, 1 << 17, 1 << 21, True), (8, 1, 1 << 17, (1 << 21) + 1, False),
    (8, 1, (1 << 17) + 1, 1 << 18, False), (8, 1, 100_000, 99_999, False), (4, 4, 1 << 17, (1 << 17) + 3, True),
    (8, 4, 90_001, 300_001, True), (4, 1, (1 << 18) + 1, 1 << 19, False)])
def test_edges(kw, nc, nr, ns, flat):
    import torch
    rng = np.random.default_rng(nr + ns)
    keys = np.unique(workloads.mix64(np.arange(1, 2 * nr * nc + 1, dtype=np.uint64)).astype(np.uint32 if kw == 4 else np.uint64))
    keys = rng.permutation(keys)
    keys = keys[:len(keys) // nc * nc].reshape(-1, nc)
    r, s = keys[:nr], keys[rng.integers(0, len(keys), ns)]
    r, s = [r[:, c].copy() for c in range(nc)], [s[:, c].copy() for c in range(nc)]
    want = np_join(workloads.reference_rows(r), workloads.reference_rows(s))
    dr, ds = workloads.to_device(r), workloads.to_device(s)
    ctx = vjoin.Context(0)
    m = len(want[0])
    for opts in (vjoin.join_opts(), vjoin.join_opts(), vjoin.join_opts(tile=vjoin.TILE_LARGE)):
        o = [torch.full((m + 1,), -1, dtype=torch.int32, device="cuda") for _ in range(2)]
        rc, n = ctx.join_into(vjoin.table(dr), vjoin.table(ds), opts, *o)
        assert rc == 0 and n == m
        assert (ctx.summary()["partitions"] == 1) == (flat and opts.tile == 0)
        got = sorted_pairs(o[0][:n].cpu().numpy().view(np.uint32), o[1][:n].cpu().numpy().view(np.uint32))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    ctx.close()
