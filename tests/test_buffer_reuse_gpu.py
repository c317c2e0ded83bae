"""GPU tests of the kept output buffers: results stay right when buffers of
other sizes and other contexts are handed out again, from several threads and
streams, and the buffers are given back with the last context."""
import threading

import numpy as np
import pytest

import vjoin
import workloads
from joinref import np_join, sorted_pairs

pytestmark = pytest.mark.gpu


def _inputs(nr, ns, seed):
    rng = np.random.default_rng(seed)
    r = rng.permutation(nr).astype(np.uint32)
    s = rng.integers(0, 2 * nr, ns).astype(np.uint32)
    return r, s, np_join(r.reshape(-1, 1).astype(np.uint64), s.reshape(-1, 1).astype(np.uint64))


def _check(ctx, r, s, want, opts):
    dr, ds = workloads.to_device([r]), workloads.to_device([s])
    a, b = ctx.join(vjoin.table(dr), vjoin.table(ds), opts)
    got = sorted_pairs(a.cpu().numpy().view(np.uint32), b.cpu().numpy().view(np.uint32))
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


def test_results_over_changing_sizes_contexts_and_regrown_outputs():
    a, b = vjoin.Context(0), vjoin.Context(0)
    try:
        for k, (nr, ns) in enumerate([(3000, 50000), (3000, 50000), (2900, 31000), (20000, 90001), (10, 20), (3000, 50000)]):
            r, s, want = _inputs(nr, ns, k)
            for c in (a, b):
                _check(c, r, s, want, vjoin.join_opts())
                _check(c, r, s, want, vjoin.join_opts(out_capacity_hint=7))  # too small: grown again
    finally:
        a.close()
        b.close()


def test_threads_with_streams_of_their_own():
    import torch
    work = [_inputs(4000 + 100 * k, 60000 + 999 * k, 50 + k) for k in range(4)]
    failed = []

    def one(k):
        try:
            c = vjoin.Context(0)
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(5):
                    _check(c, *work[k], vjoin.join_opts())
            c.close()
        except Exception as e:  # reported by the main thread
            failed.append((k, repr(e)))
    threads = [threading.Thread(target=one, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


def test_kept_buffers_go_back_with_the_last_context():
    import gc
    import torch
    gc.collect()  # contexts of earlier tests
    r, s, want = _inputs(1000, 4000, 9)
    c = vjoin.Context(0)
    _check(c, r, s, want, vjoin.join_opts())
    before = torch.cuda.mem_get_info()[0]
    hint = 48 << 20  # two columns of 192 MiB
    _check(c, r, s, want, vjoin.join_opts(out_capacity_hint=hint))
    held = before - torch.cuda.mem_get_info()[0]
    assert held <= 1 << 30  # what is kept is bounded
    _check(c, r, s, want, vjoin.join_opts(out_capacity_hint=hint))
    assert before - torch.cuda.mem_get_info()[0] <= held + (16 << 20)  # and used again
    c.set_budget(4 << 30)  # a budget: buffers of this context's own
    _check(c, r, s, want, vjoin.join_opts(out_capacity_hint=hint))
    assert before - torch.cuda.mem_get_info()[0] <= held + (16 << 20)
    c.close()
    alive = [o for o in gc.get_objects() if type(o) is vjoin.Context and o.ptr]
    if not alive:
        assert before - torch.cuda.mem_get_info()[0] < 192 << 20
