"""GPU test of a join's device time where it comes from the device's clock: in
every form of the one-pass pipeline it is positive, within the time the host
waited, and close to what events around the same stages say."""
import time

import pytest

import vjoin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,ns,form", [(1 << 10, 1 << 13, "one launch"), (1 << 16, 1 << 20, "flat"),
                                        (1 << 20, 1 << 23, "partitioned"), (1 << 20, 1 << 23, "replayed")])
def test_device_time(nr, ns, form):
    import torch
    ctx = vjoin.Context(0)
    r = torch.randperm(nr, device="cuda").to(torch.int32)
    s = torch.randint(0, 2 * nr, (ns,), device="cuda", dtype=torch.int32)
    o = [torch.empty(ns, dtype=torch.int32, device="cuda") for _ in range(2)]
    opts = vjoin.join_opts()
    clock = []
    for rep in range(6):
        torch.cuda.synchronize()
        t = time.perf_counter()
        rc, n = ctx.join_into(vjoin.table([r]), vjoin.table([s]), opts, *o)
        host = (time.perf_counter() - t) * 1e3
        assert rc == 0
        sm = ctx.summary()
        assert 0 < sm["ms_total"] < host, (rep, sm["ms_total"], host)
        clock.append(sm["ms_total"])
        if form == "replayed" and rep > 2:
            assert sm["graph_replay"] == 1
    if form == "partitioned":
        ctx.set_profiling(True)
        events = []
        for rep in range(5):
            rc, n = ctx.join_into(vjoin.table([r]), vjoin.table([s]), opts, *o)
            events.append(ctx.summary()["ms_total"])
        # the same kernels; events add the launches' gaps (some us each) to some 150 us
        assert 0.4 < min(clock) / min(events) < 1.1, (clock, events)
    ctx.close()
