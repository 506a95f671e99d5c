"""Requests of a server are planned by several threads at once: results must be
those of a request submitted alone, whatever thread submits and whichever plan
is ready first, an error stays with its request, and a server that is closed
with requests still to plan ends."""
import threading

import numpy as np
import pytest

import kate_amd as K
from kate_amd import workloads as W
from test_gpu_server import make_requests

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count,submitters", [(1, 1), (9, 1), (40, 4)])
def test_concurrent_planning_is_bitwise_the_same(gpu, count, submitters):
    print("server planners", count, submitters, flush=True)
    reqs = make_requests(count, 11, 12, 18)
    with K.Server(dtype="c128", streams=4, max_active=16, hbm_budget_bytes=2 << 30) as srv:
        alone = [srv.wait(srv.submit(K.Circuit(n, g), m, tp))[0] for n, g, tp, m in reqs]
    got = [None] * count
    with K.Server(dtype="c128", streams=4, max_active=16, hbm_budget_bytes=2 << 30) as srv:

        def run(first):
            mine = range(first, count, submitters)
            ids = [(i, srv.submit(K.Circuit(reqs[i][0], reqs[i][1]), reqs[i][3], reqs[i][2])) for i in mine]
            for i, rid in ids:
                got[i] = srv.wait(rid)[0]

        threads = [threading.Thread(target=run, args=(k,)) for k in range(submitters)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    for a, b in zip(alone, got):
        assert np.array_equal(a, b)


def test_refused_request_between_others_and_close_with_a_queue(gpu):
    print("server planners: budget, close", flush=True)
    reqs = make_requests(6, 13, 12, 14)
    srv = K.Server(dtype="c128", streams=2, max_active=4, hbm_budget_bytes=64 << 20)
    ids = [srv.submit(K.Circuit(n, g), m, tp) for n, g, tp, m in reqs[:3]]
    big = srv.submit(K.Circuit(24, W.layered(24, 2, 5)), [1])
    ids += [srv.submit(K.Circuit(n, g), m, tp) for n, g, tp, m in reqs[3:]]
    with pytest.raises(K.KateError):
        srv.wait(big)
    for rid in ids:
        z, _ = srv.wait(rid)
        assert np.all(np.isfinite(z))
    for _ in range(3):
        for n, g, tp, m in reqs:
            srv.submit(K.Circuit(n, g), m, tp)
    srv.close()
