"""Workspaces of destroyed plans are handed to later plans on the same graph:
results do not depend on what a block held before, on plans that live at the
same time, on threads, or on work a destroyed plan had not been waited for."""
import threading

import numpy as np
import pytest

from test_gpu_parity import same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g12(C, O):
    g = C.Graph.rmat(12, 8, weights=True)
    off, adj, w = g.csr(weights=True)
    return g, O.OracleGraph(off, adj, weights=w)


def cases(C, O, g, og):
    out = []
    for i, (n, fan, bias) in enumerate([(1, [3], 0), (900, [10, 5], 1), (40, [4, 4, 4], 2), (0, [5, 5], 0), (300, [64], 2),
                                        (2000, [25, 10], 0), (7, [], 1)]):
        seeds = g.seeds(n, request=i)
        want = O.sample(og, seeds, fan, bias=bias, request=i) if fan else None
        out.append((seeds, fan, bias, i, want))
    return out


def check(C, g, c):
    seeds, fan, bias, i, want = c
    got = C.sample(g, seeds, fan, bias=bias, request=i)
    if want is None:
        assert len(got["src"]) == 0
    else:
        same(got, want, f"request {i}")


def test_blocks_reused_in_any_order(C, O, g12):
    g, og = g12
    cs = cases(C, O, g, og)
    rng = np.random.default_rng(1)
    for _ in range(40):
        check(C, g, cs[rng.integers(len(cs))])


def test_threads_share_one_graph(C, O, g12):
    g, og = g12
    cs = cases(C, O, g, og)
    for c in cs:
        check(C, g, c)  # what the graph builds once, before the threads
    errors = []

    def work(k):
        try:
            for t in range(12):
                check(C, g, cs[(k + t) % len(cs)])
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors[0]


def test_plans_alive_together_and_unwaited(C, O, g12):
    g, og = g12
    cs = [c for c in cases(C, O, g, og) if c[4] is not None]
    spec = lambda c: {"seeds": c[0], "fanouts": c[1], "bias": c[2], "request": c[3]}  # noqa: E731
    plans = [C.Plan(g, [spec(c)], mode=m, cdf_cache=k) for c in cs for m in (0, 1) for k in (False, True)]
    for p in plans:
        p.run()
    for p, c in zip(plans, [c for c in cs for _ in range(4)]):
        same(p.result(0), c[4])
        p.close()
    for c in cs * 3:
        p = C.Plan(g, [spec(c)], mode=C.MODE_BATCHED, cdf_cache=True, use_graph=True)
        p.run(sync=False)
        p.close()  # its block goes back only once the work is done
        check(C, g, c)


def test_plan_outlives_its_graph(C):
    g = C.Graph.rmat(8, 4)
    p = C.Plan(g, [{"seeds": g.seeds(10), "fanouts": [3], "bias": 0}], mode=C.MODE_PLAIN)
    p.run()
    want = p.result(0)
    g.close()
    got = p.result(0)
    for k in want:
        assert np.array_equal(got[k], want[k])
    p.close()
