"""csaw_plan_copy_device fills caller-owned device buffers with the same edge
lists csaw_plan_copy returns on the host.  The buffers come from the HIP
runtime the library itself links (libamdhip64.so.7): a framework that hands
its own device memory to the library must share that runtime."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Hip:
    def __init__(self):
        self.L = ctypes.CDLL("libamdhip64.so.7")
        self.L.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
        self.L.hipFree.argtypes = [ctypes.c_void_p]
        self.L.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]

    def alloc(self, nbytes):
        p = ctypes.c_void_p()
        assert self.L.hipMalloc(ctypes.byref(p), max(nbytes, 4)) == 0
        return p

    def to_host(self, p, n, dtype):
        out = np.zeros(max(n, 1), dtype)
        assert self.L.hipMemcpy(out.ctypes.data, p, n * out.itemsize, 2) == 0  # device to host
        return out[:n]


def test_plan_copy_device(C):
    hip = Hip()
    g = C.Graph.rmat(14, 8, weights=True)
    specs = []
    for i, (fan, bias) in enumerate([([5, 3], 0), ([4, 2, 2], 1), ([6], 2), ([3, 0], 1)]):
        specs.append({"seeds": g.seeds(300 + 50 * i, request=i), "fanouts": fan, "bias": bias, "dedup": 1,
                      "key": 42, "request": i})
    for mode in (C.MODE_PLAIN, C.MODE_BATCHED):
        p = C.Plan(g, specs, mode=mode)
        p.run()
        for r, spec in enumerate(specs):
            want = p.result(r)
            n = p.n_edges(r)
            S, D = len(spec["seeds"]), len(spec["fanouts"])
            bufs = [hip.alloc(4 * n), hip.alloc(4 * n), hip.alloc(4 * n), hip.alloc(8 * D * (S + 1))]
            try:
                st = C.lib().csaw_plan_copy_device(p.h, r, bufs[0], bufs[1], bufs[2], bufs[3], None, 1)
                assert st == 0, C.last_error()
                got = {"src": hip.to_host(bufs[0], n, np.int32), "dst": hip.to_host(bufs[1], n, np.int32),
                       "smp": hip.to_host(bufs[2], n, np.int32),
                       "hop_off": hip.to_host(bufs[3], D * (S + 1), np.int64).reshape(D, S + 1)}
                for k in ("src", "dst", "smp", "hop_off"):
                    assert np.array_equal(got[k], want[k]), (mode, r, k)
            finally:
                for b in bufs:
                    hip.L.hipFree(b)
        p.close()


@pytest.mark.parametrize("shift", [0, 1, 2, 3])
@pytest.mark.parametrize("sync", [True, False])
def test_plan_copy_device_alignments(C, shift, sync):
    """Requests of 1 to 13 samples packed one after another from `shift`
    elements into the buffers: every alignment of source and destination, heads
    and tails shorter than four elements, a request without edges, and the
    bounds of a run that was not waited for by the call itself."""
    hip = Hip()
    g = C.Graph.rmat(10, 4)
    off, adj = g.csr()
    deg = np.diff(off)
    specs = [{"seeds": g.seeds(n, request=n), "fanouts": [3, 2], "bias": n % 2, "dedup": n % 2, "request": n}
             for n in range(1, 14)]
    specs.append({"seeds": np.nonzero(deg == 0)[0][:5].astype(np.int32), "fanouts": [2, 2], "bias": 0, "request": 20})
    p = C.Plan(g, specs, mode=C.MODE_BATCHED, use_graph=True, cdf_cache=True)
    p.run(sync=sync)
    if not sync:
        assert hip.L.hipDeviceSynchronize() == 0
    want = [p.result(r) for r in range(len(specs))]
    total = sum(len(w["src"]) for w in want) + shift
    bufs = [hip.alloc(4 * (total + 4)) for _ in range(3)]
    try:
        at = shift
        for r in range(len(specs)):
            st = C.lib().csaw_plan_copy_device(p.h, r, bufs[0].value + 4 * at, bufs[1].value + 4 * at,
                                               bufs[2].value + 4 * at, None, None, 1)
            assert st == 0, C.last_error()
            at += len(want[r]["src"])
        for buf, k in zip(bufs, ("src", "dst", "smp")):
            got = hip.to_host(buf, at, np.int32)[shift:]
            assert np.array_equal(got, np.concatenate([w[k] for w in want])), k
    finally:
        for b in bufs:
            hip.L.hipFree(b)
    p.close()
