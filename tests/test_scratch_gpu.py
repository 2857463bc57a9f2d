"""Memory that small calls give back to their stream (csrc/host_calls.cpp, Scratch): threads that share a stream, and recorded calls."""
import threading

import pytest

from conftest import load

pytestmark = pytest.mark.gpu


def calls(seed):
    import torch
    integer, types = load("integer"), load("types")
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    # two launches over the scratch, one, and the 16-bit path with a quantizer in front
    made = [(integer.prepareB(torch.randn(k, n, device="cuda", generator=g) * 0.02, types.Type[t]), torch.randn(m, k, device="cuda", generator=g))
            for m, k, n, t in ((300, 1024, 512, "intgemm8"), (16, 512, 512, "intgemm8"), (200, 1024, 2048, "intgemm16"))]
    return lambda: [integer.dot(x, w) for w, x in made]


def test_threads_that_share_a_stream():
    import torch
    work = [calls(s) for s in range(4)]
    want = [w() for w in work]
    torch.cuda.synchronize()
    bad = []

    def run(i):
        for _ in range(60):
            if any(not torch.equal(a, b) for a, b in zip(work[i](), want[i])):
                bad.append(i)
    threads = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_recorded_calls_share_nothing():
    import torch
    work = [calls(s) for s in range(2)]
    want = [w() for w in work]
    graphs, outs = [], []
    for w in work:
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            outs.append(w())
    for _ in range(3):
        for g in graphs:
            g.replay()
        again = work[0]()
        torch.cuda.synchronize()
        for got, w in zip(outs + [again], want + [want[0]]):
            assert all(torch.equal(a, b) for a, b in zip(got, w))
            for t in got:
                t.zero_()
