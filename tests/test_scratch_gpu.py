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


def test_scratch_is_bounded_and_given_back():
    """A piece of the size that is asked for, a stream at a time, of a bounded number of streams, until it is asked back."""
    import torch
    integer = load("integer")
    release = integer.Backend.releaseScratch
    w = integer.prepareB(torch.randn(512, 512, device="cuda") * 0.02)
    streams = [torch.cuda.Stream() for _ in range(24)]
    xs = {m: torch.randn(m, 512, device="cuda") for m in (1, 300, 64)}

    def grown(m, over):
        """bytes that stay after calls of m rows"""
        for s in over:
            with torch.cuda.stream(s):
                out = integer.dot(xs[m], w)
            s.synchronize()
            del out
        return torch.cuda.memory_allocated() - before
    for s in streams:   # workspaces, which are kept for good
        with torch.cuda.stream(s):
            integer.affine_f32(xs[1], w)
        s.synchronize()
    release()
    before = torch.cuda.memory_allocated()
    assert 0 < grown(1, streams[:1]) <= 4096
    assert 4096 < grown(300, streams[:1]) <= 256 << 10          # a larger piece takes its place
    assert grown(64, streams[:1]) <= 256 << 10                  # and serves smaller calls
    assert grown(1, streams) <= (256 << 10) + 15 * 4096          # sixteen streams at the most
    release()
    assert torch.cuda.memory_allocated() == before
    assert 0 < grown(1, streams[-1:]) <= 4096                   # and again
    big = torch.randn(2300, 512, device="cuda")                  # more than a piece: never kept
    release()
    before = torch.cuda.memory_allocated()
    out = integer.dot(big, w)
    torch.cuda.synchronize()
    del out
    assert torch.cuda.memory_allocated() == before
