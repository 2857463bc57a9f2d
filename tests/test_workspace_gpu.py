"""The workspace of the calls that take an abs-max (csrc/quantize_common.h): what one launch leaves for the next lies apart from what the
workgroups of a launch exchange, so a launch that exchanges may come in between."""
import pytest

from conftest import load

pytestmark = pytest.mark.gpu

FILL = 0xA5


def test_partials_and_exchanged_words_lie_apart():
    import torch
    integer = load("integer")
    be = integer.Backend.get("cuda:0")
    lib, n = be.lib, be.workspace_bytes
    ws = torch.empty(n, device="cuda", dtype=torch.uint8)
    x = torch.randn(4096, 1024, device="cuda")   # prepareA: 256 workgroups
    w = torch.randn(1024, 1032, device="cuda")   # prepareB: two tiles to a workgroup
    v = torch.randn(1024, 8192, device="cuda")   # prepareB in two launches, as many partials as there are
    few, Bq = x[:64].contiguous(), integer.prepareB(w)
    out = torch.empty(4 << 20 | 256, device="cuda", dtype=torch.int8)
    big = torch.empty(8 << 20 | 256, device="cuda", dtype=torch.int8)
    y = torch.empty(64, 1032, device="cuda")

    def prepare_a():
        return lib.marian_hip_int8_prepare_a(x.data_ptr(), out.data_ptr(), 4096, 1024, ws.data_ptr(), n, be.stream())

    def prepare_b(m):
        return lib.marian_hip_int8_prepare_b(m.data_ptr(), big.data_ptr(), m.shape[0], m.shape[1], ws.data_ptr(), n, be.stream())

    def affine():
        return lib.marian_hip_int8_affine_f32(few.data_ptr(), out.data_ptr(), Bq.data.data_ptr(), None, None, 0, y.data_ptr(), 64, 1024, 1032,
                                              1.0, 0, ws.data_ptr(), n, be.stream())

    def written(*calls, run=lambda f: f()):
        ws.fill_(FILL)
        for c in calls:
            assert run(c) == 0
        torch.cuda.synchronize()
        return (ws.view(torch.int32) != torch.full((4,), FILL, device="cuda", dtype=torch.uint8).view(torch.int32)).cpu()

    def replayed(call):
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            status = call()
        graph.replay()
        return status

    partials = written(lambda: prepare_b(v))
    words = written(prepare_a, lambda: prepare_b(w), affine)
    recorded = written(prepare_a, lambda: prepare_b(w), run=replayed)
    assert partials.sum() >= 900 and words.sum() >= 1024 and recorded.sum() > 1024
    assert not (partials & words).any() and not (partials & recorded).any()


def test_quantizer_of_as_many_partials_as_there_are(orc, synth):
    """two launches; the largest value in the first, in the last and in a middle share"""
    import numpy as np
    import torch
    integer = load("integer")
    K, N = 1088, 4096
    W = synth.normal(77, synth.STREAM_W, (K, N), 0.02)
    for at in (0, K * N - 1, 991 * 1024 * 4 + 17, 992 * 1024 * 4 + 5):
        big = W.copy()
        big.flat[at] = np.float32(0.75)
        assert np.array_equal(integer.prepareB(torch.from_numpy(big).cuda()).file_bytes(), orc.prepare_b(big)), at


def test_threads_that_share_a_stream_and_its_partials():
    """Calls of two launches, the first of which leaves partials for the second, made by threads at once."""
    import threading

    import torch
    integer = load("integer")
    g = torch.Generator(device="cuda")
    g.manual_seed(5)

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, device="cuda", generator=g) * scale

    def work(scale):
        w, x = normal(1024, 8192, scale=scale), normal(64, 1024, scale=scale)
        three = [(integer.prepareB(normal(1024, 1024, scale=0.02)), None) for _ in range(3)]
        return lambda: [integer.prepareB(w).data[:w.numel() + 4], *integer.affine_f32_grouped(x, three)[0]]
    work = [work(scale) for scale in (1.0, 0.25, 4.0, 0.02)]
    want = [w() for w in work]
    torch.cuda.synchronize()
    bad, start = [], threading.Barrier(len(work))

    def run(i):
        start.wait()
        for n in range(40):
            if not all(torch.equal(a, b) for a, b in zip(work[i](), want[i])):
                bad.append((i, n))
    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
