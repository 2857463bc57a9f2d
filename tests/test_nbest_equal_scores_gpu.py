"""Log-softmax and n-best in one launch: waves in which none, one or several threads hold scores that reach the bound, one or several of a thread's
values among them, and as many candidates as can be collected, one fewer and one more - against the separate launches."""
import pytest

from conftest import load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [4100, 32000, 32768])
@pytest.mark.parametrize("N", [1, 6, 16])
def test_threads_of_a_wave(vocab, N):
    import torch
    ops = load("ops")
    g = torch.Generator(device="cuda")
    g.manual_seed(vocab + N)
    last = vocab // 4 - 1
    # of thread t of 1024 and its vector j, word 4 (1024 j + t)
    held = {"one thread of a wave": [0], "two of a wave": [64, 127], "two of one wave, one of another": [128, 190, 512], "all of a wave": range(192, 256),
            "one of every wave": range(5, 1024, 64), "two of every wave": [64 * w + i for w in range(16) for i in (0, 63)], "the last vector": [last, 1],
            "1023": range(1023), "1024": range(1024), "1025": list(range(1024)) + [last]}
    for name, vectors in held.items():
        for values in ((0,), (3,), (0, 1, 2, 3)):
            if len(values) > 1 and name[0] == "1":
                continue
            print("threads of a wave", vocab, N, name, values, flush=True)
            x = torch.randn(1, 2, vocab, device="cuda", generator=g)
            at = torch.tensor([4 * v + e for v in vectors for e in values], device="cuda")
            x[0, 0, at] = 9.0
            x[0, 1, at] = 9.0 + 0.25 * torch.randint(0, 3, (len(at),), device="cuda", generator=g)
            want_lp = ops.logsoftmax(x)
            want = ops.getNBestListOfBeams(want_lp, N)
            got = ops.logsoftmaxNBestOfBeams(x, N)
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), name
