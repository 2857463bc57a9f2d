"""Log-softmax and n-best in one launch where its collection of candidates can go wrong: equal scores within a thread's values, within a wave
and over all of them, best words that lie side by side, rows that end within a vector, more than can be collected, NaN and infinities -
against the separate launches."""
import pytest

from conftest import load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [4100, 8192, 16388, 32000, 32768])
@pytest.mark.parametrize("N", [1, 6, 16])
def test_collection(vocab, N):
    import torch
    ops = load("ops")
    beam, batch = 2, 3
    g = torch.Generator(device="cuda")
    g.manual_seed(vocab + N)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)

    def forms():
        yield "spread", r(beam, batch, vocab)
        x = r(beam, batch, vocab)
        x[..., 1000:1000 + 40] += 20.0                       # best words of neighbouring threads, several to a thread
        yield "side by side", x
        yield "few values", (r(beam, batch, vocab) * 1.5).round()
        x = torch.zeros(beam, batch, vocab, device="cuda")
        yield "all equal", x
        x = r(beam, batch, vocab)
        x[..., 4096 * 0 + 5::4096] = 9.0                     # one thread's values
        yield "one thread", x
        x = r(beam, batch, vocab)
        x[..., -1], x[..., -4] = 30.0, 31.0                  # the row's last vector
        yield "last", x
        x = r(beam, batch, vocab) * 1e-3 + 1e4               # differences below the score's last place
        yield "rounded together", x
        x = r(beam, batch, vocab)
        x[0, 0, 17], x[1, 1, 18], x[0, 2, 19] = float("nan"), float("inf"), float("-inf")
        x[1, 2] = float("-inf")
        yield "not finite", x

    for name, x in forms():
        for scores in (None, r(beam, batch)):
            print("collection", vocab, N, name, scores is not None, flush=True)
            lp = ops.logsoftmax(x)
            want_lp = lp
            if scores is not None:
                lp = lp + scores[..., None]
            want = ops.getNBestListOfBeams(lp, N)
            got = ops.logsoftmaxNBestOfBeams(x, N, pathScores=scores, want_logprobs=True)
            for a, b in zip(got[:2], want):
                assert torch.equal(a, b) or (torch.equal(torch.isnan(a.float()), torch.isnan(b.float()))
                                             and torch.equal(torch.nan_to_num(a.float()), torch.nan_to_num(b.float()))), name
            assert torch.equal(torch.nan_to_num(got[2]), torch.nan_to_num(want_lp)) and torch.equal(torch.isnan(got[2]), torch.isnan(want_lp))
            again = ops.logsoftmaxNBestOfBeams(x, N, pathScores=scores)
            assert all(torch.equal(torch.nan_to_num(a.float()), torch.nan_to_num(b.float())) for a, b in zip(again[:2], got[:2])), name
