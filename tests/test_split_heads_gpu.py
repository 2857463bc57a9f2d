"""Keys and values as SplitHeads leaves them - views of an affine call's output, a position's heads side by side - in the
calls that are made for caches of memory of their own: the same results, the same refusals."""
import pytest

from conftest import load

pytestmark = pytest.mark.gpu


def same(a, b):
    import torch
    return a.shape == b.shape and torch.equal(a.contiguous().view(torch.int32), b.contiguous().view(torch.int32))


def inputs(hyps, sentences, heads, length, seed):
    """x [M, K], three projections, a source mask and the rows whose heads are keys and values"""
    import torch
    integer = load("integer")
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    K = heads * 64
    weights = [(integer.prepareB(r(K, K) * 0.02), r(K) if i != 1 else None) for i in range(3)]
    mask = -1e8 * (torch.rand(sentences, length, device="cuda", generator=g) < 0.3).float()
    mask[:, 0] = 0.0
    return r, r(hyps * sentences, K), weights, mask, r(1, sentences, length, K), r(1, sentences, length, K)


@pytest.mark.parametrize("hyps,sentences,heads,length,used", [
    (1, 1, 2, 1, None), (6, 1, 8, 23, None), (4, 3, 16, 96, 95), (1, 7, 4, 97, None), (3, 2, 8, 512, 300), (5, 2, 2, 9, 1)])
def test_query_projection_over_views(hyps, sentences, heads, length, used):
    ops = load("ops")
    _, x, weights, mask, keys, values = inputs(hyps, sentences, heads, length, 100 * hyps + length)
    mask = mask[:, :used].contiguous()
    k, v = ops.SplitHeads(keys, heads), ops.SplitHeads(values, heads)
    assert length == 1 or not k.is_contiguous()
    args = dict(kvLen=used, mask=mask, want_absmax=True, want_projections=True)
    got = ops.ProjectedAttention(x, weights[:1], k, v, heads, **args)
    want = ops.ProjectedAttention(x, weights[:1], k.contiguous(), v.contiguous(), heads, **args)
    assert same(got[0], want[0]) and same(got[3][0], want[3][0])
    assert got[2].data.max().item() == want[2].data.max().item()


def test_query_projection_over_views_refuses_what_it_refuses_over_copies():
    import torch
    integer, ops = load("integer"), load("ops")
    r, x, weights, mask, keys, values = inputs(2, 3, 8, 20, 5)
    wide = [(integer.prepareB(r(512, 1024) * 0.02), None)]
    long = [(integer.prepareB(r(576, 512) * 0.02), None)]
    heads8 = [ops.SplitHeads(t, 8) for t in (keys, values)]
    heads16 = [ops.SplitHeads(t, 16) for t in (keys, values)]
    other = ops.SplitHeads(r(1, 3, 19, 512), 8)
    calls = [(x, weights[:1], *heads8, 4, None),       # heads of another number than the weights'
             (x, wide, *heads8, 8, None),              # columns of another number than the heads'
             (x, weights[:1], *heads16, 16, None),     # heads of 32
             (x[:, :448], weights[:1], *heads8, 8, None), (x[:, :448], weights[:1], *heads8, 7, None),
             (x, weights[:1], heads8[0], other, 8, None),
             (x, weights[:1], heads8[0].double(), heads8[1].double(), 8, None),
             (x, weights[:1], *heads8, 8, 21), (x, weights[:1], *heads8, 8, 0),
             (torch.ones(6, 576, device="cuda"), long, *heads8, 8, None)]
    for a, w, k, v, heads, used in calls:
        for caches in ((k, v), (k.contiguous(), v.contiguous())):
            with pytest.raises(RuntimeError):
                ops.ProjectedAttention(a, w, *caches, heads, kvLen=used, mask=mask[:, :used].contiguous() if used else mask)
