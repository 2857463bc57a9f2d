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


def test_projections_over_views_refuse_what_they_refuse_over_copies():
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
    with pytest.raises(RuntimeError):   # (six rows, the caches of three sentences)
        ops.ProjectedAttention(x, weights, *heads8, 8)
    for a, w, k, v, heads, used in calls:
        for caches in ((k, v), (k.contiguous(), v.contiguous())):
            with pytest.raises(RuntimeError):
                ops.ProjectedAttention(a, w, *caches, heads, kvLen=used, mask=mask[:, :used].contiguous() if used else mask)


@pytest.mark.parametrize("rows,heads,length,used", [(1, 2, 2, None), (6, 8, 23, 12), (65, 8, 34, 34), (3, 16, 130, 129), (2, 4, 512, 1)])
@pytest.mark.parametrize("masked", [False, True])
def test_three_projections_over_views(rows, heads, length, used, masked):
    """self-attention: the same results as over copies, the new position in the views"""
    ops = load("ops")
    r, x, weights, mask, keys, values = inputs(1, rows, heads, length, rows + length)
    mask = mask[:, :used].contiguous() if masked else None
    k, v = ops.SplitHeads(keys, heads), ops.SplitHeads(values, heads)
    kc, vc = k.contiguous(), v.contiguous()
    args = dict(kvLen=used, mask=mask, want_absmax=True, want_projections=True)
    want = ops.ProjectedAttention(x, weights, kc, vc, heads, **args)
    before = r(rows, heads * 64), r(rows, heads * 64)
    got = ops.ProjectedAttention(x, weights, k, v, heads, **args)
    assert same(got[0], want[0]) and all(same(p, q) for p, q in zip(got[3], want[3]))
    assert got[2].data.max().item() == want[2].data.max().item()
    assert same(k, kc) and same(v, vc)
    assert (got[1].numpy() == want[1].numpy()).all()
    # with the layer norm in front, over a cache of which one half is a view
    (a, add), ln = before, (1 + 0.1 * r(heads * 64), 0.1 * r(heads * 64))
    want = ops.ProjectedAttentionOfLayerNorm(a, add, ln, weights, kc, vc, heads, kvLen=used, mask=mask)
    got = ops.ProjectedAttentionOfLayerNorm(a, add, ln, weights, k, v.contiguous(), heads, kvLen=used, mask=mask)
    assert same(got[0], want[0]) and same(got[1], want[1]) and same(k, kc)


@pytest.mark.parametrize("sentences,heads,dk,cap,used", [
    (1, 2, 64, 2, None), (5, 8, 64, 33, 20), (3, 4, 64, 130, 129), (2, 16, 64, 40, 1), (2, 4, 32, 12, 11), (3, 2, 80, 70, None),
    (2, 3, 6, 9, 5)])   # (6: rows that are not a multiple of 16 bytes)
@pytest.mark.parametrize("masked", [False, True])
def test_attention_appends_to_views(sentences, heads, dk, cap, used, masked):
    """the same output as over copies, the new position in the views, nothing else of theirs touched"""
    import torch
    ops = load("ops")
    g = torch.Generator(device="cuda")
    g.manual_seed(cap + dk)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    keys, values = r(1, sentences, cap, heads * dk), r(1, sentences, cap, heads * dk)
    k, v = ops.SplitHeads(keys, heads), ops.SplitHeads(values, heads)
    assert not k.is_contiguous() and k.data_ptr() == keys.data_ptr()
    kc, vc = k.clone(memory_format=torch.contiguous_format), v.clone(memory_format=torch.contiguous_format)
    n, L = sentences * heads, used or cap
    q, kn, vn = r(n, 1, dk), r(n, dk), r(n, dk)
    mask = r(sentences, L) if masked else None
    args = dict(mask=mask, rowsPerMask=heads, want_absmax=True, kNew=kn, vNew=vn, kvLen=used)
    want, wmax = ops.Attention(q, kc, vc, **args)
    # (the call moves one position of each tensor, not the tensors)
    before = torch.cuda.memory_stats()["allocated_bytes.all.allocated"]
    got, gmax = ops.Attention(q, k, v, **args)
    taken = torch.cuda.memory_stats()["allocated_bytes.all.allocated"] - before
    assert dk % 4 != 0 or keys.numel() < 30000 or taken < 4 * keys.numel(), taken
    assert same(got, want) and same(k, kc) and same(v, vc)
    assert gmax.data.max().item() == wmax.data.max().item()


def test_attention_refuses_appends_it_cannot_place():
    import torch
    ops = load("ops")
    keys = torch.zeros(1, 3, 10, 512, device="cuda")
    k, v = ops.SplitHeads(keys, 8), ops.SplitHeads(keys.clone(), 8)
    one = lambda *s: torch.ones(*s, device="cuda")
    good = dict(q=one(24, 1, 64), k=k, v=v, kNew=one(24, 64), vNew=one(24, 64))
    long = ops.SplitHeads(torch.zeros(1, 1, 4097, 128, device="cuda"), 2)
    for bad in (dict(q=one(24, 2, 64)), dict(q=one(16, 1, 64)), dict(q=one(24, 1, 32)), dict(kNew=one(23, 64)), dict(vNew=one(24, 32)),
                dict(kvLen=0), dict(kvLen=11), dict(v=v[:, :, :9]), dict(v=v[..., ::2]), dict(k=k.transpose(2, 3)),
                dict(k=k.contiguous().view(24, 10, 64)), dict(k=long, v=long, q=one(2, 1, 64), kNew=one(2, 64), vNew=one(2, 64))):
        with pytest.raises(RuntimeError):
            ops.Attention(**{**good, **bad})
    assert not keys.any() and not v.any()   # (nothing was written for a call that is refused)
