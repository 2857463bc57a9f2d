"""Attention of many heads with several query rows each (attention_heads_kernel): bit for bit the three operators, at the edges of its
blocks of sixteen keys and rows, and of its shared-reciprocal divisions."""
import pytest

from conftest import load

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(integer):
    return load("ops")


def three_operators(ops, q, k, v, mask, rpm):
    return ops.bdot_legacy(ops.softmax(ops.bdot_legacy(q, k, transB=True, scalar=0.125), mask, rowsPerMask=rpm), v)


@pytest.mark.parametrize("batch,m,L", [(72, 17, 32), (72, 16, 15), (72, 1 + 16, 33), (72, 33, 48), (72, 49, 49), (72, 64, 64), (72, 65, 80), (36, 80, 66),
                                       (36, 81, 96), (36, 96, 81), (36, 97, 97), (36, 128, 128), (18, 200, 113), (72, 8, 8), (72, 9, 1), (72, 8, 40), (72, 20, 120), (72, 70, 20)])
@pytest.mark.parametrize("how", ["none", "head", "rows", "infinite", "far apart"])
def test_heads_that_fill_the_chip(ops, batch, m, L, how):
    import torch
    heads = 4
    g = torch.Generator(device="cuda")
    g.manual_seed(131 * m + L)
    # (heads side by side: rows of a head lie heads * 64 values apart; values past the last row are NaN)
    def side_by_side(n, scale):
        t = torch.full((batch * n * heads * 64 + 4096,), float("nan"), device="cuda")
        t[:batch * n * heads * 64] = torch.randn(batch * n * heads * 64, device="cuda", generator=g) * scale
        return t[:batch * n * heads * 64].view(1, batch, n, heads * 64)
    # far apart: weights of all magnitudes down to the smallest, and zeros
    x, y, z = side_by_side(m, 8.0 if how == "far apart" else 1.0), side_by_side(L, 2.0 if how == "far apart" else 1.0), side_by_side(L, 1.0)
    rpm, mask = heads * m, torch.zeros(batch, L, device="cuda")
    if how == "rows":
        rpm = 3
        mask = -1e8 * (torch.rand((batch * heads * m + 2) // 3, L, device="cuda", generator=g) < 0.4).float()
        mask[:, L // 2] = 0.0
    if how == "head":
        mask[:, max(1, L // 3):] = -99999999.0
    if how == "infinite":
        mask[:, max(1, L // 2):] = -float("inf")
        mask[1] = -float("inf")
    qh, kh, vh = (ops.SplitHeads(t, heads) for t in (x, y, z))
    slots = batch * heads * m <= 2048
    got = ops.Attention(qh, kh, vh, None if how == "none" else mask, rowsPerMask=rpm, want_absmax=slots)
    got, amax = got if slots else (got, None)
    apart = [t.contiguous().reshape(-1, t.shape[2], 64) for t in (qh, kh, vh)]
    want = three_operators(ops, *apart, None if how == "none" else mask, rpm)
    got = got.contiguous().reshape(-1, m, 64)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
    if how != "infinite":
        assert not got.isnan().any()
        if slots:
            assert float(amax.data.max()) == float(got.abs().max())
