"""Attention of one query position over rows that a workgroup holds in LDS or in registers (no more than 96): bit for bit the
attention of rows that have their caches to themselves, which reads them from memory."""
import pytest

from conftest import load

pytestmark = pytest.mark.gpu


def same(got, want):
    import torch
    got, want = got.reshape(-1), want.reshape(-1)
    nan = torch.isnan(want)
    return torch.equal(torch.isnan(got), nan) and torch.equal(got[~nan], want[~nan])


# blocks of sixteen positions, one or two positions to a lane of the wave, passes of 32 while staging
LENGTHS = (1, 2, 3, 4, 13, 14, 15, 16, 17, 29, 30, 31, 32, 33, 46, 47, 48, 49, 63, 64, 65, 66, 79, 80, 81, 94, 95, 96)


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("batch,hyps", [(4, 4), (5, 2), (8, 2), (3, 8)])
def test_shared_rows(integer, batch, hyps, special):
    import torch
    ops = load("ops")
    M, heads, K = batch * hyps, 2, 128
    g = torch.Generator(device="cuda")
    g.manual_seed(100 * batch + hyps)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    w, x = (integer.prepareB(r(K, K) * 0.02), r(K) * 0.01), r(M, K)
    q, _ = integer.affine_f32(x, *w)
    for L in LENGTHS:
        print("shared rows", batch, hyps, L, special, flush=True)
        kc, vc = r(batch * heads, L, 64), r(batch * heads, L, 64)
        mask = (torch.arange(L, device="cuda")[None, :] >= torch.randint(1, L + 1, (batch,), device="cuda", generator=g)[:, None]).float() * -99999999.0
        if special:   # a sentence that is masked throughout, values that are not finite at either end
            mask[0] = torch.finfo(torch.float32).min
            vc[:, -1, ::7], vc[:, 0, 3::11], kc[-1, L // 2, 5] = float("inf"), float("-inf"), float("nan")
        own = lambda c: c.view(batch, heads, L, 64).repeat(hyps, 1, 1, 1).view(M * heads, L, 64)
        want = ops.Attention(q.view(M * heads, 1, 64), own(kc), own(vc), mask.repeat(hyps, 1), rowsPerMask=heads)
        got = ops.ProjectedAttention(x, [w], kc, vc, heads, mask=mask)[0]
        assert same(got, want), ("projected", L)
        got = ops.Attention(q.view(M * heads, 1, 64), kc, vc, mask, rowsPerMask=heads)
        assert same(got, want), ("on its own", L)


@pytest.mark.parametrize("M", [3, 40])
def test_held_rows(integer, M):
    """histories of every length modulo a block's sixteen, the newest row and its neighbours not finite"""
    import torch
    ops = load("ops")
    heads, K = 2, 128
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    ws, x = [(integer.prepareB(r(K, K) * 0.02), r(K) * 0.01) for _ in range(3)], r(M, K)
    ws[2][1][::9] = float("inf")
    (q, k, v), _ = integer.affine_f32_grouped(x, ws)
    for T in list(range(1, 36)) + list(range(45, 66)):
        print("held rows", M, T, flush=True)
        kc, vc = r(M * heads, T + 3, 64), r(M * heads, T + 3, 64)
        kc2, vc2 = kc.clone(), vc.clone()
        want = ops.Attention(q.view(M * heads, 1, 64), kc, vc, kNew=k.view(M * heads, 64), vNew=v.view(M * heads, 64), kvLen=T)
        got = ops.ProjectedAttention(x, ws, kc2, vc2, heads, kvLen=T)[0]
        assert same(got, want), T
