"""Multiplications of more rows than the decode forms take, in small tiles (csrc/c_abi.hip, small_tiles): sizes around the edges of
32x64 and 64x64 tiles and of the ranges that take them, against the checker, and bit for bit against the larger tiles (measurement id 340)."""
import numpy as np
import pytest

from conftest import load
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# (workgroups of 32x64 and of 64x64 tiles on a chip of 256 CUs: the form)
SHAPES = [
    (257, 128, 8),        # the stream form: one sub-step to a wave
    (520, 128, 8),        # 17: 32x64, one K block
    (288, 1024, 1024),    # the stream form: eight sub-steps to a wave
    (288, 1280, 1024),    # 144: 32x64, whole tiles
    (511, 2048, 1024),    # 256: 32x64, the last size, a row short
    (513, 2048, 1024),    # 272, 144: 64x64, a row more
    (1024, 384, 1024),    # 64x64, whole tiles, the last size, fewer blocks than stages
    (1025, 512, 1032),    # 289: 64x64, several to a CU, a row and eight columns more
    (961, 512, 4096),     # 1024: the last of those
    (700, 768, 2056),     # 363: K = 768
    (65, 2048, 520),      # few rows, long ones: 32x64
    (200, 4096, 4104),    # 260: no small tiles
    (129, 2048, 3000),    # 32x64, 235
    (300, 576, 512),      # K no whole number of blocks: no small tiles
]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_multiplication_in_small_tiles(M, K, N):
    import torch
    integer, lib = load("integer"), load("_lib")
    rng = np.random.default_rng(M + K + N)
    x = rng.standard_normal((M, K)).astype(np.float32)
    W = (0.02 * rng.standard_normal((K, N))).astype(np.float32)
    bias = (0.01 * rng.standard_normal(N)).astype(np.float32)
    dx, db = torch.from_numpy(x).cuda(), torch.from_numpy(bias).cuda()
    Aq, Bq = integer.prepareA(dx), integer.prepareB(torch.from_numpy(W).cuda())
    relu = M % 2 == 0
    out = integer.multiply(Aq, Bq, db, scale=0.5, relu=relu)
    want = orc.affine(orc.prepare_a(x), orc.prepare_b(W), bias, M, K, N, 0.5, relu)[0]
    assert np.allclose(out.cpu().numpy(), want, rtol=1e-5, atol=1e-6)   # (whole accumulators, three roundings)
    with lib.forced_kernel(340):
        assert torch.equal(integer.multiply(Aq, Bq, db, scale=0.5, relu=relu), out)
    y, _, amax = integer.affine_f32(dx, Bq, db, scale=0.5, relu=relu, want_absmax=True)
    assert torch.equal(y, out) and float(amax.data.max()) == float(out.abs().max())
    ids = torch.arange(0, N, 2 if N > 8 else 1, device="cuda", dtype=torch.int32)[:max(8, N // 16 * 8)]
    assert torch.equal(integer.multiply(Aq, Bq, db, scale=0.5, relu=relu, shortlist=ids), out[:, ids.long()])


@pytest.mark.parametrize("M,K,Ns", [(257, 256, (8, 64, 72)), (300, 1024, (1024, 8, 520)), (640, 1024, (512, 512, 512)),
                                    (1000, 512, (512, 1032)), (1100, 768, (1544, 64))])
def test_matrices_side_by_side_in_small_tiles(M, K, Ns):
    import torch
    integer = load("integer")
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K)
    x = torch.randn(M, K, device="cuda", generator=g)
    weights = [(integer.prepareB(torch.randn(K, n, device="cuda", generator=g) * 0.02),
                torch.randn(n, device="cuda", generator=g) if i % 2 == 0 else None) for i, n in enumerate(Ns)]
    outs, _ = integer.affine_f32_grouped(x, weights)
    for out, (w, b) in zip(outs, weights):
        assert torch.equal(out, integer.affine_f32(x, w, b)[0])
