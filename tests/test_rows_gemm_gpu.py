"""The multiplication whose waves each quantize their own share of the activations (csrc/gemm_rows_kernel.h: 8, 16 or 32
rows to a workgroup, one to eight pairs of K sub-steps to a wave), against the CPU checker: outputs, quantized activations and
their quantMult bit for bit."""
import numpy as np
import pytest

from conftest import load

pytestmark = pytest.mark.gpu
f32 = np.float32

SIZES = [
    # 8 rows (K = 64: fewer sub-steps than waves, another form)
    (9, 64, 8), (9, 256, 8), (17, 448, 24), (23, 512, 512), (40, 576, 264), (64, 1024, 1024), (12, 1600, 72), (30, 2048, 512), (20, 2624, 96),
    (33, 3136, 128), (9, 4032, 40), (31, 4096, 40),
    # 16 rows
    (127, 512, 1024), (128, 1088, 1000), (16, 1536, 4096), (100, 4096, 1000), (128, 3520, 1024), (113, 2560, 1024), (128, 2880, 1000),
    # 32 rows
    (256, 512, 1000), (255, 960, 1024), (200, 2048, 1048), (250, 1216, 1000),
]


def upload(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


@pytest.mark.parametrize("kind", ["normal", "zero", "infinite"])
@pytest.mark.parametrize("M,K,N", SIZES)
def test_affine_with_known_absmax(integer, orc, synth, M, K, N, kind):
    ops = load("ops")
    z = synth.normal(900 + M + K, synth.STREAM_A, (M, K), 1.0)
    if kind == "infinite":   # a row of NaN and infinities: an infinite abs-max, every product zero or NaN
        z[M // 2, K // 2] = np.inf
    gamma, beta = np.ones(K, f32), np.zeros(K, f32)
    x, absmax = ops.layerNorm(upload(z if kind != "zero" else np.ones_like(z)), upload(gamma), upload(beta), eps=1e-6, want_absmax=True)
    if kind == "infinite":
        x[M // 2, 3] = float("inf")
        absmax.data[0] = float("inf")
    A = x.cpu().numpy()
    W, bias = synth.normal(900 + N, synth.STREAM_W, (K, N), 0.02), synth.normal(900 + N, synth.STREAM_BIAS, (N,), 0.01)
    Aq_h, Bq_h = orc.prepare_a(A), orc.prepare_b(W)
    relu = M % 2 == 1
    want, _ = orc.affine(Aq_h, Bq_h, bias, M, K, N, 0.5, relu)
    Bq = integer.prepareB(upload(W))
    out, Aq, omax = integer.affine_f32(x, Bq, upload(bias), scale=0.5, relu=relu, absmax=absmax, want_absmax=True)
    assert np.array_equal(Aq.numpy(), Aq_h)
    assert np.array_equal(out.cpu().numpy(), want, equal_nan=True)
    if kind == "normal":
        assert omax.data.max().item() == np.abs(want).max()
        # several matrices, and a shortlist, take the same rows
        outs, _ = integer.affine_f32_grouped(x, [(Bq, upload(bias)), (Bq, None)], scale=0.5, relu=relu, absmax=absmax)
        assert np.array_equal(outs[0].cpu().numpy(), want)
        assert np.array_equal(outs[1].cpu().numpy(), orc.affine(Aq_h, Bq_h, None, M, K, N, 0.5, relu)[0])
        idx = np.arange(0, N, 2, dtype=np.uint32)[: N // 2 // 8 * 8]
        if idx.size:
            short, _ = integer.affine_f32(x, Bq, upload(bias), scale=0.5, relu=relu, absmax=absmax, shortlist=upload(idx.view(np.int32)))
            assert np.array_equal(short.cpu().numpy(), want[:, idx])


@pytest.mark.parametrize("kernel", [0, 630, 702])
@pytest.mark.parametrize("M,K,N", [(64, 2048, 8), (128, 576, 264), (64, 1024, 1024), (9, 1984, 2056), (30, 2048, 512), (128, 1088, 1000),
                                   (113, 2048, 1024), (255, 960, 1024), (200, 2048, 1048), (250, 1216, 1000)])
def test_affine_that_takes_its_absmax(integer, orc, synth, M, K, N, kernel):
    """The abs-max taken by the launch that multiplies (id 630: by a launch in front; 702: every workgroup scans all activations
    itself), at one to 256 workgroups, the largest value in the last workgroup's share; twice, since a call leaves words for the next."""
    import contextlib
    W, bias = synth.normal(940 + N, synth.STREAM_W, (K, N), 0.02), synth.normal(940 + N, synth.STREAM_BIAS, (N,), 0.01)
    Bq_h, Bq = orc.prepare_b(W), integer.prepareB(upload(W))
    with load("_lib").forced_kernel(kernel) if kernel else contextlib.nullcontext():
        for turn in range(2):
            A = synth.normal(940 + M + K + turn, synth.STREAM_A, (M, K), 1.0 + turn)
            A.flat[A.size - 1 - 3 * turn] = -9.5 - turn
            Aq_h = orc.prepare_a(A)
            out, Aq = integer.affine_f32(upload(A), Bq, upload(bias))
            assert np.array_equal(Aq.numpy(), Aq_h)
            assert np.array_equal(out.cpu().numpy(), orc.affine(Aq_h, Bq_h, bias, M, K, N, 1.0, False)[0])


@pytest.mark.parametrize("kind", ["zero", "infinite", "nan", "tiny"])
@pytest.mark.parametrize("kernel", [0, 702])
@pytest.mark.parametrize("M,K,N", [(64, 1024, 1024), (128, 1088, 1000), (250, 1216, 1000)])
def test_absmax_that_is_none_of_the_usual(integer, orc, synth, M, K, N, kernel, kind):
    """What is exchanged is a zero, an infinity, a maximum beside NaNs (which count for nothing) or a denormal number: the bytes and
    outputs of the checker, with the values in the share of the last workgroup."""
    import contextlib
    A = synth.normal(980 + M, synth.STREAM_A, (M, K), 1.0)
    if kind == "zero":
        A[:] = 0.0
    elif kind == "infinite":
        A[-1, -2] = -np.inf
    elif kind == "nan":
        A[-1, -2:], A[0, 0] = np.nan, np.nan
        A[-1, -5] = 7.25
    else:
        A *= f32(1e-41)
    W, bias = synth.normal(980 + N, synth.STREAM_W, (K, N), 0.02), synth.normal(980 + N, synth.STREAM_BIAS, (N,), 0.01)
    Aq_h, Bq_h = orc.prepare_a(A), orc.prepare_b(W)
    want = orc.affine(Aq_h, Bq_h, bias, M, K, N, 1.0, False)[0]
    Bq = integer.prepareB(upload(W))
    with load("_lib").forced_kernel(kernel) if kernel else contextlib.nullcontext():
        out, Aq = integer.affine_f32(upload(A), Bq, upload(bias))
    assert np.array_equal(Aq.numpy(), Aq_h)
    assert np.array_equal(out.cpu().numpy(), want, equal_nan=True)


@pytest.mark.parametrize("gx,gy", [(32, 8), (64, 4), (16, 5), (3, 7), (8, 1), (1, 8), (24, 3), (48, 2), (100, 2), (16, 16), (5, 32), (2, 13)])
def test_tiles_are_each_taken_once(integer, synth, orc, gx, gy):
    """every split of the tiles over the XCDs: 8, 16 or 32 rows by 32 columns, one output wrong per tile missed (K = 512: the form
    whose waves split K in eight, where the columns leave room for it)"""
    M, K, N = 16 * gy, 512, 32 * gx
    A, W = synth.normal(gx, synth.STREAM_A, (M, K), 1.0), synth.normal(gy, synth.STREAM_W, (K, N), 0.02)
    want, _ = orc.affine(orc.prepare_a(A), orc.prepare_b(W), None, M, K, N, 1.0, False)
    x = upload(A)
    absmax = integer.AbsMax(x.device)
    absmax.data.fill_(float(np.abs(A).max()))
    out, _ = integer.affine_f32(x, integer.prepareB(upload(W)), None, absmax=absmax)
    assert np.array_equal(out.cpu().numpy(), want)
