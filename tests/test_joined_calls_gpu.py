"""Calls that take several steps in one launch - a layer norm with the multiplication behind it, several matrices behind many
rows - against the separate calls: the same bits."""
import importlib

import pytest

PKG = "marian-dev_amd"


def load(name):
    return importlib.import_module(PKG + "." + name)


pytestmark = pytest.mark.gpu


def same(a, b):
    import torch
    return a.shape == b.shape and torch.equal(a.view(torch.int32), b.view(torch.int32))


def inputs(M, K, seed, kind="normal"):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    a, add, gamma, beta = r(M, K), r(M, K), 1 + 0.1 * r(K), 0.1 * r(K)
    if kind == "constant":     # rows without variance and a zero shift: every output is zero, the quantMult infinite
        a, add, beta = torch.ones_like(a), torch.ones_like(a), torch.zeros_like(beta)
    if kind == "infinite":
        a[0, K // 2] = float("inf")
    return r, a, add, (gamma, beta)


@pytest.mark.parametrize("kind", ["normal", "constant", "infinite"])
@pytest.mark.parametrize("M,K,N", [
    (1, 64, [8]), (8, 64, [40]), (3, 128, [32, 8, 200]), (6, 512, [2048]), (6, 512, [512, 512, 512]), (8, 512, [4000]),
    (2, 576, [576]), (7, 768, [3072]), (8, 1024, [1024, 1024, 1024]), (8, 1024, [4096]), (5, 256, [8192]), (4, 1024, [16384]),
    (3, 448, [32000]), (1, 512, [40000]), (2, 320, [33000, 40000]),
    (9, 512, [512]), (4, 1088, [64, 64])])   # (the last two: separate calls)
def test_affine_of_layer_norm(M, K, N, kind):
    import torch
    integer, ops = load("integer"), load("ops")
    r, a, add, ln = inputs(M, K, 7 * M + K + len(N), kind)
    weights = [(integer.prepareB(r(K, n) * 0.02), r(n) if i != 1 else None) for i, n in enumerate(N)]
    relu, want = len(N) == 1, len(N) == 1
    for eps in (1e-6, 1e-9):
        x, outs, omax = ops.affineOfLayerNorm(a, add, ln, weights, eps=eps, relu=relu, want_absmax=want)
        x_s, xmax = ops.layerNorm(a, *ln, eps=eps, add=add, want_absmax=True)
        assert same(x, x_s)
        for (w, b), out in zip(weights, outs):
            assert same(out, integer.affine_f32(x_s, w, b, relu=relu, absmax=xmax)[0])
        if want:
            assert omax.data.max().item() == outs[0].abs().max().item() or torch.isnan(outs[0]).any()


@pytest.mark.parametrize("hyps,sentences,heads,length", [
    (1, 1, 2, 1), (6, 1, 8, 23), (1, 8, 4, 33), (4, 2, 16, 96), (2, 3, 8, 64), (8, 1, 12, 97), (3, 2, 16, 5), (5, 2, 8, 9)])
def test_projected_attention_of_layer_norm(hyps, sentences, heads, length):
    import torch
    integer, ops = load("integer"), load("ops")
    M, K = hyps * sentences, heads * 64
    r, a, add, ln = inputs(M, K, M + K + length)
    weights = [(integer.prepareB(r(K, K) * 0.02), r(K)) for _ in range(3)]
    x_s, xmax = ops.layerNorm(a, *ln, eps=1e-6, add=add, want_absmax=True)
    # over complete caches, `hyps` hypotheses to a sentence
    k, v = r(sentences * heads, length, 64), r(sentences * heads, length, 64)
    mask = -1e8 * (torch.rand(sentences, length, device="cuda") < 0.3).float()
    mask[:, 0] = 0.0
    x, out, omax, proj = ops.ProjectedAttentionOfLayerNorm(a, add, ln, weights[:1], k, v, heads, mask=mask, want_projections=True)
    out_s, _, omax_s, proj_s = ops.ProjectedAttention(x_s, weights[:1], k, v, heads, mask=mask, absmax=xmax, want_absmax=True,
                                                      want_projections=True)
    assert same(x, x_s) and same(out, out_s) and same(proj[0], proj_s[0])
    assert omax.data.max().item() == omax_s.data.max().item()
    # self-attention: the new key and value are appended
    k, v = r(M * heads, length + 2, 64), r(M * heads, length + 2, 64)
    k_s, v_s = k.clone(), v.clone()
    x, out, omax, proj = ops.ProjectedAttentionOfLayerNorm(a, add, ln, weights, k, v, heads, kvLen=length)
    out_s, _, omax_s = ops.ProjectedAttention(x_s, weights, k_s, v_s, heads, kvLen=length, absmax=xmax, want_absmax=True)
    assert same(x, x_s) and same(out, out_s) and same(k, k_s) and same(v, v_s) and proj is None
    assert omax.data.max().item() == omax_s.data.max().item()


def test_refused_arguments():
    import ctypes
    import torch
    lib, L = load("_lib").lib(), load("_lib")

    class Norm(ctypes.Structure):
        _fields_ = [(n, ctypes.c_void_p) for n in ("add", "gamma", "beta", "out")] + [("eps", ctypes.c_float)]
    t = torch.zeros(16, 2048, device="cuda")
    p = t.data_ptr()
    one = lambda v: (ctypes.c_void_p * 1)(v)
    n64 = (ctypes.c_int64 * 1)(64)

    def call(norm, M=4, K=64, A=p):
        return lib.marian_hip_int8_affine_f32_normed(A, ctypes.byref(norm), 1, one(p), None, one(p + 65536), n64, M, K, 1.0, 0, None, None)
    good = dict(add=p, gamma=p, beta=p, out=p + 32768, eps=1e-6)
    assert call(Norm(**good), M=9) == L.ERR_SHAPE
    assert call(Norm(**good), K=1088) == L.ERR_SHAPE
    assert call(Norm(**{**good, "beta": None})) == L.ERR_NULL
    assert call(Norm(**{**good, "out": p + 4})) == L.ERR_ALIGN
    assert call(Norm(**{**good, "out": p + 16})) == L.ERR_ALIAS
    assert call(Norm(**good), M=0) == L.OK


def test_rows_and_biases_that_are_too_short():
    """refused before anything is launched: the kernels take their lengths from the other operands"""
    import torch
    integer, ops = load("integer"), load("ops")
    one = lambda *s: torch.ones(*s, device="cuda")
    q, k, v = one(24, 1, 64), one(24, 10, 64), one(24, 10, 64)
    for new in ((one(23, 64), one(24, 64)), (one(24, 64), one(1, 64)), (one(24, 32), one(24, 64))):
        with pytest.raises(RuntimeError):
            ops.Attention(q, k, v, kNew=new[0], vNew=new[1])
    w = integer.prepareB(one(512, 512))
    x, short, k, v = one(3, 512), [(w, one(504))], one(24, 10, 64), one(24, 10, 64)
    for weights in (short, 3 * short, 2 * [(w, None)] + short):
        with pytest.raises(RuntimeError):
            ops.ProjectedAttention(x, weights, k, v, 8)
        with pytest.raises(RuntimeError):
            ops.ProjectedAttentionOfLayerNorm(x, x, (one(512), one(512)), weights, k, v, 8)
    ops.ProjectedAttention(x, [(w, one(1, 512))], k, v, 8)
    assert (k == 1).all() and (v == 1).all()


def test_back_pointers_and_tables_on_another_device():
    import torch
    ops = load("ops")
    table, parents = torch.zeros(4, 8, dtype=torch.int32, device="cuda"), torch.zeros(4, dtype=torch.int32, device="cuda")
    for par, out in ((parents.cpu(), table.clone()), (parents.long().cpu(), table.clone()), (parents, table.cpu())):
        with pytest.raises(RuntimeError):
            ops.advanceAncestors(table, par, 3, out)
    assert ops.advanceAncestors(table, parents.long(), 3, table.clone())[:, 3].tolist() == [0, 1, 2, 3]


@pytest.mark.parametrize("M,K,N", [
    (4096, 1024, [1024, 1024, 1024]), (2048, 1536, [2048, 1024, 3072, 256]),                   # tile pairs
    (3000, 512, [512, 512, 512]), (2050, 384, [1000, 8, 2056]), (4096, 1664, [1024, 1024]),     # a 128x128 tile per CU
    (257, 128, [8, 8]), (600, 1024, [1024, 1024, 1024]), (1000, 512, [512, 0, 72, 200]),        # 128x64 tiles
    (300, 576, [64, 128])])                                                                     # K not in whole blocks
@pytest.mark.parametrize("relu", [False, True])
def test_grouped_matrices_behind_many_rows(M, K, N, relu):
    import torch
    integer = load("integer")
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K)
    x = torch.randn(M, K, device="cuda", generator=g)
    weights = [(integer.prepareB(torch.randn(K, n, device="cuda", generator=g) * 0.02) if n else
                integer.QTensor(torch.zeros(256, dtype=torch.int8, device="cuda"), (K, 0), load("types").Type.intgemm8, True),
                torch.randn(n, device="cuda", generator=g) if i != 1 else None) for i, n in enumerate(N)]
    outs, _ = integer.affine_f32_grouped(x, weights, relu=relu)
    for (w, b), out, n in zip(weights, outs, N):
        assert out.shape == (M, n)
        if n:
            assert same(out, integer.affine_f32(x, w, b, relu=relu)[0])


@pytest.mark.parametrize("M,K,N", [(17, 2048, 512), (23, 1088, 8), (64, 2048, 512), (57, 3008, 520), (33, 4096, 1000), (25, 1536, 2048)])
@pytest.mark.parametrize("known", [False, True])
def test_few_long_rows_equal_the_separate_passes(M, K, N, known):
    """8-row tiles (rows of more than 1024 values, so few that CUs idle) against the quantizer and the multiplication as two launches"""
    import torch
    integer, L = load("integer"), load("_lib")
    r, x, _, (gamma, _) = inputs(M, K, M + K + N)
    w, b = integer.prepareB(r(K, N) * 0.02), r(N)
    xmax = None
    if known:
        x, xmax = load("ops").layerNorm(x, gamma, want_absmax=True)
    with L.forced_kernel(600):
        want, want_q = integer.affine_f32(x, w, b, relu=True)
    out, q, omax = integer.affine_f32(x, w, b, relu=True, absmax=xmax, want_absmax=True)
    assert same(out, want) and torch.equal(q.data[:M * K + 4], want_q.data[:M * K + 4])
    assert omax.data.max().item() == out.abs().max().item()


@pytest.mark.parametrize("M,heads,length,cap", [(1, 2, 1, 1), (6, 8, 12, 12), (8, 16, 65, 70), (37, 4, 33, 40), (128, 16, 21, 30), (64, 2, 130, 130),
                                                (257, 2, 9, 9), (5, 8, 513, 520)])   # (the last two: separate calls)
@pytest.mark.parametrize("norm", [False, True])
def test_projected_attention_by_ancestors(M, heads, length, cap, norm):
    import torch
    integer, ops = load("integer"), load("ops")
    K = heads * 64
    r, a, add, ln = inputs(M, K, M + K + length)
    weights = [(integer.prepareB(r(K, K) * 0.02), r(K) if i != 2 else None) for i in range(3)]
    k, v = r(M * heads, cap, 64), r(M * heads, cap, 64)
    k_s, v_s = k.clone(), v.clone()
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    anc = torch.randint(0, M + 2, (M, cap), device="cuda", generator=g).to(torch.int32)   # (entries past the last hypothesis: clamped)
    x, xmax = ops.layerNorm(a, *ln, eps=1e-6, add=add, want_absmax=True)
    args = (a, weights, k, v, anc, length, add, ln) if norm else (x, weights, k, v, anc, length)
    got_x, out, omax, proj = ops.ProjectedAttentionByAncestors(*args, absmax=None if norm else xmax, want_projections=True)
    qkv, _ = integer.affine_f32_grouped(x, weights, absmax=xmax)
    out_s, omax_s = ops.AttentionByAncestors(qkv[0], k_s, v_s, anc, length, qkv[1], qkv[2], want_absmax=True)
    assert same(got_x, x) and same(out, out_s.view(out.shape)) and same(k, k_s) and same(v, v_s)
    assert all(same(p, q) for p, q in zip(proj, qkv)) and omax.data.max().item() == omax_s.data.max().item()
