"""Host mirror of the float operators between the int8 GEMMs of a transformer decode step,
running on the HIP library (include/marian_hip_ops.h).

Mirrors, name for name:
  reference src/graph/expression_operators.cpp:901-913   layerNorm(x, gamma, beta, eps = 1e-9)
  reference src/graph/expression_operators.cpp           softmax(a), logsoftmax(a),
                                                         transpose(a, {0, 2, 1, 3}),
                                                         bdot_legacy(a, b, transA, transB, scalar)
  reference src/models/transformer.h:145-170             SplitHeads, JoinHeads
  reference src/graph/expression_operators.cpp           rows(a, indices)
  reference src/graph/node_initializers.cpp:224-226      sinusoidalPositionEmbeddings(start)
  reference src/models/transformer.h:93,110-117          scaledEmbeddings: sqrt(dimEmb) * rows(E, ids) + signal

Tensors are torch float32 tensors on the GPU (device memory and streams only); every arithmetic
step is a call into the C ABI.  There is no CPU fallback.
"""
import torch

from . import _lib
from .integer import _abort_if, _backend_of, _host, _on_gpu, _taken


def _f32c(x, what):
    _abort_if(x.dtype != torch.float32, "{} expects float32, got {}", what, x.dtype)
    if x.device.type == "cuda" and _heads_side_by_side(x):   # its copy head by head is the 0213 transpose
        return transpose0213(x.transpose(1, 2))
    return x.contiguous()


def _heads_side_by_side(t):
    """SplitHeads' view of rows"""
    return t.dim() == 4 and not t.is_contiguous() and t.transpose(1, 2).is_contiguous()


def layerNorm(x, gamma, beta=None, eps=1e-9, add=None, want_absmax=False):
    """reference src/graph/expression_operators.cpp:901-913; `add` fuses the skip connection in
    front of it (out = layerNorm(x + add)).  want_absmax: also return the AbsMax of the output
    for the affine calls that read it."""
    out = _host.layer_norm(x, gamma, beta, eps, add, want_absmax)
    if out is not None:
        return out
    x = _f32c(x, "layerNorm")
    _on_gpu(x)
    cols = x.shape[-1]
    gamma = _f32c(gamma, "layerNorm").reshape(-1)
    _abort_if(gamma.numel() not in (1, cols), "layerNorm: gamma must have {} or 1 values", cols)
    if beta is not None:
        beta = _f32c(beta, "layerNorm").reshape(-1)
        _abort_if(beta.numel() not in (1, cols), "layerNorm: beta must have {} or 1 values", cols)
    if add is not None:
        add = _f32c(add, "layerNorm")
        _abort_if(tuple(add.shape) != tuple(x.shape), "layerNorm: skip input shape {} vs {}", tuple(add.shape), tuple(x.shape))
    return _taken(_host.layer_norm(x, gamma, beta, eps, add, want_absmax), "layerNorm")


def scaledEmbeddings(E, ids, scale=1.0, signal=None, rowsPerSignal=1, want_absmax=False, out=None):
    """scale * E[ids] (+ signal): the embedding step in front of the first layer (reference
    src/layers/embedding.cpp:161-168 and src/models/transformer.h:93,117) as one launch.  E
    [vocab, dimEmb]; ids: integer tensor on the device, any shape; signal: None or [n, dimEmb],
    output row r taking signal row (r / rowsPerSignal) % n.  Returns [*ids.shape, dimEmb] (`out`
    when given: a contiguous float32 tensor of that many values that does not overlap E)."""
    res = _host.embed(E, ids, scale, signal, rowsPerSignal, want_absmax, out)
    if res is not None:
        return res
    E = _f32c(E, "scaledEmbeddings")
    _on_gpu(E)
    _abort_if(E.dim() != 2, "scaledEmbeddings: the table has to be a matrix, got shape {}", tuple(E.shape))
    _abort_if(ids.dtype not in (torch.int32, torch.int64, torch.uint32) or ids.device != E.device,
              "scaledEmbeddings: indices have to be an integer tensor on the table's device")
    words = ids.contiguous()
    if words.dtype == torch.int64:   # the reference's IndexType has 32 bits
        words = words.to(torch.int32)
    if signal is not None:
        signal = _f32c(signal, "scaledEmbeddings").reshape(-1, E.shape[1])
    if out is not None:
        _abort_if(out.dtype != torch.float32 or not out.is_contiguous() or out.device != E.device or
                  out.numel() != ids.numel() * E.shape[1], "scaledEmbeddings: out has to be a contiguous float32 "
                  "tensor of {} x {} values on the table's device", ids.numel(), E.shape[1])
        lo, hi = out.data_ptr(), out.data_ptr() + 4 * out.numel()
        _abort_if(lo < E.data_ptr() + 4 * E.numel() and E.data_ptr() < hi, "scaledEmbeddings: out overlaps the table")
    return _taken(_host.embed(E, words, scale, signal, rowsPerSignal, want_absmax, out), "scaledEmbeddings")


def rows(a, indices, out=None):
    """reference rows(a, indices) (CopyRows, src/tensors/cpu/tensor_operators.cpp:577-603); also
    the selection of the surviving hypotheses' decoder states between two steps of the beam search
    (reference src/rnn/types.h:22-42)"""
    return scaledEmbeddings(a, indices.reshape(-1), out=out)


def selectState(state, indices, out, used=None):
    """The decoder state of the surviving hypotheses (reference src/models/states.h:87-107,
    src/rnn/types.h:22-42): out[r, s, :used] = state[indices[r], s, :used] for a state [entries,
    segments, capacity] whose segments (the cached positions of a head) are in use up to `used`
    values (None: entirely); out [len(indices), segments, capacity] is a tensor of its own."""
    res = _host.select_state(state, indices, out, used)
    if res is not None:
        return res
    _abort_if(state.dtype != torch.float32 or out.dtype != torch.float32 or state.dim() != 3 or out.dim() != 3 or
              not state.is_contiguous() or not out.is_contiguous(), "selectState expects contiguous float32 "
              "tensors [entries, segments, capacity], got {} and {}", tuple(state.shape), tuple(out.shape))
    _on_gpu(state)
    _abort_if(tuple(out.shape) != (indices.numel(),) + tuple(state.shape[1:]), "selectState: out has shape {}, not {}",
              tuple(out.shape), (indices.numel(),) + tuple(state.shape[1:]))
    _abort_if(indices.dtype not in (torch.int32, torch.int64, torch.uint32) or indices.device != state.device,
              "selectState: indices have to be an integer tensor on the state's device")
    ids = indices.contiguous()
    if ids.dtype == torch.int64:
        ids = ids.to(torch.int32)
    return _taken(_host.select_state(state, ids, out, used), "selectState")


def sinusoidalPositionEmbeddings(dimWords, dimEmb, start=0, device=None):
    """The constant [dimWords, 1, dimEmb] of reference src/models/transformer.h:110-111, made on the
    host by the library (reference src/tensors/cpu/tensor_operators.cpp:1733-1746) and copied to
    `device` when one is given."""
    out = torch.empty((dimWords, 1, dimEmb), dtype=torch.float32)
    _lib.check(_lib.lib().marian_hip_sinusoidal_position_embeddings(out.data_ptr(), dimWords, dimEmb, start),
               "sinusoidalPositionEmbeddings")
    return out if device is None else out.to(device)


def softmax(a, mask=None, rowsPerMask=1):
    """softmax over the last axis; `mask` [n, cols] fuses the `a + mask` in front of it, row r of
    `a` taking mask row (r / rowsPerMask) % n (reference src/models/transformer.h:264,772-774)."""
    a = _f32c(a, "softmax")
    be = _backend_of(a)
    cols = a.shape[-1]
    rows = a.numel() // cols if a.numel() else 0
    n_masks = 0
    if mask is not None:
        mask = _f32c(mask, "softmax").reshape(-1, cols)
        n_masks = mask.shape[0]
    out = torch.empty_like(a)
    st = be.lib.marian_hip_softmax(a.data_ptr(), None if mask is None else mask.data_ptr(), n_masks,
                                   rowsPerMask, out.data_ptr(), rows, cols, be.stream())
    _lib.check(st, "softmax")
    return out


def logsoftmax(a):
    a = _f32c(a, "logsoftmax")
    be = _backend_of(a)
    cols = a.shape[-1]
    rows = a.numel() // cols if a.numel() else 0
    out = torch.empty_like(a)
    _lib.check(be.lib.marian_hip_logsoftmax(a.data_ptr(), out.data_ptr(), rows, cols, be.stream()),
               "logsoftmax")
    return out


def transpose0213(a):
    """transpose(a, {0, 2, 1, 3}) of a 4-d tensor.  With a middle dimension of 1 (the single
    target position of a decoding step) the transposed tensor has the same memory image, so it
    is returned as a view and no kernel runs."""
    a = _f32c(a, "transpose")
    _abort_if(a.dim() != 4, "transpose0213 expects a 4-d tensor, got {} dimensions", a.dim())
    be = _backend_of(a)
    d0, d1, d2, d3 = a.shape
    if d1 == 1 or d2 == 1:
        return a.reshape(d0, d2, d1, d3)
    out = torch.empty((d0, d2, d1, d3), dtype=torch.float32, device=a.device)
    _lib.check(be.lib.marian_hip_transpose0213(a.data_ptr(), out.data_ptr(), d0, d1, d2, d3, be.stream()),
               "transpose")
    return out


def SplitHeads(input, dimHeads):
    """reference src/models/transformer.h:145-156: [beam, batch, steps, model] ->
    [batch * beam, heads, steps, depth].  The result is a view (the heads of a position side by side, as
    the affine call wrote them): Attention reads it as it is, and what needs it head by head copies.
    Memory of its own, head by head - for .view(), or for a cache that is appended to while `input` is
    still needed - is SplitHeads(..).contiguous()."""
    out = _host.split_heads(input, dimHeads)
    if out is not None:
        return out
    dimBeam, dimBatch, dimSteps, dimModel = input.shape
    return transpose0213(input.reshape(dimBatch * dimBeam, dimSteps, dimHeads, dimModel // dimHeads))


def JoinHeads(input, dimBeam=1):
    """reference src/models/transformer.h:158-170; a view of `input` where the heads of a position lie side by side (the
    output of Attention on SplitHeads' views)"""
    out = _host.join_heads(input, dimBeam)
    if out is not None:
        return out
    dimBatchBeam, dimHeads, dimSteps, dimDepth = input.shape
    out = transpose0213(input)
    return out.reshape(dimBeam, dimBatchBeam // dimBeam, dimSteps, dimHeads * dimDepth)


def bdot_legacy(a, b, transA=False, transB=False, scalar=1.0):
    """reference src/tensors/cpu/prod.cpp:233-330: batch entry i uses a[i % batchA], b[i % batchB]"""
    a, b = _f32c(a, "bdot"), _f32c(b, "bdot")
    be = _backend_of(a)
    batchA = a.numel() // (a.shape[-1] * a.shape[-2])
    batchB = b.numel() // (b.shape[-1] * b.shape[-2])
    m, k = a.shape[-2], a.shape[-1]
    if transA:
        m, k = k, m
    l, n = b.shape[-2], b.shape[-1]
    if transB:
        l, n = n, l
    _abort_if(l != k, "Matrix product requires inner dimensions to match: {} vs {}", k, l)
    lead = tuple(a.shape[:-2]) if batchA >= batchB else tuple(b.shape[:-2])
    out = torch.empty(lead + (m, n), dtype=torch.float32, device=a.device)
    st = be.lib.marian_hip_bdot_legacy(a.data_ptr(), b.data_ptr(), out.data_ptr(), batchA, batchB,
                                       m, n, k, int(transA), int(transB), scalar, be.stream())
    _lib.check(st, "bdot")
    return out


def Attention(q, k, v, mask=None, rowsPerMask=1, want_absmax=False, kNew=None, vNew=None, kvLen=None):
    """reference src/models/transformer.h:241-280 (inference: no dropout, weights not kept):
    softmax(bdot_legacy(q, k, false, true, 1/sqrt(dk)) + mask) then bdot_legacy(weights, v), in
    one launch.  q: [batch*beam, heads, tgt, dk]; k, v: [batch(*beam), heads, len, dk].
    kNew, vNew [batch*beam*heads, dk]: key and value of the newest position of a decoding step;
    they stand for position len - 1 and are also stored there in k and v (the concatenation onto
    the cached positions, src/models/transformer.h:683-700); where k and v are SplitHeads' views, in the
    tensors they are views of.  The output lies in memory as q does.
    kvLen: k and v have room for k.shape[-2] positions per entry, of which the first kvLen are in
    use (caches that stay in place from step to step); None: all of them."""
    m = q.shape[-2]
    if kNew is None and (m >= 8 or not (q.is_contiguous() and k.is_contiguous() and v.is_contiguous())):
        out = _host.attention_rows(q, k, v, mask, rowsPerMask, kvLen, want_absmax)
        if out is not None:
            return out
    if m < 8 or kNew is not None or want_absmax or kvLen is not None:
        out = _host.attention(q, k, v, mask, rowsPerMask, want_absmax, kNew, vNew, kvLen)
        if out is not None:
            return out
    q = _f32c(q, "Attention")
    _abort_if(k.dtype != torch.float32 or v.dtype != torch.float32, "Attention expects float32, got {}", k.dtype)
    if kNew is None:
        k, v = _f32c(k, "Attention"), _f32c(v, "Attention")
    else:
        _abort_if(not all(t.is_contiguous() or _heads_side_by_side(t) for t in (k, v)),
                  "Attention: the key/value cache must be contiguous{}", "")
        kNew, vNew = _f32c(kNew, "Attention"), _f32c(vNew, "Attention")
        if not (k.is_contiguous() and v.is_contiguous()):
            return _attention_appending_to_views(q, k, v, mask, rowsPerMask, want_absmax, kNew, vNew, kvLen)
    _on_gpu(q)
    dk, cap = q.shape[-1], k.shape[-2]
    L = cap if kvLen is None else int(kvLen)
    _abort_if(not 0 < L <= cap, "Attention: {} positions in use of {} the cache has room for", L, cap)
    _abort_if(k.shape[-1] != dk or tuple(v.shape) != tuple(k.shape), "Attention: key/value shapes {} {} vs dk {}",
              tuple(k.shape), tuple(v.shape), dk)
    if m >= 8 and kNew is None and not want_absmax and L == cap:
        # Many query positions per head and another head size, or more than 256 keys: the three operators share a head's keys
        # and values through LDS tiles; the one-launch form gives every query row a wave that walks
        # them on its own.
        batchQ, batchKV = q.numel() // (m * dk), k.numel() // (cap * dk)
        scores = bdot_legacy(q.reshape(batchQ, m, dk), k.reshape(batchKV, L, dk), False, True, 1.0 / float(dk) ** 0.5)
        weights = softmax(scores, mask, rowsPerMask)
        return bdot_legacy(weights, v.reshape(batchKV, L, dk)).reshape(q.shape)
    if mask is not None:
        mask = _f32c(mask, "Attention").reshape(-1, L)
    return _taken(_host.attention(q, k, v, mask, rowsPerMask, want_absmax, kNew, vNew, L), "Attention")


def _attention_appending_to_views(q, k, v, mask, rowsPerMask, want_absmax, kNew, vNew, kvLen):
    """Attention with a new key and value over SplitHeads' views: the one position is written where the views have
    it, and the attention reads them as they are (with the bits of the call on caches of their own)."""
    _abort_if(tuple(v.shape) != tuple(k.shape) or q.shape[-1] != k.shape[-1], "Attention: key/value shapes {} {} vs dk {}",
              tuple(k.shape), tuple(v.shape), q.shape[-1])
    entries, heads, cap, dk = k.shape
    L = cap if kvLen is None else int(kvLen)
    _abort_if(not 0 < L <= min(cap, 4096), "Attention: {} positions in use of {} the cache has room for", L, cap)
    _abort_if(q.shape[-2] != 1 or any(t.numel() != entries * heads * dk for t in (q, kNew, vNew)),
              "Attention: one query, new key and new value of {} values per cache entry", dk)
    _abort_if(want_absmax and entries * heads > _lib.ABSMAX_SLOTS, "Attention: the abs-max of up to {} query rows, got {}",
              _lib.ABSMAX_SLOTS, entries * heads)
    if mask is not None:
        mask = _f32c(mask, "Attention").reshape(-1, L)
    k[:, :, L - 1].copy_(kNew.view(entries, heads, dk))
    v[:, :, L - 1].copy_(vNew.view(entries, heads, dk))
    return Attention(q, k, v, mask, rowsPerMask, want_absmax, kvLen=L)


def ProjectedAttention(x, weights, k, v, heads, kvLen=None, mask=None, absmax=None, want_absmax=False,
                       want_projections=False):
    """The projections in front of an attention and the attention itself for one new target
    position, in one launch (reference src/models/transformer.h:279-348: MultiHead's affine nodes
    for q - and, in self-attention, k and v - then the head split and Attention()).
    x [M, K] float32; weights: [(Wq, bq)] - attention over caches that are complete (the encoder's
    keys and values) - or [(Wq, bq), (Wk, bk), (Wv, bv)] - self-attention: the new key and value
    are appended to the caches k, v at position kvLen - 1 (quantized weights, bias or None each).
    k, v [entries, capacity, 64] with kvLen positions in use; mask [n, len] or None, one row per
    sentence (query row r of [M * heads] uses row (r // heads) % n).  absmax: the AbsMax the producer
    of x left.  Returns (out [M, heads * 64], aQuant) and, when asked for, the AbsMax of out and
    the projections themselves - bit for bit what affine_f32_grouped / affine_f32 followed by
    Attention give (and faster than those up to 128 rows, level at 256, slower at 512)."""
    res = _host.proj_attention(x, weights, k, v, heads, kvLen, mask, absmax, want_absmax, want_projections)
    if res is not None:
        return res
    from . import integer
    x = _f32c(x, "ProjectedAttention")
    _on_gpu(x)
    n = len(weights)
    _abort_if(n not in (1, 3), "ProjectedAttention: one projection (q) or three (q, k, v), got {}", n)
    K, N = x.shape[-1], heads * 64
    # caches that are SplitHeads' views: the separate calls, which read them as they are and append where they have the position
    views = not (k.is_contiguous() and v.is_contiguous())
    strided = k.dim() == 4 if n == 1 else all(t.is_contiguous() or _heads_side_by_side(t) for t in (k, v))
    _abort_if((views and not strided) or k.dtype != torch.float32 or v.dtype != torch.float32,
              "ProjectedAttention: the key/value caches must be contiguous float32{}", "")
    _abort_if(k.shape[-1] != 64 or tuple(k.shape) != tuple(v.shape), "ProjectedAttention: head size 64, got caches {} {}",
              tuple(k.shape), tuple(v.shape))
    L = k.shape[-2] if kvLen is None else int(kvLen)
    for bQuant, _ in weights:
        integer._check_weights(bQuant)
        _abort_if(integer.rows(bQuant) != K or integer.cols(bQuant) != N, "ProjectedAttention: weights {} vs [{}, {}]",
                  tuple(bQuant.shape), K, N)
    if views:
        # (the limits of the one-launch form, which refuses them itself)
        _abort_if(K % 128 != 0 or K > 1024 or not 0 < L <= min(k.shape[-2], 512), "ProjectedAttention: rows of {} values over "
                  "{} of {} positions", K, L, k.shape[-2])
        qkv, aq = integer.affine_f32_grouped(x, weights, absmax=absmax)
        rows = qkv[0].numel() // 64
        q, kNew, vNew = [t.view(rows, 64) for t in qkv] if n == 3 else (qkv[0].view(rows, 64), None, None)
        o = Attention(q.view(rows, 1, 64), k, v, mask, heads, want_absmax, kNew, vNew, L)
        o, omax = o if want_absmax else (o, None)
        return (o.view(qkv[0].shape), aq) + ((omax,) if want_absmax else ()) + ((qkv,) if want_projections else ())
    weights = [(bQuant, None if bias is None else _f32c(bias, "ProjectedAttention")) for bQuant, bias in weights]
    if mask is not None:
        mask = _f32c(mask, "ProjectedAttention").reshape(-1, L)
    return _taken(_host.proj_attention(x, weights, k, v, heads, kvLen, mask, absmax, want_absmax, want_projections),
                  "ProjectedAttention")


def affineOfLayerNorm(a, add, ln, weights, eps=1e-6, relu=False, want_absmax=False):
    """x = layerNorm(a, *ln, eps, add=add) and x through one or several weight matrices (affine_f32, or
    affine_f32_grouped for several): one launch for up to eight rows of up to 1024 values
    (marian_hip_int8_affine_f32_normed), otherwise the separate calls, with the same bits.
    Returns (x, [out, ..], AbsMax of the only out or None)."""
    res = _host.affine_f32_normed(a, add, ln, eps, weights, 1.0, relu, want_absmax)
    if res is not None:
        return res
    from . import integer
    x, xmax = layerNorm(a, *ln, eps=eps, add=add, want_absmax=True)
    if len(weights) > 1:
        _abort_if(want_absmax, "affineOfLayerNorm: the abs-max of one output only{}", "")
        return x, integer.affine_f32_grouped(x, weights, relu=relu, absmax=xmax)[0], None
    res = integer.affine_f32(x, *weights[0], relu=relu, absmax=xmax, want_absmax=want_absmax)
    return x, [res[0]], res[2] if want_absmax else None


def ProjectedAttentionOfLayerNorm(a, add, ln, weights, k, v, heads, kvLen=None, mask=None, eps=1e-6, want_projections=False):
    """x = layerNorm(a, *ln, eps, add=add) and ProjectedAttention(x, ..): one launch for up to eight rows
    (marian_hip_int8_proj_attention_normed), otherwise the two calls, with the same bits.
    Returns (x, out, AbsMax of out, the projections when asked for or None)."""
    res = _host.proj_attention_normed(a, add, ln, eps, weights, k, v, heads, kvLen, mask, want_projections)
    if res is not None:
        return res
    x, xmax = layerNorm(a, *ln, eps=eps, add=add, want_absmax=True)
    res = ProjectedAttention(x, weights, k, v, heads, kvLen, mask, xmax, True, want_projections)
    return x, res[0], res[2], res[3] if want_projections else None


def ProjectedAttentionByAncestors(a, weights, k, v, ancestors, kvLen, add=None, ln=None, eps=1e-6, absmax=None, want_projections=False):
    """Self-attention of one new position per hypothesis over caches that stay where they were written: the
    projections q, k, v of x and AttentionByAncestors in one launch (up to 256 hypotheses, where it pays, of up to
    1024 values, 512 positions), otherwise as separate calls, with the same bits.  x is a [M, K], or with `add` and
    ln = (gamma, beta) layerNorm(a, *ln, eps, add=add).  Returns (x, out [M, K], AbsMax of out, the projections
    when asked for or None)."""
    if len(ancestors) <= 256:
        res = _host.proj_attention_ancestors(a, add, ln, eps, weights, k, v, ancestors, kvLen, absmax, want_projections)
        if res is not None:
            return res
    from . import integer
    if add is not None:
        a, absmax = layerNorm(a, *ln, eps=eps, add=add, want_absmax=True)
        if len(ancestors) <= 256:
            res = _host.proj_attention_ancestors(a, None, None, eps, weights, k, v, ancestors, kvLen, absmax, want_projections)
            if res is not None:
                return res
    qkv, _ = integer.affine_f32_grouped(a, weights, absmax=absmax)
    o, omax = AttentionByAncestors(qkv[0], k, v, ancestors, kvLen, qkv[1], qkv[2], want_absmax=True)
    return a, o.view(a.shape), omax, qkv if want_projections else None


def AttentionByAncestors(q, k, v, ancestors, kvLen, kNew, vNew, want_absmax=False):
    """Self-attention of a decoding step on caches that are never moved (no counterpart in the
    reference, which copies the surviving hypotheses' states, src/rnn/types.h:22-42): cached
    position p of hypothesis h is read from the cache entry of hypothesis ancestors[h, p].
    q [hyps * heads, 1, dk]; k, v [hyps * heads, capacity, dk]; ancestors int32 [hyps, capacity];
    kNew, vNew [hyps * heads, dk] become position kvLen - 1 of the hypotheses' own entries."""
    out = _host.attention_ancestors(q, k, v, ancestors, kvLen, kNew, vNew, want_absmax)
    if out is not None:
        return out
    q, kNew, vNew = _f32c(q, "AttentionByAncestors"), _f32c(kNew, "AttentionByAncestors"), _f32c(vNew, "AttentionByAncestors")
    _on_gpu(q)
    _abort_if(k.dtype != torch.float32 or v.dtype != torch.float32 or not (k.is_contiguous() and v.is_contiguous()) or
              k.dim() != 3 or tuple(k.shape) != tuple(v.shape), "AttentionByAncestors: the caches have to be contiguous "
              "float32 tensors [entries, capacity, dk], got {} and {}", tuple(k.shape), tuple(v.shape))
    entries, cap, dk = k.shape
    _abort_if(ancestors.dtype not in (torch.int32, torch.uint32) or ancestors.dim() != 2 or ancestors.shape[1] != cap or
              not ancestors.is_contiguous() or entries % ancestors.shape[0] != 0,
              "AttentionByAncestors: ancestors have to be a contiguous int32 tensor [hypotheses, {}]", cap)
    _abort_if(q.numel() != entries * dk or kNew.numel() != entries * dk or vNew.numel() != entries * dk,
              "AttentionByAncestors: one query, key and value row of {} values per cache entry", dk)
    return _taken(_host.attention_ancestors(q, k, v, ancestors, kvLen, kNew, vNew, want_absmax), "AttentionByAncestors")


def advanceAncestors(prev, parents, lenPrev, out):
    """the table of ancestors of the next step: out[h, p] = prev[parents[h], p] for p < lenPrev,
    out[h, lenPrev] = h (prev, out: int32 [hypotheses, capacity], two tensors)"""
    res = _host.ancestors_advance(prev, parents, lenPrev, out)
    if res is not None:
        return res
    _abort_if(prev.dtype != torch.int32 or out.dtype != torch.int32 or tuple(prev.shape) != tuple(out.shape) or
              prev.dim() != 2 or not (prev.is_contiguous() and out.is_contiguous()),
              "advanceAncestors expects two contiguous int32 tensors [hypotheses, capacity]{}", "")
    _on_gpu(prev)
    par = parents.contiguous()
    if par.dtype == torch.int64:
        par = par.to(torch.int32)
    _abort_if(par.dtype not in (torch.int32, torch.uint32) or par.numel() != prev.shape[0],
              "advanceAncestors: one int32 back-pointer per hypothesis{}", "")
    return _taken(_host.ancestors_advance(prev, par, lenPrev, out), "advanceAncestors")


def getNBestList(scores, N):
    """reference src/translator/nth_element.cpp:26-67: scores [dimBatch, 1, beam, vocab]; returns
    (pathScores, keys) of dimBatch * N entries, keys = position in the flattened tensor."""
    out = _host.nbest(scores, N)
    if out is not None:
        return out
    scores = _f32c(scores, "getNBestList")
    _on_gpu(scores)
    return _taken(_host.nbest(scores, N), "getNBestList")


def getNBestWords(scores, N, ids=None):
    """the N best of every row of scores [.., cols] and the words they stand for: the positions in the
    row, or the shortlist's ids [cols] there; returns (scores [rows, N], int64 words [rows, N])"""
    out = _host.nbest_words(scores, N, ids)
    if out is not None:
        return out
    scores = _f32c(scores, "getNBestWords")
    _on_gpu(scores)
    return _taken(_host.nbest_words(scores, N, ids), "getNBestWords")


def getNBestListOfBeams(scores, N):
    """reference src/translator/beam_search.cpp:472 + :492: swapAxes(expandedPathScores, 0, 2)
    followed by getNBestList, without the transposed copy.  scores [beam, 1, dimBatch, vocab] (or
    [beam, dimBatch, vocab]); returns what getNBestList returns for the transposed tensor."""
    out = _host.nbest_beams(scores, N)
    if out is not None:
        return out
    scores = _f32c(scores, "getNBestListOfBeams")
    _on_gpu(scores)
    return _taken(_host.nbest_beams(scores, N), "getNBestListOfBeams")


def logsoftmaxNBestOfBeams(logits, N, pathScores=None, want_logprobs=False):
    """The end of a beam-search step in one call: logsoftmax over the vocabulary (reference
    src/tensors/cpu/tensor_operators.cpp:474-526), + the hypotheses' path scores
    (src/translator/beam_search.cpp:433-436), then what getNBestListOfBeams does (:472, :492).
    logits [beam, 1, dimBatch, vocab] (or [beam, dimBatch, vocab]); pathScores: None or one value
    per row [beam, dimBatch]; returns (vals, keys), and the log-probabilities as a third value when
    asked for.  Bit for bit what the separate calls give."""
    out = _host.logsoftmax_nbest_beams(logits, N, pathScores, want_logprobs)
    if out is not None:
        return out
    logits = _f32c(logits, "logsoftmaxNBestOfBeams")
    _on_gpu(logits)
    beam, vocab = logits.shape[0], logits.shape[-1]
    dimBatch = logits.numel() // (beam * vocab) if beam * vocab else 0
    if not (vocab % 4 == 0 and 4096 < vocab <= 32768 and logits.data_ptr() % 16 == 0):
        # sizes the one-launch form does not take: the separate calls
        lp = logsoftmax(logits)
        scored = lp if pathScores is None else lp + _f32c(pathScores, "logsoftmaxNBestOfBeams").reshape(
            (beam,) + (1,) * (logits.dim() - 3) + (dimBatch, 1))
        vals, keys = getNBestListOfBeams(scored, N)
        return (vals, keys, lp) if want_logprobs else (vals, keys)
    if pathScores is not None:
        pathScores = _f32c(pathScores, "logsoftmaxNBestOfBeams").reshape(-1)
        _abort_if(pathScores.numel() != beam * dimBatch, "one path score per hypothesis, got {}", pathScores.numel())
    return _taken(_host.logsoftmax_nbest_beams(logits, N, pathScores, want_logprobs), "logsoftmaxNBestOfBeams")
