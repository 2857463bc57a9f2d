"""The merge of the hypotheses' n-best lists at the end of a beam-search step (csrc/decode_ops.hip, nbest_hand_over): numbers of candidates
around the 64 that one wave merges from registers, with equal scores within and across hypotheses, against a stable sort."""
import numpy as np
import pytest

from conftest import load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beam,N", [(1, 1), (1, 16), (7, 9), (8, 8), (16, 4), (13, 5), (9, 8), (12, 12)])
@pytest.mark.parametrize("batch,vocab", [(1, 4100), (5, 8192)])
def test_merge_of_candidates(beam, N, batch, vocab):
    import torch
    ops = load("ops")
    rng = np.random.default_rng(beam * 100 + N)
    x = torch.from_numpy(rng.standard_normal((beam, 1, batch, vocab)).astype(np.float32)).cuda()
    x[:, 0, 0, ::257] = 5.0   # equal logits in a row and, rows being alike below, across hypotheses
    if beam > 1:
        x[1] = x[0]
    lp = ops.logsoftmax(x)
    for _ in range(3):   # (the counters are left at zero)
        vals, keys = ops.logsoftmaxNBestOfBeams(x, N)
        flat = lp.permute(2, 1, 0, 3).reshape(batch, -1).cpu().numpy()
        order = np.argsort(-flat, axis=1, kind="stable")[:, :N]
        assert np.array_equal(vals.cpu().numpy().reshape(batch, N), np.take_along_axis(flat, order, 1))
        want = order + np.arange(batch)[:, None] * flat.shape[1]
        assert np.array_equal(keys.cpu().numpy().view(np.uint32).reshape(batch, N).astype(np.int64), want)
        assert torch.equal(ops.getNBestListOfBeams(lp, N)[1], keys)
