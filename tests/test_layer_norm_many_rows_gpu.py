"""Layer norm with a skip input, scale and shift of more rows than there are abs-max slots, up to rows that its workgroups come back for: bits, the abs-max
and what lies behind the last row.  Whole numbers in pairs of either sign, so that numpy's float32 operations give every bit."""
import numpy as np
import pytest

from conftest import load

pytestmark = pytest.mark.gpu
f32 = np.float32
SLOTS = 2048


@pytest.mark.parametrize("cols", [4, 64, 1000, 1024])
@pytest.mark.parametrize("rows", [1, 2048, 2049, 2500, 8192, 8193, 8300])
@pytest.mark.parametrize("form", ["skip", "alone"])
def test_rows_beyond_the_slots(integer, rows, cols, form):
    import torch
    lib = load("_lib")
    print("layer norm", rows, cols, form, flush=True)
    rng = np.random.default_rng(10 * cols + rows)
    gamma, beta = rng.standard_normal(cols).astype(f32), rng.standard_normal(cols).astype(f32)
    half = rng.integers(1, 16, (rows, cols // 2))
    x = np.concatenate([half, -half], axis=1).astype(f32)
    x = x[:, rng.permutation(cols)]
    part = rng.integers(-15, 16, (rows, cols)).astype(f32)
    var = ((x.astype(np.float64) ** 2).sum(1).astype(f32) / f32(cols)).astype(f32)
    sigma = np.sqrt((var + f32(1e-6)).astype(f32)).astype(f32)
    want = (gamma * (x / sigma[:, None]).astype(f32)).astype(f32) + beta
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    skip = form == "skip"
    a, add, g, b = dev(x - part if skip else x), dev(part), dev(gamma), dev(beta)
    out, slots = torch.full((rows * cols + 2048,), 7.0, device="cuda"), torch.full((SLOTS + 64,), float("nan"), device="cuda")
    lib.check(lib.lib().marian_hip_layer_norm(a.data_ptr(), add.data_ptr() if skip else None, g.data_ptr(), cols, b.data_ptr(), cols, out.data_ptr(), rows, cols,
                                              1e-6, slots.data_ptr(), torch.cuda.current_stream().cuda_stream), "layer_norm")
    got, slots = out.cpu().numpy(), slots.cpu().numpy()
    assert np.array_equal(got[:rows * cols].reshape(rows, cols), want)
    assert (got[rows * cols:] == 7.0).all(), "written past the rows"
    assert np.isnan(slots[SLOTS:]).all(), "written past the slots"
    assert (slots[:SLOTS] >= 0).all() and slots[:SLOTS].max() == np.abs(want).max()
