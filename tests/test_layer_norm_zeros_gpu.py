"""Layer norm of rows with values equal to their mean - single ones, rows of zeros or of one value, beside values too small for the shared
reciprocal: the bits of the division, signs of zeros among them.  Whole numbers times a power of two with mean zero, so that numpy's
float32 operations give every bit."""
import numpy as np
import pytest

from conftest import load

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.mark.parametrize("cols", [4, 64, 512, 1000, 1024])
@pytest.mark.parametrize("rows", [1, 8, 300])
def test_values_equal_to_the_mean(rows, cols):
    import torch
    ops = load("ops")
    rng = np.random.default_rng(1000 * cols + rows)
    gamma = rng.standard_normal(cols).astype(f32)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    half = rng.integers(1, 16, (rows, cols // 2))
    plain = np.concatenate([half, -half], axis=1)
    plain = np.take_along_axis(plain, rng.random((rows, cols)).argsort(1), 1).astype(f32)
    signs = np.where(rng.random((rows, cols)) < 0.5, f32(0.0), f32(-0.0))
    signs[:, 0] = f32(0.0)   # (a row of negative zeros alone has a mean of positive zero all the same)

    def with_zeros(x, pairs):   # that many values and their opposites
        x = x.copy()
        for r in range(rows):
            for _ in range(pairs):
                at = rng.integers(cols)
                other = (x[r] == -x[r, at]).argmax()
                x[r, at], x[r, other] = signs[r, at], signs[r, other]
        return x

    forms = {"one pair": with_zeros(plain, 1), "many": with_zeros(plain, cols // 3), "zeros": signs,
             "every other row": np.where(np.arange(rows)[:, None] % 2 == 0, signs, plain),
             "tiny beside zeros": with_zeros(plain, 1) * f32(2.0) ** f32(-64), "tiny": plain * f32(2.0) ** f32(-64),
             "least": with_zeros(plain, 1) * f32(2.0) ** f32(-60)}
    for name, x in forms.items():
        print("layer norm", rows, cols, name, flush=True)
        var = ((x.astype(np.float64) ** 2).sum(1).astype(f32) / f32(cols)).astype(f32)
        sigma = np.sqrt((var + f32(1e-6)).astype(f32)).astype(f32)
        want = (gamma * (x / sigma[:, None]).astype(f32)).astype(f32)
        got = ops.layerNorm(dev(x), dev(gamma), eps=1e-6).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), name
        beta = rng.standard_normal(cols).astype(f32)
        got = ops.layerNorm(dev(x), dev(gamma), dev(beta), eps=1e-6, add=dev(np.zeros_like(x))).cpu().numpy()
        assert np.array_equal(got, want + beta), name
    constant = np.full((rows, cols), f32(3.0))
    got = ops.layerNorm(dev(constant), dev(gamma), eps=1e-6).cpu().numpy()
    assert np.array_equal(got, np.zeros_like(constant))
