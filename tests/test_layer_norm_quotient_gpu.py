"""The layer norm of a wave's row divides by a shared reciprocal where no step under- or overflows: its bits are those of the
division.  Rows of whole numbers in pairs of either sign, times a power of two, have the same mean and variance in any order of
summation, so numpy's float32 operations give every bit."""
import numpy as np
import pytest

from conftest import load

pytestmark = pytest.mark.gpu
f32 = np.float32


def expected(x, gamma, beta, eps):
    with np.errstate(all="ignore"):
        sq = (x.astype(np.float64) ** 2).sum(1)   # (exact: whole numbers below 2^53 times a power of two)
        var = (sq.astype(f32) / f32(x.shape[1])).astype(f32)
        sigma = np.sqrt((var + f32(eps)).astype(f32)).astype(f32)
        return (gamma * (x / sigma[:, None]).astype(f32)).astype(f32) + beta


@pytest.mark.parametrize("cols", [4, 64, 256, 512, 1000, 1024])
@pytest.mark.parametrize("rows", [1, 37, 2500])
def test_bits_of_the_division(rows, cols):
    import torch
    ops = load("ops")
    rng = np.random.default_rng(1000 * cols + rows)
    gamma, beta = rng.standard_normal(cols).astype(f32), rng.standard_normal(cols).astype(f32)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    # magnitudes at and past the edges of the quotient's range (2^-60 .. , divisors 2^-40 .. 2^40), with zeros of either sign among them
    for exponent in (-64, -61, -60, -58, -40, -20, 0, 20, 36, 40, 45, 56, 60, 61):
        for zero in (False, True):
            print("layer norm", rows, cols, exponent, zero, flush=True)
            half = rng.integers(1, 16, (rows, cols // 2))
            x = np.concatenate([half, -half], axis=1)
            x = np.take_along_axis(x, rng.random((rows, cols)).argsort(1), 1).astype(f32) * f32(2.0) ** f32(exponent)
            if zero:
                lost = x[np.arange(rows), np.arange(rows) % cols].copy()
                other = (x == -lost[:, None]).argmax(1)
                x[np.arange(rows), np.arange(rows) % cols], x[np.arange(rows), other] = f32(0.0), f32(-0.0)
            eps = 1e-6 if exponent > -40 else 1e-30
            want = expected(x, gamma, beta, eps)
            got = ops.layerNorm(dev(x), dev(gamma), dev(beta), eps=eps)
            assert np.array_equal(got.cpu().numpy(), want), (exponent, zero)
            # with a skip input (all loads as buffers), in whole numbers as well; nothing is written past the rows
            part = rng.integers(-15, 16, (rows, cols)).astype(f32) * f32(2.0) ** f32(exponent)
            got = ops.layerNorm(dev(x - part), dev(gamma), dev(beta), eps=eps, add=dev(part))
            assert np.array_equal(got.cpu().numpy(), want), (exponent, zero, "skip")
