"""The abs-max that the workgroups of a launch exchange (marian-dev_amd/csrc/onepass_exchange.h): numbers of workgroups around those at which
the words take another line, the maximum in the first, the last and a middle workgroup's share, and the call again on other values."""
import numpy as np
import pytest

from conftest import load
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def values(rng, rows, cols, at):
    x = rng.standard_normal((rows, cols)).astype(np.float32)
    x.flat[at] = np.float32(9.5)
    return x


# 1024 threads hold 16 values each: workgroups of prepareA, a CU's worth of a 256-CU chip at the most
@pytest.mark.parametrize("groups", [3, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256])
def test_prepare_a_of_so_many_workgroups(groups):
    import torch
    integer = load("integer")
    rng = np.random.default_rng(groups)
    rows, cols = (groups - 1) * 256 + 1, 64   # (one row of the last workgroup's 256)
    for at in (0, rows * cols - 1, (groups // 2) * 16384 + 5):
        x = values(rng, rows, cols, at)
        assert np.array_equal(integer.prepareA(torch.from_numpy(x).cuda()).numpy(), orc.prepare_a(x)), (groups, at)


# tiles of 8, 16 or 32 rows and 32 columns; rows of more than 2048 values, which exchange it up to a workgroup to two CUs
@pytest.mark.parametrize("M,K,N", [(9, 4096, 1000), (40, 3072, 768), (100, 4096, 1024), (128, 2112, 1024), (64, 4096, 512), (256, 1024, 1000)])
def test_multiplication_that_takes_the_absmax(M, K, N):
    import torch
    integer = load("integer")
    rng = np.random.default_rng(M + K)
    W = (0.02 * rng.standard_normal((K, N))).astype(np.float32)
    Bq = integer.prepareB(torch.from_numpy(W).cuda())
    for at in (0, M * K - 1, M * K // 2 + 3):
        x = values(rng, M, K, at)
        out, Aq = integer.affine_f32(torch.from_numpy(x).cuda(), Bq)
        Aq_h, Bq_h = orc.prepare_a(x), orc.prepare_b(W)
        assert np.array_equal(Aq.numpy(), Aq_h), at
        want = orc.affine(Aq_h, Bq_h, None, M, K, N, 1.0, False)[0]
        assert np.allclose(out.cpu().numpy(), want, rtol=1e-5, atol=1e-6), at   # (whole accumulators, two roundings)


@pytest.mark.parametrize("M,K,N,exchanged", [
    (40, 3072, 768, True),      # 120 workgroups
    (64, 4096, 512, True),      # 128
    (64, 4096, 544, False),     # 136: more than one to two CUs of long rows
    (100, 4096, 1024, False),
    (128, 2112, 1024, False),
    (256, 2048, 256, True),     # 256 of shorter rows
    (256, 1024, 1000, True),
])
def test_which_multiplications_exchange_it(M, K, N, exchanged):
    """told by the words that an exchange leaves in the workspace, behind the partials"""
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the numbers are those of 256 CUs")
    integer = load("integer")
    x, w = torch.randn(M, K, device="cuda"), integer.prepareB(torch.randn(K, N, device="cuda") * 0.02)
    torch.cuda.synchronize()
    words = integer.Backend.get("cuda:0").workspace[4096:]
    words.fill_(0x25)
    integer.dot(x, w)
    torch.cuda.synchronize()
    assert bool((words != 0x25).any()) == exchanged
