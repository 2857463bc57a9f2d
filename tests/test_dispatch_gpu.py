"""Which form a multiplication takes (csrc/c_abi.hip, launch_gemm), where a rule's line lies: told by the number of workgroups that leave an
abs-max, on a chip of 256 CUs.  The sizes beside each were measured on both sides of the line."""
import pytest

from conftest import load

pytestmark = pytest.mark.gpu


def workgroups(M, K, N):
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the numbers are those of 256 CUs")
    integer = load("integer")
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K + N)
    x = torch.randn(M, K, device="cuda", generator=g)
    w = integer.prepareB(torch.randn(K, N, device="cuda", generator=g) * 0.02)
    y, _, top = integer.affine_f32(x, w, want_absmax=True)
    assert float(top.data.max()) == float(y.abs().max())
    return int(top.data.count_nonzero())


@pytest.mark.parametrize("M,K,N,tiles", [
    (2048, 1024, 4096, 512),   # 128x128, two to a CU, one round of them
    (2000, 768, 4096, 512),
    (1000, 2048, 8192, 512),
    (2050, 1024, 4096, 144),   # a row of tiles more: 256x256
    (3000, 768, 3072, 144),
    (2500, 512, 4096, 640),    # short rows: 128x128
])
def test_two_tiles_to_a_cu(M, K, N, tiles):
    assert workgroups(M, K, N) == tiles
