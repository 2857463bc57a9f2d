"""Multiplications of 65 to 256 rows (csrc/c_abi.hip, launch_gemm): outputs of few columns in small tiles, wide ones in the tiles of the
large-M forms, around the edges of each range, bit for bit against the forms they take the place of (measurement id 340)."""
import pytest

from conftest import load

pytestmark = pytest.mark.gpu

# (on a chip of 256 CUs)
SHAPES = [
    (64, 768, 2048),      # the stream form
    (65, 512, 2048),      # the stream form: two sub-steps to a wave
    (65, 512, 8200),      # 128x64, three stages
    (128, 1024, 4096),    # the stream form, its last width
    (128, 1024, 4104),    # 64x64
    (129, 1024, 1032),    # the stream form: four sub-steps to a wave
    (129, 1280, 1032),    # 32x64: five
    (256, 512, 2048),     # the stream form
    (257, 512, 2048),     # the stream form: two waves, eight sub-steps each
    (257, 384, 2048),     # 64x64: six
    (65, 768, 776),       # the stream form: three sub-steps to a wave
    (65, 1536, 776),      # 32x64: six
    (128, 640, 16384),    # 128x64, its last width
    (128, 640, 16392),    # 128x128
    (100, 1024, 32776),   # 128x128, ragged rows short of 14 MB
    (128, 256, 32776),    # 128x128, plain stores behind ragged rows from 14 MB on
    (128, 1152, 16384),   # 128x64, four stages, one to a CU
    (77, 1152, 16392),    # 128x64, three stages, two to a CU
    (80, 1152, 32776),    # 128x128, more than one to a CU
    (129, 1024, 8200),    # the forms of more rows
    (256, 1024, 16392),   # 128x128, and 128x64 for the last columns
    (256, 1024, 20000),   # 128x128 alone
    (200, 1152, 8200),    # long rows
    (130, 576, 8200),     # K no whole number of blocks
]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_multiplication_of_65_to_256_rows(M, K, N):
    import torch
    integer, lib = load("integer"), load("_lib")
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K + N)
    x = torch.randn(M, K, device="cuda", generator=g)
    w = integer.prepareB(torch.randn(K, N, device="cuda", generator=g) * 0.02)
    b = torch.randn(N, device="cuda", generator=g) * 0.01
    Aq = integer.prepareA(x)
    out = integer.multiply(Aq, w, b, scale=0.5, relu=M % 2 == 0)
    with lib.forced_kernel(340):
        assert torch.equal(integer.multiply(Aq, w, b, scale=0.5, relu=M % 2 == 0), out)
        want = integer.affine_f32(x, w)[0]
    assert torch.equal(integer.affine_f32(x, w)[0], want)
    y, _, top = integer.affine_f32(x, w, b, scale=0.5, relu=M % 2 == 0, want_absmax=True)
    assert torch.equal(y, out) and float(top.data.max()) == float(out.abs().max())
