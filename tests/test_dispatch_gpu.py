"""Which form a multiplication takes (csrc/c_abi.hip, launch_gemm), where a rule's line lies: told by the number of workgroups that leave an
abs-max, on a chip of 256 CUs.  The sizes beside each were measured on both sides of the line."""
import ctypes

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


# rows, K, columns, and the rows and columns of a tile (None: the stream form, whose waves leave a value each, eight to a workgroup)
@pytest.mark.parametrize("M,K,N,tile", [
    (65, 384, 512, None),       # eight waves, two sub-steps each
    (200, 1024, 1024, None),    # four
    (129, 2048, 1536, None),    # eight
    (300, 512, 1024, None),     # four waves, four
    (100, 4096, 768, None),     # eight waves, two rounds of eight
    (65, 256, 3000, None),      # four waves, two
    (200, 512, 3000, None),     # two waves, eight
    (100, 1280, 1032, (32, 64)),    # eight waves, five
    (128, 3072, 512, (32, 64)),     # twelve
    (129, 1536, 1032, (32, 64)),    # six
    (160, 768, 3072, (32, 64)),     # four waves, six
    (160, 2048, 2048, (32, 64)),    # two rounds of eight
    (200, 384, 3072, (64, 64)),     # two waves, six
    (128, 512, 8192, (64, 64)),     # 128 rows to a workgroup in the stream form
])
def test_stream_form_or_small_tiles(M, K, N, tile):
    lib = load("_lib")
    with lib.forced_kernel(600):   # (quantized first: affine_f32 of so few rows may quantize on the way instead)
        found = workgroups(M, K, N)
    tiles = lambda rows, columns: -(-M // rows) * -(-N // columns)
    if tile:
        assert found == tiles(*tile)
    else:
        assert found > 2 * tiles(32, 64)


@pytest.mark.parametrize("M,K,N,tile", [
    (512, 768, 4096, (128, 64)),    # one to a CU
    (2048, 768, 768, (128, 64)),
    (600, 640, 3072, (128, 64)),
    (1500, 768, 1536, (64, 64)),    # 128x64 would be 288
    (1500, 512, 1024, (64, 64)),    # shorter rows
    (160, 512, 8192, (128, 64)),    # mostly weights
    (192, 384, 8192, (64, 64)),
    (512, 512, 8192, (128, 128)),   # four of 64x64 to a CU
    (300, 384, 12000, (64, 64)),    # 128x128 would be 282
    (1000, 512, 4096, (64, 64)),    # fewer of them weights
    (340, 640, 6144, (64, 64)),     # longer rows, nine to four CUs
])
def test_small_tiles_several_to_a_cu_or_taller_ones(M, K, N, tile):
    with load("_lib").forced_kernel(600):
        assert workgroups(M, K, N) == -(-M // tile[0]) * -(-N // tile[1])


@pytest.mark.parametrize("M,K,N,tiles", [
    (256, 1024, 16448, 256 + 2),        # two rows of 128 whole 128x128 tiles, and one of 128x64 each for the last columns
    (256, 512, 16504, 256 + 4),
    (384, 1024, 10928, 255 + 3),
    (256, 1024, 20000, 2 * 157),        # two rounds either way: 128x128 alone
])
def test_a_little_more_than_a_tile_to_a_cu(M, K, N, tiles):
    with load("_lib").forced_kernel(600):
        assert workgroups(M, K, N) == tiles


class KernelNode(ctypes.Structure):
    """hipKernelNodeParams"""
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint * 3),
                ("params", ctypes.c_void_p), ("lds", ctypes.c_uint)]


def launches(call, kernels=False):
    """the workgroups of the launches that a call makes, recorded, or their kernels"""
    import torch
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64.so" in line))
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    raw, n = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    found = []
    for node in nodes:
        p = KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        found.append(p.func if kernels else p.grid[0] * p.grid[1] * p.grid[2])
    return found


@pytest.mark.parametrize("M,K,Ns,tile", [
    (300, 768, (2048, 2048, 2048), (64, 64)),   # 128x64 would be 288; 480 of these
    (1500, 512, (512, 512, 512), (64, 64)),     # 576
    (600, 768, (1536, 1536, 1536), (64, 64)),   # 720
    (1024, 512, (1000, 1000, 1000), (128, 64)),  # 768: three to a CU
    (768, 768, (768, 768, 768), (128, 64)),     # 216 of 128x64
    (768, 256, (768, 768, 768), (64, 64)),      # short rows
    (600, 512, (512, 512), (64, 64)),           # one to a CU
])
def test_matrices_side_by_side(M, K, Ns, tile):
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the numbers are those of 256 CUs")
    integer = load("integer")
    x = torch.randn(M, K, device="cuda")
    weights = [(integer.prepareB(torch.randn(K, n, device="cuda") * 0.02), None) for n in Ns]
    assert launches(lambda: integer.affine_f32_grouped(x, weights))[-1] == -(-M // tile[0]) * sum(-(-n // tile[1]) for n in Ns)


@pytest.mark.parametrize("M,N,streamed", [
    (2100, 3968, True),    # 31.8 MB
    (2050, 4096, False),   # 32.03 MB: what reads the output would pay for the stores
    (2500, 4096, False),
])
def test_stores_of_large_outputs(M, N, streamed):
    """256x256 tiles with edges, and the same kernel as an output of 64 MB, or another"""
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the form is that of 256 CUs")
    integer = load("integer")

    def kernel(m, k, n):
        Aq, w = integer.prepareA(torch.randn(m, k, device="cuda")), integer.prepareB(torch.randn(k, n, device="cuda") * 0.02)
        return launches(lambda: integer.multiply(Aq, w), kernels=True)[-1]
    assert (kernel(M, 2048, N) != kernel(4090, 2048, 4096)) == streamed
