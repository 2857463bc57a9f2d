"""Abs-max slots that attention_heads_kernel leaves: the largest magnitude of every wave's sixteen query rows, zeros for waves without rows
and behind the last wave.  Through the C entry point: the host mirror asks for no abs-max of so many rows."""
import ctypes

import pytest

from conftest import load

pytestmark = pytest.mark.gpu
SLOTS = 2048


def attend(heads, m, L, slots):
    import torch
    lib = load("_lib")
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 * m + L)
    q, k, v = (torch.randn(heads, n, 64, device="cuda", generator=g) for n in (m, L, L))
    out = torch.full((heads * m * 64 + 4096,), 7.0, device="cuda")
    strides = [(ctypes.c_int64 * 3)(n * 64, n * 64, 64) for n in (m, L, L, m)]
    lib.check(lib.lib().marian_hip_attention_rows(q.data_ptr(), strides[0], k.data_ptr(), strides[1], v.data_ptr(), strides[2], None, 1, 1, out.data_ptr(),
                                                  strides[3], heads, heads, 1, m, L, 64, 0.125, None if slots is None else slots.data_ptr(),
                                                  torch.cuda.current_stream().cuda_stream), "attention_rows")
    torch.cuda.synchronize()
    assert bool((out[heads * m * 64:] == 7.0).all()), "written past the rows"
    return out[:heads * m * 64].view(heads, m, 64)


# heads x rows x keys, waves of a workgroup (None: their slots would be too many, and the other form takes the call)
@pytest.mark.parametrize("heads,m,L,waves", [(288, 17, 32, 2), (288, 8, 20, 2), (288, 33, 48, 3), (288, 48, 33, 3), (288, 49, 64, 4), (288, 64, 50, 4),
                                             (255, 65, 80, 3), (200, 96, 96, 3), (255, 97, 128, 4), (144, 48, 64, 4), (512, 64, 64, 4), (250, 112, 80, None)])
def test_slots(integer, heads, m, L, waves):
    import torch
    print("slots", heads, m, L, flush=True)
    slots = torch.full((SLOTS + 64,), float("nan"), device="cuda")
    out = attend(heads, m, L, slots)
    assert torch.equal(out, attend(heads, m, L, None))
    assert bool(slots[SLOTS:].isnan().all()), "written past the slots"
    slots = slots[:SLOTS]
    assert float(slots.max()) == float(out.abs().max()) and bool((slots >= 0).all())
    if waves:
        rows = waves * 16
        groups = -(-m // rows)
        padded = torch.zeros(heads, groups * rows, 64, device="cuda")
        padded[:, :m] = out.abs()
        want = torch.zeros(SLOTS, device="cuda")
        want[:heads * groups * waves] = padded.view(heads * groups * waves, 16 * 64).max(1).values
        assert torch.equal(slots, want)
