"""GPU: the hardware's f32 -> bf16 conversion rounds to nearest even and keeps
NaN, infinities, zeros' signs and denormals as the integer arithmetic
u + 0x7FFF + ((u >> 16) & 1), >> 16 does."""
import numpy as np
import pytest
import torch

from _parity import to_dev
from t2h import ops

pytestmark = pytest.mark.gpu

# under every upper half: exact, just above, around and at the tie, just below
LOW = [0, 1, 2, 0x3FFF, 0x4000, 0x7FFE, 0x7FFF, 0x8000, 0x8001, 0x8002, 0xBFFF, 0xC000, 0xFFFE, 0xFFFF]


def _rounded(u):
    return ((u.astype(np.uint64) + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


@pytest.mark.parametrize("cols", [1024, 1023])
def test_rounding_over_all_upper_halves(dev, cols):
    """modulate of x = 0 stores its f32 shift rounded: pairs in 16-byte pieces
    (1,024 columns) and one value at a time (1,023)."""
    u = (np.arange(1 << 16, dtype=np.uint32)[:, None] << 16 | np.array(LOW, np.uint32)).reshape(-1)
    rows = -(-u.size // cols)
    u = np.concatenate([u, np.zeros(rows * cols - u.size, np.uint32)])
    shift = torch.from_numpy(u.view(np.float32).reshape(rows, cols)).to(dev)
    x = torch.zeros((rows, cols), dtype=torch.bfloat16, device=dev)
    got = ops.modulate(x, shift, torch.zeros_like(shift), rows_per_batch=1)
    got = got.view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1)
    nan = np.isnan(u.view(np.float32))
    assert np.all((got[nan] & 0x7FFF) > 0x7F80)                      # NaN stays NaN
    want = np.where(u == 0x80000000, np.uint16(0), _rounded(u))      # 0 * 1 + -0 = 0
    assert np.array_equal(got[~nan], want[~nan])
