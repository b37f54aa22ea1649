"""GPU: t2h_qkv_linear_pack's cos/sin, looked up in a block's table or computed
for tokens outside it, in blocks that walk several 256-token tiles. The phase
table of the same positions must give the same bits."""
import numpy as np
import pytest
import torch

from _parity import to_dev
from t2h import nn, ops

pytestmark = pytest.mark.gpu

# around the table's ends (167 positions for 21 frequencies, 256 at
# most), around 16 bits, and the ends of int32
ODD = np.array([-1, -77, 127, 128, 160, 161, 166, 167, 168, 255, 256, 5000, 32767, 32768, -32767, -32768, -32769,
                1 << 24, (1 << 31) - 1, -(1 << 31)], np.int64).astype(np.int32)


def _both(dev, rows, heads, hd, pos_dim, kt, pad, **pos):
    g = torch.Generator(device=dev).manual_seed(7)
    k = 192
    x = torch.randn((rows, k), generator=g, device=dev).half()
    w = (torch.randn((3 * heads * hd, k), generator=g, device=dev) * 0.1).half()
    b = torch.randn((3 * heads * hd,), generator=g, device=dev) * 0.02
    gam = torch.randn((2, heads, hd), generator=g, device=dev) * 0.02 + 1
    fr = nn.rope_freqs(hd, pos_dim)
    kw = dict(bias=b, gamma_q=gam[0], gamma_k=gam[1], mp=pad, lp=pad, freqs=fr, k_transposed=kt, pos_dim=pos_dim)
    ph = ops.rope_phases(rows, hd, fr, pos_dim=pos_dim, device=dev, **pos)
    return ops.qkv_linear_pack(x, w, heads, **pos, **kw), ops.qkv_linear_pack(x, w, heads, phases=ph, **kw)


# 360 and 288 tiles of 256 x 256 (256 CUs), the last token tile ragged, pads
# past it
@pytest.mark.parametrize("rows,heads,hd", [(5001, 12, 128), (6001, 16, 64)])
@pytest.mark.parametrize("kt", [True, False])
@pytest.mark.parametrize("pos_dim,share", [(3, 0), (3, 9), (3, 1), (1, 9), (2, 9), (4, 9)])
def test_coords_over_several_tiles(dev, rows, heads, hd, kt, pos_dim, share):
    """No token, every ninth or every token with a coordinate outside."""
    rng = np.random.default_rng(rows + pos_dim + share)
    c = rng.integers(0, 48, (rows, 1 + pos_dim)).astype(np.int32)
    if share:
        odd = rng.choice(rows, rows // share, replace=False)
        c[odd, 1 + rng.integers(0, pos_dim, odd.size)] = rng.choice(ODD, odd.size)
    for got, want in zip(*_both(dev, rows, heads, hd, pos_dim, kt, 6656, coords=to_dev(c, dev))):
        assert torch.equal(got, want)


@pytest.mark.parametrize("res", [16, 200, 40_000])
@pytest.mark.parametrize("rows", [70, 33_001])
def test_dense_grid(dev, rows, res):
    """Positions of the dense grid inside the table, past it, and (the last
    axis of row 32,768 on) past 16 bits; 128- and 256-token tiles."""
    for got, want in zip(*_both(dev, rows, 2, 128, 3, False, (rows + 303) // 8 * 8, grid_res=res)):
        assert torch.equal(got, want)
