"""GPU: every tile size the weight GEMM chooses from (t2h_linear,
t2h_linear_gate_residual, t2h_qkv_linear_pack), at ragged row counts, k
remainders and row strides past the 32-bit offsets.

The operands are -1, 0 and 1, so every product and partial sum is exact and
the results equal the C oracle's bit for bit; where operands are random, two
calls that must give the same bits are compared with each other.
"""
import numpy as np
import pytest
import torch

import oracle as orc
from _parity import host, to_dev
from t2h import nn, ops

pytestmark = pytest.mark.gpu

# row counts, none a multiple of its tile, that at N = 1536 and K = 128 or 192
# take 32 x 64 (two), 64 x 64, 128 x 64, 128 x 128, 256 x 128, 256 x 256 and
# 256 x 128 tiles on 256 CUs, the last two or three to a block. (At K = 1536
# the last takes 256 x 256.)
ROWS = [1, 301, 501, 1001, 2001, 4101, 8001, 12001]


def _signs(rng, shape):
    return rng.integers(-1, 2, shape).astype(np.float32)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_linear_every_tile_exact(dev, rows, dtype):
    """Bias and ReLU in the store, f32 and 16-bit outputs; k = 192: a last
    stage of half the k of a 64 x 64 or smaller tile's."""
    rng = np.random.default_rng(rows)
    n, k = 1536, 192
    a, w, b = _signs(rng, (rows, k)), _signs(rng, (n, k)), rng.integers(-3, 4, (n,)).astype(np.float32)
    want = orc.linear(a, w, bias=b)
    assert np.abs(want).max() < 256                      # exact in bf16 too
    ad, wd, bd = to_dev(a, dev, dtype), to_dev(w, dev, dtype), to_dev(b, dev)
    assert np.array_equal(host(ops.linear(ad, wd, bd, out_dtype=torch.float32)), want)
    assert np.array_equal(host(ops.linear(ad, wd, bd)), want)
    assert np.array_equal(host(ops.linear(ad, wd, bd, act=ops.ACT_RELU)), np.maximum(want, 0))


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("res_dtype", [torch.float16, torch.float32])
def test_gate_residual_every_tile_exact(dev, rows, res_dtype):
    """Three batches with borders inside tiles, power-of-two gates, in place."""
    rng = np.random.default_rng(100 + rows)
    n, k = 1536, 128
    a, w, b = _signs(rng, (rows, k)), _signs(rng, (n, k)), rng.integers(-3, 4, (n,)).astype(np.float32)
    gate = (2.0 ** rng.integers(-1, 2, (3, n))).astype(np.float32)
    res = rng.integers(-8, 9, (rows, n)).astype(np.float32)
    cuts = np.array([0, rows // 3, rows // 3, rows], np.int64)      # the second batch is empty
    want = orc.gate_residual(res, orc.linear(a, w), gate, cuts, b)
    rd = to_dev(res, dev, res_dtype)
    got = ops.linear_gate_residual(to_dev(a, dev, torch.float16), to_dev(w, dev, torch.float16), rd, bias=to_dev(b, dev),
                                   gate=to_dev(gate, dev), offsets=to_dev(cuts, dev), out=rd)
    assert got is rd and np.array_equal(host(rd), want)


@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 1536])
@pytest.mark.parametrize("rows", [9, 700, 2100, 9000])
def test_k_steps_exact(dev, rows, k):
    """One step to many, odd and even, on 32 x 64 (two row counts), 128 x 64
    and 256 x 128 tiles (every size: test_every_tile_at_few_k_steps)."""
    rng = np.random.default_rng(k + rows)
    a, w = _signs(rng, (rows, k)), _signs(rng, (512, k))
    got = ops.linear(to_dev(a, dev, torch.float16), to_dev(w, dev, torch.float16), out_dtype=torch.float32)
    assert np.array_equal(host(got), orc.linear(a, w))


def _exact(a, w, b=None):
    """a w^T + b of small integers: exact in f32 in any order."""
    out = a @ w.T
    return out if b is None else out + b


@pytest.mark.parametrize("k", [64, 128, 192, 320, 448])
@pytest.mark.parametrize("rows", [9, 1501, 3001, 6001, 12_001, 16_501])
def test_every_tile_at_few_k_steps(dev, rows, k):
    """N = 512: 32 x 64, 64 x 64, 128 x 64, 128 x 128, 256 x 128 and 256 x 256
    tiles at 1 to 7 k steps: fewer than their stages, odd and even, the linear
    and the residual in both stream types."""
    rng = np.random.default_rng(1000 + k + rows)
    a, w, b = _signs(rng, (rows, k)), _signs(rng, (512, k)), rng.integers(-3, 4, (512,)).astype(np.float32)
    ad, wd, bd = to_dev(a, dev, torch.float16), to_dev(w, dev, torch.float16), to_dev(b, dev)
    want = _exact(a, w, b)
    assert np.array_equal(host(ops.linear(ad, wd, bd, out_dtype=torch.float32)), want)
    assert np.array_equal(host(ops.linear(ad, wd, bd)), want)
    res = rng.integers(-8, 9, (rows, 512)).astype(np.float32)
    for dt in (torch.float16, torch.float32):
        assert np.array_equal(host(ops.linear_gate_residual(ad, wd, to_dev(res, dev, dt), bias=bd)), res + want)


@pytest.mark.parametrize("res_dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("rows,k", [(16_741, 192), (12_001, 192), (16_741, 4096)])
def test_residual_of_several_tiles_per_block(dev, rows, k, res_dtype):
    """396 tiles of 256 x 256 (564 of 256 x 128 at 12,001 rows) on 256 CUs: a
    block's residual rows, gate row and next operands overlap from tile to
    tile. Batches end inside tiles and at their edges, the join is in place;
    K = 4096 groups two token tiles instead of four."""
    rng = np.random.default_rng(2000 + rows + k)
    n = 1536
    a, w, b = _signs(rng, (rows, k)), _signs(rng, (n, k)), rng.integers(-3, 4, (n,)).astype(np.float32)
    cuts = np.array([0, 100, 256, 5000, 5000, 2 * rows // 3, rows], np.int64)
    gate = (2.0 ** rng.integers(-1, 2, (6, n))).astype(np.float32)
    res = rng.integers(-8, 9, (rows, n)).astype(np.float32)
    want = res + _exact(a, w, b) * np.repeat(gate, np.diff(cuts), axis=0)
    assert np.abs(want).max() < 1024                       # halves are exact in f16
    rd = to_dev(res, dev, res_dtype)
    ops.linear_gate_residual(to_dev(a, dev, torch.float16), to_dev(w, dev, torch.float16), rd, bias=to_dev(b, dev),
                             gate=to_dev(gate, dev), offsets=to_dev(cuts, dev), out=rd)
    assert np.array_equal(host(rd), want)


def test_rows_do_not_depend_on_the_row_count(dev):
    """Every tile size sums over k in the same order: the first rows of a call
    have the same bits whatever the call's size (random operands)."""
    g = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn((12001, 1536), generator=g, device=dev).half()
    w = (torch.randn((1536, 1536), generator=g, device=dev) * 0.025).half()
    full = ops.linear(x, w, out_dtype=torch.float32)
    for rows in ROWS[:-1]:
        assert torch.equal(ops.linear(x[:rows], w, out_dtype=torch.float32), full[:rows]), rows


def test_row_strides_past_32_bit_offsets(dev):
    """Token rows 2^22 + 8 elements apart: the same bits as packed rows."""
    rows, k, ldx = 5, 128, (1 << 22) + 8
    g = torch.Generator(device=dev).manual_seed(6)
    buf = torch.zeros((rows - 1) * ldx + k, dtype=torch.float16, device=dev)
    x = buf.as_strided((rows, k), (ldx, 1))
    x.copy_(torch.randn((rows, k), generator=g, device=dev))
    w = (torch.randn((768, k), generator=g, device=dev) * 0.1).half()
    assert torch.equal(ops.linear(x, w), ops.linear(x.contiguous(), w))
    for got, want in zip(ops.qkv_linear_pack(x, w, 2, use_rope=False, mp=8, lp=8),
                         ops.qkv_linear_pack(x.contiguous(), w, 2, use_rope=False, mp=8, lp=8)):
        assert torch.equal(got, want)
    gate = torch.randn((1, 768), generator=g, device=dev)
    for dt in (torch.float16, torch.float32):
        res = torch.randn((rows, 768), generator=g, device=dev).to(dt)
        assert torch.equal(ops.linear_gate_residual(x, w, res, gate=gate),
                           ops.linear_gate_residual(x.contiguous(), w, res, gate=gate))


@pytest.mark.parametrize("rows", [70, 1700, 3001])
@pytest.mark.parametrize("heads,hd", [(4, 128), (8, 64)])
@pytest.mark.parametrize("kt", [True, False])
def test_qkv_positions_in_and_out_of_the_lookup(dev, rows, heads, hd, kt):
    """cos/sin looked up in the block's table, and computed for tokens whose
    coordinates it does not hold (negative, 5,000): the same bits as from the
    phase table of the same coordinates. 128-token tiles, one to a block (the
    others: test_gpu_qkv_positions.py)."""
    rng = np.random.default_rng(rows + hd)
    c = rng.integers(0, 128, (rows, 4)).astype(np.int32)
    odd = rng.choice(rows, rows // 9, replace=False)
    c[odd, 1 + rng.integers(0, 3, odd.size)] = rng.choice(np.array([-1, -77, 127, 128, 129, 5000], np.int32), odd.size)
    g = torch.Generator(device=dev).manual_seed(7)
    k = 192
    x = torch.randn((rows, k), generator=g, device=dev).half()
    w = (torch.randn((3 * heads * hd, k), generator=g, device=dev) * 0.1).half()
    gam = torch.randn((2, heads, hd), generator=g, device=dev) * 0.02 + 1
    cd, fr, pad = to_dev(c, dev), nn.rope_freqs(hd), (rows + 7) // 8 * 8
    kw = dict(gamma_q=gam[0], gamma_k=gam[1], mp=pad, lp=pad, freqs=fr, k_transposed=kt)
    got = ops.qkv_linear_pack(x, w, heads, coords=cd, **kw)
    want = ops.qkv_linear_pack(x, w, heads, phases=ops.rope_phases(rows, hd, fr, coords=cd), **kw)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
