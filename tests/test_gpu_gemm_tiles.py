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

# one row count per tile size for N = 1536 on 256 CUs (32 x 64, 64 x 64,
# 128 x 64, 128 x 128, 256 x 128, 256 x 256, the last with more tiles than CUs),
# none a multiple of its tile
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
    """One step to many, odd and even, on tiles of every stage depth."""
    rng = np.random.default_rng(k + rows)
    a, w = _signs(rng, (rows, k)), _signs(rng, (512, k))
    got = ops.linear(to_dev(a, dev, torch.float16), to_dev(w, dev, torch.float16), out_dtype=torch.float32)
    assert np.array_equal(host(got), orc.linear(a, w))


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


@pytest.mark.parametrize("rows", [70, 1700, 3001])
@pytest.mark.parametrize("heads,hd", [(4, 128), (8, 64)])
@pytest.mark.parametrize("kt", [True, False])
def test_qkv_positions_in_and_out_of_the_lookup(dev, rows, heads, hd, kt):
    """cos/sin looked up in the block's table, and computed for tokens whose
    coordinates it does not hold (negative, 128, large): the same bits as from
    the phase table of the same coordinates."""
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
