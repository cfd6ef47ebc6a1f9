"""Quantize's two routes, chosen per wave: reciprocal divisions where the inputs
are finite and the scales of ordinary size, divisions as written elsewhere.
Codes, scales and biases are the oracle's bit for bit on both, so there is no
tolerance; inputs sit on and around rounding ties of the quotients, at scales
past the reciprocal's range, and in waves that hold a non-finite group among
ordinary ones."""

import numpy as np
import pytest
import torch

import mlxturbo_amd as mq
from oracle import oracle as O
from qmm_helpers import TORCH_DTYPE, from_dev

pytestmark = pytest.mark.gpu


def _values(rng, n, gs, bits, dtype):
    """n groups: plain ones, grids of half steps (every quotient a tie or an
    integer, before rounding to dtype), half steps moved by one float, tiny
    values beside one large one, and all of them over many magnitudes."""
    nb = (1 << bits) - 1
    w = rng.standard_normal((n, gs)).astype(np.float32)
    half = rng.integers(0, 2 * nb + 1, (n, gs)).astype(np.float32) / 2
    half[:, 0], half[:, 1] = 0, nb
    off = rng.integers(-nb, 1, (n, 1)).astype(np.float32)
    grid = half + off
    kind = rng.integers(0, 5, n)
    w[kind == 1] = grid[kind == 1]
    near = np.nextafter(grid, np.where(rng.random((n, gs)) < 0.5, -np.inf, np.inf).astype(np.float32))
    w[kind == 2] = near[kind == 2]
    tiny = w * np.float32(1e-30)
    tiny[:, 3] = 1.7
    w[kind == 3] = tiny[kind == 3]
    lim = 6 if dtype == "float16" else 100
    scale = np.exp2(rng.integers(-20, lim, n)).astype(np.float32)
    third = np.where(rng.random(n) < 0.5, np.float32(1), np.float32(1) / 3).astype(np.float32)
    return w * (scale * third)[:, None]


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("bits, gs, rows", [
    (4, 32, 257), (4, 64, 1), (8, 64, 130), (8, 128, 65), (2, 32, 63), (3, 64, 40), (5, 128, 31),
    (6, 64, 33),
])
def test_quantize_routes(bits, gs, rows, dtype):
    rng = np.random.default_rng(bits * 1000 + gs + rows)
    G = 7                                       # a wave holds groups of several rows
    w = _values(rng, rows * G, gs, bits, dtype).reshape(rows, G * gs)
    if rows > 1:                                # whole waves of both routes, and mixed ones
        w[rows // 2, 5] = np.inf
        w[rows // 3, gs + 1] = np.nan
        if dtype != "float16":
            w[rows - 1] *= np.float32(2.0 ** 20)
    w = O.to_f32(O.from_f32(w, dtype), dtype)
    t = torch.from_numpy(w).cuda().to(TORCH_DTYPE[dtype])
    got = mq.quantize(t, group_size=gs, bits=bits)
    want = O.quantize(w, gs, bits, dtype)
    np.testing.assert_array_equal(from_dev(got[0]), want[0])
    for g, e in zip(got[1:], want[1:]):
        e = O.to_f32(e, dtype)
        np.testing.assert_array_equal(g.float().cpu().numpy(), e)   # NaN equals NaN


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("from_bits, from_gs, bits, gs, N, K", [
    (8, 64, 4, 64, 130, 640), (8, 128, 4, 32, 33, 384), (8, 32, 2, 128, 7, 1152),
    (4, 32, 8, 64, 65, 192), (4, 64, 3, 32, 40, 320), (4, 128, 6, 64, 1, 128),
    (8, 64, 5, 128, 63, 256), (4, 64, 4, 64, 257, 64),
])
def test_requantize_is_dequantize_then_quantize(from_bits, from_gs, bits, gs, N, K, dtype):
    """One pass over the codes: the bytes of the two operators, with scales of
    either sign, out of the reciprocal's range, infinite and NaN."""
    g = torch.Generator(device="cuda").manual_seed(N + K + bits)
    w = torch.randint(-2**31, 2**31, (N, K * from_bits // 32), generator=g, device="cuda",
                      dtype=torch.int64).to(torch.int32).view(torch.uint32)
    s = torch.randn((N, K // from_gs), generator=g, device="cuda")
    b = torch.randn((N, K // from_gs), generator=g, device="cuda") * 8
    if N > 1:
        s[0] = 1e-30
        s[N // 2, 0] = float("inf")
        b[N // 3, 0] = float("nan")
        s[N - 1] *= 1e4 if dtype == "float16" else 1e34
    s, b = s.to(TORCH_DTYPE[dtype]), b.to(TORCH_DTYPE[dtype])
    kw = dict(group_size=gs, bits=bits)
    got = mq.ops._requantize(w, s, b, from_gs, from_bits, gs, bits)
    want = mq.quantize(mq.dequantize(w, s, b, group_size=from_gs, bits=from_bits), **kw)
    for x, y in zip(got, want):
        assert x.shape == y.shape and x.dtype == y.dtype
        assert torch.equal(x.view(torch.int32) if x.dtype == torch.uint32 else x.view(torch.int16),
                           y.view(torch.int32) if y.dtype == torch.uint32 else y.view(torch.int16))
    assert mq.ops._requantize(w, s, b, from_gs, from_bits, gs, 7) is None
    assert mq.ops._requantize(w, s.float(), b.float(), from_gs, from_bits, gs, bits) is None
