"""The 256-column MFMA tile whose weights go from memory through registers into
MFMA operands: the wide kernel of quantized_matmul and the thin grouped kernel
of 8-bit banks, at the edges of its rows, columns, k-steps and scale loads, and
at every tile height (test_launch_model.py checks on the CPU that TALL's shapes
are planned as written).

References are float64 products of the dequantized weights, rounded to the
output type.  Tolerance: a float32 sum of K terms is off by about sqrt(K) 2^-24
of the output's size, which moves that part of a 16-bit rounding step's worth
of outputs by one step: below 2e-4 of the norm for bfloat16, less for float16;
1e-3 is the bound of oracle.check_output for the whole."""

import pytest
import torch

import mlxturbo_amd as mq

pytestmark = pytest.mark.gpu

BF16, F16 = torch.bfloat16, torch.float16


def _quantized(rows, K, bits, gs, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = (torch.randn((rows, K), generator=g, device="cuda") * 0.05).to(dtype)
    return g, mq.quantize(w, group_size=gs, bits=bits)


def _check(out, ref):
    ref = ref.to(out.dtype).double()
    assert ((out.double() - ref).norm() / ref.norm()).item() < 1e-3


def _shifted(t):
    """t at an odd element address: its values are loaded one by one."""
    d = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
    d[1:].copy_(t.reshape(-1))
    return d[1:]


@pytest.mark.parametrize("M, N, K, bits, gs, dtype", [
    (65, 257, 64, 4, 64, BF16),        # one k-step, one column past a tile
    (127, 255, 320, 4, 64, BF16),      # steps of scales one by one (K = 64 odd)
    (129, 1000, 640, 8, 128, F16),     # two by two
    (193, 264, 1152, 4, 32, BF16),     # two groups per step, two by two
    (257, 250, 512, 8, 32, F16),       # one row past four tiles, four by four
    (300, 5121, 2048, 4, 128, BF16),   # N odd: stores of single values
    (96, 512, 4096, 8, 64, BF16),      # K split over workgroups
    (385, 768, 8192, 4, 64, F16),
    (1030, 513, 256, 4, 64, BF16),     # one round of four steps
])
def test_wide_edges(M, N, K, bits, gs, dtype):
    """Small matrices, all planned as 64-row tiles."""
    _wide(M, N, K, bits, gs, dtype)


# M, N, K, bits, group size, dtype; then the plan: rows of a tile, steps per load
# of scales, whether K is split.  Odd N stores values one by one.
TALL = [
    (70, 40007, 192, 4, 64, BF16, 128, 1, False),     # three steps: no whole four
    (200, 17408, 448, 8, 32, F16, 128, 1, False),     # one whole four and three
    (70, 8200, 2880, 4, 32, BF16, 128, 1, True),      # eleven fours and one, split
    (70, 40007, 384, 4, 64, BF16, 128, 2, False),
    (70, 8200, 2944, 8, 128, BF16, 128, 2, True),
    (200, 17413, 512, 8, 32, F16, 128, 4, False),
    (200, 17408, 512, 4, 64, F16, 128, 4, False),
    (70, 8200, 4096, 4, 32, BF16, 128, 4, True),
    (450, 17413, 64, 4, 64, BF16, 192, 1, False),     # one step
    (450, 17408, 320, 8, 32, F16, 192, 1, False),
    (129, 8200, 2880, 4, 64, BF16, 192, 1, True),
    (450, 17413, 128, 8, 64, BF16, 192, 2, False),
    (450, 17408, 384, 4, 32, BF16, 192, 2, False),
    (129, 8200, 2944, 8, 128, F16, 192, 2, True),
    (385, 17408, 512, 4, 128, F16, 192, 4, False),
    (129, 8200, 5120, 4, 64, BF16, 192, 4, True),
    (600, 17413, 320, 4, 64, BF16, 256, 1, False),
    (200, 17408, 2880, 8, 32, BF16, 256, 1, True),
    (600, 17408, 384, 4, 128, F16, 256, 2, False),
    (200, 17413, 4224, 8, 64, BF16, 256, 2, True),
    (600, 17413, 512, 4, 64, BF16, 256, 4, False),
    (600, 17408, 512, 8, 64, F16, 256, 4, False),
    (200, 17408, 5120, 4, 128, BF16, 256, 4, True),
]


@pytest.mark.parametrize("M, N, K, bits, gs, dtype, bm, unit, split", TALL)
def test_wide_heights(M, N, K, bits, gs, dtype, bm, unit, split):
    """Tiles of 128, 192 and 256 rows, with scales loaded for four, two and one
    steps, fours of steps with and without a rest; with the scales at an odd
    address every height runs its one-step loads."""
    _wide(M, N, K, bits, gs, dtype)


def _wide(M, N, K, bits, gs, dtype):
    g, (w, s, b) = _quantized(N, K, bits, gs, dtype, M + N + K)
    x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
    ref = x.double() @ mq.dequantize(w, s, b, group_size=gs, bits=bits).double().T
    out = mq.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    _check(out, ref)
    _check(out[-1:], ref[-1:])
    _check(out[:, -1:], ref[:, -1:])
    for r in range(0, M, 64):                  # a wrong tile shows in its own rows
        _check(out[r:r + 64], ref[r:r + 64])
    # scales at an odd address; the C entry has no workspace, so no K split
    ss, sb = _shifted(s), _shifted(b)
    got = torch.full_like(out, float("nan"))
    rc = mq._lib.lib().mq_quantized_matmul(
        x.data_ptr(), w.data_ptr(), ss.data_ptr(), sb.data_ptr(), got.data_ptr(), M, N, K, gs,
        bits, 0 if dtype == BF16 else 1, 1, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    for r in range(0, M, 64):
        _check(got[r:r + 64], ref[r:r + 64])


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("E, T, top, M, N, K, gs, dtype", [
    (16, 64, 16, 1, 256, 64, 64, BF16),     # one k-step, 64 rows per expert
    (24, 260, 4, 1, 257, 320, 64, F16),     # K = 64 odd, N odd
    (40, 300, 4, 1, 136, 640, 128, BF16),   # K = 128 odd, one ragged column tile
    (64, 128, 8, 3, 264, 512, 32, BF16),    # three rows per pair
    (32, 200, 8, 1, 512, 2048, 64, F16),
])
def test_thin_grouped_edges(bits, E, T, top, M, N, K, gs, dtype):
    g, (w, s, b) = _quantized(E * N, K, bits, gs, dtype, E + T + N + K)
    w, s, b = (t.reshape(E, N, -1) for t in (w, s, b))
    x = torch.randn((T, 1, M, K), generator=g, device="cuda").to(dtype)
    # expert 0 takes every token (segments of several tiles), the last ones few,
    # and some pairs an expert that is not there (zero rows)
    idx = torch.randint(0, E, (T, top), generator=g, device="cuda", dtype=torch.int32)
    idx[:, 0] = 0
    idx[::7, 1] = E
    out = mq.gather_qmm(x, w, s, b, rhs_indices=idx, group_size=gs, bits=bits)
    assert out.shape == (T, top, M, N)
    deq = mq.dequantize(w, s, b, group_size=gs, bits=bits)
    for e in range(E):
        t, j = (idx == e).nonzero(as_tuple=True)
        if len(t):
            ref = x[t, 0].double() @ deq[e].double().T
            _check(out[t, j], ref)
            _check(out[t, j][..., -1:], ref[..., -1:])
    assert not out[idx == E].any()
