"""Scales with |s| >= 2^100 through every matmul kernel.

The kernels dequantize with s * 2^24 folded into one fma (exact while
|s| < 2^100); larger scales must take the plain float route and still give
MLX's values.  The skinny kernel and the thin kernel of 4-bit banks choose per
step, the tiles of the wide kernels and of the thin kernel of 8-bit banks run
the fast route and recompute a tile that met such a scale.  Rows with huge
scales and ordinary rows are checked against the oracle (the larger shapes
against float64 products of the dequantized weights, within the 1e-3 of
oracle.check_output) separately: the tolerance scales with each set's own
magnitude.
"""

import numpy as np
import pytest
import torch

import mlxturbo_amd as mq
from oracle import oracle as O
from mlxturbo_amd import ops
from qmm_helpers import TORCH_DTYPE, act, bits16, from_dev, quantized, to_dev

pytestmark = pytest.mark.gpu


def _huge(s, rows, group):
    s_f = O.to_f32(s, "bfloat16")
    s_f[rows, group] = 2.0 ** 110
    return O.from_f32(s_f, "bfloat16")


def _check_split(out, ref, huge_rows):
    rest = np.setdiff1d(np.arange(ref.shape[-1]), huge_rows)
    for cols in (huge_rows, rest):
        res = O.check_output(out[..., cols], ref[..., cols])
        assert res["ok"], res


@pytest.mark.parametrize("M", [1, 8, 40, 300])
def test_qmm_huge_scales(M):
    rng = np.random.default_rng(M)
    N, K, gs = 512, 1024, 64
    w, s, b = quantized(rng, N, K, gs)
    huge_rows = np.array([3, 260, 511])
    s = _huge(s, huge_rows, 5)
    x = act(rng, (M, K))
    out = from_dev(mq.quantized_matmul(to_dev(x, "bfloat16"), to_dev(w), to_dev(s, "bfloat16"),
                                       to_dev(b, "bfloat16"), group_size=gs))
    ref = O.quantized_matmul_ref(x, w, s, b, gs)
    assert np.all(np.isfinite(out))
    _check_split(out, ref, huge_rows)


@pytest.mark.parametrize("M", [6, 16, 24])
def test_qmm_huge_scales_shared_x(M):
    """5-32 rows on a matrix of 48+ rows per CU: one workgroup per CU of three
    wave groups (x resident in LDS for 6 rows, staged per step for 16, two
    16-row A tiles for 24)."""
    rng = np.random.default_rng(40 + M)
    N, K, gs = 12288, 1024, 64
    w, s, b = quantized(rng, N, K, gs)
    huge_rows = np.array([3, 6000, 12287])
    s = _huge(s, huge_rows, 5)
    x = act(rng, (M, K))
    out = from_dev(mq.quantized_matmul(to_dev(x, "bfloat16"), to_dev(w), to_dev(s, "bfloat16"),
                                       to_dev(b, "bfloat16"), group_size=gs))
    ref = O.quantized_matmul_ref(x, w, s, b, gs)
    assert np.all(np.isfinite(out))
    _check_split(out, ref, huge_rows)


def test_grouped_gather_huge_scales():
    # prefill-width gather (grouped MFMA tiles) with one expert's scales huge
    rng = np.random.default_rng(5)
    E, N, K, P = 6, 256, 512, 1200
    parts = [quantized(rng, N, K, 64) for _ in range(E)]
    w, s, b = (np.stack([p[i] for p in parts]) for i in range(3))
    huge_rows = np.array([0, 100, 255])
    s[2] = _huge(s[2], huge_rows, 1)
    idx = np.sort(rng.integers(0, E, P)).astype(np.int32)
    x = act(rng, (P, 1, K))
    out = from_dev(mq.gather_qmm(to_dev(x, "bfloat16"), to_dev(w), to_dev(s, "bfloat16"),
                                 to_dev(b, "bfloat16"),
                                 rhs_indices=torch.from_numpy(idx).cuda(), sorted_indices=True))
    ref = O.gather_qmm_ref(x, w, s, b, np.arange(P), idx)
    assert np.all(np.isfinite(out))
    hot = idx == 2
    _check_split(out[hot], ref[hot], huge_rows)
    res = O.check_output(out[~hot], ref[~hot])
    assert res["ok"], res


def _rows(*shape, bits, gs, dtype, seed, huge):
    """Random codes of ``shape`` (..., N, K) whose rows ``huge`` hold a scale of
    2^110 (float16: infinity) in their first and last groups."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    *lead, K = shape
    w = torch.randint(-2**31, 2**31, (*lead, K * bits // 32), generator=g, device="cuda",
                      dtype=torch.int64).to(torch.int32).view(torch.uint32)
    s = torch.rand((*lead, K // gs), generator=g, device="cuda") * 0.02
    b = torch.rand((*lead, K // gs), generator=g, device="cuda") * 0.01 - 0.005
    top = 2.0 ** 110 if dtype == "bfloat16" else float("inf")
    s[..., huge, 0] = top
    s[..., huge, -1] = top
    return w, s.to(TORCH_DTYPE[dtype]), b.to(TORCH_DTYPE[dtype])


def _sets_close(out, ref, huge, dtype):
    """Columns ``huge`` and the others within the tolerance, each of its own
    norm (float16's huge ones: not finite on either side)."""
    rest = torch.ones(out.shape[-1], dtype=torch.bool, device="cuda")
    rest[huge] = False
    if dtype == "float16":
        assert not torch.isfinite(out[..., ~rest]).any()
        sets = (rest,)
    else:
        sets = (rest, ~rest)
    for cols in sets:
        o, r = out[..., cols].double(), ref[..., cols].to(out.dtype).double()
        assert torch.isfinite(o).all()
        assert ((o - r).norm() / r.norm()).item() < 1e-3


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("M, N, K, bits, gs", [
    (70, 1031, 320, 8, 64),      # 64-row tiles, scales of one step
    (70, 1031, 320, 4, 32),      # two groups per step
    (70, 1031, 384, 8, 32),      # scales of two steps
    (70, 1031, 640, 4, 128),     # a group over two steps
    (100, 1031, 1024, 8, 32),    # scales of four steps, K split
    (70, 40007, 384, 4, 32),     # 128-row tiles
    (200, 17413, 320, 8, 64),    # one step
    (257, 30001, 192, 4, 64),    # 192-row tiles, one step
    (450, 17413, 384, 8, 64),    # two steps
    (600, 17413, 320, 4, 32),    # 256-row tiles, one step
    (600, 17413, 512, 8, 128),   # four steps
])
def test_wide_tile_huge_scales(M, N, K, bits, gs, dtype):
    """The streaming tile's second route: its own addresses of codes and scales
    for each width, group size, load of scales and tile height."""
    huge = [3, 37, 69, 255, 256 + 17, N - 40, N - 1]
    w, s, b = _rows(N, K, bits=bits, gs=gs, dtype=dtype, seed=M + K + bits, huge=huge)
    x = to_dev(act(np.random.default_rng(K), (M, K), dtype), dtype)
    out = mq.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    ref = x.double() @ mq.dequantize(w, s, b, group_size=gs, bits=bits).double().T
    _sets_close(out, ref, huge, dtype)


@pytest.mark.parametrize("bits, gs, K", [(8, 32, 384), (8, 64, 320), (8, 128, 512), (4, 64, 320)])
def test_thin_gather_huge_scales(bits, gs, K):
    """The thin kernels (64 rows per expert): one bank's huge rows among
    ordinary ones, and the fused gate, up and SwiGLU launch, where a block of
    the gate and one of the up bank are recomputed together, against its two
    gathers and the SwiGLU pass bit for bit."""
    E, T, top, N = 16, 128, 8, 264
    rng = np.random.default_rng(gs + K)
    hot = {"gate": [1, 40, 130], "up": [33, 100, 263]}
    banks = {}
    for i, (name, huge) in enumerate(hot.items()):
        banks[name] = _rows(E, N, K, bits=bits, gs=gs, dtype="bfloat16", seed=K + i, huge=huge)
    idx = np.stack([rng.choice(E, top, replace=False) for _ in range(T)]).astype(np.int32)
    rhs = torch.from_numpy(idx).cuda()
    x = to_dev(act(rng, (T, 1, 1, K)), "bfloat16")
    kw = dict(group_size=gs, bits=bits)
    tables = ops.gather_tables(rhs, E)
    assert tables is not None
    parts = {}
    for name, bank in banks.items():
        parts[name] = out = ops.gather_qmm(x, *bank, rhs_indices=rhs, tables=tables, **kw)
        deq = mq.dequantize(*bank, **kw)
        ref = torch.empty(out.shape, dtype=torch.float64, device="cuda")
        for e in range(E):
            t, j = (rhs == e).nonzero(as_tuple=True)
            ref[t, j] = x[t, 0].double() @ deq[e].double().T
        _sets_close(out, ref, hot[name], "bfloat16")
    got = ops.gather_swiglu(x, banks["gate"], banks["up"], rhs, tables, **kw)
    want = ops.swiglu(parts["gate"], parts["up"])
    np.testing.assert_array_equal(bits16(got), bits16(want))
