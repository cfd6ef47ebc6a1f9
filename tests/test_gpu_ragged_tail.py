"""Weights that end where their memory ends, at K that is not whole steps of
the streaming tile: the last step of the last rows reads nothing past them.

The arrays are whole 2 MiB pages and large enough to be segments of their own
in torch's allocator, so there may be nothing mapped behind them.  Results
against float64 products of the dequantized weights (the tolerance of
oracle.check_output's relL2)."""

import pytest
import torch

import mlxturbo_amd as mq

pytestmark = pytest.mark.gpu


def _quantized(rows, K, bits, gs, dtype):
    g = torch.Generator(device="cuda").manual_seed(rows + K + bits)
    w = (torch.randn((rows, K), generator=g, device="cuda") * 0.02).to(dtype)
    return mq.quantize(w, group_size=gs, bits=bits)


def _rel(out, ref):
    ref = ref.to(out.dtype).double()
    return ((out.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("bits, gs, K, N", [
    (4, 64, 448, 65536),      # 7 groups, steps of 4; 14 MiB of codes
    (4, 32, 1152, 32768),     # 36 groups, steps of 8
    (8, 64, 320, 65536),      # 5 groups, steps of 4
    (4, 128, 640, 65536),     # 5 groups, steps of 4 (512 codes)
])
@pytest.mark.parametrize("M", [2, 8, 16])
def test_skinny_ragged_tail(bits, gs, K, N, M):
    w, s, b = _quantized(N, K, bits, gs, torch.bfloat16)
    assert w.numel() * 4 % (2 << 20) == 0
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
    out = mq.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    ref = x.double() @ mq.dequantize(w, s, b, group_size=gs, bits=bits).double().T
    assert _rel(out, ref) < 1e-3
    assert _rel(out[:, -64:], ref[:, -64:]) < 1e-3
    # scales at an odd address: no scale copy, the tail's scales one by one
    # (the step loads of every other step, and of all of them, must agree)
    shifted = [torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda") for t in (s, b)]
    for d, t in zip(shifted, (s, b)):
        d[1:].copy_(t.reshape(-1))
    got = torch.empty_like(out)
    lib = mq._lib.lib()
    rc = lib.mq_quantized_matmul(x.data_ptr(), w.data_ptr(), shifted[0].data_ptr() + 2,
                                 shifted[1].data_ptr() + 2, got.data_ptr(), M, N, K, gs, bits, 0,
                                 1, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert _rel(got, ref) < 1e-3


@pytest.mark.parametrize("bits, gs, K", [(4, 64, 448), (8, 64, 448), (4, 32, 1152)])
@pytest.mark.parametrize("T", [1, 8, 40])
def test_gather_ragged_tail(bits, gs, K, T):
    E, N, k = 64, 1024, 4
    w, s, b = (t.reshape(E, N, -1) for t in _quantized(E * N, K, bits, gs, torch.bfloat16))
    assert w.numel() * 4 % (2 << 20) == 0
    x = torch.randn((T, 1, 1, K), device="cuda").to(torch.bfloat16)
    idx = torch.randint(0, E, (T, k), device="cuda", dtype=torch.int32)
    idx[:, 0] = E - 1                          # the last expert, at the arrays' end
    out = mq.gather_qmm(x, w, s, b, rhs_indices=idx, group_size=gs, bits=bits)
    deq = mq.dequantize(w, s, b, group_size=gs, bits=bits)
    for t in range(T):
        for j in range(k):
            ref = x[t, 0].double() @ deq[int(idx[t, j])].double().T
            assert _rel(out[t, j], ref) < 1e-3
