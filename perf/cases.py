"""Performance cases: the work that a program using this package has it do.

Every case is one call, or one block of calls, of a language model's decode,
verify or prefill pass over MLX-format quantized weights, through the
package's public modules and operators:

* ``linear``: one ``nn.QuantizedLinear`` (an attention projection, the head);
* ``mlp``: the dense MLP block, gate and up projections, ``ops.swiglu``, down
  projection;
* ``moe``: ``nn.SwitchGLU`` with router scores (decode and prefill widths);
* ``block``: ``ops.moe_block``, the decode MoE block with its routing, shared
  expert's gate and merge;
* ``rebit``: ``rebit.requantize`` of a layer, dequantize and quantize.

Weights are normal matrices of standard deviation 0.02 quantized per group
between their group's minimum and maximum, as a checkpoint's are;
activations are standard normal; routing follows a Zipf law over the experts
or is uniform.
"""

from __future__ import annotations

import math

import torch

import mlxturbo_amd as mq
from mlxturbo_amd import nn, ops, rebit

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # The smallest call: one attention projection of a 4096-wide model for
        # one decoded token.
        {"name": "proj_m1", "kind": "linear", "M": 1, "K": 4096, "N": 4096,
         "bits": 4, "gs": 64, "dtype": "bf16"},
        # One decoded token through a 27B-class model's MLP (5120 <-> 17408).
        {"name": "mlp_m1", "kind": "mlp", "M": 1, "K": 5120, "N": 17408,
         "bits": 4, "gs": 64, "dtype": "bf16"},
        # A speculative-verify step of 8 drafted tokens through the same MLP.
        {"name": "mlp_m8", "kind": "mlp", "M": 8, "K": 5120, "N": 17408,
         "bits": 4, "gs": 64, "dtype": "bf16"},
        # A decode batch of 45 sequences, fp16 activations, finer groups.
        {"name": "mlp_m45_fp16_g32", "kind": "mlp", "M": 45, "K": 5120, "N": 17408,
         "bits": 4, "gs": 32, "dtype": "fp16"},
        # A short prompt's prefill, an odd number of tokens.
        {"name": "mlp_m509", "kind": "mlp", "M": 509, "K": 5120, "N": 17408,
         "bits": 4, "gs": 64, "dtype": "bf16"},
        # The largest: a whole prefill chunk of 8192 tokens.
        {"name": "mlp_m8192", "kind": "mlp", "M": 8192, "K": 5120, "N": 17408,
         "bits": 4, "gs": 64, "dtype": "bf16"},
        # The 8-bit language-model head on the two last rows of a verify step.
        {"name": "lm_head_b8_m2", "kind": "linear", "M": 2, "K": 5120, "N": 248320,
         "bits": 8, "gs": 64, "dtype": "bf16"},
        # One decoded token through a 512-expert MoE block, routing included.
        {"name": "moe_block_t1", "kind": "block", "T": 1, "k": 8, "E": 512, "H": 2048, "I": 512,
         "bits": 4, "gs": 64, "dtype": "bf16", "zipf": True},
        # Eight verified tokens through the MoE layer with the fused decode route.
        {"name": "moe_t8", "kind": "moe", "T": 8, "k": 8, "E": 512, "H": 2048, "I": 512,
         "bits": 4, "gs": 64, "dtype": "bf16", "zipf": True, "fused": True},
        # A ragged prompt's prefill over 8-bit experts, evenly spread routing.
        {"name": "moe_t301_b8", "kind": "moe", "T": 301, "k": 8, "E": 128, "H": 2048, "I": 768,
         "bits": 8, "gs": 64, "dtype": "bf16", "zipf": False, "fused": False},
        # A prefill chunk of 2048 tokens over 512 experts, skewed routing.
        {"name": "moe_t2048", "kind": "moe", "T": 2048, "k": 8, "E": 512, "H": 2048, "I": 512,
         "bits": 4, "gs": 64, "dtype": "bf16", "zipf": True, "fused": False},
        # Loading: an 8-bit layer requantized to 4 bits in groups of 32.
        {"name": "rebit_8to4", "kind": "rebit", "K": 5120, "N": 17408, "bits": 8, "gs": 64,
         "to_bits": 4, "to_gs": 32, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes log-uniform over the ranges that the listed ones
    stand for, formats as checkpoints come (4 bits and groups of 64 most)."""
    kind = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "mlp", "moe", "moe", "moe",
                       "block", "rebit"])
    c = {"kind": kind, "bits": rng.choice([4, 4, 4, 8]), "gs": rng.choice([32, 64, 64, 128]),
         "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if kind == "linear":
        c["K"] = 128 * _log(rng, 1024 / 128, 21504 / 128)
        c["N"] = _log(rng, 512, 36000)                    # any row count
        c["M"] = _log(rng, 1, 8192)
    elif kind == "mlp":
        c["K"] = 128 * _log(rng, 1024 / 128, 6144 / 128)
        c["N"] = 128 * _log(rng, 2048 / 128, 21504 / 128)
        c["M"] = _log(rng, 1, 8192 * min(1.0, 5120 * 17408 / (c["K"] * c["N"])))
    elif kind == "moe":
        c["E"] = rng.choice([64, 128, 256, 512])
        c["k"] = rng.choice([4, 6, 8])
        c["H"] = 128 * _log(rng, 1024 / 128, 3072 / 128)
        c["I"] = 128 * _log(rng, 256 / 128, 1024 / 128)
        c["T"] = _log(rng, 1, 4096)
        c["zipf"], c["fused"] = rng.random() < 0.5, rng.random() < 0.5
    elif kind == "block":
        c["E"], c["k"], c["T"] = rng.choice([64, 128, 256, 512]), rng.choice([4, 6, 8]), \
            rng.randint(1, 8)
        c["H"] = 128 * _log(rng, 1024 / 128, 3072 / 128)
        c["I"] = 128 * _log(rng, 256 / 128, 1024 / 128)
        c["zipf"] = rng.random() < 0.5
    else:
        c["K"] = 128 * _log(rng, 1024 / 128, 21504 / 128)
        c["N"] = _log(rng, 512, 17408)
        c["to_bits"] = rng.choice([4, 4, 8, 3, 6])
        c["to_gs"] = rng.choice([32, 64, 128])
    return c


# ---- inputs -----------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _weights(g, lead, K, bits, gs, dtype):
    """Quantized N(0, 0.02) weights ``(w, scales, biases)`` of shape
    ``(*lead, K)``: per group the affine grid between minimum and maximum,
    codes packed low bits first (little-endian words)."""
    rows = math.prod(lead)
    w = torch.empty((rows, K * bits // 32), dtype=torch.int32, device="cuda")
    s = torch.empty((rows, K // gs), dtype=dtype, device="cuda")
    b = torch.empty_like(s)
    step = max(1, (1 << 28) // K)
    top = float((1 << bits) - 1)
    for r0 in range(0, rows, step):
        r1 = min(rows, r0 + step)
        v = torch.randn((r1 - r0, K // gs, gs), generator=g, device="cuda").mul_(0.02)
        lo, hi = v.amin(-1, keepdim=True), v.amax(-1, keepdim=True)
        sc = ((hi - lo) / top).to(dtype)
        lo = lo.to(dtype)
        q = v.sub_(lo.float()).div_(sc.float()).round_().clamp_(0, top).to(torch.uint8)
        q = q.reshape(r1 - r0, K)
        if bits == 4:
            q = q[:, 0::2] | (q[:, 1::2] << 4)
        w[r0:r1] = q.contiguous().view(torch.int32)
        s[r0:r1], b[r0:r1] = sc.squeeze(-1), lo.squeeze(-1)
    return (w.view(torch.uint32).reshape(*lead, -1), s.reshape(*lead, -1), b.reshape(*lead, -1))


def _deq64(w, s, b, bits, gs):
    """The weights that (w, s, b) stand for, ``T(float(s) * q + float(b))``,
    in float64."""
    u8 = w.view(torch.int32).contiguous().view(torch.uint8)
    if bits == 4:
        u8 = torch.stack([u8 & 15, u8 >> 4], dim=-1).reshape(*u8.shape[:-1], -1)
    q = u8.reshape(*s.shape, gs).float()
    v = (q.double() * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).float().to(s.dtype)
    return v.reshape(*s.shape[:-1], -1).double()


def _x(g, *shape, dtype):
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _routing(g, c):
    """Router logits whose top-k follow the case's law over the experts
    (Gumbel perturbation: draws without replacement)."""
    E = c["E"]
    if c["zipf"]:
        p = torch.arange(1, E + 1, device="cuda", dtype=torch.float32).pow_(-1.1).log_()
        p = p[torch.randperm(E, generator=g, device="cuda")]
    else:
        p = torch.zeros(E, device="cuda")
    u = torch.rand((c["T"], E), generator=g, device="cuda").clamp_(1e-7, 1 - 1e-7)
    return p - torch.log(-torch.log(u))


def _inputs(c, seed):
    """The case's tensors, made from the seed alone."""
    g, dt = _gen(seed), _DTYPES[c["dtype"]]
    bits, gs, kind = c["bits"], c["gs"], c["kind"]
    if kind == "linear":
        return {"w": _weights(g, (c["N"],), c["K"], bits, gs, dt),
                "x": _x(g, c["M"], c["K"], dtype=dt)}
    if kind == "mlp":
        return {"gate": _weights(g, (c["N"],), c["K"], bits, gs, dt),
                "up": _weights(g, (c["N"],), c["K"], bits, gs, dt),
                "down": _weights(g, (c["K"],), c["N"], bits, gs, dt),
                "x": _x(g, c["M"], c["K"], dtype=dt)}
    if kind == "rebit":
        return {"w": _weights(g, (c["N"],), c["K"], bits, gs, dt)}
    E, H, I = c["E"], c["H"], c["I"]
    d = {"gate": _weights(g, (E, I), H, bits, gs, dt), "up": _weights(g, (E, I), H, bits, gs, dt),
         "down": _weights(g, (E, H), I, bits, gs, dt), "x": _x(g, c["T"], H, dtype=dt),
         "logits": _routing(g, c)}
    if kind == "block":
        d["sgw"] = (_x(g, H, dtype=torch.float32) / math.sqrt(H)).to(dt)
        d["shared"] = _x(g, c["T"], H, dtype=dt)
    else:
        top, idx = d["logits"].topk(c["k"], dim=-1)
        d["idx"], d["scores"] = idx.int(), top.softmax(-1)
    return d


def prepare(case, seed):
    """What a program holds before the call: its layers, loaded once, and the
    step's activations and routing."""
    c, d = case, _inputs(case, seed)
    q = {"group_size": c["gs"], "bits": c["bits"]}
    state = {"case": c, "x": d.get("x")}
    if c["kind"] in ("linear", "rebit"):
        state["layer"] = nn.QuantizedLinear(*d["w"], **q)
    elif c["kind"] == "mlp":
        for k in ("gate", "up", "down"):
            state[k] = nn.QuantizedLinear(*d[k], **q)
    elif c["kind"] == "moe":
        state["layer"] = nn.SwitchGLU(*[nn.QuantizedSwitchLinear(*d[k], **q)
                                        for k in ("gate", "up", "down")],
                                      fuse_gate_up=c["fused"])
        state["idx"], state["scores"] = d["idx"], d["scores"]
    else:
        state.update(d)
    return state


def run(state):
    """One pass through the package's modules and operators."""
    c, kind, x = state["case"], state["case"]["kind"], state["x"]
    if kind == "linear":
        return state["layer"](x)
    if kind == "mlp":
        h = ops.swiglu(state["gate"](x), state["up"](x))
        return {"h": h, "y": state["down"](h)}
    if kind == "moe":
        return state["layer"](x, state["idx"], state["scores"])
    if kind == "block":
        return ops.moe_block(x, state["logits"], c["k"], state["gate"], state["up"],
                             state["down"], sgw=state["sgw"], shared=state["shared"],
                             group_size=c["gs"], bits=c["bits"])
    new = rebit.requantize(state["layer"], c["to_bits"], c["to_gs"])
    return {"w": new.weight.view(torch.int32), "scales": new.scales, "biases": new.biases}


# ---- what a pass needs ------------------------------------------------------

def _bank(n, c):
    """Bytes of n quantized weights with their scales and biases."""
    return n * c["bits"] / 8 + 4 * n / c["gs"]


def _experts(c):
    """Distinct experts that T tokens of k are expected to reach."""
    E, k, T = c["E"], c["k"], c["T"]
    if c["zipf"]:
        z = [r ** -1.1 for r in range(1, E + 1)]
        t = sum(z)
        p = [min(1.0, k * v / t) for v in z]
    else:
        p = [k / E] * E
    return max(min(k, E), sum(1 - (1 - v) ** T for v in p))


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": _bank(N * K, c) + 2 * M * (K + N), "flops": 2 * M * N * K}
    if kind == "mlp":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": _bank(3 * N * K, c) + 2 * M * (2 * K + N), "flops": 6 * M * N * K}
    if kind == "rebit":
        n = c["N"] * c["K"]
        return {"bytes": _bank(n, c) + n * c["to_bits"] / 8 + 4 * n / c["to_gs"], "flops": 4 * n}
    T, k, H, I = c["T"], c["k"], c["H"], c["I"]
    b = _bank(3 * _experts(c) * H * I, c) + 4 * T * H + 8 * T * k
    if kind == "block":
        b += 4 * T * c["E"] + 2 * T * H + 2 * H
    return {"bytes": b, "flops": 6 * T * k * H * I}


def tolerance(case):
    """About four times what outputs were measured off `exact`: rel 1.7e-3
    (linear) and 3.9e-3 (an MLP's or a MoE layer's, whose intermediates are
    rounded too, so that flips of h travel into the next product) in bf16,
    2.1e-4 and 4.8e-4 in fp16; max is two roundings of the type for a linear
    layer.  Requantized codes and their scales are defined bit for bit."""
    if case["kind"] == "rebit":
        return "exact"
    fine = case["dtype"] == "fp16"
    if case["kind"] == "linear":
        return {"rel": 1e-3, "max": 2e-3} if fine else {"rel": 7e-3, "max": 1.6e-2}
    return {"rel": 2e-3, "max": 1e-2} if fine else {"rel": 1.4e-2, "max": 8e-2}


# ---- the same in 64 bits ----------------------------------------------------

def _silu_mul(g, u):
    return g / (1 + torch.exp(-g)) * u


def exact(case, seed):
    """`run` on the same inputs in float64 (the weights being what their codes
    stand for in the checkpoint's type)."""
    c, kind = case, case["kind"]
    if kind == "rebit":
        return None                          # codes, compared bit for bit
    d, bits, gs = _inputs(c, seed), c["bits"], c["gs"]

    def mm(x, bank):
        """x @ deq(bank)^T, in slices of rows (the head's weights are 10 GB)."""
        step = max(1, (1 << 28) // c["K"])
        return torch.cat([x @ _deq64(*[t[r:r + step] for t in bank], bits, gs).T
                          for r in range(0, bank[0].shape[0], step)], dim=-1)

    x = d["x"].double()
    if kind == "linear":
        return mm(x, d["w"])
    if kind == "mlp":
        h = _silu_mul(mm(x, d["gate"]), mm(x, d["up"]))
        return {"h": h, "y": mm(h, d["down"])}
    if kind == "block":
        top, idx = d["logits"].double().topk(c["k"], dim=-1)
        wts = top.softmax(-1)
    else:
        idx, wts = d["idx"].long(), d["scores"].double()
    y = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        t, j = (idx == e).nonzero(as_tuple=True)
        wg, wu, wd = (_deq64(*[v[e] for v in d[n]], bits, gs) for n in ("gate", "up", "down"))
        h = _silu_mul(x[t] @ wg.T, x[t] @ wu.T)
        y.index_add_(0, t, (h @ wd.T) * wts[t, j].unsqueeze(-1))
    if kind == "block":
        gate = torch.sigmoid(x @ d["sgw"].double())
        y += gate.unsqueeze(-1) * d["shared"].double()
    return y
