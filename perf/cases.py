"""Workloads of the quantised mixture-of-experts library, as its users call it: whole FFN layers from one token to a
full prefill batch in each weight format, the expert weight gradients of a training step, and the MX round trip of a
weight tensor.

A case is a dict of plain values.  `listed()` names the fixed ones, `draw(rng)` gives more of the same ranges,
`prepare(case, seed)` makes what a program holds before the call (weights in the layouts `matmul` prefers, precision
configs, activations, logits), `run(state)` is one pass through the public entry points, launched eagerly, and `work(case)` the
bytes and operations that pass cannot do without.

Kinds:

  mxfp4        bf16 activations, MXFP4 weights, bf16 biases, swiglu: router, both expert GEMMs and the top-k combine
               (`moe_mlp`); decode and prefill differ only in the number of tokens
  mxfp8        the same layer with activations quantised to MXFP8 in front of each GEMM (prefill)
  fp8          e4m3 weights with a scale per output channel, activations quantised to e4m3 with a scale per token
  bf16         bf16 weights and biases
  weight_grad  dW1 and dW2 of a bf16 layer from the expert-sorted activations and output gradients (ragged K)
  mx           a weight tensor quantised along K to an MX format and expanded again
"""
from __future__ import annotations

import math
import random

import torch

from triton_kernels.legacy import matmul_ogs, routing
from triton_kernels.matmul import Epilogue, FnName, FnSpecs, FusedActivation, PrecisionConfig, matmul
from triton_kernels.moe_decode import moe_mlp
from triton_kernels.numerics_details.mxfp import downcast_to_mxfp, quantize_mxfp8_fn, upcast_from_mxfp
from triton_kernels.numerics_details.rowwise_fp8 import quantize_fp8_rowwise
from triton_kernels.swiglu import swiglu_fn
from triton_kernels.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
from triton_kernels.tensor_details.layout import (make_default_matmul_fp8_w_layout, make_default_matmul_mxfp4_w_layout,
                                                  make_default_matmul_mxfp4_w_scale_layout)

DEVICE = "cuda:0"
MX_TYPES = {"e2m1": torch.uint8, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
FLOATS = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _layer(name, kind, tokens, d_model, d_ff, experts, top_k, skew=0.0):
    return dict(name=name, kind=kind, tokens=tokens, d_model=d_model, d_ff=d_ff, experts=experts, top_k=top_k, skew=skew)


def listed():
    return [
        # one token of one sequence: the latency of a layer in an interactive decode loop
        _layer("mxfp4_t1", "mxfp4", 1, 2880, 2880, 128, 4, skew=1.5),
        # a small and a fuller decode batch, experts loaded unevenly
        _layer("mxfp4_t16", "mxfp4", 16, 2880, 2880, 128, 4, skew=1.5),
        _layer("mxfp4_t61", "mxfp4", 61, 2880, 2880, 128, 4, skew=1.5),
        # a large decode batch or a chunk of a prompt: a dozen rows per expert
        _layer("mxfp4_t300", "mxfp4", 300, 2880, 2880, 128, 4),
        # a full prefill batch
        _layer("mxfp4_t4096", "mxfp4", 4096, 2880, 2880, 128, 4),
        _layer("mxfp8_t4096", "mxfp8", 4096, 2880, 2880, 128, 4),
        # few large experts in fp8: a decode batch and a full prefill batch
        _layer("fp8_t32", "fp8", 32, 4096, 14336, 8, 2),
        _layer("fp8_t8192", "fp8", 8192, 4096, 14336, 8, 2),
        # a small and a larger layer in bf16, as in fine-tuning or on unquantised checkpoints
        _layer("bf16_t128", "bf16", 128, 512, 1024, 8, 2),
        _layer("bf16_t2048", "bf16", 2048, 2048, 2048, 16, 2),
        # backward of a training step: weight gradients of 128 experts
        dict(name="weight_grad", kind="weight_grad", rows=16384, d_model=2880, d_ff=2880, experts=128),
        # quantising a stack of expert weights at load time, and reading it back
        dict(name="mx_round_trip", kind="mx", batch=32, k=2880, n=5760, to="e2m1", dtype="bf16"),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dim(rng: random.Random, lo: int, hi: int, step: int) -> int:
    return max(lo, _log_int(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(["mxfp4", "mxfp4", "mxfp4", "mxfp8", "fp8", "fp8", "bf16", "weight_grad", "mx"])
    if kind in ("mxfp4", "mxfp8"):
        # half of them at the listed layer's sizes, the others from small to that
        if rng.random() < 0.5:
            d, f, e, k = 2880, 2880, 128, 4
        else:
            d, f = _dim(rng, 512, 2880, 32), _dim(rng, 512, 2880, 32)
            e, k = rng.choice([16, 32, 64, 96, 128]), rng.choice([2, 4, 8])
        tokens = _log_int(rng, 1 if kind == "mxfp4" else 128, 16384 // k)
        return _layer_drawn(kind, tokens, d, f, e, k, rng.choice([0.0, 1.5]))
    if kind == "fp8":
        d, f = _dim(rng, 1024, 4096, 128), _dim(rng, 1024, 14336, 128)
        return _layer_drawn(kind, _log_int(rng, 16, 8192), d, f, rng.choice([8, 16]), 2, 0.0)
    if kind == "bf16":
        d, f = _dim(rng, 256, 2048, 32), _dim(rng, 256, 2048, 32)
        return _layer_drawn(kind, _log_int(rng, 16, 2048), d, f, rng.choice([8, 16, 32]), rng.choice([1, 2, 4]), 0.0)
    if kind == "weight_grad":
        return dict(kind=kind, rows=_log_int(rng, 256, 16384), d_model=_dim(rng, 256, 2880, 32), d_ff=_dim(rng, 256, 2880, 32),
                    experts=rng.choice([8, 16, 32, 64, 128]))
    n = _log_int(rng, 64, 5760)
    return dict(kind=kind, batch=_log_int(rng, 1, 32), k=_dim(rng, 64, 2880, 32), n=n if rng.random() < 0.25 else max(64, n // 16 * 16),
                to=rng.choice(sorted(MX_TYPES)), dtype=rng.choice(sorted(FLOATS)))


def _layer_drawn(kind, tokens, d_model, d_ff, experts, top_k, skew):
    c = _layer("", kind, tokens, d_model, d_ff, experts, top_k, skew)
    del c["name"]
    return c


def _rand(g, shape, scale, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=dtype).mul_(scale)


def _swiglu():
    return FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))


def _mxfp4_weights(g, e, k, n):
    """Expert weights `[e, k, n]` as a model loader leaves them: MXFP4 in the layouts `matmul` prefers."""
    q, s = downcast_to_mxfp(_rand(g, (e, k, n), 0.02), torch.uint8, axis=1)
    return (convert_layout(wrap_torch_tensor(q, dtype=FP4), make_default_matmul_mxfp4_w_layout(mx_axis=1)),
            convert_layout(wrap_torch_tensor(s), make_default_matmul_mxfp4_w_scale_layout(mx_axis=1)))


def _fp8_weights(g, e, k, n):
    """e4m3 expert weights in the layout `matmul` prefers, with their scale per output channel `[e, n]`."""
    q = torch.empty((e, n, k), dtype=torch.float8_e4m3fn, device=DEVICE)
    s = torch.empty((e, n), dtype=torch.float32, device=DEVICE)
    for i in range(e):
        w = _rand(g, (n, k), 0.02, torch.float32)
        s[i] = w.abs().amax(dim=1) / 448.0
        q[i] = (w / s[i][:, None]).clamp_(-448, 448).to(torch.float8_e4m3fn)
    return convert_layout(wrap_torch_tensor(q.transpose(1, 2)), make_default_matmul_fp8_w_layout()), s


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    st = dict(case)
    if kind == "mx":
        w = _rand(g, (case["batch"], case["k"], case["n"]), 0.02, FLOATS[case["dtype"]])
        # one weight in a thousand is an outlier of magnitude 4 to 16
        out = torch.empty(w.shape, dtype=w.dtype, device=DEVICE).uniform_(-1, 1, generator=g)
        st["w"] = torch.where(torch.rand(w.shape, generator=g, device=DEVICE) < 1e-3, out.sign() * (4 + 12 * out.abs()), w)
        return st
    d, f, e = case["d_model"], case["d_ff"], case["experts"]
    if kind == "weight_grad":
        r = case["rows"]
        cuts = torch.sort(torch.randint(0, r + 1, (e - 1, ), generator=g, device=DEVICE)).values
        ends = torch.tensor([0, r], device=DEVICE)
        sizes = torch.diff(torch.cat([ends[:1], cuts, ends[1:]])).to(torch.int32)
        st.update(md=make_ragged_tensor_metadata(sizes, r), x=_rand(g, (r, d), 1.0), dh=_rand(g, (r, 2 * f), 1.0), h=_rand(g, (r, f), 1.0),
                  dy=_rand(g, (r, d), 1.0))
        return st
    t = case["tokens"]
    st["x"] = _rand(g, (t, d), 1.0)
    logits = torch.randn((t, e), generator=g, device=DEVICE)
    st["logits"] = logits + case["skew"] * torch.randn((e, ), generator=g, device=DEVICE)
    st["act"] = _swiglu()
    if kind in ("mxfp4", "mxfp8", "bf16"):
        st["b1"], st["b2"] = _rand(g, (e, 2 * f), 0.01), _rand(g, (e, d), 0.01)
    if kind in ("mxfp4", "mxfp8"):
        st["w1"], st["s1"] = _mxfp4_weights(g, e, d, 2 * f)
        st["w2"], st["s2"] = _mxfp4_weights(g, e, f, d)
        st["pc1"], st["pc2"] = PrecisionConfig(b_mx_scale=st["s1"]), PrecisionConfig(b_mx_scale=st["s2"])
    if kind == "mxfp8":
        st["h_scale"] = torch.empty((t * case["top_k"], f // 32), dtype=torch.uint8, device=DEVICE)
        st["epilogue"] = Epilogue(FnSpecs(FnName.QUANTIZE_MXFP8.name, quantize_mxfp8_fn, (), ()), tuple(), tuple(), effective_itemsize=1.0)
    elif kind == "fp8":
        st["w1"], st["s1"] = _fp8_weights(g, e, d, 2 * f)
        st["w2"], st["s2"] = _fp8_weights(g, e, f, d)
    elif kind == "bf16":
        # [e, k, n] with unit stride along k, the form `matmul` uses in place
        st["w1"], st["w2"] = _rand(g, (e, 2 * f, d), 0.02).transpose(1, 2), _rand(g, (e, d, f), 0.02).transpose(1, 2)
        st["pc1"], st["pc2"] = PrecisionConfig(), PrecisionConfig()
    return st


def run(st):
    kind = st["kind"]
    if kind == "mx":
        q, s = downcast_to_mxfp(st["w"], MX_TYPES[st["to"]], axis=1)
        return {"values": q, "scales": s, "back": upcast_from_mxfp(q, s, st["w"].dtype, axis=1)}
    if kind == "weight_grad":
        md = st["md"]
        return {"dw1": matmul(st["x"].t(), st["dh"], None, a_ragged_metadata=md, b_ragged_metadata=md),
                "dw2": matmul(st["h"].t(), st["dy"], None, a_ragged_metadata=md, b_ragged_metadata=md)}
    x, logits, k, act = st["x"], st["logits"], st["top_k"], st["act"]
    if kind == "mxfp4":
        return moe_mlp(x, logits, k, st["w1"], st["b1"], st["w2"], st["b2"], st["pc1"], st["pc2"], act)
    rdata, gather, scatter = routing(logits, k)
    routed = {"hist": rdata.expt_hist, "expert": rdata.expt_indx}
    if kind == "mxfp8":
        xq, xs = downcast_to_mxfp(x, torch.float8_e4m3fn, axis=-1)
        pc1 = PrecisionConfig(a_mx_scale=xs, b_mx_scale=st["s1"], c_mx_scale=st["h_scale"], out_dtype=torch.float8_e4m3fn)
        h = matmul(xq, st["w1"], st["b1"], rdata.expt_data, gather_indx=rdata.token_indx, precision_config=pc1, fused_activation=act,
                   epilogue=st["epilogue"])
        pc2 = PrecisionConfig(a_mx_scale=st["h_scale"], b_mx_scale=st["s2"], out_dtype=torch.bfloat16)
        return {"out": matmul_ogs(h, st["w2"], st["b2"], rdata, scatter_indx=scatter, precision_config=pc2, gammas=rdata.gate_scal), **routed}
    if kind == "fp8":
        xq, sx = quantize_fp8_rowwise(x)
        pc1 = PrecisionConfig(a_mx_tensor_scale=sx, b_mx_tensor_scale=st["s1"], out_dtype=torch.bfloat16)
        h = matmul_ogs(xq, st["w1"], None, rdata, gather_indx=gather, precision_config=pc1, fused_activation=act)
        hq, sh = quantize_fp8_rowwise(h)
        pc2 = PrecisionConfig(a_mx_tensor_scale=sh, b_mx_tensor_scale=st["s2"], out_dtype=torch.bfloat16)
        return {"out": matmul_ogs(hq, st["w2"], None, rdata, scatter_indx=scatter, precision_config=pc2, gammas=rdata.gate_scal), **routed}
    h = matmul_ogs(x, st["w1"], st["b1"], rdata, gather_indx=gather, precision_config=st["pc1"], fused_activation=act)
    return {"out": matmul_ogs(h, st["w2"], st["b2"], rdata, scatter_indx=scatter, precision_config=st["pc2"], gammas=rdata.gate_scal), **routed}


def _active_experts(case):
    """Experts that a batch of these sizes typically touches (one fixed sample of the logits' distribution)."""
    g = torch.Generator().manual_seed(0)
    t, e = case["tokens"], case["experts"]
    logits = torch.randn((t, e), generator=g) + case["skew"] * torch.randn((e, ), generator=g)
    return int(torch.unique(torch.topk(logits, case["top_k"], dim=1).indices).numel())


def work(case):
    if case["kind"] == "mx":
        n = case["batch"] * case["k"] * case["n"]
        packed = (0.5 if case["to"] == "e2m1" else 1.0) + 1 / 32
        return {"bytes": 2 * n * (2 + packed), "flops": 0}
    d, f = case["d_model"], case["d_ff"]
    if case["kind"] == "weight_grad":
        r, e = case["rows"], case["experts"]
        return {"bytes": 2.0 * (r * (2 * d + 3 * f) + e * 3 * d * f), "flops": 2.0 * r * 3 * d * f}
    t, e, k = case["tokens"], case["experts"], case["top_k"]
    per_weight = {"mxfp4": 17 / 32, "mxfp8": 17 / 32, "fp8": 1.0, "bf16": 2.0}[case["kind"]]
    per_expert = 3 * d * f * per_weight + (0 if case["kind"] == "fp8" else 2 * (2 * f + d))
    # x and logits in, out written once; the hidden activations need not leave the chip
    return {"bytes": _active_experts(case) * per_expert + 2 * 2.0 * t * d + 4.0 * t * e, "flops": 2.0 * t * k * 3 * d * f}


def tolerance(case):
    if case["kind"] == "mx":
        return "exact"
    # bf16 results of fp32 sums; where the hidden activations are quantised again between the GEMMs, a code next to a
    # rounding threshold may fall on either side of it
    return {"rel": 1e-2}
