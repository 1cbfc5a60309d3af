"""The native host path against the general Python path, bit for bit, over the forms of a call that it serves and at its edges: both fill
a descriptor for the same kernels, so values, shapes, strides and types have to agree; and calls it has to leave to the general path."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _same(a, b):
    if isinstance(a, torch.Tensor):
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and a._version == b._version == 0
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
    elif isinstance(a, (list, tuple)):
        assert type(a) is type(b) and len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
    else:
        assert a == b and type(a) is type(b)


def _both(monkeypatch, f, served=True):
    """f() through the native path and through the general one."""
    from triton_amd import _native as nt
    real, seen = nt.host(), []

    class Watch:
        def __getattr__(self, name):
            def call(*args):
                r = getattr(real, name)(*args)
                seen.append((name, r is not None))
                return r
            return call

    with monkeypatch.context() as m:
        m.setattr(nt, "host", lambda: Watch())
        fast = f()
    assert seen and all(ok == served for _, ok in seen), seen
    with monkeypatch.context() as m:
        m.setattr(nt, "host", lambda: None)
        slow = f()
    _same(fast, slow)
    return fast


@pytest.mark.parametrize("tokens, e, k", [(1, 1, 1), (1, 128, 4), (3, 20, 2), (300, 128, 8), (33, 700, 32)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_routing(device, monkeypatch, tokens, e, k, dtype):
    from triton_amd.legacy import routing
    logits = torch.randn((tokens, e), generator=torch.Generator().manual_seed(e)).to(dtype).to(device)
    for softmax in (True, False):
        rd, gather, scatter = routing(logits, k, softmax)
        from triton_amd import _native as nt
        with monkeypatch.context() as m:
            m.setattr(nt, "host", lambda: None)
            rd2, gather2, scatter2 = routing(logits, k, softmax)
        md, md2 = rd.expt_data, rd2.expt_data
        _same([gather.src_indx, gather.dst_indx, scatter.src_indx, scatter.dst_indx], [gather2.src_indx, gather2.dst_indx, scatter2.src_indx, scatter2.dst_indx])
        _same([rd.gate_scal, rd.expt_hist, rd.token_indx, rd.expt_indx, rd.gate_vals, rd.all_rows_live, rd.n_expts_tot, rd.n_expts_act],
              [rd2.gate_scal, rd2.expt_hist, rd2.token_indx, rd2.expt_indx, rd2.gate_vals, rd2.all_rows_live, rd2.n_expts_tot, rd2.n_expts_act])
        _same([md.slice_offs, md.block_offs_data, md.block_schedule_data, md.n_slices], [md2.slice_offs, md2.block_offs_data, md2.block_schedule_data, md2.n_slices])
    with pytest.raises(ValueError):
        routing(logits, 3)


def _weights(kind, e, k, n, g, device):
    from triton_amd.numerics_details.mxfp import downcast_to_mxfp
    from triton_amd.tensor import FP4, convert_layout, wrap_torch_tensor
    from triton_amd.tensor_details import layout as L
    w = (torch.randn((e, n, k), generator=g) * 0.1).to(device)
    if kind in ("bf16", "fp16"):
        return w.to(torch.bfloat16 if kind == "bf16" else torch.float16).transpose(1, 2), None
    if kind == "fp8":
        return convert_layout(wrap_torch_tensor(w.to(torch.float8_e4m3fn).transpose(1, 2)), L.make_default_matmul_fp8_w_layout()), None
    q, s = downcast_to_mxfp(w.to(torch.bfloat16).transpose(1, 2), torch.uint8, axis=1)
    return (convert_layout(wrap_torch_tensor(q, dtype=FP4), L.make_default_matmul_mxfp4_w_layout(mx_axis=1)),
            convert_layout(wrap_torch_tensor(s), L.make_default_matmul_mxfp4_w_scale_layout(mx_axis=1)))


@pytest.fixture
def gemm_descriptors(monkeypatch):
    """What the GEMM entry of the library gets from either host path, recorded on the way to it."""
    import ctypes

    from triton_amd import _native as nt
    real, seen = nt.lib(), []

    @ctypes.CFUNCTYPE(ctypes.c_int32, ctypes.POINTER(nt.GemmDesc), ctypes.c_void_p)
    def entry(d, stream):
        seen.append({name: getattr(d.contents, name) for name, _ in nt.GemmDesc._fields_})
        return real.tk_moe_gemm(d, stream)

    class Library:
        tk_moe_gemm = entry

        def __getattr__(self, name):
            return getattr(real, name)

    with monkeypatch.context() as m:
        m.setattr(nt, "_lib", Library())
        m.setattr(nt, "_host", None)  # bound again, to this library
        yield seen
    nt._host = None
    nt.host()


def _same_descriptors(fast, slow):
    """Every number, and every pointer to the caller's operands; buffers made by the call are there or not."""
    made = {"y", "combine_out"}
    for name, value in fast.items():
        assert (bool(value), bool(slow[name])) == (True, True) if name in made and value else value == slow[name], (name, value, slow[name])


# 16 experts, 2 choices.  The row blocks that the rules choose, and with them every kernel that a layer can meet: 16-bit weights the general
# kernel (16) and both tiles of the memory-to-LDS one, e4m3 those two, MXFP4 the decode (16), streaming (32), prefill (64, 128) and wide
# (256) kernels, MXFP8 activations the prefill and the wide kernel (with K of 256 and 320 the form of the prefill kernel for a short K).
SMALL, LARGE = (256, 320), (512, 544)
LAYERS = [
    *[(kind, tokens, dims, bm) for kind in ("bf16", "fp16") for tokens, dims, bm in ((1, SMALL, 16), (40, LARGE, 16), (200, SMALL, 128), (1600, LARGE, 256))],
    *[("fp8", tokens, dims, bm) for tokens, dims, bm in ((1, SMALL, 128), (40, LARGE, 128), (1600, LARGE, 256))],
    *[("mxfp4", tokens, dims, bm) for tokens, dims, bm in ((1, SMALL, 16), (40, LARGE, 16), (140, SMALL, 32), (150, LARGE, 32), (300, LARGE, 64),
                                                           (560, LARGE, 128), (700, LARGE, 256), (1600, SMALL, 128))],
    *[(kind, tokens, dims, bm) for kind in ("mxfp8", "mxfp8_out") for tokens, dims, bm in ((1, SMALL, 256), (40, LARGE, 128), (700, LARGE, 256),
                                                                                         (1600, LARGE, 128), (1600, SMALL, 128))],
]


@pytest.mark.parametrize("kind, tokens, dims, block_m", LAYERS)
def test_layer_gemms(device, monkeypatch, gemm_descriptors, kind, tokens, dims, block_m):
    """Both GEMMs of a layer, with activation and gather, scatter and combine: the same descriptor from both host paths, with the row
    block that is written above, and the same result."""
    import triton_amd.matmul as mm
    from triton_amd.legacy import matmul_ogs, routing
    from triton_amd.numerics_details.mxfp import downcast_to_mxfp, quantize_mxfp8_fn
    from triton_amd.numerics_details.rowwise_fp8 import quantize_fp8_rowwise
    from triton_amd.swiglu import swiglu_fn
    (d, f), e, k = dims, 16, 2
    g = torch.Generator().manual_seed(tokens)
    x = torch.randn((tokens, d), generator=g).to(torch.float16 if kind == "fp16" else torch.bfloat16).to(device)
    rd, gather, scatter = routing(torch.randn((tokens, e), generator=g).to(device), k)
    w1, s1 = _weights(kind, e, d, 2 * f, g, device)
    w2, s2 = _weights(kind, e, f, d, g, device)
    b1, b2 = torch.randn((e, 2 * f), generator=g).to(device), torch.randn((e, d), generator=g).to(torch.bfloat16).to(device)
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
    P, bf16, e4m3 = mm.PrecisionConfig, torch.bfloat16, torch.float8_e4m3fn
    epi = None
    if kind == "fp8":
        x, sx = quantize_fp8_rowwise(x)
        col = torch.rand((e, 2 * f), generator=g).to(device)
        pc1 = P(a_mx_tensor_scale=sx, b_mx_tensor_scale=col, out_dtype=bf16)
    elif kind.startswith("mxfp8"):
        x, sx = downcast_to_mxfp(x, e4m3, axis=-1)
        pc1 = P(a_mx_scale=sx, b_mx_scale=s1, out_dtype=bf16)
        if kind == "mxfp8_out":
            pc1.c_mx_scale, pc1.out_dtype = torch.zeros((tokens * k, f // 32), dtype=torch.uint8, device=device), e4m3
            epi = mm.Epilogue(mm.FnSpecs(mm.FnName.QUANTIZE_MXFP8.name, quantize_mxfp8_fn, (), ()), (), (), effective_itemsize=1.0)
    else:
        pc1 = P(b_mx_scale=s1) if s1 is not None else None
    h = _both(monkeypatch, lambda: matmul_ogs(x, w1, b1, rd, gather_indx=gather, precision_config=pc1, fused_activation=act, epilogue=epi))
    if kind == "fp8":
        h, sh = _both(monkeypatch, lambda: quantize_fp8_rowwise(h))
        pc2 = P(a_mx_tensor_scale=sh, out_dtype=bf16)
    elif kind == "mxfp8":
        h, sh = _both(monkeypatch, lambda: downcast_to_mxfp(h, e4m3, axis=-1))
        pc2 = P(a_mx_scale=sh, b_mx_scale=s2, out_dtype=bf16)
    elif kind == "mxfp8_out":
        pc2 = P(a_mx_scale=pc1.c_mx_scale, b_mx_scale=s2, out_dtype=bf16)
    else:
        pc2 = P(b_mx_scale=s2) if s2 is not None else P()
    gam = rd.gate_scal
    _both(monkeypatch, lambda: matmul_ogs(h, w2, b2, rd, scatter_indx=scatter, precision_config=pc2, gammas=gam))
    assert [c["block_m"] for c in gemm_descriptors] == [block_m] * 4
    for fast, slow in (gemm_descriptors[:2], gemm_descriptors[2:]):
        _same_descriptors(fast, slow)
    # left to the general path: operands and options that are not of the plain form
    xt = x.t().contiguous().t()
    _both(monkeypatch, lambda: matmul_ogs(xt, w1, b1, rd, gather_indx=gather, precision_config=pc1, fused_activation=act, epilogue=epi), served=tokens == 1)
    with pytest.raises(AssertionError):
        matmul_ogs(x[:, :-32], w1, b1, rd, gather_indx=gather, precision_config=P(b_mx_scale=s1, out_dtype=bf16), fused_activation=act)


@pytest.mark.parametrize("shape, axis", [((1, 32), 1), ((3, 64), -1), ((64, 5), 0), ((2, 96, 7), 1), ((2, 96, 64), -2), ((1, 32, 1), 1), ((4, 3, 32), 2)])
@pytest.mark.parametrize("to", [torch.uint8, torch.float8_e4m3fn, torch.float8_e5m2])
def test_mx(device, monkeypatch, shape, axis, to):
    from triton_amd.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
    x = torch.randn(shape, generator=torch.Generator().manual_seed(sum(shape))).to(torch.bfloat16).to(device)
    q, s = _both(monkeypatch, lambda: downcast_to_mxfp(x, to, axis=axis))
    _both(monkeypatch, lambda: upcast_from_mxfp(q, s, torch.float16, axis=axis))


@pytest.mark.parametrize("m, n, sizes", [(8, 40, [3, 0, 17]), (64, 64, [0, 4])])
def test_ragged_k(device, monkeypatch, m, n, sizes):
    from triton_amd.matmul import matmul
    from triton_amd.tensor import make_ragged_tensor_metadata
    g, r = torch.Generator().manual_seed(m), sum(sizes)
    a, b = torch.randn((r, m), generator=g).to(torch.bfloat16).to(device), torch.randn((r, n), generator=g).to(torch.bfloat16).to(device)
    md = make_ragged_tensor_metadata(torch.tensor(sizes, dtype=torch.int32, device=device), r)
    _both(monkeypatch, lambda: matmul(a.t(), b, None, a_ragged_metadata=md, b_ragged_metadata=md))


@pytest.mark.parametrize("tokens, skip_bias", [(8, False), (61, True)])
def test_decode_layer(device, monkeypatch, tokens, skip_bias):
    import triton_amd.matmul as mm
    from triton_amd.moe_decode import moe_mlp
    from triton_amd.swiglu import swiglu_fn
    e, k, d, f = 32, 4, 256, 320
    g = torch.Generator().manual_seed(tokens)
    (w1, s1), (w2, s2) = _weights("mxfp4", e, d, 2 * f, g, device), _weights("mxfp4", e, f, d, g, device)
    x, logits = torch.randn((tokens, d), generator=g).to(torch.bfloat16).to(device), torch.randn((tokens, e), generator=g).to(device)
    b1 = None if skip_bias else torch.randn((e, 2 * f), generator=g).to(device)
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
    pc1, pc2 = mm.PrecisionConfig(b_mx_scale=s1), mm.PrecisionConfig(b_mx_scale=s2)
    _both(monkeypatch, lambda: moe_mlp(x, logits, k, w1, b1, w2, None, pc1, pc2, act))


@pytest.mark.parametrize("reduction_n", [None, 1, 4, "2", 1 << 70])
def test_activations_of_another_form_are_refused_by_the_general_path(device, reduction_n):
    import triton_amd.matmul as mm
    from triton_amd.swiglu import swiglu_fn
    from triton_amd.tensor import make_ragged_tensor_metadata
    x, w = torch.zeros((4, 64), dtype=torch.bfloat16, device=device), torch.zeros((1, 32, 64), dtype=torch.bfloat16, device=device).transpose(1, 2)
    md = make_ragged_tensor_metadata(torch.tensor([4], dtype=torch.int32, device=device), 4)
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=reduction_n), (1.702, 7.0))
    with pytest.raises(NotImplementedError):
        mm.matmul(x, w, None, md, fused_activation=act)


@pytest.mark.parametrize("dtype, swiglu", [(torch.bfloat16, False), (torch.float16, True)])
def test_rows_of_a_token_are_summed_by_the_same_call(device, monkeypatch, dtype, swiglu):
    """The GEMM's native call launches the combine too; results are seen by a dispatch mode, and filled in deterministic mode, as torch's own are."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from triton_amd.legacy import matmul_ogs, routing
    from triton_amd.matmul import FnSpecs, FusedActivation
    from triton_amd.swiglu import swiglu_fn
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn((40, 72), generator=g).to(dtype).to(device), torch.randn((6, 24, 72), generator=g).to(dtype).to(device).transpose(1, 2)
    bias, logits = torch.randn((6, 24), generator=g).to(device), torch.randn((40, 6), generator=g).to(device)
    act = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None
    rd, gather, scatter = routing(logits, 2)

    def run():
        return matmul_ogs(x, w, bias, rd, gather_indx=gather, scatter_indx=scatter, gammas=rd.gate_scal, fused_activation=act)
    plain = _both(monkeypatch, run)
    assert plain.shape == (40, 12 if swiglu else 24)

    class Seen(TorchDispatchMode):
        ops = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.ops.append(func)
            return func(*args, **(kwargs or {}))
    with Seen() as mode:
        _same(run(), plain)
    assert mode.ops.count(torch.ops.aten.empty.memory_format) == 2
    with torch.inference_mode():
        assert run().is_inference()
    torch.use_deterministic_algorithms(True)
    try:
        filled = run()
    finally:
        torch.use_deterministic_algorithms(False)
    assert torch.equal(filled, plain) and filled._version == 1  # (the fill)
