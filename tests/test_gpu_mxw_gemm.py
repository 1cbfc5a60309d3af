"""GPU parity of the wide MXFP4 GEMM (tiles of 160 rows x 512 columns; bf16 and MXFP8 activations) against the CPU oracle at the sizes
where it can go wrong: row blocks around 32, 80 (the shortest full block) and 160 rows, four stages of K (the fewest it takes), every remainder of the
scales' groups of four stages and a last group moved back into its row, columns around the tile of 512 and a wave's 64, several tiles a workgroup."""
import pytest
import torch

from oracle import moe as omoe
from oracle import mxfp as omx
from oracle.checks import assert_allclose_gate

pytestmark = pytest.mark.gpu

SHAPES = [
    (512, 32, [0, 1, 31, 32, 33, 0, 65]),
    (544, 512, [80, 81, 160, 0, 161]),
    (672, 520, [240, 241, 1, 320]),
    (736, 1088, [159, 64, 97]),
    (928, 576, [33] * 5),
    (512, 96, [(i * 29) % 37 for i in range(256)]),
    (1056, 1504, [17, 40, 130] * 40),
]


def _case(device, k, n, sizes, mx8):
    from triton_amd.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
    from triton_amd.tensor_details.layout import make_default_matmul_mxfp4_w_layout, make_default_matmul_mxfp4_w_scale_layout
    g = torch.Generator().manual_seed(k + n)
    E, m = len(sizes), sum(sizes)
    sizes = torch.tensor(sizes, dtype=torch.int32)
    # blocks of very different magnitudes, so that a scale that belongs to another row or block shows; none above 1, so that a sum's
    # terms add up to at most about K * 0.08 = 80 and the matrix instruction's rounding of them (2^-14 of the larger ones, 0.005) stays
    # inside the gate's 0.01 also where the sum cancels and swiglu's gate is steep
    x = (torch.randn((m, k), generator=g) * torch.exp2(torch.randint(-8, 1, (m, k // 32), generator=g).float()).repeat_interleave(32, 1)).to(torch.bfloat16)
    wq, ws = omx.downcast_to_mxfp((torch.randn((E, k, n), generator=g) * 0.1).to(torch.bfloat16), torch.uint8, axis=1)
    c = dict(E=E, m=m, sizes=sizes, x=x, wq=wq, ws=ws, bias=torch.randn((E, n), generator=g), gam=torch.rand((m, ), generator=g) + 0.5,
             gi=torch.randint(0, m, (m, ), generator=g).to(torch.int32), sc=torch.randperm(m, generator=g).to(torch.int32),
             md=make_ragged_tensor_metadata(sizes.to(device), m),
             w_dev=convert_layout(wrap_torch_tensor(wq.to(device), dtype=FP4), make_default_matmul_mxfp4_w_layout(mx_axis=1)),
             s_dev=convert_layout(wrap_torch_tensor(ws.to(device)), make_default_matmul_mxfp4_w_scale_layout(mx_axis=1)))
    if mx8:
        c["xq"], c["xs"] = omx.downcast_to_mxfp(x, torch.float8_e4m3fn, axis=1)
        c["x"] = omx.upcast_from_mxfp(c["xq"], c["xs"], torch.float32, axis=1)
    return c


@pytest.mark.parametrize("k, n, sizes", SHAPES)
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("mx8", [False, True])
def test_wide_gemm(device, k, n, sizes, swiglu, mx8):
    import triton_amd.matmul as mm
    from triton_amd.swiglu import swiglu_fn
    c = _case(device, k, n, sizes, mx8)
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None
    out = torch.full((c["m"], n // 2 if swiglu else n), float("nan"), dtype=torch.bfloat16, device=device)
    pc = mm.PrecisionConfig(b_mx_scale=c["s_dev"], a_mx_scale=c["xs"].to(device) if mx8 else None, out_dtype=torch.bfloat16)
    with mm.scoped_opt_flags_constraints({"block_m": 256}):
        mm.matmul((c["xq"] if mx8 else c["x"]).to(device), c["w_dev"], c["bias"].to(device), c["md"], gather_indx=c["gi"].to(device),
                  scatter_indx=c["sc"].to(device), gammas=c["gam"].to(device), precision_config=pc, fused_activation=act, c=out)
    ref = omoe.matmul(c["x"], c["wq"], c["bias"], c["sizes"], gather_indx=c["gi"], w_mx_scale=c["ws"], out_dtype=torch.float32)
    ref = (omoe.swiglu(ref, 1.702, 7.0).float() if swiglu else ref) * c["gam"][:, None]
    want = torch.empty_like(ref)
    want[c["sc"].long()] = ref
    assert_allclose_gate(want, out, what="wide GEMM")


@pytest.mark.parametrize("swiglu", [False, True])
def test_wide_gemm_quantised_output(device, swiglu):
    """The MX-quantised output holds what the same kernel's bf16 output does, to a rounding of e4m3 (2^-4 of a value, or half
    the smallest step, 2^-10 of the block's scale)."""
    import triton_amd.matmul as mm
    from triton_amd.numerics_details.mxfp import quantize_mxfp8_fn, upcast_from_mxfp
    from triton_amd.swiglu import swiglu_fn
    c = _case(device, 736, 1088, [159, 64, 97, 0, 161], True)
    n_out = 544 if swiglu else 1088
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None
    scale = torch.zeros((c["m"], n_out // 32), dtype=torch.uint8, device=device)
    epi = mm.Epilogue(mm.FnSpecs(mm.FnName.QUANTIZE_MXFP8.name, quantize_mxfp8_fn, (), ()), tuple(), tuple(), effective_itemsize=1.0)
    args = (c["xq"].to(device), c["w_dev"], c["bias"].to(device), c["md"])
    with mm.scoped_opt_flags_constraints({"block_m": 256}):
        plain = mm.matmul(*args, precision_config=mm.PrecisionConfig(b_mx_scale=c["s_dev"], a_mx_scale=c["xs"].to(device), out_dtype=torch.bfloat16),
                          fused_activation=act).float()
        q = mm.matmul(*args, precision_config=mm.PrecisionConfig(b_mx_scale=c["s_dev"], a_mx_scale=c["xs"].to(device), c_mx_scale=scale,
                                                                 out_dtype=torch.float8_e4m3fn), fused_activation=act, epilogue=epi)
    back = upcast_from_mxfp(q, scale, torch.float32, axis=-1)
    step = torch.exp2(scale.float() - 127).repeat_interleave(32, 1)
    # (2^-8: the bf16 value's own rounding)
    assert torch.all((back - plain).abs() <= plain.abs() * (2.0**-4 + 2.0**-8) + step * 2.0**-10)
