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


# mean rows per slice, slices, K, N, sizes dealt in turn: every tile that the rules name, at the edges of its row blocks (one more, one less, none at
# all), of its columns and of a wave's 64, with four stages of K (the fewest), remainders of K and of the scales' groups
RULED = [
    ("bf16", "64x512", 256, 544, 1056, [0, 1, 31, 32, 33, 5, 2, 9, 64, 65]),
    ("bf16", "32x256", 192, 736, 1072, [0, 1, 31, 32, 33, 5, 2, 9]),
    ("bf16", "32x256", 256, 512, 2080, [0, 1, 3, 2, 0, 33, 0, 0, 0, 0]),
    ("bf16", "32x256", 256, 512, 2080, [0, 1, 31, 2, 0, 33, 0, 0, 0, 0]),
    ("bf16", "64x512", 256, 512, 1056, [0, 1, 31, 2, 9, 33, 0, 65, 0, 0, 0, 0]),
    ("bf16", "32x256", 40, 512, 528, [0, 1, 31, 32, 33, 2, 13]),
    ("bf16", "64x256", 64, 544, 1056, [63, 64, 65, 1, 0, 33, 127, 128, 129]),
    ("bf16", "64x256", 64, 1312, 1040, [95, 32, 31, 97]),
    ("bf16", "64x512", 256, 512, 544, [0, 1, 31, 32, 33, 63, 64, 65, 10]),
    ("bf16", "96x512", 256, 736, 528, [95, 96, 97, 1, 33, 65, 64, 100]),
    ("bf16", "160x512", 256, 512, 576, [159, 160, 161, 81, 80, 1, 33]),
    ("mxfp8", "32x256", 128, 512, 576, [0, 1, 31, 32, 33, 2, 13]),
    ("mxfp8", "128x512", 128, 672, 544, [0, 1, 31, 32, 33, 63, 64, 65, 10]),
    ("mxfp8", "64x512", 128, 672, 544, [0, 1, 31, 32, 33, 63, 64, 65, 10, 0]),
    ("mxfp8", "64x512", 256, 544, 1088, [0, 1, 31, 32, 63, 64, 65, 10, 2, 1, 0]),
    ("mxfp8", "128x512", 128, 736, 576, [95, 96, 97, 1, 33, 65, 40]),
    ("mxfp8", "128x512", 128, 928, 544, [127, 128, 129, 65, 64, 1, 33, 97, 96]),
    ("mxfp8", "128x512", 64, 544, 1024, [127, 128, 129, 150, 255, 256, 1, 160]),
]
# MXFP8 rows of more than 104 a slice, by what the tiles cost
RULED += [
    ("mxfp8", "64x512", 32, 608, 864, [127, 128, 129, 192, 193, 130]),
    ("mxfp8", "128x512", 16, 672, 2112, [255, 256, 257, 300, 260, 268]),
    ("mxfp8", "160x512", 16, 672, 1856, [480, 481, 560, 640, 641, 340]),
]


@pytest.mark.parametrize("kind, tile, e, k, n, sizes", RULED)
@pytest.mark.parametrize("swiglu, routed", [(True, True), (False, False), (False, True)])
def test_tiles_by_the_rules(device, kind, tile, e, k, n, sizes, swiglu, routed):
    """The tile of the wide kernel that the rules name gives, bit for bit, what the kernel for row blocks of 128 gives (whose sums over K run in the
    same order): gathered and scattered rows, gate weights, rows without a destination, a quantised output."""
    import triton_amd._native as nt
    import triton_amd.matmul as mm
    from triton_amd.numerics_details.mxfp import downcast_to_mxfp, quantize_mxfp8_fn
    from triton_amd.swiglu import swiglu_fn
    from triton_amd.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
    from triton_amd.tensor_details.layout import make_default_matmul_mxfp4_w_layout, make_default_matmul_mxfp4_w_scale_layout
    g = torch.Generator(device=device).manual_seed(k + n)
    sizes = torch.tensor([sizes[i % len(sizes)] for i in range(e)], dtype=torch.int32, device=device)
    m = int(sizes.sum())
    mx8 = kind == "mxfp8"
    assert nt.rules().wide_block_n(m, e, k, n, m * k, mx8) == int(tile.split("x")[1])
    x = torch.randn((m, k), generator=g, device=device).to(torch.bfloat16)
    wq, ws = downcast_to_mxfp((torch.randn((e, k, n), generator=g, device=device) * 0.1).to(torch.bfloat16), torch.uint8, axis=1)
    w = convert_layout(wrap_torch_tensor(wq, dtype=FP4), make_default_matmul_mxfp4_w_layout(mx_axis=1))
    s = convert_layout(wrap_torch_tensor(ws), make_default_matmul_mxfp4_w_scale_layout(mx_axis=1))
    bias = torch.randn((e, n), generator=g, device=device)
    args = dict(fused_activation=mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None)
    if routed:
        args.update(gammas=torch.rand((m, ), generator=g, device=device) + 0.5, gather_indx=torch.randint(0, m, (m, ), generator=g, device=device).to(torch.int32),
                    scatter_indx=torch.randperm(m, generator=g, device=device).to(torch.int32))
        args["scatter_indx"][::7] = -1
    md = make_ragged_tensor_metadata(sizes, m)
    n_out = n // 2 if swiglu else n
    quantised = mx8 and n_out % 32 == 0

    def run():
        out = torch.zeros((m, n_out), dtype=torch.bfloat16, device=device)
        a, pc = x, mm.PrecisionConfig(b_mx_scale=s, out_dtype=torch.bfloat16)
        if mx8:
            a, pc.a_mx_scale = downcast_to_mxfp(x, torch.float8_e4m3fn, axis=-1)
        got = [mm.matmul(a, w, bias, md, precision_config=pc, c=out, **args).clone()]
        if quantised:
            pc.c_mx_scale, pc.out_dtype = torch.zeros((m, n_out // 32), dtype=torch.uint8, device=device), torch.float8_e4m3fn
            epi = mm.Epilogue(mm.FnSpecs(mm.FnName.QUANTIZE_MXFP8.name, quantize_mxfp8_fn, (), ()), tuple(), tuple(), effective_itemsize=1.0)
            q = torch.zeros((m, n_out), dtype=torch.float8_e4m3fn, device=device)
            got += [mm.matmul(a, w, bias, md, precision_config=pc, epilogue=epi, c=q, **args).view(torch.uint8).clone(), pc.c_mx_scale]
        return got
    by_rule = run()
    with mm.scoped_opt_flags_constraints({"block_m": 128}):
        want = run()
    for a, b in zip(by_rule, want):
        assert torch.equal(a, b)
    assert not torch.isnan(by_rule[0]).any() and by_rule[0].any()


# slices, K, N, sizes: each tile with MXFP8 rows (32, 64, 128 and 160 rows; eight, sixteen and twenty rows' scales a wave)
SCALED = [(128, 544, 576, [0, 1, 31, 32, 33, 2, 13]), (256, 672, 544, [33, 63, 64, 65, 10, 1]), (128, 800, 544, [95, 96, 97, 1, 33, 65, 40]), (128, 928, 544, [159, 160, 161, 33, 97])]


@pytest.mark.parametrize("e, k, n, sizes", SCALED)
@pytest.mark.parametrize("offset, pad", [(0, 0), (1, 3), (2, 1), (3, 6), (1, 7)])
def test_scales_at_any_byte(device, e, k, n, sizes, offset, pad):
    """Rows of activation scales that begin at any byte, between bytes that are no scales (NaN): the result is, bit for bit, that of scales in a
    tensor of their own, and nothing of a neighbour gets into the last blocks of a row."""
    import triton_amd.matmul as mm
    from triton_amd.numerics_details.mxfp import downcast_to_mxfp
    from triton_amd.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
    from triton_amd.tensor_details.layout import make_default_matmul_mxfp4_w_layout, make_default_matmul_mxfp4_w_scale_layout
    g = torch.Generator(device=device).manual_seed(k + n + offset)
    sizes = torch.tensor([sizes[i % len(sizes)] for i in range(e)], dtype=torch.int32, device=device)
    m = int(sizes.sum())
    a, scale = downcast_to_mxfp(torch.randn((m, k), generator=g, device=device).to(torch.bfloat16), torch.float8_e4m3fn, axis=-1)
    wq, ws = downcast_to_mxfp((torch.randn((e, k, n), generator=g, device=device) * 0.1).to(torch.bfloat16), torch.uint8, axis=1)
    w = convert_layout(wrap_torch_tensor(wq, dtype=FP4), make_default_matmul_mxfp4_w_layout(mx_axis=1))
    s = convert_layout(wrap_torch_tensor(ws), make_default_matmul_mxfp4_w_scale_layout(mx_axis=1))
    md, gather = make_ragged_tensor_metadata(sizes, m), torch.randint(0, m, (m, ), generator=g, device=device).to(torch.int32)

    def run(x_scale):
        return mm.matmul(a, w, None, md, gather_indx=gather, precision_config=mm.PrecisionConfig(a_mx_scale=x_scale, b_mx_scale=s, out_dtype=torch.bfloat16))
    with mm.scoped_opt_flags_constraints({"block_m": 128}):
        want = run(scale)
    stride = k // 32 + pad
    room = torch.full((offset + m * stride, ), 255, dtype=torch.uint8, device=device)
    view = room[offset:].view(m, stride)[:, :k // 32]
    view.copy_(scale)
    got = run(view)
    assert torch.equal(got, want) and not torch.isnan(got).any()


@pytest.mark.parametrize("e, k, n, sizes", [(16, 1792, 2048, [81, 104, 97, 90]), (8, 576, 1056, [96, 128, 64, 100, 33, 129, 90, 95])])
def test_mxfp8_rows_without_a_wide_tile(device, e, k, n, sizes):
    """81 to 104 rows a slice where the tiles of 128 x 256 are one round: they run, and give what the wide kernel's 160 x 512 give, bit for bit."""
    import triton_amd._native as nt
    import triton_amd.matmul as mm
    from triton_amd.swiglu import swiglu_fn
    c = _case(device, k, n, [sizes[i % len(sizes)] for i in range(e)], True)
    assert 80 * e < c["m"] <= 104 * e
    assert nt.rules().wide_block_n(c["m"], e, k, n, c["m"] * k, 1) == 0 and nt.rules().wide_block_m(c["m"], e, k, n, c["m"] * k, 1) == 128
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
    pc = mm.PrecisionConfig(b_mx_scale=c["s_dev"], a_mx_scale=c["xs"].to(device), out_dtype=torch.bfloat16)
    args = dict(gather_indx=c["gi"].to(device), scatter_indx=c["sc"].to(device), gammas=c["gam"].to(device), precision_config=pc, fused_activation=act)
    out = mm.matmul(c["xq"].to(device), c["w_dev"], c["bias"].to(device), c["md"], **args)
    with mm.scoped_opt_flags_constraints({"block_m": 256}):
        wide = mm.matmul(c["xq"].to(device), c["w_dev"], c["bias"].to(device), c["md"], **args)
    assert torch.equal(out, wide) and out.any()
