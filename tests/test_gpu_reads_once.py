"""Weights of over 128 MiB with about one row block per slice are fetched with the non-temporal hint: bit for bit what the same kernels give for each
half of the slices, whose weights are below that line."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _weights(kind, e, k, n, g, device):
    from triton_amd.tensor import FP4, convert_layout, wrap_torch_tensor
    from triton_amd.tensor_details.layout import make_default_matmul_fp8_w_layout, make_default_matmul_mxfp4_w_layout, make_default_matmul_mxfp4_w_scale_layout
    if kind.startswith("mx"):
        v = torch.randint(0, 256, (e, n, k // 2), dtype=torch.uint8, generator=g, device=device).transpose(1, 2)
        s = torch.randint(118, 122, (e, n, k // 32), dtype=torch.uint8, generator=g, device=device).transpose(1, 2)
        return lambda part: (convert_layout(wrap_torch_tensor(v[part], dtype=FP4), make_default_matmul_mxfp4_w_layout(mx_axis=1)),
                             convert_layout(wrap_torch_tensor(s[part]), make_default_matmul_mxfp4_w_scale_layout(mx_axis=1)))
    w = torch.randn((e, n, k), generator=g, device=device) * 0.1
    if kind == "e4m3":
        w = w.to(torch.float8_e4m3fn)
        return lambda part: (convert_layout(wrap_torch_tensor(w[part].transpose(1, 2)), make_default_matmul_fp8_w_layout()), None)
    w = w.to(getattr(torch, kind))
    return lambda part: (w[part].transpose(1, 2), None)


@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("kind, block_m, e, k, n", [("bfloat16", 128, 70, 1048, 1000), ("float16", 256, 70, 1048, 1000), ("e4m3", 128, 140, 1040, 1000),
                                                    ("e4m3", 256, 140, 1040, 1000), ("mxfp4", 256, 128, 1536, 1512), ("mxfp8", 256, 128, 1536, 1512)])
def test_whole_against_halves(device, kind, block_m, e, k, n, swiglu):
    import triton_amd.matmul as mm
    from triton_amd.numerics_details.mxfp import downcast_to_mxfp
    from triton_amd.swiglu import swiglu_fn
    from triton_amd.tensor import make_ragged_tensor_metadata
    assert e * k * n * {"e4m3": 1, "mxfp4": 0.5, "mxfp8": 0.5}.get(kind, 2) > 128 * 2**20
    g = torch.Generator(device=device).manual_seed(e + k)
    sizes = torch.randint(0, 150 if block_m == 256 else 75, (e, ), generator=g, device=device, dtype=torch.int32)
    sizes[:4] = torch.tensor([0, 300, 1, 129], dtype=torch.int32)
    m = int(sizes.sum())
    x = torch.randn((m, k), generator=g, device=device)
    x = x.to(torch.float8_e4m3fn) if kind == "e4m3" else x.to(torch.float16 if kind == "float16" else torch.bfloat16)
    bias = torch.randn((e, n), generator=g, device=device)
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None
    weights = _weights(kind, e, k, n, g, device)

    def run(part, rows):
        w, s = weights(part)
        a, xs = downcast_to_mxfp(x[rows], torch.float8_e4m3fn, axis=1) if kind == "mxfp8" else (x[rows], None)
        pc = mm.PrecisionConfig(b_mx_scale=s, a_mx_scale=xs, out_dtype=torch.float16 if kind == "float16" else torch.bfloat16)
        with mm.scoped_opt_flags_constraints({"block_m": block_m}):
            return mm.matmul(a, w, bias[part], make_ragged_tensor_metadata(sizes[part].contiguous(), a.shape[0]), precision_config=pc, fused_activation=act)
    cut = int(sizes[:e // 2].sum())
    halves = torch.cat([run(slice(0, e // 2), slice(0, cut)), run(slice(e // 2, e), slice(cut, m))])
    assert torch.equal(run(slice(0, e), slice(0, m)), halves)
