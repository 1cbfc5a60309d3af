"""GPU parity of the streaming bf16 x tiled MXFP4 GEMM (row blocks of 32) against the CPU oracle at the sizes where it can go wrong:
row blocks around 32 rows, one stage of K, a stage and a remainder and more stages than buffers, columns around the tile of 256 and
its waves' 64, few tiles and several rounds of them."""
import pytest
import torch

from oracle import moe as omoe
from oracle import mxfp as omx
from oracle.checks import assert_allclose_gate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k, n, sizes", [
    (32, 32, [0, 1, 31, 32, 33, 0, 65]),
    (128, 264, [5, 0, 32, 64, 1]),
    (160, 576, [33] * 5),
    (544, 96, [(i * 29) % 37 for i in range(256)]),
    (416, 1504, [17, 40] * 60),
])
@pytest.mark.parametrize("swiglu", [False, True])
def test_streaming_gemm(device, k, n, sizes, swiglu):
    import triton_amd.matmul as mm
    from triton_amd.swiglu import swiglu_fn
    from triton_amd.tensor import FP4, convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
    from triton_amd.tensor_details.layout import make_default_matmul_mxfp4_w_layout, make_default_matmul_mxfp4_w_scale_layout
    g = torch.Generator().manual_seed(k + n)
    E, m = len(sizes), sum(sizes)
    sizes = torch.tensor(sizes, dtype=torch.int32)
    x = torch.randn((m, k), generator=g).to(torch.bfloat16)
    wq, ws = omx.downcast_to_mxfp((torch.randn((E, k, n), generator=g) * 0.1).to(torch.bfloat16), torch.uint8, axis=1)
    bias, gam = torch.randn((E, n), generator=g), torch.rand((m, ), generator=g) + 0.5
    gi, sc = torch.randint(0, m, (m, ), generator=g).to(torch.int32), torch.randperm(m, generator=g).to(torch.int32)
    w_dev = convert_layout(wrap_torch_tensor(wq.to(device), dtype=FP4), make_default_matmul_mxfp4_w_layout(mx_axis=1))
    s_dev = convert_layout(wrap_torch_tensor(ws.to(device)), make_default_matmul_mxfp4_w_scale_layout(mx_axis=1))
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None
    out = torch.full((m, n // 2 if swiglu else n), float("nan"), dtype=torch.bfloat16, device=device)
    with mm.scoped_opt_flags_constraints({"block_m": 32}):
        mm.matmul(x.to(device), w_dev, bias.to(device), make_ragged_tensor_metadata(sizes.to(device), m), gather_indx=gi.to(device),
                  scatter_indx=sc.to(device), gammas=gam.to(device), precision_config=mm.PrecisionConfig(b_mx_scale=s_dev),
                  fused_activation=act, c=out)
    ref = omoe.matmul(x, wq, bias, sizes, gather_indx=gi, w_mx_scale=ws, out_dtype=torch.float32)
    ref = (omoe.swiglu(ref, 1.702, 7.0).float() if swiglu else ref) * gam[:, None]
    want = torch.empty_like(ref)
    want[sc.long()] = ref
    assert_allclose_gate(want, out, what="streaming GEMM")
