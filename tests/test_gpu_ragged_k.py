"""GPU parity of the ragged-K GEMM (the expert weight gradient, `matmul(..., b_ragged_metadata=...)`) through the C ABI
against the CPU oracle.

Mirrors the `inner_expt_opt` cases of python/triton_kernels/tests/test_matmul.py:311-320,469-500: the reduction
dimension is split into slices (10, one of them empty), either operand's slices may be padded ("pad_a" / "pad_b", so
the two operands carry different slice offsets), no bias.  Operands are bf16 or fp16; a is taken both k-slow (x^T of a
row-major x: the weight-gradient layout) and k-contiguous, b both row-major and transposed.  Tolerance: the rtol 2e-2 /
atol 1e-2 gate for 16-bit outputs (accumulation order differs from torch's), tighter for fp32 outputs."""
import pytest
import torch

from oracle import moe as omoe
from oracle.checks import assert_allclose_gate

pytestmark = pytest.mark.gpu


def _slices(k_total, n_slices, g):
    cuts = torch.sort(torch.randint(0, k_total + 1, (n_slices - 1, ), generator=g)).values
    sizes = torch.diff(torch.cat([torch.tensor([0]), cuts, torch.tensor([k_total])]))
    if n_slices > 2:
        sizes[n_slices // 2 + 1] += sizes[n_slices // 2]  # one empty slice
        sizes[n_slices // 2] = 0
    return sizes.to(torch.int32)


def _metadata(sizes, offs, device):
    from triton_amd.tensor import RaggedTensorMetadata, make_ragged_tensor_metadata
    md = make_ragged_tensor_metadata(sizes.to(device), int(offs[-1]))
    return RaggedTensorMetadata(md.slice_sizes, offs.to(torch.int32).to(device), md.block_offs_data, md.block_schedule_data)


def _offsets(sizes, pad):
    """Start of every slice (+ the end): dense, or each slice padded to a multiple of `pad`."""
    offs = [0]
    for s in sizes.tolist():
        step = s if pad is None else (s + pad - 1) // pad * pad
        offs.append(offs[-1] + step)
    return torch.tensor(offs, dtype=torch.int32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("m, n, k", [(300, 400, 416), (128, 256, 1024), (720, 576, 768), (17, 40, 100), (256, 8, 64)])
@pytest.mark.parametrize("pad", [None, "pad_a", "pad_b"])
@pytest.mark.parametrize("a_k_slow, b_transposed", [(True, False), (False, False), (True, True), (False, True)])
def test_ragged_k_matmul(device, dtype, m, n, k, pad, a_k_slow, b_transposed):
    import triton_amd.matmul as mm
    g = torch.Generator().manual_seed(m * 31 + n * 7 + k)
    sizes = _slices(k, 10, g)
    a_offs = _offsets(sizes, 16 if pad == "pad_a" else None)
    b_offs = _offsets(sizes, 16 if pad == "pad_b" else None)
    ka, kb = int(a_offs[-1]), int(b_offs[-1])
    # the padding holds garbage that must not reach the output (NaN would poison a sum that read it)
    a = torch.randn((m, ka), generator=g).to(dtype)
    b = torch.randn((kb, n), generator=g).to(dtype)
    for e, s in enumerate(sizes.tolist()):
        a[:, int(a_offs[e]) + s:int(a_offs[e + 1])] = float("nan")
        b[int(b_offs[e]) + s:int(b_offs[e + 1]), :] = float("nan")
    ref = omoe.matmul_ragged_k(a, b, sizes, a_offs, b_offs)
    a_dev = a.to(device)
    if a_k_slow:  # x^T of a row-major [k, m] tensor
        a_dev = a.t().contiguous().to(device).t()
        assert a_dev.stride(0) == 1
    b_dev = b.to(device)
    if b_transposed:
        b_dev = b.t().contiguous().to(device).t()
    out = mm.matmul(a_dev, b_dev, None, a_ragged_metadata=_metadata(sizes, a_offs, device),
                    b_ragged_metadata=_metadata(sizes, b_offs, device))
    assert out.shape == (10, m, n) and out.dtype == dtype
    assert not torch.isnan(out).any()
    assert_allclose_gate(ref, out, what="ragged-K matmul")
    assert out[5].abs().max() == 0  # the empty slice


def test_ragged_k_fp32_output_and_weight_gradient_identity(device):
    """dW[e] = x_e^T @ dy_e at a MoE-like shape with fp32 output, and the identity sum_e dW[e] = x^T @ dy."""
    import triton_amd.matmul as mm
    g = torch.Generator().manual_seed(3)
    rows, hidden, n, E = 1024, 360, 200, 8
    sizes = _slices(rows, E, g)
    offs = _offsets(sizes, None)
    x = torch.randn((rows, hidden), generator=g).to(torch.bfloat16)
    dy = torch.randn((rows, n), generator=g).to(torch.bfloat16)
    md = _metadata(sizes, offs, device)
    pc = mm.PrecisionConfig(out_dtype=torch.float32)
    out = mm.matmul(x.to(device).t(), dy.to(device), None, a_ragged_metadata=md, b_ragged_metadata=md, precision_config=pc)
    ref = omoe.matmul_ragged_k(x.t(), dy, sizes, offs, offs, out_dtype=torch.float32)
    torch.testing.assert_close(out.cpu(), ref, rtol=1e-4, atol=1e-3)
    torch.testing.assert_close(out.cpu().sum(0).double(), x.double().t() @ dy.double(), rtol=1e-4, atol=2e-3)


def test_ragged_k_rejections(device):
    import triton_amd.matmul as mm
    sizes = torch.tensor([4, 4], dtype=torch.int32)
    md = _metadata(sizes, _offsets(sizes, None), device)
    a = torch.zeros((8, 8), dtype=torch.bfloat16, device=device)
    with pytest.raises(NotImplementedError):
        mm.matmul(a, a, torch.zeros((2, 8), device=device), a_ragged_metadata=md, b_ragged_metadata=md)
    with pytest.raises(NotImplementedError):
        mm.matmul(a.float(), a.float(), None, a_ragged_metadata=md, b_ragged_metadata=md)
    with pytest.raises(ValueError):
        mm.matmul(a, a, None, b_ragged_metadata=md)


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("m, n", [(8, 8), (128, 136), (264, 1032)])
def test_ragged_k_stage_and_tile_edges(device, m, n, out_dtype):
    """Aligned k-slow operands (transposed by the LDS reads): slice lengths around the 16-row stages and the five stage
    buffers, tiles around 128, more and fewer tiles than XCDs, each output type."""
    import triton_amd.matmul as mm
    g = torch.Generator().manual_seed(m + n)
    sizes = torch.tensor([0, 1, 15, 16, 17, 48, 64, 65, 80, 81, 96, 200], dtype=torch.int32)
    offs = _offsets(sizes, 24)
    k = int(offs[-1])
    a, b = torch.randn((k, m), generator=g).to(torch.bfloat16), torch.randn((k, n), generator=g).to(torch.bfloat16)
    for e, s in enumerate(sizes.tolist()):
        a[int(offs[e]) + s:int(offs[e + 1])] = float("nan")
        b[int(offs[e]) + s:int(offs[e + 1])] = float("nan")
    out = torch.full((len(sizes), m, n), float("nan"), dtype=out_dtype, device=device)
    md = _metadata(sizes, offs, device)
    mm.matmul(a.to(device).t(), b.to(device), None, a_ragged_metadata=md, b_ragged_metadata=md, c=out,
              precision_config=mm.PrecisionConfig(out_dtype=out_dtype))
    ref = omoe.matmul_ragged_k(a.t(), b, sizes, offs, offs, out_dtype=torch.float32)
    assert_allclose_gate(ref, out.float(), what="ragged-K matmul")


@pytest.mark.parametrize("n_slices, m, n", [(70, 2040, 2168), (64, 2048, 2048), (63, 2040, 2168), (64, 1920, 2168)])
def test_operands_asked_for_ahead(device, n_slices, m, n):
    """From 64 slices and 32 tiles of a slice per XCD on, tiles ask for lines of later slices: some of these are empty, some long, the last
    ones have no successor, and both sides of the line.  The sum is exact but for its order (fp32) and the result's rounding to bf16, half of 2^-8."""
    import triton_amd.matmul as mm
    g = torch.Generator().manual_seed(n_slices + m)
    sizes = torch.randint(0, 12, (n_slices, ), generator=g).to(torch.int32)
    sizes[3], sizes[5], sizes[-1] = 0, 250, 200
    offs = _offsets(sizes, None)
    a, b = torch.randn((int(offs[-1]), m), generator=g).to(torch.bfloat16).to(device), torch.randn((int(offs[-1]), n), generator=g).to(torch.bfloat16).to(device)
    md = _metadata(sizes, offs, device)
    out = mm.matmul(a.t(), b, None, a_ragged_metadata=md, b_ragged_metadata=md)
    for e in range(n_slices):
        k = slice(int(offs[e]), int(offs[e + 1]))
        ref = a[k].float().t() @ b[k].float()
        assert ((out[e].float() - ref).abs() <= ref.abs() * 2**-8 + 1e-4).all(), e


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("n_slices, m, n, rest", [(12, 264, 1032, 300), (9, 8, 136, 2000), (128, 520, 264, 170), (1, 264, 520, 700), (128, 520, 776, 170), (129, 264, 264, 170)])
def test_long_slices(device, n_slices, m, n, rest, out_dtype):
    """Slices long enough on average for the kernel of long ones: lengths around its stages of 32 and its four buffers, empty ones, tiles of 128 and
    of 256 with remainders, more and fewer tiles than workgroups and XCDs, one slice more than it keeps.  The sum is exact but for its order (fp32: some
    2000 terms of size one, 2^-24 each time, far below the gate) and the result's rounding."""
    import triton_amd.matmul as mm
    g = torch.Generator().manual_seed(n_slices + m + n)
    sizes = torch.full((n_slices, ), rest, dtype=torch.int32)
    edges = [0, 1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 3 * rest]
    for i, s in enumerate(edges[:n_slices if n_slices > 1 else 0]):
        sizes[(i * 5) % n_slices] = s
    offs = _offsets(sizes, 8)
    k = max(int(offs[-1]), 160 * n_slices + 8)  # (some rows belong to no slice)
    a, b = torch.randn((k, m), generator=g).to(torch.bfloat16), torch.randn((k, n), generator=g).to(torch.bfloat16)
    used = torch.zeros(k, dtype=torch.bool)
    for e, s in enumerate(sizes.tolist()):
        used[int(offs[e]):int(offs[e]) + s] = True
    a[~used], b[~used] = float("nan"), float("nan")
    out = torch.full((n_slices, m + 8, n + 8), float("nan"), dtype=out_dtype, device=device)
    md = _metadata(sizes, offs, device)
    mm.matmul(a.to(device).t(), b.to(device), None, a_ragged_metadata=md, b_ragged_metadata=md, c=out[:, :m, :n],
              precision_config=mm.PrecisionConfig(out_dtype=out_dtype))
    ref = omoe.matmul_ragged_k(a.t(), b, sizes, offs, offs, out_dtype=torch.float32)
    assert_allclose_gate(ref, out[:, :m, :n].float(), what="ragged-K matmul")
    assert torch.isnan(out[:, m:]).all() and torch.isnan(out[:, :, n:]).all()  # nothing written beside the result


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("m, n, beside", [(8, 8, 8), (72, 56, 8), (136, 200, 0), (120, 328, 24), (264, 120, 16)])
def test_short_slices_rows_of_broken_lines(device, m, n, beside, out_dtype):
    """Results whose rows begin and end inside a 128-byte line, tiles that end inside a wave's rows or columns: nothing is written beside them.  One
    rounding of a sum of at most 40 terms."""
    import triton_amd.matmul as mm
    g = torch.Generator().manual_seed(m * n)
    sizes = torch.tensor([0, 1, 17, 40, 16], dtype=torch.int32)
    offs = _offsets(sizes, 8)
    k = int(offs[-1])
    a, b = torch.randn((k, m), generator=g).to(torch.bfloat16), torch.randn((k, n), generator=g).to(torch.bfloat16)
    out = torch.full((len(sizes), m + 8, n + beside), float("nan"), dtype=out_dtype, device=device)
    md = _metadata(sizes, offs, device)
    mm.matmul(a.to(device).t(), b.to(device), None, a_ragged_metadata=md, b_ragged_metadata=md, c=out[:, :m, :n],
              precision_config=mm.PrecisionConfig(out_dtype=out_dtype))
    ref = omoe.matmul_ragged_k(a.t(), b, sizes, offs, offs, out_dtype=torch.float32)
    assert_allclose_gate(ref, out[:, :m, :n].float(), what="ragged-K matmul")
    assert torch.isnan(out[:, m:]).all() and torch.isnan(out[:, :, n:]).all()


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("n_slices, m, n, rest, tile", [(12, 264, 1032, 300, 128), (128, 520, 776, 170, 256)])
def test_long_slices_of_fp16(device, n_slices, m, n, rest, tile, out_dtype):
    """fp16 operands by either tile of the kernel for long slices.  A sum of at most 900 products of values below 5 in size: far inside fp16's range, and
    its order's error (2^-24 a term) far below the gate."""
    import triton_amd._native as nt
    import triton_amd.matmul as mm
    g = torch.Generator().manual_seed(n_slices + n)
    sizes = torch.full((n_slices, ), rest, dtype=torch.int32)
    for i, s in enumerate([0, 1, 31, 33, 64, 97, 129, 3 * rest]):
        sizes[(i * 5) % n_slices] = s
    offs = _offsets(sizes, 8)
    k = max(int(offs[-1]), 160 * n_slices + 8)
    assert nt.rules().ragged_k_tile(k // n_slices, m, n, n_slices) == tile
    a, b = torch.randn((k, m), generator=g).to(torch.float16), torch.randn((k, n), generator=g).to(torch.float16)
    out = torch.full((n_slices, m, n), float("nan"), dtype=out_dtype, device=device)
    md = _metadata(sizes, offs, device)
    mm.matmul(a.to(device).t(), b.to(device), None, a_ragged_metadata=md, b_ragged_metadata=md, c=out, precision_config=mm.PrecisionConfig(out_dtype=out_dtype))
    ref = omoe.matmul_ragged_k(a.t(), b, sizes, offs, offs, out_dtype=torch.float32)
    assert_allclose_gate(ref, out.float(), what="ragged-K matmul")
