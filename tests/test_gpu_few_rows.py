"""GPU parity of the expert GEMM for few rows per expert (bf16, fp16; 32 or 64 columns a workgroup) against the CPU oracle, where the rule
takes it: row blocks that are empty, around every number of 16-row fragments, full and walked more than once; one chunk of K, fewer chunks
than waves, a remainder, more chunks than buffers; columns around a workgroup's; the epilogue's options; with and without ragged metadata."""
import pytest
import torch

from oracle import moe as omoe
from oracle.checks import assert_allclose_gate

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 250, 0, 20, 20, 20]  # 650 rows of 16 slices: the 250 are walked in turns


def _operands(sizes, k, n, dtype):
    g = torch.Generator().manual_seed(k * 7 + n)
    e, m = len(sizes), sum(sizes)
    x, w = torch.randn((m, k), generator=g).to(dtype), (torch.randn((e, n, k), generator=g) * 0.1).to(dtype)
    bias, gam = torch.randn((e, n), generator=g), torch.rand((m, ), generator=g) + 0.5
    gi, sc = torch.randint(0, m, (m, ), generator=g).to(torch.int32), torch.randperm(m, generator=g).to(torch.int32)
    return torch.tensor(sizes, dtype=torch.int32), x, w, bias, gam, gi, sc


@pytest.fixture
def columns(monkeypatch):
    """The columns a workgroup that each call of the library's GEMM entry asks for, by either host path."""
    import ctypes

    from triton_amd import _native as nt
    real, seen = nt.lib(), []

    @ctypes.CFUNCTYPE(ctypes.c_int32, ctypes.POINTER(nt.GemmDesc), ctypes.c_void_p)
    def entry(d, stream):
        seen.append(d.contents.block_n)
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


@pytest.mark.parametrize("k, n, block_n", [(8, 8, 32), (64, 250, 32), (136, 520, 64), (200, 256, 32), (520, 776, 64), (1032, 40, 32)])
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tile_and_chunk_edges(device, monkeypatch, columns, dtype, swiglu, k, n, block_n):
    import triton_amd.matmul as mm
    from triton_amd import _native as nt
    from triton_amd.swiglu import swiglu_fn
    from triton_amd.tensor import make_ragged_tensor_metadata
    sizes, x, w, bias, gam, gi, sc = _operands(SIZES, k, n, dtype)
    m = x.shape[0]
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None
    wd = w.to(device).transpose(1, 2)
    md = make_ragged_tensor_metadata(sizes.to(device), m)

    def run():
        return mm.matmul(x.to(device), wd, bias.to(device), md, gather_indx=gi.to(device), scatter_indx=sc.to(device), gammas=gam.to(device), fused_activation=act)
    native = run()
    with monkeypatch.context() as p:
        p.setattr(nt, "host", lambda: None)
        general = run()
    assert columns == [block_n] * 2
    ref = omoe.matmul(x, w.transpose(1, 2), bias, sizes, gather_indx=gi, out_dtype=torch.float32)
    ref = (omoe.swiglu(ref, 1.702, 7.0).float() if swiglu else ref) * gam[:, None]
    want = torch.empty_like(ref)
    want[sc.long()] = ref
    assert_allclose_gate(want, native, what=f"{dtype} K {k} N {n}")
    assert torch.equal(native, general)


@pytest.mark.parametrize("n", [24, 520])
def test_epilogue_options(device, columns, n):
    """betas, out_alpha, an accumulator to add, rows that go nowhere, an output of wider rows; scales per row and column."""
    import triton_amd.matmul as mm
    from triton_amd.tensor import make_ragged_tensor_metadata
    sizes, x, w, bias, gam, gi, sc = _operands(SIZES, 520, n, torch.bfloat16)
    m = x.shape[0]
    g = torch.Generator().manual_seed(n)
    betas, acc = torch.rand((m, ), generator=g) + 0.5, torch.randn((m, n), generator=g).to(torch.bfloat16)
    wide = torch.full((m, n + 3), float("nan"), dtype=torch.bfloat16, device=device)  # (rows that take no vector stores)
    md = make_ragged_tensor_metadata(sizes.to(device), m)
    args = (x.to(device), w.to(device).transpose(1, 2), bias.to(device), md)
    mm.matmul(*args, gammas=gam.to(device), betas=betas.to(device), out_alpha=0.75, c_acc_in=acc.to(device), c=wide[:, :n])
    ref = omoe.matmul(x, w.transpose(1, 2), None, sizes, out_dtype=torch.float32)
    rows = torch.repeat_interleave(torch.arange(len(SIZES)), sizes.long())
    want = (ref + bias[rows] * betas[:, None]) * 0.75 * gam[:, None] + acc.float()
    assert_allclose_gate(want, wide[:, :n], what="betas, out_alpha, c_acc_in")
    assert torch.isnan(wide[:, n:]).all()
    sc[::5] = -1
    out = torch.full((m, n), 7.0, dtype=torch.bfloat16, device=device)
    mm.matmul(*args, scatter_indx=sc.to(device), c=out)
    want = torch.full((m, n), 7.0)
    want[sc[sc >= 0].long()] = (ref + bias[rows])[sc >= 0]
    assert_allclose_gate(want, out, what="rows that go nowhere")
    row, col = torch.rand((m, ), generator=g) + 0.5, torch.rand((len(SIZES), n), generator=g) + 0.5
    pc = mm.PrecisionConfig(a_mx_tensor_scale=row.to(device), b_mx_tensor_scale=col.to(device))
    assert_allclose_gate(ref * row[:, None] * col[rows] + bias[rows], mm.matmul(*args, precision_config=pc), what="scales per row and column")
    assert columns == [32 if n == 24 else 64] * 3


def test_not_ragged_and_idle_units(device, columns):
    """One slice without metadata; with compute units to leave idle another kernel runs."""
    import triton_amd.matmul as mm
    _, x, w, bias, _, _, _ = _operands([60], 640, 136, torch.float16)
    want = omoe.matmul(x, w.transpose(1, 2), bias, torch.tensor([60], dtype=torch.int32), out_dtype=torch.float32)
    args = (x.to(device), w.to(device).transpose(1, 2), bias.to(device))
    assert_allclose_gate(want, mm.matmul(*args), what="not ragged")
    mm.matmul_set_idle_sms(8)
    try:
        assert_allclose_gate(want, mm.matmul(*args), what="idle units")
    finally:
        mm.matmul_set_idle_sms(0)
    assert columns == [32, 0]
