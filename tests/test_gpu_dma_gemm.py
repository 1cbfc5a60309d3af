"""GPU parity of the expert GEMM that stages both operands by memory-to-LDS transfers (bf16, fp16, e4m3; row blocks of 128 and 256)
against the CPU oracle, at the sizes where it can go wrong: row blocks that are empty, nearly empty, nearly and exactly
full; one stage of K, a stage and a remainder, more stages than LDS buffers; columns around the tile; all its slice registers."""
import pytest
import torch

from oracle import moe as omoe
from oracle.checks import assert_allclose_gate

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 31, 33, 127, 128, 129, 0, 255, 256, 257, 390]


def _check(device, dtype, block_m, sizes, k, n, swiglu=False):
    import triton_amd.matmul as mm
    from triton_amd.swiglu import swiglu_fn
    from triton_amd.tensor import convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
    from triton_amd.tensor_details.layout import make_default_matmul_fp8_w_layout
    g = torch.Generator().manual_seed(k * 7 + n)
    E, m = len(sizes), sum(sizes)
    sizes = torch.tensor(sizes, dtype=torch.int32)
    x, w = torch.randn((m, k), generator=g), torch.randn((E, n, k), generator=g) * 0.1
    bias, gam = torch.randn((E, n), generator=g), torch.rand((m, ), generator=g) + 0.5
    gi, sc = torch.randint(0, m, (m, ), generator=g).to(torch.int32), torch.randperm(m, generator=g).to(torch.int32)
    pc, scales = mm.PrecisionConfig(), {}
    if dtype == "e4m3":
        scales = dict(x_row_scale=torch.rand((m, ), generator=g) + 0.5, w_col_scale=torch.rand((E, n), generator=g) + 0.5)
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn).transpose(1, 2)
        w_dev = convert_layout(wrap_torch_tensor(w.transpose(1, 2).contiguous().to(device).transpose(1, 2)), make_default_matmul_fp8_w_layout())
        pc = mm.PrecisionConfig(a_mx_tensor_scale=scales["x_row_scale"].to(device), b_mx_tensor_scale=scales["w_col_scale"].to(device),
                                out_dtype=torch.bfloat16)
        out_dtype = torch.bfloat16
    else:
        out_dtype = getattr(torch, dtype)
        x, w = x.to(out_dtype), w.to(out_dtype).transpose(1, 2)
        w_dev = w.transpose(1, 2).contiguous().to(device).transpose(1, 2)
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None
    out = torch.full((m, n // 2 if swiglu else n), float("nan"), dtype=out_dtype, device=device)
    with mm.scoped_opt_flags_constraints({"block_m": block_m}):
        mm.matmul(x.to(device), w_dev, bias.to(device), make_ragged_tensor_metadata(sizes.to(device), m), gather_indx=gi.to(device),
                  scatter_indx=sc.to(device), gammas=gam.to(device), precision_config=pc, fused_activation=act, c=out)
    ref = omoe.matmul(x, w, bias, sizes, gather_indx=gi, out_dtype=torch.float32, **scales)
    ref = (omoe.swiglu(ref, 1.702, 7.0).float() if swiglu else ref) * gam[:, None]
    want = torch.empty_like(ref)
    want[sc.long()] = ref
    assert_allclose_gate(want, out, what=f"{dtype} block_m {block_m}")


@pytest.mark.parametrize("k, n", [(32, 8), (64, 264), (208, 520), (1040, 248)])
@pytest.mark.parametrize("block_m", [128, 256])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "e4m3"])
def test_tile_and_stage_edges(device, dtype, block_m, k, n):
    _check(device, dtype, block_m, SIZES, k, n)


@pytest.mark.parametrize("block_m", [128, 256])
@pytest.mark.parametrize("dtype", ["bfloat16", "e4m3"])
def test_swiglu(device, dtype, block_m):
    _check(device, dtype, block_m, SIZES, 272, 528, swiglu=True)


@pytest.mark.parametrize("n_slices", [64, 65, 256, 257])
def test_slice_registers(device, n_slices):
    """257 slices run on the kernel without registers for them."""
    _check(device, "e4m3", 128, [(i * 37) % 9 for i in range(n_slices)], 192, 160)
    _check(device, "bfloat16", 128, [(i * 37) % 9 for i in range(n_slices)], 192, 160)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("stride", [0, 8, 56])
def test_overlapping_rows(device, monkeypatch, dtype, stride):
    """Rows closer together than their length (one row expanded, sliding windows) with as many of them per slice as take row blocks of
    256 otherwise: they run on the general kernel, from the native host path and from the general one, gathered and not."""
    import triton_amd.matmul as mm
    from triton_amd import _native as nt
    from triton_amd.tensor import make_ragged_tensor_metadata
    g = torch.Generator().manual_seed(stride)
    sizes, k, n = torch.tensor([300, 0, 129, 400], dtype=torch.int32), 64, 72
    m, out_dtype = int(sizes.sum()), getattr(torch, dtype)
    base = torch.randn((m * stride + k, ), generator=g).to(out_dtype)
    x, xd = base.as_strided((m, k), (stride, 1)), base.to(device).as_strided((m, k), (stride, 1))
    w = (torch.randn((4, n, k), generator=g) * 0.1).to(out_dtype)
    wd = w.to(device).transpose(1, 2)
    md = make_ragged_tensor_metadata(sizes.to(device), m)
    for gi in (None, torch.randint(0, m, (m, ), generator=g).to(torch.int32)):
        gd = None if gi is None else gi.to(device)
        want = omoe.matmul(x, w.transpose(1, 2), None, sizes, gather_indx=gi, out_dtype=torch.float32)
        native = mm.matmul(xd, wd, None, md, gather_indx=gd)
        with monkeypatch.context() as p:
            p.setattr(nt, "host", lambda: None)
            general = mm.matmul(xd, wd, None, md, gather_indx=gd)
        assert_allclose_gate(want, native, what=f"{dtype} row stride {stride}")
        assert torch.equal(native, general)
    assert_allclose_gate(omoe.matmul(x, w[:1].transpose(1, 2), None, torch.tensor([m], dtype=torch.int32), out_dtype=torch.float32),
                         mm.matmul(xd, wd[:1], None), what="not ragged")


@pytest.mark.parametrize("sizes", [[300, 0, 129, 400], [1100, 1030, 1000]])
@pytest.mark.parametrize("stride", [0, 16])
def test_overlapping_rows_tiled_e4m3(device, monkeypatch, sizes, stride):
    """The same with tiled e4m3 weights, on the kernel that takes rows anywhere: row blocks of 128, and from 1024 rows per slice on of 256."""
    import triton_amd.matmul as mm
    from triton_amd import _native as nt
    from triton_amd.tensor import convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
    from triton_amd.tensor_details.layout import make_default_matmul_fp8_w_layout
    g = torch.Generator().manual_seed(stride + len(sizes))
    E, m, k, n = len(sizes), sum(sizes), 272, 72
    sizes = torch.tensor(sizes, dtype=torch.int32)
    base = torch.randn((m * stride + k, ), generator=g).to(torch.float8_e4m3fn)
    x, xd = base.as_strided((m, k), (stride, 1)), base.to(device).as_strided((m, k), (stride, 1))
    w = (torch.randn((E, n, k), generator=g) * 0.1).to(torch.float8_e4m3fn)
    wd = convert_layout(wrap_torch_tensor(w.to(device).transpose(1, 2)), make_default_matmul_fp8_w_layout())
    gi, pc, md = torch.randint(0, m, (m, ), generator=g).to(torch.int32), mm.PrecisionConfig(out_dtype=torch.bfloat16), make_ragged_tensor_metadata(sizes.to(device), m)
    native = mm.matmul(xd, wd, None, md, gather_indx=gi.to(device), precision_config=pc)
    with monkeypatch.context() as p:
        p.setattr(nt, "host", lambda: None)
        general = mm.matmul(xd, wd, None, md, gather_indx=gi.to(device), precision_config=pc)
    want = omoe.matmul(x.contiguous(), w.transpose(1, 2), None, sizes, gather_indx=gi, out_dtype=torch.float32)
    assert_allclose_gate(want, native, what=f"e4m3 row stride {stride}")
    assert torch.equal(native, general)


@pytest.mark.parametrize("dtype", ["bfloat16", "e4m3"])
def test_few_large_tiles_run_as_small_ones(device, monkeypatch, dtype):
    """Where the rows say 256 x 256 and the chip would have few such tiles: the unforced choice against the oracle and, bit for bit, against
    the small tiles asked for by name, from both host paths."""
    import triton_amd.matmul as mm
    from triton_amd import _native as nt
    from triton_amd.tensor import convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
    from triton_amd.tensor_details.layout import make_default_matmul_fp8_w_layout
    g = torch.Generator().manual_seed(11)
    sizes, k, n = torch.tensor([0, 250, 700, 129, 513], dtype=torch.int32), 272, 264
    m, e = int(sizes.sum()), len(sizes)
    assert nt.rules().dma_block_m(m, k, n, e) == 256 and nt.rules().dma_block_n(m, n, e, 256) == 128
    dt = torch.bfloat16 if dtype == "bfloat16" else torch.float8_e4m3fn
    x, w = torch.randn((m, k), generator=g).to(dt), (torch.randn((e, n, k), generator=g) * 0.1).to(dt)
    wd = w.to(device).transpose(1, 2)
    wd = wd if dtype == "bfloat16" else convert_layout(wrap_torch_tensor(wd), make_default_matmul_fp8_w_layout())
    md, pc = make_ragged_tensor_metadata(sizes.to(device), m), mm.PrecisionConfig(out_dtype=torch.bfloat16)
    native = mm.matmul(x.to(device), wd, None, md, precision_config=pc)
    with monkeypatch.context() as p:
        p.setattr(nt, "host", lambda: None)
        general = mm.matmul(x.to(device), wd, None, md, precision_config=pc)
    with mm.scoped_opt_flags_constraints({"block_m": 128}):
        small = mm.matmul(x.to(device), wd, None, md, precision_config=pc)
    assert_allclose_gate(omoe.matmul(x, w.transpose(1, 2), None, sizes, out_dtype=torch.float32), native, what=f"{dtype} few large tiles")
    assert torch.equal(native, general) and torch.equal(native, small)


@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("k", [32, 160, 272, 400])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "e4m3"])
def test_narrow_tiles_of_short_row_blocks(device, dtype, k, swiglu):
    """256 full tiles, one round, and short row blocks of 1, 128, 64 and 31 rows in tiles of 128 columns behind them: an odd and an even number of
    stages' halves, and less than one."""
    _check(device, dtype, 256, [257, 384, 320, 0, 31, 256, 256, 512, 256], k, 8184, swiglu=swiglu)


# slices, K, N, sizes dealt in turn: what the rules name at row blocks of 320 rows (one less, all of them, one more; half of one, which makes a short
# block of what is left, and one more; none), at K of less than a stage, one, a remainder behind one, an odd and an even number, columns around the tile and a wave's
TALL = [
    ("320x128", 16, 40, 2040, [320, 256, 161, 321, 0, 319, 288, 257, 224]),
    ("320x128", 16, 136, 1608, [160, 256, 481, 1, 289]),
    ("320x128", 8, 320, 2048, [320, 640, 480, 641, 479]),
    ("320x256", 16, 64, 2312, [320, 320, 161, 321, 0, 319, 288, 319, 321, 320, 289]),
    ("320x256", 16, 72, 2056, [160, 320, 481, 1, 320, 320]),
    ("320x256", 32, 448, 1344, [256, 240, 272, 288, 255]),
]


@pytest.mark.parametrize("tile, e, k, n, sizes", TALL)
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("swiglu, routed", [(True, True), (False, False), (False, True)])
def test_tiles_of_320_rows(device, monkeypatch, tile, e, k, n, sizes, dtype, swiglu, routed):
    """The tile of 320 rows that the rules name gives, bit for bit, what row blocks of 128 give (whose sums over K run in the same order), from both
    host paths: gathered and scattered rows, gate weights, rows without a destination.  (Not compared with row blocks of 256: where their last tile hangs over N
    the compiler contracts bias and gate weight differently, and one value in 100000 is the neighbouring fp16 number.)"""
    import triton_amd.matmul as mm
    from triton_amd import _native as nt
    from triton_amd.swiglu import swiglu_fn
    from triton_amd.tensor import make_ragged_tensor_metadata
    g = torch.Generator(device=device).manual_seed(k + n)
    sizes = torch.tensor([sizes[i % len(sizes)] for i in range(e)], dtype=torch.int32, device=device)
    m, dt = int(sizes.sum()), getattr(torch, dtype)
    assert nt.rules().dma_block_m(m, 2 * k, n, e) == 256 and nt.rules().dma_block_n_16bit(m, n, e, 256) == int(tile.split("x")[1])
    x = torch.randn((m, k), generator=g, device=device).to(dt)
    w = (torch.randn((e, n, k), generator=g, device=device) * 0.1).to(dt).transpose(1, 2)
    args = dict(fused_activation=mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None)
    if routed:
        args.update(gammas=torch.rand((m, ), generator=g, device=device) + 0.5, gather_indx=torch.randint(0, m, (m, ), generator=g, device=device).to(torch.int32),
                    scatter_indx=torch.randperm(m, generator=g, device=device).to(torch.int32))
        args["scatter_indx"][::7] = -1
    bias, md = torch.randn((e, n), generator=g, device=device), make_ragged_tensor_metadata(sizes, m)

    def run():
        return mm.matmul(x, w, bias, md, c=torch.zeros((m, n // 2 if swiglu else n), dtype=dt, device=device), **args).clone()
    by_rule = run()
    with monkeypatch.context() as p:
        p.setattr(nt, "host", lambda: None)
        general = run()
    with mm.scoped_opt_flags_constraints({"block_m": 128}):
        want = run()
    assert torch.equal(by_rule, want) and torch.equal(general, want)
    assert not torch.isnan(want).any() and want.any()


@pytest.mark.parametrize("e, k, n, sizes", [
    (16, 136, 2048, [1100, 20, 0, 511, 130, 1, 700, 31, 257, 640, 90, 320, 5, 0, 33, 258]),  # where 320 x 128 is more than a round
    (32, 72, 2312, [700, 129, 1, 384, 0, 256, 33, 512]),                                     # 320 x 256: full square tiles, short ones beside them
    (16, 400, 4096, [257, 384, 320, 0, 31, 256, 512, 230]),                                  # ... and in narrow tiles behind them
])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("swiglu", [False, True])
def test_square_tiles_where_a_routing_divides_worse_into_tall_ones(device, dtype, e, k, n, sizes, swiglu):
    """The rows that a tile of 320 is meant for, dealt so that the kernel goes by 256 x 256 tiles: against the oracle on a row of every row block's kind."""
    import triton_amd.matmul as mm
    from triton_amd import _native as nt
    from triton_amd.swiglu import swiglu_fn
    from triton_amd.tensor import make_ragged_tensor_metadata
    sizes = [sizes[i % len(sizes)] for i in range(e)]
    m, dt = sum(sizes), getattr(torch, dtype)
    cols = nt.rules().dma_block_n_16bit(m, n, e, 256)
    assert cols in (128, 256)
    tall, square = (sum(-(-s // b) for s in sizes) * -(-n // c) / 256 for b, c in ((320, cols), (256, 256)))  # rounds on 256 compute units
    assert (tall > 1) if cols == 128 else 0.73 * square < (tall if tall < 1 else int(tall) + (0.43 if tall > int(tall) else 0))
    g = torch.Generator(device=device).manual_seed(k + n)
    x = torch.randn((m, k), generator=g, device=device).to(dt)
    w = (torch.randn((e, n, k), generator=g, device=device) * 0.1).to(dt).transpose(1, 2)
    bias, gam = torch.randn((e, n), generator=g, device=device), torch.rand((m, ), generator=g, device=device) + 0.5
    gi, sc = torch.randint(0, m, (m, ), generator=g, device=device).to(torch.int32), torch.randperm(m, generator=g, device=device).to(torch.int32)
    act = mm.FusedActivation(mm.FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0)) if swiglu else None
    out = torch.full((m, n // 2 if swiglu else n), float("nan"), dtype=dt, device=device)
    mm.matmul(x, w, bias, make_ragged_tensor_metadata(torch.tensor(sizes, dtype=torch.int32, device=device), m), gather_indx=gi, scatter_indx=sc, gammas=gam, fused_activation=act, c=out)
    assert not torch.isnan(out).any()
    first = [sum(sizes[:i]) for i in range(e)]
    pick = sorted({r for i, s in enumerate(sizes) for r in (first[i], first[i] + s // 2, first[i] + s - 1) if s})
    counts = torch.tensor([sum(first[i] <= r < first[i] + s for r in pick) for i, s in enumerate(sizes)], dtype=torch.int32)
    rows = torch.tensor(pick)
    ref = omoe.matmul(x.cpu(), w.cpu(), bias.cpu(), counts, gather_indx=gi.cpu()[rows], out_dtype=torch.float32)
    ref = (omoe.swiglu(ref, 1.702, 7.0).float() if swiglu else ref) * gam.cpu()[rows][:, None]
    assert_allclose_gate(ref, out.cpu()[sc.cpu()[rows].long()], what=f"{dtype} square tiles")


@pytest.mark.parametrize("sizes", [[0, 1, 31, 32, 33, 63, 64, 40], [2, 0, 31, 33, 64, 65, 129, 2], [5], [96, 97, 128, 161, 192, 1, 0, 95]])
@pytest.mark.parametrize("k, n", [(32, 8), (144, 264), (528, 1032), (1040, 72)])
@pytest.mark.parametrize("dtype, swiglu", [("e4m3", False), ("e4m3", True), ("bfloat16", True), ("float16", False)])
def test_narrow_tiles_of_few_rows(device, sizes, k, n, dtype, swiglu):
    """Few rows a slice, or few tiles in all: row blocks of 64 by 64 columns and twice the K a stage."""
    _check(device, dtype, 128, sizes, k, n, swiglu=swiglu)


@pytest.mark.parametrize("k, n", [(32, 1032), (208, 1288), (528, 1032)])
@pytest.mark.parametrize("dtype, swiglu", [("e4m3", False), ("bfloat16", False), ("bfloat16", True), ("float16", False)])
def test_tiles_of_128_columns(device, k, n, dtype, swiglu):
    """More columns than the small tiles are for: the row blocks of 128 at the edges of tiles and stages."""
    _check(device, dtype, 128, SIZES, k, n, swiglu=swiglu)


@pytest.mark.parametrize("dtype", ["bfloat16", "e4m3"])
def test_small_tiles_of_one_round(device, monkeypatch, dtype):
    """More large tiles than the chip would leave CUs without, but one round of small ones: both host paths choose these, whose results are those of small
    tiles asked for by name, bit for bit, and agree with the oracle."""
    import triton_amd.matmul as mm
    from triton_amd import _native as nt
    from triton_amd.tensor import convert_layout, make_ragged_tensor_metadata, wrap_torch_tensor
    from triton_amd.tensor_details.layout import make_default_matmul_fp8_w_layout
    g = torch.Generator().manual_seed(12)
    sizes, k, n = torch.tensor([272, 250, 300, 129, 400, 256, 257, 320], dtype=torch.int32), 48, 2056
    m, e = int(sizes.sum()), len(sizes)
    assert nt.rules().dma_block_m(m, k, n, e) == 256 and nt.rules().dma_block_n(m, n, e, 256) == 128 and nt.rules().dma_block_n_16bit(m, n, e, 256) == 128
    assert nt.rules().dma_block_n(m, 2 * n, e, 256) == 0
    dt = torch.bfloat16 if dtype == "bfloat16" else torch.float8_e4m3fn
    x, w = torch.randn((m, k), generator=g).to(dt), (torch.randn((e, n, k), generator=g) * 0.1).to(dt)
    wd = w.to(device).transpose(1, 2)
    wd = wd if dtype == "bfloat16" else convert_layout(wrap_torch_tensor(wd), make_default_matmul_fp8_w_layout())
    md, pc = make_ragged_tensor_metadata(sizes.to(device), m), mm.PrecisionConfig(out_dtype=torch.bfloat16)
    native = mm.matmul(x.to(device), wd, None, md, precision_config=pc)
    with monkeypatch.context() as p:
        p.setattr(nt, "host", lambda: None)
        general = mm.matmul(x.to(device), wd, None, md, precision_config=pc)
    with mm.scoped_opt_flags_constraints({"block_m": 128}):
        small = mm.matmul(x.to(device), wd, None, md, precision_config=pc)
    assert_allclose_gate(omoe.matmul(x, w.transpose(1, 2), None, sizes, out_dtype=torch.float32), native, what=f"{dtype} small tiles")
    assert torch.equal(native, general) and torch.equal(native, small)
