"""Host-side mirror of the reference's operator interface: names, data classes, layouts, tile constraints and
the argument checks that run before any kernel is launched.  CPU only."""
import importlib

import pytest
import torch

import triton_kernels  # noqa: F401  (alias package: triton_kernels.X is triton_amd.X)
from triton_kernels.matmul_details import opt_flags as of
from triton_kernels.tensor import (BIT, FP4, UINT8, RaggedTensorMetadata, Tensor, convert_layout, empty, wrap_torch_tensor)
from triton_kernels.tensor_details.layout import StridedLayout
from triton_kernels.tensor_details.layout_details.strided import repack


def test_reference_module_names_resolve():
    # the import lines of the reference's benchmark and tests (bench/bench_mlp.py:1-25, tests/test_matmul.py:1-40)
    names = {
        "triton_kernels.matmul": ["matmul", "PrecisionConfig", "FlexCtx", "FnSpecs", "FusedActivation", "Epilogue"],
        "triton_kernels.topk": ["topk"],
        "triton_kernels.reduce": ["reduce"],
        "triton_kernels.swiglu": ["swiglu", "swiglu_fn", "PrecisionConfig"],
        "triton_kernels.numerics_details.mxfp": ["downcast_to_mxfp", "upcast_from_mxfp", "DequantScaleRoundingMode", "MXFP_BLOCK_SIZE"],
        "triton_kernels.tensor": ["SparseMatrix", "RaggedTensor", "make_ragged_tensor_metadata", "make_bitmatrix_metadata", "wrap_torch_tensor",
                                  "convert_layout", "FP4", "Tensor", "Storage"],
        "triton_kernels.tensor_details.layout": ["StridedLayout", "make_default_matmul_mxfp4_w_layout", "make_default_matmul_mxfp4_w_scale_layout"],
        "triton_kernels.matmul_details.opt_flags": ["make_opt_flags", "scoped_opt_flags_constraints", "update_opt_flags_constraints",
                                                    "reset_opt_flags_constraints", "InapplicableConstraint", "OptFlags"],
        "triton_kernels.legacy": ["routing", "RoutingData", "GatherIndx", "ScatterIndx", "matmul_ogs"],
        "triton_kernels.target_info": ["is_hip", "is_hip_cdna4", "is_cuda"],
    }
    for mod, attrs in names.items():
        m = importlib.import_module(mod)
        for a in attrs:
            assert hasattr(m, a), f"{mod}.{a}"
    import triton_amd.matmul
    assert importlib.import_module("triton_kernels.matmul") is triton_amd.matmul


@pytest.mark.parametrize(("logical_shape", "is_fp4", "layout", "storage_shape"), [
    ((3, 258, 514), True, StridedLayout(-2), [3, 129, 514]),
    ((0, 64), True, StridedLayout(-2), [0, 64]),
    ((3, 258, 514), True, StridedLayout(-1), [3, 258, 257]),
    ((3, 70, 65), False, StridedLayout(-2), [3, 70, 65]),
])
def test_layout_storage_shape_matches_conversion(logical_shape, is_fp4, layout, storage_shape):
    # tests/test_tensor.py:85-118 (the strided rows of its table)
    t = empty(logical_shape, dtype=FP4 if is_fp4 else UINT8, device="meta")
    converted = convert_layout(t, layout)
    assert layout.storage_shape(list(logical_shape), is_fp4) == storage_shape
    assert list(converted.storage.data.shape) == storage_shape


@pytest.mark.parametrize("major_dim", [-1, -2])
@pytest.mark.parametrize("other_size", [0, 2])
def test_strided_layout_rejects_odd_fp4_packing_dim(major_dim, other_size):
    # tests/test_tensor.py:128-135
    shape = [other_size, other_size]
    shape[major_dim] = 1
    with pytest.raises(ValueError):
        StridedLayout(major_dim).storage_shape(shape, True)


def test_strided_layout_order_and_errors():
    assert StridedLayout(-1).order(3) == [2, 1, 0]
    assert StridedLayout(-2).order(3) == [1, 2, 0]
    assert StridedLayout(0).order(3) == [0, 1, 2]
    with pytest.raises(ValueError):
        StridedLayout(3).order(3)
    with pytest.raises(TypeError):
        StridedLayout("k")


def test_wrap_fp4_doubles_the_unit_stride_dim():
    # tensor.py:216-233: uint8 storage of FP4 has two elements per byte along the contiguous dimension
    w = torch.zeros((4, 16, 6), dtype=torch.uint8).transpose(1, 2).contiguous().transpose(1, 2)  # strides (96, 1, 16)
    t = wrap_torch_tensor(w, dtype=FP4)
    assert t.shape == [4, 32, 6] and t.storage.layout == StridedLayout(-2)
    t = wrap_torch_tensor(torch.zeros((4, 16, 6), dtype=torch.uint8), dtype=FP4)
    assert t.shape == [4, 16, 12] and t.storage.layout == StridedLayout(-1)
    with pytest.raises(ValueError):
        Tensor(t.storage, dtype=FP4)  # sub-byte types need an explicit shape
    assert BIT.bitwidth == 1 and FP4.bitwidth == 4


def test_repack_moves_nibbles_between_dims():
    g = torch.Generator().manual_seed(0)
    vals = torch.randint(0, 16, (3, 8, 6), generator=g, dtype=torch.uint8)  # one nibble per logical element
    pack_last = vals[..., 0::2] | (vals[..., 1::2] << 4)  # [3, 8, 3]
    pack_mid = vals[:, 0::2, :] | (vals[:, 1::2, :] << 4)  # [3, 4, 6]
    assert torch.equal(repack(pack_last, -1, -2, True), pack_mid)
    assert torch.equal(repack(pack_mid, -2, -1, True), pack_last)
    assert repack(pack_last, -1, -1, True) is pack_last
    with pytest.raises(TypeError):
        repack(pack_last.to(torch.float32), -1, -2, True)


def test_convert_layout_round_trip_fp4():
    g = torch.Generator().manual_seed(1)
    data = torch.randint(0, 256, (2, 6, 8), generator=g, dtype=torch.uint8)
    t = wrap_torch_tensor(data, dtype=FP4)  # logical [2, 6, 16], packed along the last dim
    k_major = convert_layout(t, StridedLayout(-2))
    assert list(k_major.storage.data.shape) == [2, 3, 16] and k_major.storage.data.stride(1) == 1
    back = convert_layout(k_major, StridedLayout(-1))
    assert torch.equal(back.storage.data, data)
    assert convert_layout(t, StridedLayout(-1)) is t


def test_ragged_metadata_static_helpers():
    # ragged_tensor.py:73-89
    assert RaggedTensorMetadata.block_sizes() == [16, 32, 64, 128, 256]
    assert RaggedTensorMetadata.n_blocks(128, 16384, 16) == 1144
    assert RaggedTensorMetadata.max_n_blocks(128, 16384) == 1144
    assert RaggedTensorMetadata.n_blocks(8, 3, 64) == 3


def test_opt_flags_constraints_scope_and_tiles():
    of.reset_opt_flags_constraints()
    flags = of.make_opt_flags(None, None, FP4, None, 1, 16384, 5760, 2880, None)
    assert (flags.block_m, flags.block_n, flags.block_k, flags.split_k, flags.is_persistent) == (128, 256, 128, 1, False)
    with of.scoped_opt_flags_constraints({"block_m": 16}):
        f = of.make_opt_flags(None, None, FP4, None, 1, 16384, 5760, 2880, None)
        assert (f.block_m, f.block_n, f.block_k) == (16, 128, 256)
        f = of.make_opt_flags(None, None, torch.bfloat16, None, 1, 16384, 5760, 2880, None)
        assert (f.block_m, f.block_n, f.block_k) == (16, 128, 128)
        with of.scoped_opt_flags_constraints({"block_n": 64}):
            with pytest.raises(of.InapplicableConstraint):
                of.make_opt_flags(None, None, FP4, None, 1, 64, 64, 64, None)
    assert of._get_opt_flags_constraints() == {}
    for bad in ({"is_persistent": True}, {"split_k": 4}, {"block_m": 48}, {"max_allowable_mn": 1024}):
        with of.scoped_opt_flags_constraints(bad):
            with pytest.raises(of.InapplicableConstraint):
                of.make_opt_flags(None, None, FP4, None, 1, 64, 64, 64, None)
    with of.scoped_opt_flags_constraints({"no_such_knob": 1}):
        with pytest.raises(AssertionError):
            of.make_opt_flags(None, None, FP4, None, 1, 64, 64, 64, None)
    of.update_opt_flags_constraints({"block_m": 32})
    assert of.make_opt_flags(None, None, FP4, None, 1, 4096, 64, 64, None).block_m == 32
    of.reset_opt_flags_constraints()


def test_default_block_m_follows_rows_per_expert():
    class Md:
        n_slices = 128
        expected_slice_size = None

    assert of.default_block_m(16384, Md()) == 128
    assert of.default_block_m(64 * 4, Md()) == 16
    assert of.default_block_m(40, None) == 64
    Md.expected_slice_size = 20
    assert of.default_block_m(16384, Md()) == 32


def test_constraints_are_per_context():
    import contextvars
    of.reset_opt_flags_constraints()

    def inner():
        of.update_opt_flags_constraints({"block_m": 64})
        return of._get_opt_flags_constraints()

    assert contextvars.copy_context().run(inner) == {"block_m": 64}
    assert of._get_opt_flags_constraints() == {}


def test_cpu_tensors_are_refused_not_computed():
    # there is no CPU path: every operator refuses host tensors before doing anything
    from triton_kernels.matmul import matmul
    from triton_kernels.numerics_details.mxfp import downcast_to_mxfp, upcast_from_mxfp
    from triton_kernels.reduce import reduce
    from triton_kernels.swiglu import PrecisionConfig, swiglu
    from triton_kernels.topk import topk
    x = torch.zeros((32, 64), dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="HIP device"):
        matmul(x, torch.zeros((64, 32), dtype=torch.bfloat16), None)
    with pytest.raises(RuntimeError, match="HIP device"):
        topk(torch.zeros((4, 8)), 2)
    with pytest.raises(RuntimeError, match="HIP device"):
        downcast_to_mxfp(x, torch.uint8, axis=1)
    with pytest.raises(RuntimeError, match="HIP device"):
        upcast_from_mxfp(torch.zeros((32, 32), dtype=torch.uint8), torch.zeros((32, 2), dtype=torch.uint8), torch.bfloat16, axis=1)
    with pytest.raises(RuntimeError, match="HIP device"):
        swiglu(x, 1.0, PrecisionConfig(limit=None))
    with pytest.raises(RuntimeError, match="HIP device"):
        reduce(x.view(16, 2, 64), dim=1)


def test_mx_argument_checks_match_the_reference():
    # mxfp.py:39-47: axis range and divisibility are checked before any work
    from triton_kernels.numerics_details.mxfp import downcast_to_mxfp
    with pytest.raises((AssertionError, ValueError)):
        downcast_to_mxfp(torch.zeros((4, 8), dtype=torch.bfloat16), torch.uint8, axis=2)
    with pytest.raises((AssertionError, ValueError)):
        downcast_to_mxfp(torch.zeros((4, 7), dtype=torch.bfloat16), torch.uint8, axis=1)


def test_weight_relayout_cache_key_and_invalidation():
    """The K-contiguous copy `matmul` keeps on an N-contiguous weight tensor follows in-place torch updates through the
    version counter; writes through `.data` do not bump it (checked here), so `invalidate_weight_cache` is the
    documented way to drop the copy after such a write.  Inference-mode tensors have no counter and must not raise."""
    from triton_amd.matmul import _cache_key, _k_contiguous, invalidate_weight_cache
    w = torch.randn(2, 8, 16)
    c0 = _k_contiguous(w)
    assert c0.stride(-2) == 1 and torch.equal(c0, w)
    assert _k_contiguous(w) is c0  # cached
    w.add_(1.0)  # visible to the version counter: a new copy
    c1 = _k_contiguous(w)
    assert c1 is not c0 and torch.equal(c1, w)
    v = w._version
    w.data.mul_(2.0)  # NOT visible
    assert w._version == v and _k_contiguous(w) is c1 and not torch.equal(c1, w)
    invalidate_weight_cache(w)
    c2 = _k_contiguous(w)
    assert c2 is not c1 and torch.equal(c2, w)
    # a different storage under the same Python object (set_) changes the key as well
    w.set_(torch.randn(2, 8, 16))
    assert torch.equal(_k_contiguous(w), w)
    with torch.inference_mode():
        wi = torch.randn(2, 8, 16)
    assert _cache_key(wi)[1] is None
    assert torch.equal(_k_contiguous(wi), wi)
    # already K-contiguous weights are used in place
    wk = torch.randn(2, 16, 8).transpose(1, 2)
    assert _k_contiguous(wk) is wk


def test_routing_data_records_whether_every_token_has_all_its_rows():
    from triton_amd.legacy import RoutingData
    assert RoutingData.__dataclass_fields__["all_rows_live"].default is False


@pytest.fixture
def gemm_calls(monkeypatch):
    """The descriptors `matmul` hands to the library, with host tensors in the place of device ones and nothing launched."""
    from triton_amd import _native as nt
    nt.rules()
    real, calls = nt.lib(), []

    class Recorder:
        def tk_moe_gemm(self, d, stream):
            calls.append({name: getattr(d, name) for name, _ in d._fields_})
            return nt.TK_OK

        def __getattr__(self, name):
            return getattr(real, name)

    recorder = Recorder()
    monkeypatch.setattr(nt, "lib", lambda: recorder)
    monkeypatch.setattr(nt, "require_gpu", lambda *_: None)
    monkeypatch.setattr(nt, "stream_ptr", lambda *_: 0)
    return calls


def _metadata(n_slices, rows):
    i32 = dict(dtype=torch.int32)
    width = RaggedTensorMetadata.max_n_blocks(n_slices, rows)
    return RaggedTensorMetadata(torch.zeros(n_slices, **i32), torch.zeros(n_slices + 1, **i32), torch.zeros((5, n_slices + 1), **i32),
                                torch.zeros((5, width), **i32))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ragged", [True, False])
def test_overlapping_rows_stay_off_the_256_row_blocks(gemm_calls, dtype, ragged):
    # rows closer together than their length: the kernel with row blocks of 256 does not run on them and the general one ends at 128
    from triton_amd.matmul import matmul, scoped_opt_flags_constraints
    n_slices, rows, k, n = (16, 4096, 512, 1024) if ragged else (1, 4096, 512, 1024)
    w = torch.zeros((n_slices, n, k), dtype=dtype).transpose(1, 2)
    md = _metadata(n_slices, rows) if ragged else None
    base = torch.zeros(rows * 512, dtype=dtype)
    for stride, want in ((512, 256), (0, 128), (256, 128), (504, 128)):
        x = base.as_strided((rows, k), (stride, 1))
        matmul(x, w, None, md)
        assert (gemm_calls[-1]["x_stride_m"], gemm_calls[-1]["block_m"]) == (stride, want)
        with scoped_opt_flags_constraints({"block_m": 256}):
            matmul(x, w, None, md)
        assert gemm_calls[-1]["block_m"] == want
    one = torch.zeros((1, k), dtype=dtype).expand(rows, k)
    matmul(one, w, None, md)
    assert gemm_calls[-1]["block_m"] == 128


def _tiled(kind, n_slices, k, n):
    from triton_amd.tensor_details import layout as L
    if kind == "fp8":
        w = torch.zeros((n_slices, n, k), dtype=torch.float8_e4m3fn).transpose(1, 2)
        return convert_layout(wrap_torch_tensor(w), L.make_default_matmul_fp8_w_layout()), None
    w, s = torch.zeros((n_slices, n, k // 2), dtype=torch.uint8).transpose(1, 2), torch.zeros((n_slices, n, k // 32), dtype=torch.uint8).transpose(1, 2)
    return (convert_layout(wrap_torch_tensor(w, dtype=FP4), L.make_default_matmul_mxfp4_w_layout(mx_axis=1)),
            convert_layout(wrap_torch_tensor(s), L.make_default_matmul_mxfp4_w_scale_layout(mx_axis=1)))


@pytest.mark.parametrize("kind, n_slices, per_slice, want, overlapping", [
    ("fp8", 4, 250, 256, 128), ("fp8", 4, 1023, 256, 128), ("fp8", 4, 1024, 256, 256), ("fp8", 4, 64, 128, 128), ("fp8", 257, 200, 128, 128),
    ("mxfp4", 16, 30, 64, 32), ("mxfp4", 16, 60, 128, 64), ("mxfp4", 16, 162, 256, 128), ("mxfp4", 257, 60, 64, 64),
    ("mxfp8", 16, 162, 256, 128), ("mxfp8", 16, 250, 128, 128), ("mxfp8", 257, 60, 256, 256),
])
def test_row_blocks_follow_the_kernel_that_runs(gemm_calls, kind, n_slices, per_slice, want, overlapping):
    # the rules measured for the kernels that address x through a buffer resource hold where those run (not with overlapping rows, not
    # with more than 256 slices); elsewhere the other kernels' own rules do
    from triton_amd.matmul import PrecisionConfig, matmul
    k, n, rows = 512, 64, n_slices * per_slice
    w, s = _tiled(kind, n_slices, k, n)
    dtype = torch.bfloat16 if kind == "mxfp4" else torch.float8_e4m3fn
    xs = torch.zeros((rows, k // 32), dtype=torch.uint8) if kind == "mxfp8" else None
    pc, md = PrecisionConfig(a_mx_scale=xs, b_mx_scale=s, out_dtype=torch.bfloat16), _metadata(n_slices, rows)
    for stride, block_m in ((k, want), (0, overlapping), (k - 16, overlapping)):
        matmul(torch.zeros(rows * k, dtype=dtype).as_strided((rows, k), (stride, 1)), w, None, md, precision_config=pc)
        assert (gemm_calls[-1]["x_stride_m"], gemm_calls[-1]["block_m"]) == (stride, block_m)


@pytest.mark.parametrize("kind, block_m", [("bf16", 16), ("bf16", 32), ("bf16", 64), ("bf16", 128), ("mxfp4", 16), ("mxfp4", 64), ("mxfp4", 128), ("fp8", 128)])
def test_a_callers_row_block_is_the_one_that_runs(gemm_calls, kind, block_m):
    # named by a constraint or by flags of the caller's own, where the rules would take 256
    import dataclasses
    from triton_amd.matmul import PrecisionConfig, matmul, scoped_opt_flags, scoped_opt_flags_constraints
    n_slices, rows, k, n = 4, 1000, 512, 64
    w, s = (torch.zeros((n_slices, n, k), dtype=torch.bfloat16).transpose(1, 2), None) if kind == "bf16" else _tiled(kind, n_slices, k, n)
    x = torch.zeros((rows, k), dtype=torch.float8_e4m3fn if kind == "fp8" else torch.bfloat16)
    pc, md = PrecisionConfig(b_mx_scale=s, out_dtype=torch.bfloat16), _metadata(n_slices, rows)
    matmul(x, w, None, md, precision_config=pc)
    assert gemm_calls[-1]["block_m"] == 256
    with scoped_opt_flags_constraints({"block_m": block_m}):
        matmul(x, w, None, md, precision_config=pc)
    assert gemm_calls[-1]["block_m"] == block_m
    flags = dataclasses.replace(of.make_opt_flags(torch.bfloat16, torch.bfloat16, torch.bfloat16, pc, 1, rows, n, k, md), block_m=block_m)
    with scoped_opt_flags(flags):
        matmul(x, w, None, md, precision_config=pc)
    assert gemm_calls[-1]["block_m"] == block_m


def test_16_bit_tiles_at_256_rows_are_the_kernels_own(gemm_calls):
    # 256 x 256 with eight waves; the 128 x 128 tile stays accepted beside block_m = 256 and is then the one that runs
    from triton_amd.matmul import matmul, scoped_opt_flags_constraints
    n_slices, rows, k, n = 4, 1000, 512, 64
    w, x, md = torch.zeros((n_slices, n, k), dtype=torch.bfloat16).transpose(1, 2), torch.zeros((rows, k), dtype=torch.bfloat16), _metadata(n_slices, rows)
    for constraints, block_m, block_n in (({}, 256, 256), ({"block_n": 256}, 256, 256), ({"block_n": 256, "num_warps": 8, "block_k": 64}, 256, 256),
                                          ({"block_n": 128}, 128, 128), ({"block_k": 128, "num_warps": 4}, 128, 128)):
        with scoped_opt_flags_constraints({"block_m": 256, **constraints}):
            f = of.make_opt_flags(None, None, torch.bfloat16, None, 1, rows, n, k, md)
            assert (f.block_m, f.block_n) == (block_m, block_n)
            matmul(x, w, None, md)
        assert gemm_calls[-1]["block_m"] == block_m
    for constraints in ({"block_n": 64}, {"block_n": 256, "num_warps": 4}, {"block_n": 128, "block_k": 64}):
        with scoped_opt_flags_constraints({"block_m": 256, **constraints}), pytest.raises(of.InapplicableConstraint):
            of.make_opt_flags(None, None, torch.bfloat16, None, 1, rows, n, k, md)


@pytest.mark.parametrize("per_slice, N, n_slices, want", [
    (32, 1024, 8, 32), (32, 2048, 8, 64), (48, 1024, 16, 64), (49, 1024, 16, 0), (51, 1024, 16, 0), (48, 512, 32, 64), (51, 512, 32, 0),
    (51, 2048, 8, 64), (51, 16384, 1, 64), (51, 256, 32, 32), (51, 512, 16, 32), (62, 512, 16, 64), (62, 1024, 16, 0), (64, 1024, 8, 64), (65, 64, 8, 0)])
def test_columns_of_the_kernel_for_few_rows(per_slice, N, n_slices, want):
    """Both sides of the line: with 64 columns a second round for slices of over 64 rows costs more than the kernel gains."""
    from triton_amd import _native as nt
    assert nt.rules().few_block_n(per_slice * n_slices, N, n_slices) == want


@pytest.mark.parametrize("outer, length, inner", [
    (16, 1024, 3200), (26, 2048, 1024), (8, 2048, 3328), (2, 5120, 5120), (7, 2880, 2560), (2, 1024, 26624), (3, 2880, 5760), (4, 2880, 5760), (1, 64, 528), (260, 288, 260), (5, 32, 7)])
@pytest.mark.parametrize("e2m1", [True, False])
@pytest.mark.parametrize("down", [True, False])
def test_every_workgroup_of_the_mx_tiles_has_a_block(outer, length, inner, e2m1, down):
    """The number of workgroups is that of the tiles of the kernel that runs, above all from 96 to 128 MiB, where both the rule for reading once and the
    one for small tensors apply."""
    from triton_amd import _native as nt
    grid, blocks, _ = nt.rules().mx_tiles(outer, length, inner, e2m1, down, inner % 4 == 0)
    cols = -(-inner // 256) * outer
    assert grid % cols == 0 and (grid // cols - 1) * blocks < length // 32 <= grid // cols * blocks
    assert blocks in ((4, 8) if e2m1 else (4, ))
    if e2m1 and (outer, length, inner) == (260, 288, 260):
        assert blocks == 8


def test_sources_to_e2m1_are_read_with_the_hint():
    """From 36 MiB on: a tensor that the program did not touch lately, which a first call on loaded weights has, is read faster with it."""
    from triton_amd import _native as nt
    for outer, length, inner in [(3, 2880, 2880), (8, 2048, 2048), (2, 2880, 5760), (3, 2880, 5760), (13, 2048, 2048), (32, 2880, 5760)]:
        assert nt.rules().mx_tiles(outer, length, inner, True, True, True)[2] == 1
    assert nt.rules().mx_tiles(2, 2880, 2880, True, True, True)[2] == 0 and nt.rules().mx_tiles(16, 2048, 1093, True, True, False)[2] == 0
    assert nt.rules().mx_tiles(2, 2880, 5760, False, True, True)[2] == 0 and nt.rules().mx_tiles(4, 2880, 5760, False, True, True)[2] == 1


def test_small_mx_tiles_up_to_two_whole_line_ones_a_cu_when_expanding():
    """Beyond, half lines fetched twice cost more than the shorter chain gains; quantising takes them up to four a CU."""
    from triton_amd import _native as nt
    blocks = lambda *size: [nt.rules().mx_tiles(*size, True, down, True)[1] for down in (True, False)]
    assert blocks(2, 2880, 2880) == blocks(8, 2048, 2048) == [4, 4]
    assert blocks(2, 2880, 5760) == blocks(3, 2880, 5760) == [4, 8]
    assert blocks(8, 2880, 2880) == [8, 8]


@pytest.mark.parametrize("e2m1", [True, False])
def test_tiles_of_small_launches_fetch_all_their_bytes_together(e2m1):
    """Up to two tiles a CU nothing else runs while a tile waits for one piece after the other."""
    from triton_amd import _native as nt
    together = lambda *size: nt.rules().mx_tiles(*size, e2m1, False, False)[::2]
    for size in [(1, 64, 5), (1, 960, 517), (2, 1024, 517), (1, 2880, 517), (8, 1024, 1024)]:
        assert together(*size)[1] == 1
    assert together(4, 2048, 2048) == (512, 1) and together(2, 2880, 2880) == (552, 0)
    assert together(2, 2880, 5760)[1] == 0


def test_small_sources_with_rows_at_any_address_are_quantised_by_columns():
    """Up to 70 tiles, whose longer chain is all that there is to see, except where the last columns are few."""
    from triton_amd import _native as nt
    by = nt.rules().mx_by_columns
    for size in [(1, 64, 33), (1, 480, 1093), (1, 960, 517), (1, 960, 1093), (2, 1024, 517), (1, 2880, 517), (1, 512, 2049), (1, 960, 577), (1, 2880, 261)]:
        assert by(*size), size
    for size in [(1, 2880, 1093), (4, 960, 517), (6, 1632, 1093), (1, 480, 65), (1, 960, 193), (1, 480, 897)]:
        assert not by(*size), size


def test_mxfp8_row_blocks_of_256_only_where_the_wide_kernel_has_a_tile():
    """A row block of 256 without columns is that kernel's largest tile; where the rules name none of its tiles the other kernel runs, whose row blocks are 128."""
    from triton_amd import _native as nt
    rules, without = nt.rules(), 0
    for n_slices in (1, 2, 8, 16, 32, 64, 128):
        for K in (576, 960, 1792, 2880):
            for N in (256, 960, 2048, 2880, 5760):
                for per_slice in (1, 24, 40, 64, 80, 81, 90, 96, 97, 104, 105, 122, 152, 176, 300, 640, 1000):
                    rows = per_slice * n_slices
                    if not rules.wide_block_n(rows, n_slices, K, N, rows * K, 1):
                        without += 1
                        assert rules.wide_block_m(rows, n_slices, K, N, rows * K, 1) == 128, (n_slices, K, N, per_slice)
    assert without > 100


def test_decode_layers_up_to_16_tokens_read_the_weights_with_the_hint():
    """Read once by the whole grid, whatever their size: another layer's weights come in between.  Beyond 16 tokens plain loads (0), or as the routing has it (2)."""
    from triton_amd import _native as nt
    blocks = lambda d, f: (2 * f // 32) * -(-d // 128) + (d // 32) * -(-f // 128)
    for T in (1, 10, 16):
        for E, k, d in [(16, 4, 2048), (8, 4, 2880), (32, 8, 1024), (64, 8, 768), (128, 4, 2880)]:
            assert nt.rules().decode_fetch(T, k, E, blocks(d, d)) == 1
    assert nt.rules().decode_fetch(17, 4, 16, blocks(2048, 2048)) == 0 and nt.rules().decode_fetch(17, 4, 128, blocks(2880, 2880)) == 2


@pytest.mark.parametrize("k, m, n, n_slices, tile", [
    # the sizes that test_gpu_ragged_k.py runs by each kernel
    (160, 264, 1032, 12, 128), (160, 8, 136, 9, 128), (160, 520, 264, 128, 128), (160, 264, 520, 1, 128), (160, 520, 776, 128, 256), (160, 264, 264, 129, 0), (159, 264, 1032, 12, 0),
    # from 90 k on: rounds, and what hangs over the edges
    (128, 2880, 5760, 128, 256), (128, 2880, 2880, 128, 0), (128, 2880, 5760, 32, 256), (128, 2880, 5760, 16, 0), (93, 2880, 5760, 64, 256), (89, 2880, 5760, 128, 0), (128, 1600, 2400, 128, 0),
    (256, 2880, 5760, 8, 256), (2048, 512, 1024, 8, 128)])
def test_tile_of_a_ragged_k_gemm(k, m, n, n_slices, tile):
    """Both sides of each line: k a slice, rounds of tiles, their overhang, the slices that the kernel for long ones keeps."""
    from triton_amd import _native as nt
    assert nt.rules().ragged_k_tile(k, m, n, n_slices) == tile
