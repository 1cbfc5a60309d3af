// The host side of the common calls: a CPython extension module (`triton_amd._host`) that checks the operands, allocates the
// results, fills the descriptor of the C ABI and launches, for the calls a layer is made of (routing, the expert GEMM, the top-k
// combine, the quantisers, the ragged-K GEMM, the one-launch decode layer).
//
// What bounds it: these calls come one after another from Python, and at small sizes the GPU waits for them.  The same steps
// written in Python cost 15 us for a GEMM, 20 us for the router and 11 us for the combine, most of it attribute and tensor
// accessors at 50 to 200 ns each and about 40 ctypes fields; here they are a few ns each and what is left is the allocations
// and the launches (2 us each): a bf16 layer of 128 tokens (d 512, d_ff 1024, 8 experts) went from 65 to 37 us of host
// time, and now, with fewer launches, allocations past the dispatcher and the combine launched from the GEMM's call, takes 20.
//
// Every function returns None for a call that is not of the plain form it handles (another device, a layout, an option, a
// shape error) before it does anything; the Python code then takes the general path, which serves every option and raises the
// errors.  A call served here gets the same descriptor as it would there.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/EmptyTensor.h>
#include <ATen/detail/CUDAHooksInterface.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <array>
#include <optional>

#include "../../include/triton_amd.h"
#include "gemm_limits.h"
#include "mx_tiles.h"

namespace {

using at::ScalarType;
using at::Tensor;

// ---- objects of the Python side, set once by bind() -------------------------------------------------------------------------
struct Bound {
  decltype(&tk_moe_gemm) moe_gemm = nullptr;
  decltype(&tk_route) route = nullptr;
  decltype(&tk_route_workspace_bytes) route_workspace_bytes = nullptr;
  decltype(&tk_reduce_mid) reduce_mid = nullptr;
  decltype(&tk_quant_fp8_rows) quant_fp8_rows = nullptr;
  decltype(&tk_mx_downcast) mx_downcast = nullptr;
  decltype(&tk_mx_upcast) mx_upcast = nullptr;
  decltype(&tk_ragged_k_gemm) ragged_k_gemm = nullptr;
  decltype(&tk_moe_decode_layer) decode_layer = nullptr;
  decltype(&tk_moe_decode_layer_workspace_bytes) decode_workspace_bytes = nullptr;
  PyObject *check, *raw_stream, *current_device;              // _native.check, torch's raw stream and device getters
  PyObject *tile_counters, *combine_counters, *decode_workspace;  // per device and stream
  PyObject *tensor_type, *mx_value, *mx_scale, *fp8_value, *fp4;  // Tensor, its layouts, the FP4 data type
  PyObject *metadata_type, *routing_type, *gather_type, *scatter_type;
  PyObject *default_flex, *no_activation, *no_epilogue;
} B;

#define NAMES(X)                                                                                                            \
  X(storage) X(data) X(layout) X(shape) X(dtype) X(device) X(specs) X(fn) X(name) X(reduction_n) X(fn_args) X(flex_ctx)        \
  X(a_mx_scale) X(a_mx_tensor_scale) X(a_microblock_size) X(b_mx_scale) X(b_mx_tensor_scale) X(b_microblock_size)              \
  X(c_mx_scale) X(c_microblock_size) X(out_dtype) X(slice_sizes) X(slice_offs) X(block_offs_data) X(block_schedule_data)       \
  X(expected_slice_size) X(slice_sizes_divisibility) X(remapped_from) X(gate_scal) X(expt_hist) X(n_expts_tot) X(n_expts_act)  \
  X(expt_data) X(token_indx) X(expt_indx) X(gate_vals) X(all_rows_live) X(src_indx) X(dst_indx) X(_tk_combined)
struct Names {
#define X(n) PyObject* n;
  NAMES(X)
#undef X
} N_;

struct Ref {  // owned reference
  PyObject* p;
  explicit Ref(PyObject* q) : p(q) {}
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  ~Ref() { Py_XDECREF(p); }
  operator PyObject*() const { return p; }
};

struct PyError {};  // a Python exception is set

PyObject* attr(PyObject* o, PyObject* name) {
  PyObject* r = PyObject_GetAttr(o, name);
  if (!r) throw PyError();
  return r;
}

bool is_none(PyObject* o) { return o == Py_None; }

const Tensor* tensor_of(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

int32_t dtype_code(ScalarType t) {
  switch (t) {
    case ScalarType::Float: return TK_F32;
    case ScalarType::BFloat16: return TK_BF16;
    case ScalarType::Half: return TK_F16;
    case ScalarType::Float8_e4m3fn: return TK_E4M3;
    case ScalarType::Float8_e5m2: return TK_E5M2;
    default: return -1;
  }
}

bool f32_or_bf16(const Tensor& t) { return t.scalar_type() == ScalarType::Float || t.scalar_type() == ScalarType::BFloat16; }

// A dense tensor on the current device (which is like's: stream_of() has been asked).  Straight from the caching allocator (the router with its
// seven results 9.6 -> 6.9 us): the way through the dispatcher is taken only where something listens there (a dispatch or functional mode, a
// tracer, the fill of deterministic mode).
bool dispatcher_heard() {
  return !(c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() || at::globalContext().deterministicAlgorithms();
}
const c10::DispatchKeySet kOnDevice(c10::DispatchKey::CUDA);
Tensor empty(at::IntArrayRef sizes, ScalarType t, const Tensor& like) {
  if (dispatcher_heard()) return at::empty(sizes, at::TensorOptions().dtype(t).device(like.device()));
  return Tensor(at::detail::empty_generic(sizes, at::detail::getCUDAHooks().getCUDADeviceAllocator(), kOnDevice, t, std::nullopt));
}
Tensor empty_strided(at::IntArrayRef sizes, at::IntArrayRef strides, ScalarType t, const Tensor& like) {
  if (dispatcher_heard()) return at::empty_strided(sizes, strides, at::TensorOptions().dtype(t).device(like.device()));
  return Tensor(at::detail::empty_strided_generic(sizes, strides, at::detail::getCUDAHooks().getCUDADeviceAllocator(), kOnDevice, t));
}

// A dense tensor of `sizes` at `offset` elements of `base`.
PyObject* part_of(const Tensor& base, int64_t offset, at::IntArrayRef sizes) {
  auto t = at::detail::make_tensor<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(base.storage()), base.key_set(), base.dtype());
  t.unsafeGetTensorImpl()->set_storage_offset(base.storage_offset() + offset);
  t.unsafeGetTensorImpl()->set_sizes_contiguous(sizes);
  return THPVariable_Wrap(std::move(t));
}

// The current stream of t's device, or no value when that is not the current device.
std::optional<void*> stream_of(const Tensor& t) {
  Ref cur(PyObject_CallNoArgs(B.current_device));
  if (!cur) throw PyError();
  if (PyLong_AsLong(cur) != t.get_device()) return std::nullopt;
  Ref s(PyObject_CallOneArg(B.raw_stream, cur));
  if (!s) throw PyError();
  return PyLong_AsVoidPtr(s);
}

template <class F>
void launch(F&& f) {
  int32_t status;
  PyThreadState* st = PyEval_SaveThread();
  status = f();
  PyEval_RestoreThread(st);
  if (status != TK_OK) {
    Ref code(PyLong_FromLong(status));
    Ref r(PyObject_CallOneArg(B.check, code));
    if (r) PyErr_SetString(PyExc_RuntimeError, "a native call failed");
    throw PyError();
  }
}

PyObject* none() { Py_RETURN_NONE; }

// A dataclass instance with these fields (its __init__ would only assign them).
template <size_t n>
PyObject* instance(PyObject* type, const std::pair<PyObject*, PyObject*> (&fields)[n]) {
  auto* tp = reinterpret_cast<PyTypeObject*>(type);
  PyObject* o = tp->tp_alloc(tp, 0);
  if (!o) throw PyError();
  for (auto& f : fields)
    if (PyObject_GenericSetAttr(o, f.first, f.second)) {
      Py_DECREF(o);
      throw PyError();
    }
  return o;
}

// ---- rules ------------------------------------------------------------------------------------------------------------------

// Row blocks of the memory-to-LDS kernel: 256 (256 x 256 tiles, one workgroup per CU) or 128 (128 x 128, two per CU).  The large
// tile moves half the operand bytes per product, the small one fills the chip with fewer rows.  Measured on 8 to 32 slices: up to 64
// rows per slice the small tile is as fast or faster (e4m3, 8 rows, K 4096: 174 against 183 us), from 192 on the large one is
// (e4m3, 256 rows: 350 against 456 us); in between it depends on the large tiles there are for the 256 CUs (bf16, 128 rows, K 2048:
// N 4096, 256 tiles, 56 against 72 us; N 2048, 128 tiles, 44 against 38 us) and, with fewer, on the length of a row, which a
// tile's start and end have to be paid from (e4m3, 128 tiles, K 14336: 168 against 214 us).
int64_t dma_block_m(int64_t rows, int64_t row_bytes, int64_t N, int64_t n_slices) {
  int64_t per_slice = rows / std::max<int64_t>(n_slices, 1);
  if (per_slice <= 64) return 128;
  int64_t tiles = n_slices * ((per_slice + 255) / 256) * ((N + 255) / 256);
  return per_slice >= 192 || tiles >= 192 || row_bytes >= 8192 ? 256 : 128;
}

// 128 = the kernel's 128 x 128 tiles although the rule above says 256: where those are one round (small_tiles_one_round, gemm_limits.h), and with fewer rows
// up to 96 of the large tiles, which leave most of the 256 CUs without one.
// Measured with a random routing (us, 128 against 256): bf16, K 2048, N 2048, 8 slices of 256 rows (64 large tiles) 29 against 42; N 1536, 16
// slices (96) 34 against 41; N 2048, 16 slices (128) 51 against 49; K 1024, N 1024, 16 slices (64) 19 against 27, N 512 (32) 11 against 23;
// K 4096, N 1024, 16 slices (64) 55 against 72; e4m3, K 14336, N 2048, 8 slices (64) 92 against 126, N 4096 (128) 193 against 158.
// With 16-bit operands, columns of the tiles of 320 rows where gemm_limits.h names those.
int64_t dma_block_n(int64_t rows, int64_t N, int64_t n_slices, int64_t block_m, bool bits16) {
  const int64_t cols = block_m == 256 && bits16 ? tk::dma_tile(rows, n_slices, N).cols : 0;
  if (cols) return cols;
  const int64_t per_slice = rows / std::max<int64_t>(n_slices, 1);
  return block_m == 256 && (tk::small_tiles_one_round(rows, n_slices, N) || n_slices * ((per_slice + 255) / 256) * ((N + 255) / 256) <= 96) ? 128 : 0;
}

// Row blocks for tiled e4m3 weights: by the rule above where that kernel runs (`x_bytes` as in gemm_limits.h).  The other kernel walks a
// block of 256 rows in two passes, which pays from 1024 rows per slice on (8 slices, K 4096, N 8192: 512 rows 147 us with either, 1024
// 296 with blocks of 128 against 289 with 256; 2048 rows, N 28672: 1930 against 1853, K 14336, N 4096: 846 against 819 us) and costs up to twice
// the time below (256 rows, K 14336: 133 against 273 us; 300 slices of 256 rows, K and N 2048: 474 against 544 us).
int64_t fp8_block_m(int64_t rows, uint32_t x_bytes, int64_t K, int64_t N, int64_t n_slices) {
  if (tk::dma_runs_e4m3(x_bytes, n_slices, K, N)) return dma_block_m(rows, K, N, n_slices);
  return rows >= 1024 * n_slices ? 256 : 128;
}

// Row blocks for tiled MXFP4 weights with more routed rows than the decode kernel is made for.  32 = the streaming kernel, faster
// than the decode kernel's 16-row blocks from 160 rows on (128 slices, K 2880, N 5760: 300 tokens 210 against 232 us, 32 slices,
// 200 tokens 28 against 57 us) and than the prefill kernel's 64-row blocks up to about 20 rows per slice (18: 245 against 258 us,
// 31: 331 against 290 us); those give way to the larger ones at about 56 (47: 340 against 372 us, 62: 410 against 399 us).
// (For calls that the streaming kernel takes: x as a buffer resource, slices in registers, no row or column scales.  Where the wide kernel runs, its tiles
// (mxw_tile) come in place of all of these.)
int64_t mxfp4_block_m(int64_t rows, int64_t n_slices, int64_t otherwise) {
  int64_t per_slice = rows / std::max<int64_t>(n_slices, 1);
  return per_slice <= 20 ? 32 : per_slice <= 56 ? 64 : std::max<int64_t>(otherwise, 128);
}

// Row blocks of 128, or 256 = the wide kernel (160 x 512 tiles), for MXFP4 weights beyond the sizes above.  Measured at K 2880, N 5760 and
// 2880 (both GEMMs, 128 against 256).  bf16 rows: 64 per slice 571 against 582 us, 94 684 against 668, 162 1296 against 1131,
// 250 (16 slices) 258 against 246, 1024 754 against 716 us.  MXFP8 rows: 64 per slice 444 against 451 us; beyond 104 by mx8_tile (gemm_limits.h).
// The wide kernel takes four stages of K (the activation scales sixteen blocks), slices in registers and x as a buffer resource.
int64_t wide_block_m(int64_t rows, int64_t n_slices, int64_t K, int64_t N, uint32_t x_bytes, bool mx8) {
  n_slices = std::max<int64_t>(n_slices, 1);
  if (K <= (mx8 ? 511 : 384) || n_slices > tk::kDmaSlices || !x_bytes) return rows <= 144 * n_slices ? 256 : 128;
  if (rows <= 80 * n_slices) return 128;
  // (the wide kernel's tiles are asked for by their columns; the other kernel, wherever the rules name none of them, has row blocks of 128: its tiles are one round there, which
  // with row blocks of 256 were 160 x 512 of the wide kernel on a quarter of the CUs.  Layers, us, 16 slices of 90 rows, 1792 and 1024: 80 -> 56; 8 of 96, 2880 105 -> 65; 16 of 84, 1024
  // 65 -> 48; 32 of 96, 1024 64 -> 50.  K of 512 and 544 with up to 104 rows keep the row block of 256, which callers can see in the descriptor and are promised for the wide
  // kernel, although 128 is faster there as well: 16 slices of 87, K 512, N 1088 16.3 against 9.8, K 544, N 512 17.2 against 10.5)
  if (mx8 && (K > 544 || rows > 104 * n_slices) && !tk::mxw_tile(rows, n_slices, K, N, mx8).rows) return 128;
  return !mx8 || rows <= 176 * n_slices || rows >= 640 * n_slices ? 256 : 128;
}

// Columns of the wide kernel's tiles that gemm_limits.h names for such weights, 0 = the kernel of the row block.
int64_t wide_block_n(int64_t rows, int64_t n_slices, int64_t K, int64_t N, uint32_t x_bytes, bool mx8) {
  n_slices = std::max<int64_t>(n_slices, 1);
  return K <= (mx8 ? 511 : 384) || n_slices > tk::kDmaSlices || !x_bytes ? 0 : tk::mxw_tile(rows, n_slices, K, N, mx8).cols;
}

// Columns a workgroup of the kernel for few rows, 0 = the kernels above: up to 64 rows per slice and one workgroup per CU at most, with 32
// columns while they fit, then 64.  Measured (us, this kernel against the one that ran before; other weights each call): 8 slices of 32
// rows, N 2048: K 512 9.1 against 12.1, K 2048 20 against 28, K 8192 60 against 76; N 512: K 1024 7.6 against 15.4, K 8192 26 against 72; 64 rows, N
// 1024: K 512 9.0 against 11.6, K 8192 47 against 77; one slice of 50 rows, N 16384: K 512 10.4 against 12.3, K 8192 67 against 77; 16 slices
// of 28 rows, some of them over 64, N 1024: K 512 11.7 against 12.3, K 2048 24 against 28.  The same weights again: 8 slices of 32 rows, K 512,
// N 2048 6.3 against 9.4; 16 slices, 2 or 8 rows each, K 512, N 1024 4.2 against 6.6.
// 64 columns only up to 48 rows per slice where one row block of more than eight slices each is counted on: a slice of more than 64 rows is then a
// second round, which takes as long as the first (16 slices, N 1024, of 48 rows: K 512 11.1 against 12.7, K 2048 22 against 28; of 51: 12.4 against
// 12.7 and 29 against 28, with such a slice in every routing 15.2 against 12.3; 32 slices of 51, N 512, K 1024 19 against 18).  Eight slices seldom
// have one (of 51 rows, N 2048: K 512 11.2 against 12.8, K 2048 24 against 28), and with 32 columns it is the faster way all the same (32
// slices of 51, N 256: K 512 9.6 against 10.6, K 2048 19 against 25).  With two workgroups per CU to be
// run in turn the others are as fast or faster (16 slices, K 1024, N 2048: 8 rows 16.8 against 15.5, 32 rows 19.6 against 16.8; 8 slices of
// 125 rows, K 512, N 1024: 12.0 against 9.9).
int64_t few_block_n(int64_t rows, int64_t N, int64_t n_slices) {
  if (n_slices < 1 || rows > 64 * n_slices) return 0;
  const int64_t blocks = tk::few_row_blocks(rows, n_slices);
  if (blocks * ((N + 31) / 32) <= 256) return 32;
  return blocks * ((N + 63) / 64) <= 256 && (rows <= 48 * n_slices || n_slices <= 8 || blocks > n_slices) ? 64 : 0;
}

int64_t default_block_m(int64_t rows, int64_t n_slices) {
  int64_t per_slice = std::max<int64_t>(1, rows / std::max<int64_t>(n_slices, 1));
  return per_slice <= 16 ? 16 : per_slice <= 32 ? 32 : per_slice <= 64 ? 64 : 128;
}

int64_t n_blocks(int64_t n_slices, int64_t rows, int64_t block_m) {
  return rows <= n_slices ? rows : n_slices - 1 + (rows + 1 - n_slices + block_m - 1) / block_m;
}

// ---- operands ---------------------------------------------------------------------------------------------------------------

struct Metadata {
  const Tensor *sizes, *offs, *block_offs, *schedule;
  bool read(PyObject* md) {
    if (Py_TYPE(md) != reinterpret_cast<PyTypeObject*>(B.metadata_type)) return false;
    Ref e(attr(md, N_.expected_slice_size)), r(attr(md, N_.remapped_from)), a(attr(md, N_.slice_sizes)), b(attr(md, N_.slice_offs)),
        c(attr(md, N_.block_offs_data)), d(attr(md, N_.block_schedule_data));
    if (!is_none(e) || !is_none(r)) return false;
    sizes = tensor_of(a), offs = tensor_of(b), block_offs = tensor_of(c), schedule = tensor_of(d);  // (md keeps them alive)
    return sizes && offs && block_offs && schedule && sizes->dim() == 1 && sizes->is_contiguous() && offs->is_contiguous()
           && block_offs->dim() == 2 && schedule->dim() == 2 && block_offs->stride(1) == 1
           && (schedule->numel() == 0 || schedule->stride(1) == 1);
  }
};

// The storage of a package tensor with this layout, else null; *shape gets the last two sizes.
const Tensor* storage_of(PyObject* w, PyObject* layout_type, int64_t* shape) {
  if (Py_TYPE(w) != reinterpret_cast<PyTypeObject*>(B.tensor_type)) return nullptr;
  Ref st(attr(w, N_.storage)), layout(attr(st, N_.layout));
  if (reinterpret_cast<PyObject*>(Py_TYPE(layout.p)) != layout_type) return nullptr;
  if (shape) {
    Ref s(attr(w, N_.shape));
    if (!PyList_Check(s.p) || PyList_GET_SIZE(s.p) < 2) return nullptr;
    Py_ssize_t n = PyList_GET_SIZE(s.p);
    shape[0] = PyLong_AsLongLong(PyList_GET_ITEM(s.p, n - 2)), shape[1] = PyLong_AsLongLong(PyList_GET_ITEM(s.p, n - 1));
    if (PyErr_Occurred()) throw PyError();
  }
  Ref d(attr(st, N_.data));
  return tensor_of(d);
}

PyObject* layout_type_of(PyObject* w) {
  if (Py_TYPE(w) != reinterpret_cast<PyTypeObject*>(B.tensor_type)) return nullptr;
  Ref st(attr(w, N_.storage)), layout(attr(st, N_.layout));
  return reinterpret_cast<PyObject*>(Py_TYPE(layout.p));
}

bool named(PyObject* o, PyObject* attr_name, const char* want) {
  Ref n(attr(o, attr_name));
  return PyUnicode_Check(n.p) && PyUnicode_CompareWithASCIIString(n, want) == 0;
}

struct Activation {
  bool swiglu = false, has_limit = false;
  double alpha = 0, limit = 0;
  bool read(PyObject* act) {
    if (is_none(act) || act == B.no_activation) return true;
    Ref specs(attr(act, N_.specs)), red(attr(specs, N_.reduction_n)), args(attr(act, N_.fn_args));
    const long columns = PyLong_AsLong(red);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    if (!named(specs, N_.name, "swiglu") || columns != 2 || !PyTuple_Check(args.p)) return false;
    Py_ssize_t n = PyTuple_GET_SIZE(args.p);
    if (n < 1) return false;
    alpha = PyFloat_AsDouble(PyTuple_GET_ITEM(args.p, 0));
    if (n > 1 && !is_none(PyTuple_GET_ITEM(args.p, 1))) has_limit = true, limit = PyFloat_AsDouble(PyTuple_GET_ITEM(args.p, 1));
    if (PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    return swiglu = true;
  }
};

bool plain_index(PyObject* o, const Tensor** t) {
  *t = nullptr;
  if (is_none(o)) return true;
  *t = tensor_of(o);
  return *t && (*t)->scalar_type() == ScalarType::Int && (*t)->dim() == 1 && (*t)->is_contiguous();
}

// One expert GEMM, scatter-combine included; see gemm() for the arguments.  Null = the general path.
PyObject* run_gemm(PyObject* const* v) {
  PyObject *a_o = v[0], *b_o = v[1], *bias_o = v[2], *pc = v[6], *gam_o = v[7], *epi = v[9];
  const Tensor* a = tensor_of(a_o);
  if (!a || !a->is_cuda() || a->dim() != 2 || a->stride(1) != 1) return none();
  const ScalarType at = a->scalar_type();
  Metadata md;
  Activation act;
  const Tensor *gather, *scatter, *gammas = nullptr, *bias = nullptr;
  if (!md.read(v[3]) || !plain_index(v[4], &gather) || !plain_index(v[5], &scatter) || !act.read(v[8])) return none();
  if (!is_none(bias_o)) {
    bias = tensor_of(bias_o);
    if (!bias || bias->dim() != 2 || bias->stride(1) != 1 || !f32_or_bf16(*bias)) return none();
  }
  if (!is_none(gam_o)) {
    gammas = tensor_of(gam_o);
    if (!gammas || !gammas->is_contiguous() || !f32_or_bf16(*gammas)) return none();
  }
  // (whole numbers; the general path says what it makes of anything else, None and floats among them)
  if ((!is_none(v[10]) && !PyLong_Check(v[10])) || !PyLong_Check(v[11])) return none();
  const long combine_k = is_none(v[10]) ? 0 : PyLong_AsLong(v[10]), idle = PyLong_AsLong(v[11]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return none();
  }

  // ---- weights
  int64_t kn[2];
  const Tensor* w = tensor_of(b_o);
  const bool strided = w != nullptr;
  bool tiled = false, tiled_fp8 = false;
  if (strided) {
    if (w->dim() != 3 || w->scalar_type() != at || !(at == ScalarType::BFloat16 || at == ScalarType::Half) || w->stride(1) != 1
        || !(w->size(1) == 1 || w->stride(2) >= w->size(1)))
      return none();
    kn[0] = w->size(1), kn[1] = w->size(2);
  } else {
    PyObject* lt = layout_type_of(b_o);
    tiled = lt == B.mx_value, tiled_fp8 = lt == B.fp8_value;
    if (!tiled && !tiled_fp8) return none();
    w = storage_of(b_o, lt, kn);
    if (!w || w->scalar_type() != ScalarType::Byte || !w->is_contiguous() || w->dim() < 1) return none();
    if (tiled) {
      Ref dt(attr(b_o, N_.dtype));
      if (dt != B.fp4) return none();
    }
  }

  // ---- precision config
  const Tensor *xs = nullptr, *x_row = nullptr, *w_col = nullptr, *ws = nullptr, *ys = nullptr;
  bool mx_act = false, mx_out = false;
  ScalarType out = at;
  if (!is_none(pc)) {
    Ref flex(attr(pc, N_.flex_ctx)), axs(attr(pc, N_.a_mx_scale)), ats(attr(pc, N_.a_mx_tensor_scale)), amb(attr(pc, N_.a_microblock_size)),
        bxs(attr(pc, N_.b_mx_scale)), bts(attr(pc, N_.b_mx_tensor_scale)), bmb(attr(pc, N_.b_microblock_size)), cxs(attr(pc, N_.c_mx_scale)),
        cmb(attr(pc, N_.c_microblock_size)), od(attr(pc, N_.out_dtype));
    if (flex != B.default_flex || !is_none(amb) || !is_none(bmb) || !is_none(cmb)) return none();
    if (!is_none(od)) {
      if (!THPDtype_Check(od)) return none();
      out = reinterpret_cast<THPDtype*>(od.p)->scalar_type;
    }
    if (!is_none(axs)) {
      xs = tensor_of(axs), mx_act = true;
      if (!xs || xs->scalar_type() != ScalarType::Byte || xs->dim() != 2 || xs->stride(1) != 1) return none();
    }
    if (!is_none(ats)) {
      x_row = tensor_of(ats);
      if (!x_row || x_row->scalar_type() != ScalarType::Float || !x_row->is_contiguous()) return none();
    }
    if (!is_none(bts)) {
      w_col = tensor_of(bts);
      if (!w_col || w_col->scalar_type() != ScalarType::Float || w_col->dim() != 2 || !w_col->is_contiguous()) return none();
    }
    if (!is_none(bxs)) {
      ws = storage_of(bxs, B.mx_scale, nullptr);
      if (!ws || ws->scalar_type() != ScalarType::Byte || !ws->is_contiguous() || ws->dim() < 1) return none();
    }
    if (!is_none(cxs)) {
      ys = tensor_of(cxs), mx_out = true;
      if (!ys || ys->scalar_type() != ScalarType::Byte || ys->dim() != 2 || ys->stride(1) != 1) return none();
    }
  }
  if (is_none(epi) || epi == B.no_epilogue) {
    if (mx_out) return none();
  } else {
    Ref specs(attr(epi, N_.specs));
    if (!mx_out || !named(specs, N_.name, "QUANTIZE_MXFP8")) return none();
  }
  if (tiled != (ws != nullptr)) return none();

  // ---- shapes and types
  const int64_t K = kn[0], N = kn[1], n_slices = md.sizes->size(0), a_rows = a->size(0), a_stride = a->stride(0);
  const int64_t M = gather ? gather->size(0) : a_rows, y_rows = scatter ? scatter->size(0) : M, n_out = act.swiglu ? N / 2 : N;
  if (a->size(1) != K || w->size(0) != n_slices || M == 0 || N == 0) return none();
  if (mx_act ? !tiled || at != ScalarType::Float8_e4m3fn || x_row || xs->size(0) != a_rows || xs->size(1) != (K + 31) / 32
      : tiled_fp8 ? at != ScalarType::Float8_e4m3fn
                  : at != ScalarType::BFloat16 && !(strided && at == ScalarType::Half))
    return none();
  if (mx_out) {
    if (!mx_act || out != ScalarType::Float8_e4m3fn || n_out % 32 || ys->size(0) != y_rows || ys->size(1) != n_out / 32) return none();
  } else if (out != (at == ScalarType::Half ? ScalarType::Half : ScalarType::BFloat16)) {
    return none();
  }
  if ((x_row && x_row->numel() != a_rows) || (w_col && (w_col->size(0) != n_slices || w_col->size(1) != N))
      || (ws && ws->size(0) != n_slices))
    return none();

  // ---- row blocks
  int64_t block_m = default_block_m(M, n_slices), block_n = 0;
  const uint32_t x_bytes = tk::x_extent(a_rows, a_stride, K, a->element_size());
  if (tiled_fp8) {
    block_m = fp8_block_m(M, x_bytes, K, N, n_slices);
    if (tk::dma_runs_e4m3(x_bytes, n_slices, K, N)) block_n = dma_block_n(M, N, n_slices, block_m, false);
  } else if (mx_act) {
    block_m = wide_block_m(M, n_slices, K, N, x_bytes, true);
    block_n = wide_block_n(M, n_slices, K, N, x_bytes, true);
  } else if (tiled) {
    if (M > 256 && x_bytes && n_slices <= tk::kDmaSlices && !x_row && !w_col) {
      block_m = mxfp4_block_m(M, n_slices, block_m);
      if (n_out % 8 == 0) block_n = wide_block_n(M, n_slices, K, N, x_bytes, false);
    }
    if (block_m == 128) block_m = wide_block_m(M, n_slices, K, N, x_bytes, false);
  } else if (tk::dma_runs_16bit(x_bytes, n_slices, K, N, w->stride(2))) {
    if (idle <= 0) block_n = few_block_n(M, N, n_slices);
    if (block_m > 16) block_m = dma_block_m(M, 2 * K, N, n_slices);
    if (!block_n) block_n = dma_block_n(M, N, n_slices, block_m, true);
  }
  if (tiled && block_m >= 64 && !mx_act && n_out % 8) return none();  // (through a padded buffer)

  auto stream = stream_of(*a);
  if (!stream) return none();
  Tensor y = empty({y_rows, n_out}, out, *a), combined;
  tk_gemm_desc d{};
  d.x = a->data_ptr(), d.x_dtype = dtype_code(at), d.x_stride_m = a_stride, d.x_rows = a_rows;
  if (x_row) d.x_row_scale = static_cast<const float*>(x_row->data_ptr());
  if (mx_act) d.x_mx_scale = static_cast<const uint8_t*>(xs->data_ptr()), d.xs_stride_m = xs->stride(0);
  d.w = w->data_ptr(), d.w_stride_e = w->stride(0);
  if (strided) {
    d.w_stride_k = 1, d.w_stride_n = w->stride(2), d.w_dtype = dtype_code(at);
  } else {
    d.w_layout = TK_W_TILED, d.w_dtype = tiled ? TK_E2M1 : TK_E4M3;
    if (ws) d.w_mx_scale = static_cast<const uint8_t*>(ws->data_ptr()), d.ws_stride_e = ws->stride(0);
  }
  if (w_col) d.w_col_scale = static_cast<const float*>(w_col->data_ptr()), d.wcs_stride_e = w_col->stride(0);
  if (bias) d.bias = bias->data_ptr(), d.bias_dtype = dtype_code(bias->scalar_type()), d.bias_stride_e = bias->stride(0);
  if (gather) d.gather_indx = static_cast<const int32_t*>(gather->data_ptr());
  if (scatter) d.scatter_indx = static_cast<const int32_t*>(scatter->data_ptr()), d.scatter_len = int32_t(y_rows);
  if (gammas) d.gammas = gammas->data_ptr(), d.gammas_dtype = dtype_code(gammas->scalar_type());
  const int64_t row = 63 - __builtin_clzll(uint64_t(block_m)) - 4;  // 16 .. 256 -> 0 .. 4
  d.slice_sizes = static_cast<const int32_t*>(md.sizes->data_ptr()), d.slice_offs = static_cast<const int32_t*>(md.offs->data_ptr());
  d.block_offs = static_cast<const int32_t*>(md.block_offs->data_ptr()) + row * md.block_offs->stride(0);
  d.block_schedule = static_cast<const int32_t*>(md.schedule->data_ptr()) + row * md.schedule->stride(0);
  d.n_slices = int32_t(n_slices), d.block_m = int32_t(block_m), d.block_n = int32_t(block_n);
  d.grid_m = int32_t(std::min(n_blocks(n_slices, M, block_m), md.schedule->size(1)));
  d.M = int32_t(M), d.N = int32_t(N), d.K = int32_t(K);
  d.y = y.data_ptr(), d.y_dtype = dtype_code(out), d.y_stride_m = n_out;
  if (act.swiglu) d.activation = TK_ACT_SWIGLU, d.act_alpha = float(act.alpha), d.act_limit = float(act.limit), d.act_has_limit = act.has_limit;
  d.idle_cus = int32_t(std::max<long>(idle, 0));
  if (mx_out) d.y_mx_scale = static_cast<uint8_t*>(ys->data_ptr()), d.ys_stride_m = ys->stride(0);
  auto words = [&](PyObject* of, bool with_stream) {
    Ref dev(attr(a_o, N_.device)), s(PyLong_FromVoidPtr(*stream));
    PyObject* args[2] = {dev, s};
    Ref t(PyObject_Vectorcall(of, args, with_stream ? 2 : 1, nullptr));
    if (!t) throw PyError();
    return static_cast<int32_t*>(THPVariable_Unpack(t.p).data_ptr());  // (kept for the life of the process)
  };
  if ((tiled || tiled_fp8) && block_m >= 64 && !mx_act) d.tile_counters = words(B.tile_counters, true);
  // the combine inside the launch, by the wave that completes a token's rows: the decode kernel only
  if (combine_k > 0 && tiled && !mx_act && !act.swiglu && scatter && y_rows % combine_k == 0 && block_m == 16
      && (y_rows / combine_k) * ((N + 31) / 32) <= (1 << 16)) {
    combined = empty({y_rows / combine_k, N}, out, *a);
    d.combine_k = int32_t(combine_k), d.combine_out = combined.data_ptr(), d.combine_stride_m = N;
    d.combine_counters = words(B.combine_counters, false);
  }
  launch([&] { return B.moe_gemm(&d, *stream); });
  // or by a launch of its own, from here
  if (combine_k > 0 && !combined.defined() && scatter && y_rows > 0 && y_rows % combine_k == 0) {
    combined = empty({y_rows / combine_k, n_out}, out, *a);
    launch([&] {
      return B.reduce_mid(y.data_ptr(), dtype_code(out), y_rows / combine_k, combine_k, n_out, combine_k * n_out, n_out, nullptr, 0, 0, 0, nullptr, 0, 0,
                          0, combined.data_ptr(), n_out, *stream);
    });
  }
  PyObject* r = THPVariable_Wrap(std::move(y));
  if (r && combined.defined()) {
    Ref c(THPVariable_Wrap(std::move(combined)));
    if (!c.p || PyObject_SetAttr(r, N_._tk_combined, c)) {
      Py_DECREF(r);
      throw PyError();
    }
  }
  return r;
}

// ---- routing ----------------------------------------------------------------------------------------------------------------

// (logits, k, apply_softmax) -> (RoutingData, GatherIndx, ScatterIndx)
PyObject* run_route(PyObject* const* v) {
  const Tensor* logits = tensor_of(v[0]);
  if (!logits || !logits->is_cuda() || logits->dim() != 2 || logits->stride(1) != 1) return none();
  const ScalarType t = logits->scalar_type();
  if (t != ScalarType::Float && t != ScalarType::BFloat16 && t != ScalarType::Half) return none();
  const int64_t T = logits->size(0), E = logits->size(1), k = PyLong_AsLongLong(v[1]), R = T * k;
  const int softmax = PyObject_IsTrue(v[2]);
  if (PyErr_Occurred()) throw PyError();
  if (T == 0 || E == 0 || E >= 32768 || k < 1 || k > 32 || (k & (k - 1))) return none();
  auto stream = stream_of(*logits);
  if (!stream) return none();
  // Allocations by what a caller keeps or saves together: the [E] histogram by itself, the two permutations with the [R] gather index, and
  // the metadata ([E + 1] row offsets, [5, E + 1] block offsets, [5, width] schedules, whose readers load single words).  The kernels'
  // scratch ends with this call.
  const int64_t width = n_blocks(E, R, 16), scratch = std::max<int64_t>(1, B.route_workspace_bytes(int32_t(T), int32_t(E)));
  Tensor hist_t = empty({E}, ScalarType::Int, *logits), perm = empty({3 * R}, ScalarType::Int, *logits),
         meta = empty({6 * (E + 1) + 5 * width}, ScalarType::Int, *logits), work = empty({scratch}, ScalarType::Byte, *logits);
  Tensor vals = empty({T, k}, t, *logits), indx = empty({T, k}, ScalarType::Short, *logits), gammas = empty({R}, t, *logits);
  int32_t *perms = static_cast<int32_t*>(perm.data_ptr()), *metas = static_cast<int32_t*>(meta.data_ptr());
  const int64_t row = R, gat = 2 * R, blocks = E + 1, sched = blocks + 5 * (E + 1);
  tk_route_desc d{};
  d.logits = logits->data_ptr(), d.logits_dtype = dtype_code(t), d.logits_stride_m = logits->stride(0);
  d.n_tokens = int32_t(T), d.n_rows = -1, d.n_experts = int32_t(E), d.k = int32_t(k), d.apply_softmax = softmax;
  d.vals = vals.data_ptr(), d.indx = indx.data_ptr(), d.indx_dtype = TK_I16, d.gammas = gammas.data_ptr();
  d.col_sum = static_cast<int32_t*>(hist_t.data_ptr()), d.col_sorted_indx = perms, d.row_sorted_indx = perms + row, d.gather_indx = perms + gat;
  d.slice_offs = metas, d.block_offs = metas + blocks, d.block_offs_stride = E + 1;
  d.block_schedule = metas + sched, d.block_schedule_stride = width, d.max_n_blocks = int32_t(width);
  d.workspace = work.data_ptr();
  launch([&] { return B.route(&d, *stream); });
  Ref hist(THPVariable_Wrap(hist_t)), col_o(part_of(perm, 0, {R})), row_o(part_of(perm, row, {R})), gat_o(part_of(perm, gat, {R})),
      offs_o(part_of(meta, 0, {E + 1})), blocks_o(part_of(meta, blocks, {5, E + 1})), sched_o(part_of(meta, sched, {5, width})),
      vals_o(THPVariable_Wrap(vals)), indx_o(THPVariable_Wrap(indx)), gam_o(THPVariable_Wrap(gammas)), e_o(PyLong_FromLongLong(E));
  for (PyObject* o : {hist.p, col_o.p, row_o.p, gat_o.p, offs_o.p, blocks_o.p, sched_o.p, vals_o.p, indx_o.p, gam_o.p, e_o.p})
    if (!o) throw PyError();
  Ref md(instance(B.metadata_type, {{N_.slice_sizes, hist}, {N_.slice_offs, offs_o}, {N_.block_offs_data, blocks_o},
                                    {N_.block_schedule_data, sched_o}, {N_.expected_slice_size, Py_None}, {N_.slice_sizes_divisibility, Py_None}}));
  Ref rd(instance(B.routing_type, {{N_.gate_scal, gam_o}, {N_.expt_hist, hist}, {N_.n_expts_tot, e_o}, {N_.n_expts_act, v[1]},
                                   {N_.expt_data, md}, {N_.token_indx, gat_o}, {N_.expt_indx, indx_o}, {N_.gate_vals, vals_o},
                                   {N_.all_rows_live, Py_True}}));
  Ref gi(instance(B.gather_type, {{N_.src_indx, col_o}, {N_.dst_indx, row_o}}));
  Ref si(instance(B.scatter_type, {{N_.src_indx, row_o}, {N_.dst_indx, col_o}}));
  return PyTuple_Pack(3, rd.p, gi.p, si.p);
}

// ---- element-wise companions ----------------------------------------------------------------------------------------------------

// (y [T * k, C], k) -> [T, C], the k rows of every token summed
PyObject* run_combine(PyObject* const* v) {
  const Tensor* y = tensor_of(v[0]);
  const int64_t k = PyLong_AsLongLong(v[1]);
  if (PyErr_Occurred()) throw PyError();
  if (!y || !y->is_cuda() || y->dim() != 2 || !y->is_contiguous() || k < 1 || y->size(0) == 0 || y->size(0) % k) return none();
  const int32_t t = dtype_code(y->scalar_type());
  if (t != TK_BF16 && t != TK_F16 && t != TK_F32) return none();
  auto stream = stream_of(*y);
  if (!stream) return none();
  const int64_t A = y->size(0) / k, C = y->size(1);
  Tensor out = empty({A, C}, y->scalar_type(), *y);
  launch([&] {
    return B.reduce_mid(y->data_ptr(), t, A, k, C, k * C, C, nullptr, 0, 0, 0, nullptr, 0, 0, 0, out.data_ptr(), C, *stream);
  });
  return THPVariable_Wrap(std::move(out));
}

// x [M, K] -> (values [M, K], scales [M])
PyObject* run_quant_fp8_rows(PyObject* const* v) {
  const Tensor* x = tensor_of(v[0]);
  if (!x || !x->is_cuda() || x->dim() != 2 || x->scalar_type() != ScalarType::BFloat16 || x->stride(1) != 1 || x->numel() == 0) return none();
  auto stream = stream_of(*x);
  if (!stream) return none();
  const int64_t M = x->size(0), K = x->size(1);
  Tensor q = empty({M, K}, ScalarType::Float8_e4m3fn, *x), s = empty({M}, ScalarType::Float, *x);
  launch([&] {
    return B.quant_fp8_rows(x->data_ptr(), TK_BF16, M, K, x->stride(0), q.data_ptr(), K, static_cast<float*>(s.data_ptr()), *stream);
  });
  Ref qo(THPVariable_Wrap(std::move(q))), so(THPVariable_Wrap(std::move(s)));
  if (!qo.p || !so.p) throw PyError();
  return PyTuple_Pack(2, qo.p, so.p);
}

// [outer, rows, inner] of a dense tensor with the quantised axis last (inner = 1) or last but one
struct Axis {
  int64_t outer = 1, len = 0, inner = 1;
  bool last = false;
  bool of(const Tensor& t, int64_t axis) {
    const int64_t n = t.dim();
    if (axis < 0) axis += n;
    if (axis != n - 1 && (axis != n - 2 || axis < 0)) return false;
    last = axis == n - 1;
    for (int64_t i = 0; i < axis; ++i) outer *= t.size(i);
    len = t.size(axis), inner = last ? 1 : t.size(n - 1);
    return true;
  }
};

// Sizes with the quantised axis' length replaced; the result is dense with that axis fastest.
Tensor along(const Tensor& like, const Axis& ax, int64_t len, ScalarType t) {
  c10::SmallVector<int64_t, 5> sizes(like.sizes()), strides(like.dim());
  const int64_t n = like.dim(), a = ax.last ? n - 1 : n - 2;
  sizes[a] = len;
  strides[a] = 1;
  int64_t run = len;
  if (!ax.last) strides[n - 1] = run, run *= sizes[n - 1];
  for (int64_t i = a - 1; i >= 0; --i) strides[i] = run, run *= sizes[i];
  return empty_strided(sizes, strides, t, like);
}

// (x, kind of the values, axis, rounding) -> (values, scales)
PyObject* run_mx_downcast(PyObject* const* v) {
  const Tensor* x = tensor_of(v[0]);
  const long kind = PyLong_AsLong(v[1]), axis = PyLong_AsLong(v[2]), rounding = PyLong_AsLong(v[3]);
  if (PyErr_Occurred()) throw PyError();
  if (!x || !x->is_cuda() || x->dim() < 2 || x->dim() > 3 || !x->is_contiguous() || x->numel() == 0) return none();
  const int32_t t = dtype_code(x->scalar_type());
  Axis ax;
  if ((t != TK_BF16 && t != TK_F16 && t != TK_F32) || !ax.of(*x, axis) || ax.len % 32) return none();
  auto stream = stream_of(*x);
  if (!stream) return none();
  Tensor q = along(*x, ax, kind == TK_E2M1 ? ax.len / 2 : ax.len,
                   kind == TK_E2M1 ? ScalarType::Byte : kind == TK_E4M3 ? ScalarType::Float8_e4m3fn : ScalarType::Float8_e5m2);
  Tensor s = along(*x, ax, ax.len / 32, ScalarType::Byte);
  // one stride per collapsed dimension; 0 where a dimension has a single element
  const int64_t so = ax.outer > 1 ? ax.len * ax.inner : 0, si = ax.last ? 0 : ax.inner > 1 ? 1 : 0;
  launch([&] {
    return B.mx_downcast(x->data_ptr(), t, ax.outer, ax.len, ax.inner, ax.last ? 1 : ax.inner, so, ax.inner, si, q.data_ptr(), s.data_ptr(),
                         int32_t(kind), int32_t(rounding), *stream);
  });
  Ref qo(THPVariable_Wrap(std::move(q))), sc(THPVariable_Wrap(std::move(s)));
  if (!qo.p || !sc.p) throw PyError();
  return PyTuple_Pack(2, qo.p, sc.p);
}

// Dense with the quantised axis fastest.
bool dense_along(const Tensor& t, const Axis& ax) {
  if (ax.last) return t.is_contiguous();
  const int64_t n = t.dim(), len = t.size(n - 2), inner = t.size(n - 1);
  return (len == 1 || t.stride(n - 2) == 1) && (inner == 1 || t.stride(n - 1) == len) && (n == 2 || t.size(0) == 1 || t.stride(0) == len * inner);
}

// (values, scales, target dtype, axis) -> expanded
PyObject* run_mx_upcast(PyObject* const* v) {
  const Tensor *q = tensor_of(v[0]), *s = tensor_of(v[1]);
  const long axis = PyLong_AsLong(v[3]);
  if (PyErr_Occurred()) throw PyError();
  if (!q || !s || !THPDtype_Check(v[2]) || !q->is_cuda() || !s->is_cuda() || q->dim() < 2 || q->dim() > 3 || s->dim() != q->dim()
      || s->scalar_type() != ScalarType::Byte || q->numel() == 0)
    return none();
  const ScalarType out_t = reinterpret_cast<THPDtype*>(v[2])->scalar_type, qt = q->scalar_type();
  const int32_t out_c = dtype_code(out_t), kind = qt == ScalarType::Byte ? int32_t(TK_E2M1) : dtype_code(qt);
  Axis ax, as;
  if ((out_c != TK_BF16 && out_c != TK_F16 && out_c != TK_F32) || (kind != TK_E2M1 && kind != TK_E4M3 && kind != TK_E5M2) || !ax.of(*q, axis)
      || !as.of(*s, axis))
    return none();
  const int64_t len = ax.len * (kind == TK_E2M1 ? 2 : 1);
  if (len % 32 || as.len * 32 != len || as.outer != ax.outer || as.inner != ax.inner || !dense_along(*q, ax) || !dense_along(*s, as))
    return none();
  auto stream = stream_of(*q);
  if (!stream) return none();
  c10::SmallVector<int64_t, 5> sizes(q->sizes());
  sizes[ax.last ? q->dim() - 1 : q->dim() - 2] = len;
  Tensor out = empty(sizes, out_t, *q);
  launch([&] {
    return B.mx_upcast(q->data_ptr(), s->data_ptr(), kind, ax.outer, len, ax.inner, ax.last ? 1 : ax.inner, out.data_ptr(), out_c,
                       len * ax.inner, ax.inner, 1, *stream);
  });
  return THPVariable_Wrap(std::move(out));
}

// (a [M, R], b [R, N], a's metadata, b's metadata) -> [slices, M, N] in the operands' type
PyObject* run_ragged_k(PyObject* const* v) {
  const Tensor *a = tensor_of(v[0]), *b = tensor_of(v[1]);
  if (!a || !b || !a->is_cuda() || !b->is_cuda() || a->dim() != 2 || b->dim() != 2 || a->scalar_type() != b->scalar_type()) return none();
  const ScalarType t = a->scalar_type();
  if (t != ScalarType::BFloat16 && t != ScalarType::Half) return none();
  Metadata ma, mb;
  if (!ma.read(v[2]) || !mb.read(v[3]) || ma.sizes->size(0) != mb.sizes->size(0)) return none();
  auto stream = stream_of(*a);
  if (!stream) return none();
  const int64_t E = mb.sizes->size(0), M = a->size(0), N = b->size(1);
  Tensor y = empty({E, M, N}, t, *a);
  tk_ragged_k_desc d{};
  d.a = a->data_ptr(), d.dtype = dtype_code(t), d.a_stride_m = a->stride(0), d.a_stride_k = a->stride(1);
  d.b = b->data_ptr(), d.b_stride_k = b->stride(0), d.b_stride_n = b->stride(1);
  d.y = y.data_ptr(), d.y_dtype = d.dtype, d.y_stride_e = y.stride(0), d.y_stride_m = y.stride(1);
  d.M = int32_t(M), d.N = int32_t(N), d.n_slices = int32_t(E);
  d.a_k_extent = a->size(1), d.b_k_extent = b->size(0);
  d.slice_sizes = static_cast<const int32_t*>(mb.sizes->data_ptr());
  d.a_slice_offs = static_cast<const int32_t*>(ma.offs->data_ptr()), d.b_slice_offs = static_cast<const int32_t*>(mb.offs->data_ptr());
  launch([&] { return B.ragged_k_gemm(&d, *stream); });
  return THPVariable_Wrap(std::move(y));
}

// ---- the decode layer -----------------------------------------------------------------------------------------------------------

struct MxWeights {
  const Tensor *w, *s, *bias = nullptr;
  int64_t kn[2];
  bool read(PyObject* wo, PyObject* bo, PyObject* pc, int64_t E) {
    w = storage_of(wo, B.mx_value, kn);
    if (!w || is_none(pc)) return false;
    Ref dt(attr(wo, N_.dtype)), flex(attr(pc, N_.flex_ctx)), axs(attr(pc, N_.a_mx_scale)), ats(attr(pc, N_.a_mx_tensor_scale)),
        bxs(attr(pc, N_.b_mx_scale)), bts(attr(pc, N_.b_mx_tensor_scale)), cxs(attr(pc, N_.c_mx_scale)), od(attr(pc, N_.out_dtype));
    if (dt != B.fp4 || flex != B.default_flex || !is_none(axs) || !is_none(ats) || !is_none(bts) || !is_none(cxs)) return false;
    if (!is_none(od) && !(THPDtype_Check(od) && reinterpret_cast<THPDtype*>(od.p)->scalar_type == ScalarType::BFloat16)) return false;
    s = storage_of(bxs, B.mx_scale, nullptr);
    if (!s || w->scalar_type() != ScalarType::Byte || s->scalar_type() != ScalarType::Byte || !w->is_contiguous() || !s->is_contiguous()
        || w->dim() < 1 || w->size(0) != E || s->dim() < 1 || s->size(0) != E)
      return false;
    if (is_none(bo)) return true;
    bias = tensor_of(bo);
    return bias && bias->dim() == 2 && bias->size(0) == E && bias->size(1) == kn[1] && bias->stride(1) == 1 && f32_or_bf16(*bias);
  }
};

// (x, logits, k, w1, b1, w2, b2, pc1, pc2, activation, most rows, most experts, largest dimension) -> [T, d_model]
PyObject* run_decode_layer(PyObject* const* v) {
  const Tensor *x = tensor_of(v[0]), *lg = tensor_of(v[1]);
  const int64_t k = PyLong_AsLongLong(v[2]), max_rows = PyLong_AsLongLong(v[10]), max_e = PyLong_AsLongLong(v[11]),
                max_dim = PyLong_AsLongLong(v[12]);
  if (PyErr_Occurred()) throw PyError();
  if (!x || !lg || !x->is_cuda() || !lg->is_cuda() || x->dim() != 2 || x->scalar_type() != ScalarType::BFloat16 || lg->dim() != 2
      || !f32_or_bf16(*lg) || lg->size(0) != x->size(0) || lg->stride(1) != 1)
    return none();
  const int64_t T = lg->size(0), E = lg->size(1);
  if (T == 0 || k < 1 || T * k > max_rows || E > max_e || k > std::min<int64_t>(E, 32)) return none();
  Activation act;
  if (!act.read(v[9]) || !act.swiglu) return none();
  MxWeights w1, w2;
  if (!w1.read(v[3], v[4], v[7], E) || !w2.read(v[5], v[6], v[8], E)) return none();
  const int64_t dm = w1.kn[0], ff = w2.kn[0];
  if (x->size(1) != dm || w1.kn[1] != 2 * ff || w2.kn[1] != dm || dm > max_dim || ff > max_dim || dm % 8 || ff % 8) return none();
  if (x->stride(1) != 1 || x->stride(0) < dm || x->stride(0) % 8 || reinterpret_cast<uintptr_t>(x->data_ptr()) % 16
      || ((T - 1) * x->stride(0) + dm) * 2 > 0x7FFFFFFF)
    return none();
  auto stream = stream_of(*x);
  if (!stream) return none();
  Tensor ws;  // (row by row: this call's own; a graph's belongs to the graph)
  if (tk::decode_by_rows(T, k, ff, dm)) {
    ws = empty({B.decode_workspace_bytes(int32_t(T), int32_t(k), int32_t(E), int32_t(ff), int32_t(dm))}, ScalarType::Byte, *x);
  } else {
    Ref dev(attr(v[0], N_.device)), t_o(PyLong_FromLongLong(T)), e_o(PyLong_FromLongLong(E)), f_o(PyLong_FromLongLong(ff)),
        d_o(PyLong_FromLongLong(dm));
    PyObject* args[6] = {dev, t_o, v[2], e_o, f_o, d_o};
    Ref kept(PyObject_Vectorcall(B.decode_workspace, args, 6, nullptr));
    if (!kept) throw PyError();
    ws = THPVariable_Unpack(kept.p);
  }
  Tensor out = empty({T, dm}, ScalarType::BFloat16, *x);
  tk_decode_layer_desc d{};
  d.x = x->data_ptr(), d.x_stride_m = x->stride(0);
  d.logits = lg->data_ptr(), d.logits_dtype = dtype_code(lg->scalar_type()), d.logits_stride_m = lg->stride(0);
  d.n_tokens = int32_t(T), d.n_experts = int32_t(E), d.k = int32_t(k), d.apply_softmax = 1, d.d_model = int32_t(dm), d.d_ff = int32_t(ff);
  d.w1 = static_cast<const uint8_t*>(w1.w->data_ptr()), d.w1_mx_scale = static_cast<const uint8_t*>(w1.s->data_ptr());
  d.w1_stride_e = w1.w->stride(0), d.w1s_stride_e = w1.s->stride(0);
  d.w2 = static_cast<const uint8_t*>(w2.w->data_ptr()), d.w2_mx_scale = static_cast<const uint8_t*>(w2.s->data_ptr());
  d.w2_stride_e = w2.w->stride(0), d.w2s_stride_e = w2.s->stride(0);
  if (w1.bias) d.b1 = w1.bias->data_ptr(), d.b1_dtype = dtype_code(w1.bias->scalar_type()), d.b1_stride_e = w1.bias->stride(0);
  if (w2.bias) d.b2 = w2.bias->data_ptr(), d.b2_dtype = dtype_code(w2.bias->scalar_type()), d.b2_stride_e = w2.bias->stride(0);
  d.act_alpha = float(act.alpha), d.act_limit = float(act.limit), d.act_has_limit = act.has_limit;
  d.out = out.data_ptr(), d.out_stride_m = dm;
  d.workspace = ws.data_ptr();
  launch([&] { return B.decode_layer(&d, *stream); });
  return THPVariable_Wrap(std::move(out));
}

// ---- module -----------------------------------------------------------------------------------------------------------------

// f(args) with the number of arguments checked and C++ exceptions turned into Python's
template <PyObject* (*f)(PyObject* const*), int n>
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t given) {
  if (given != n) return PyErr_Format(PyExc_TypeError, "takes %d arguments (%zd given)", n, given);
  HANDLE_TH_ERRORS
  try {
    return f(args);
  } catch (const PyError&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// The rules and conditions for the general host path, on integers.
template <size_t n>
std::array<int64_t, n> integers(PyObject* const* v) {
  std::array<int64_t, n> a;
  for (size_t i = 0; i < n; ++i) a[i] = PyLong_AsLongLong(v[i]);
  if (PyErr_Occurred()) throw PyError();
  return a;
}
PyObject* rule_x_extent(PyObject* const* v) {
  const auto [rows, stride, K, itemsize] = integers<4>(v);
  return PyLong_FromUnsignedLong(tk::x_extent(rows, stride, K, itemsize));
}
PyObject* rule_dma_16bit(PyObject* const* v) {
  const auto [x_bytes, n_slices, K, N, w_stride_n] = integers<5>(v);
  return PyBool_FromLong(tk::dma_runs_16bit(uint32_t(x_bytes), n_slices, K, N, w_stride_n));
}
PyObject* rule_dma(PyObject* const* v) {
  const auto [rows, row_bytes, N, n_slices] = integers<4>(v);
  return PyLong_FromLongLong(dma_block_m(rows, row_bytes, N, n_slices));
}
PyObject* rule_few(PyObject* const* v) {
  const auto [rows, N, n_slices] = integers<3>(v);
  return PyLong_FromLongLong(few_block_n(rows, N, n_slices));
}
PyObject* rule_dma_n(PyObject* const* v) {
  const auto [rows, N, n_slices, block_m] = integers<4>(v);
  return PyLong_FromLongLong(dma_block_n(rows, N, n_slices, block_m, false));
}
PyObject* rule_dma_n_16bit(PyObject* const* v) {
  const auto [rows, N, n_slices, block_m] = integers<4>(v);
  return PyLong_FromLongLong(dma_block_n(rows, N, n_slices, block_m, true));
}
PyObject* rule_dma_e4m3(PyObject* const* v) {
  const auto [x_bytes, n_slices, K, N] = integers<4>(v);
  return PyBool_FromLong(tk::dma_runs_e4m3(uint32_t(x_bytes), n_slices, K, N));
}
PyObject* rule_decode_rows(PyObject* const* v) {
  const auto [T, k, d_ff, d_model] = integers<4>(v);
  return PyBool_FromLong(tk::decode_by_rows(T, k, d_ff, d_model));
}
PyObject* rule_decode_fetch(PyObject* const* v) {
  const auto [T, k, E, blocks_of_expert] = integers<4>(v);
  return PyLong_FromLong(tk::decode_fetch(T, k, E, blocks_of_expert));
}
PyObject* rule_fp8(PyObject* const* v) {
  const auto [rows, x_bytes, K, N, n_slices] = integers<5>(v);
  return PyLong_FromLongLong(fp8_block_m(rows, uint32_t(x_bytes), K, N, n_slices));
}
PyObject* rule_mxfp4(PyObject* const* v) {
  const auto [rows, n_slices, otherwise] = integers<3>(v);
  return PyLong_FromLongLong(mxfp4_block_m(rows, n_slices, otherwise));
}
PyObject* rule_wide_n(PyObject* const* v) {
  const auto [rows, n_slices, K, N, x_bytes, mx8] = integers<6>(v);
  return PyLong_FromLongLong(wide_block_n(rows, n_slices, K, N, uint32_t(x_bytes), mx8 != 0));
}
PyObject* rule_wide(PyObject* const* v) {
  const auto [rows, n_slices, K, N, x_bytes, mx8] = integers<6>(v);
  return PyLong_FromLongLong(wide_block_m(rows, n_slices, K, N, uint32_t(x_bytes), mx8 != 0));
}
PyObject* rule_ragged_k_tile(PyObject* const* v) {
  const auto [k, M, N, n_slices] = integers<4>(v);
  return PyLong_FromLong(tk::ragged_k_tile(k, M, N, n_slices));
}
PyObject* rule_mx_tiles(PyObject* const* v) {
  const auto [outer, L, inner, e2m1, down, rows8] = integers<6>(v);
  const tk::MxTiles t = tk::mx_tiles(outer, L, inner, e2m1 != 0, down != 0, rows8 != 0);
  return Py_BuildValue("(Lii)", (long long)t.grid, (int)t.blocks, (int)(down ? t.once : t.together));
}
PyObject* rule_mx_by_columns(PyObject* const* v) {
  const auto [outer, L, inner] = integers<3>(v);
  return PyBool_FromLong(tk::mx_by_columns(outer, L, inner));
}

// bind(dict): the addresses of the entry points (integers) and the Python objects above
PyObject* bind(PyObject*, PyObject* dict) {
  auto get = [&](const char* n) -> PyObject* {
    PyObject* o = PyDict_GetItemString(dict, n);
    if (!o) PyErr_Format(PyExc_KeyError, "%s", n);
    return o;
  };
#define ENTRY(field, name)                                                                   \
  if (PyObject* o = get(#name)) {                                                            \
    B.field = reinterpret_cast<decltype(B.field)>(PyLong_AsVoidPtr(o));                      \
    if (!B.field) return PyErr_Format(PyExc_ValueError, "no address for %s", #name);         \
  } else {                                                                                   \
    return nullptr;                                                                          \
  }
  ENTRY(moe_gemm, tk_moe_gemm)
  ENTRY(route, tk_route)
  ENTRY(route_workspace_bytes, tk_route_workspace_bytes)
  ENTRY(reduce_mid, tk_reduce_mid)
  ENTRY(quant_fp8_rows, tk_quant_fp8_rows)
  ENTRY(mx_downcast, tk_mx_downcast)
  ENTRY(mx_upcast, tk_mx_upcast)
  ENTRY(ragged_k_gemm, tk_ragged_k_gemm)
  ENTRY(decode_layer, tk_moe_decode_layer)
  ENTRY(decode_workspace_bytes, tk_moe_decode_layer_workspace_bytes)
#undef ENTRY
#define OBJECT(name)                            \
  if (!(B.name = get(#name))) return nullptr;   \
  Py_INCREF(B.name);
  OBJECT(check) OBJECT(raw_stream) OBJECT(current_device) OBJECT(tile_counters) OBJECT(combine_counters) OBJECT(decode_workspace)
  OBJECT(tensor_type) OBJECT(mx_value) OBJECT(mx_scale) OBJECT(fp8_value) OBJECT(fp4) OBJECT(metadata_type) OBJECT(routing_type)
  OBJECT(gather_type) OBJECT(scatter_type) OBJECT(default_flex) OBJECT(no_activation) OBJECT(no_epilogue)
#undef OBJECT
  Py_RETURN_NONE;
}

#define METHOD(name, f, n) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&call<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    // (a, b, bias, metadata, gather, scatter, precision config, gammas, activation, epilogue, combine k, idle CUs)
    METHOD("gemm", run_gemm, 12),
    METHOD("route", run_route, 3),
    METHOD("combine", run_combine, 2),
    METHOD("quant_fp8_rows", run_quant_fp8_rows, 1),
    METHOD("mx_downcast", run_mx_downcast, 4),
    METHOD("mx_upcast", run_mx_upcast, 4),
    METHOD("ragged_k", run_ragged_k, 4),
    METHOD("decode_layer", run_decode_layer, 13),
    METHOD("x_extent", rule_x_extent, 4),
    METHOD("dma_runs_16bit", rule_dma_16bit, 5),
    METHOD("dma_block_m", rule_dma, 4),
    METHOD("dma_runs_e4m3", rule_dma_e4m3, 4),
    METHOD("dma_block_n", rule_dma_n, 4),
    METHOD("dma_block_n_16bit", rule_dma_n_16bit, 4),
    METHOD("few_block_n", rule_few, 3),
    METHOD("decode_by_rows", rule_decode_rows, 4),
    METHOD("decode_fetch", rule_decode_fetch, 4),
    METHOD("fp8_block_m", rule_fp8, 5),
    METHOD("mxfp4_block_m", rule_mxfp4, 3),
    METHOD("wide_block_m", rule_wide, 6),
    METHOD("wide_block_n", rule_wide_n, 6),
    METHOD("ragged_k_tile", rule_ragged_k_tile, 4),
    METHOD("mx_tiles", rule_mx_tiles, 6),
    METHOD("mx_by_columns", rule_mx_by_columns, 3),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", "Native host path of triton_amd.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
#define X(n) N_.n = PyUnicode_InternFromString(#n);
  NAMES(X)
#undef X
  return PyModule_Create(&module_def);
}
