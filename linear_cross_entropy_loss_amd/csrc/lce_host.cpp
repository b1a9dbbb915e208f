// Host path of the Python operator (ops.py) for ordinary calls: from the tensors to one call of the C ABI (include/lce.h) and its
// results, without the interpreter in between.
//
// A step of a small problem is bound by the host: N=256, H=256, V=4096 in bf16 has 43 us of kernels and took 81 us of host time in
// Python, 51 here -- 160 and 106 where the threads of a backward, which wait for each other, sleep long enough for the processor's
// deeper idle states.
//
// What is no such call -- a tensor subclass, strides in no order of rows, a problem that the library refuses -- is not handled
// here: the functions return None before anything has been allocated or launched, and ops.py goes on as for any call, errors
// included.  Device calls go to the current device and the stream that is handed over; allocations come from torch's caching
// allocator, as the current stream's.
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/Allocator.h>

#include "../../include/lce.h"

namespace {

// The C ABI's functions, by the addresses that the loader of the library gives (bind).
struct Abi {
  decltype(&lce_check_problem) check_problem;
  decltype(&lce_workspace_bytes) workspace_bytes;
  decltype(&lce_forward) forward;
  decltype(&lce_backward) backward;
  decltype(&lce_forward_backward_workspace_bytes) forward_backward_workspace_bytes;
  decltype(&lce_forward_backward_plan) forward_backward_plan;
  decltype(&lce_forward_backward) forward_backward;
  decltype(&lce_stand_in) stand_in;
  decltype(&lce_unit_gradient) unit_gradient;
  decltype(&lce_pad_rows) pad_rows;
  decltype(&lce_transpose_rows) transpose_rows;
} abi;

template <class F> void bind_one(const py::dict& d, const char* name, F& f) { f = reinterpret_cast<F>(d[name].cast<uintptr_t>()); }
void bind(const py::dict& d) {
  bind_one(d, "lce_check_problem", abi.check_problem);
  bind_one(d, "lce_workspace_bytes", abi.workspace_bytes);
  bind_one(d, "lce_forward", abi.forward);
  bind_one(d, "lce_backward", abi.backward);
  bind_one(d, "lce_forward_backward_workspace_bytes", abi.forward_backward_workspace_bytes);
  bind_one(d, "lce_forward_backward_plan", abi.forward_backward_plan);
  bind_one(d, "lce_forward_backward", abi.forward_backward);
  bind_one(d, "lce_stand_in", abi.stand_in);
  bind_one(d, "lce_unit_gradient", abi.unit_gradient);
  bind_one(d, "lce_pad_rows", abi.pad_rows);
  bind_one(d, "lce_transpose_rows", abi.transpose_rows);
}

int dtype_code(at::ScalarType t) {
  return t == at::kBFloat16 ? LCE_BF16 : t == at::kHalf ? LCE_F16 : t == at::kFloat ? LCE_F32 : -1;
}
int64_t row_multiple(at::ScalarType t) { return t == at::kFloat ? 4 : 8; }

// A dense tensor on a GPU that is nothing but that.
bool plain(const at::Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.unsafeGetTensorImpl()->is_python_dispatch() && !t.is_neg() &&
         !t.is_conj();
}
bool aligned(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// Memory that is given back when the call's launches have been issued (the allocator hands it out again in stream order).
struct Workspace {
  c10::DataPtr data;
  explicit Workspace(size_t n) : data(n > 0 ? c10::GetAllocator(c10::DeviceType::CUDA)->allocate(n) : c10::DataPtr()) {}
};

py::object tensor_or_none(const at::Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

// Row strides of matrices that are laid out here (ops.py, _padded_cols and _dx_cols).
int64_t padded_cols(int64_t cols, at::ScalarType t) {
  int64_t m = row_multiple(t);
  if (cols % m == 0) return cols;
  if (2 * cols >= 8 * m) m *= 8;
  return (cols + m - 1) / m * m;
}
int64_t dx_cols(int64_t H, at::ScalarType t) { return H % 4 == 0 ? H : padded_cols(H, t); }

// How the kernels come to a matrix: as it is, or from a copy whose rows start on 16-byte boundaries.
enum Copy { kInPlace, kByRows, kTransposed };
struct Call {
  lce_problem p;
  Copy x, w;
};

// x: rows of H, contiguous or (`strided`) with a row stride.  At: (H, V), as the operator takes it.  False: no ordinary call.
bool describe(const at::Tensor& x, const at::Tensor& At, bool strided, Call& c) {
  memset(&c, 0, sizeof(c));
  if (!plain(x) || !plain(At) || x.dim() < 1 || At.dim() != 2 || x.device() != At.device()) return false;
  const at::ScalarType xt = x.scalar_type(), wt = At.scalar_type();
  const int xd = dtype_code(xt), wd = dtype_code(wt);
  if (xd < 0 || (wd != xd && wd != LCE_F32)) return false;
  const int64_t H = x.size(-1), V = At.size(1), m = row_multiple(wt);
  if (H <= 0 || V <= 0 || At.size(0) != H || x.numel() <= 0) return false;
  lce_problem& p = c.p;
  if (strided) {
    if (x.dim() != 2 || x.stride(1) != 1 || x.stride(0) % row_multiple(xt) != 0 || x.stride(0) < H || !aligned(x)) return false;
    p.ldx = x.stride(0);
  } else {
    if (!x.is_contiguous()) return false;
    c.x = H % row_multiple(xt) == 0 && aligned(x) ? kInPlace : kByRows;
    p.ldx = c.x == kInPlace ? H : padded_cols(H, xt);
  }
  p.N = x.numel() / H;
  p.H = H;
  p.V = V;
  p.lddx = dx_cols(H, xt);
  p.x_dtype = p.dx_dtype = xd;
  p.w_dtype = p.dw_dtype = wd;
  p.w_layout = LCE_W_HV;
  if (At.stride(1) == 1 && At.stride(0) % m == 0 && At.stride(0) >= V) {
    if (!aligned(At)) return false;
    p.ldw = At.stride(0);
  } else if (xd != LCE_F32 && H % 8 == 0 && V > 1 && At.stride(0) == 1 && At.stride(1) % m == 0 && At.stride(1) >= H) {
    if (!aligned(At)) return false;
    p.w_layout = LCE_W_VH;
    p.ldw = At.stride(1);
  } else {
    if (At.stride(1) == 1 && At.stride(0) >= V) c.w = kByRows;
    else if (At.stride(0) == 1 && At.stride(1) >= H) c.w = kTransposed;
    else return false;
    p.ldw = padded_cols(V, wt);
  }
  p.lddw = padded_cols(p.w_layout == LCE_W_VH ? H : V, wt);
  return true;
}

at::Tensor rows_of(int64_t rows, int64_t cols, int64_t ld, const at::TensorOptions& o) {
  at::Tensor t = at::empty({rows, ld}, o);
  return ld == cols ? t : t.narrow(1, 0, cols);
}
int copy_rows(Copy how, const at::Tensor& from, int64_t rows, int64_t cols, const at::Tensor& to, int64_t ld, void* stream) {
  const int d = dtype_code(to.scalar_type());
  return how == kByRows ? abi.pad_rows(from.data_ptr(), d, rows, cols, from.dim() == 2 ? from.stride(0) : cols, to.data_ptr(), ld, stream)
                        : abi.transpose_rows(from.data_ptr(), d, rows, cols, from.stride(1), to.data_ptr(), ld, stream);
}

// The loss, and with `route` (1: where the library says so, 2: wherever it fits) and a gradient wanted, that too if one evaluation of
// the logits gives both: (out5, lse, n_valid, x, y, w, layout, dx, dw, pre), as ops.py's _one_pass_impl and _forward_impl return
// them, then whether the gradients are there; (status, name) where the C ABI refused; None: not handled.  `copy_w`: a weight that
// cannot be read in place may be copied here (ops.py says so to the user once).
py::object forward(const at::Tensor& x_in, const at::Tensor& y, const at::Tensor& At, int64_t ignore_index, double z_reg, double scale,
                   int64_t n_chunk, bool monitoring, int pack, int route, bool exact, bool need_dx, bool need_dw, bool copy_w, uintptr_t stream) {
  Call c;
  lce_problem& p = c.p;
  if (!describe(x_in, At, false, c) || (c.w != kInPlace && !copy_w) || !plain(y) || y.scalar_type() != at::kLong || y.device() != x_in.device() || !y.is_contiguous() ||
      y.numel() != p.N)
    return py::none();
  p.ignore_index = ignore_index;
  p.logit_scale = (float)scale;
  p.z_reg = (float)z_reg;
  p.n_chunk = n_chunk;
  p.monitoring = monitoring ? 1 : 0;
  p.pack_rows = pack;
  const bool grads = route > 0 && (need_dx || need_dw);
  if (grads)
    p.route = (route == 2 ? LCE_ROUTE_ONE_PASS : LCE_ROUTE_AUTO) | (exact ? LCE_ROUTE_EXACT_SUMS : 0) |
              (p.x_dtype == LCE_F32 ? LCE_ROUTE_KEEP_LOGITS : 0);
  if (abi.check_problem(&p) != LCE_OK) return py::none();
  int64_t chunks = 0;
  if (grads && abi.forward_backward_plan(&p, &chunks, nullptr) != LCE_OK) return py::none();
  size_t bytes = 0;
  if ((chunks > 0 ? abi.forward_backward_workspace_bytes(&p, &bytes) : abi.workspace_bytes(&p, &bytes, nullptr)) != LCE_OK)
    return py::none();

  at::NoGradGuard no_grad;
  const auto o = x_in.options();
  const at::Tensor y1 = y.dim() == 1 ? y : y.view({p.N});
  const at::Tensor x = c.x != kInPlace ? rows_of(p.N, p.H, p.ldx, o) : x_in.dim() == 2 ? x_in : x_in.view({p.N, p.H});
  const at::Tensor w = c.w != kInPlace ? rows_of(p.H, p.V, p.ldw, At.options()) : p.w_layout == LCE_W_VH ? At.t() : At;
  at::Tensor dx, dw, pre;
  if (chunks > 0 && need_dx) dx = rows_of(p.N, p.H, p.lddx, o);
  if (chunks > 0 && need_dw) dw = rows_of(w.size(0), w.size(1), p.lddw, At.options());
  const auto f32 = o.dtype(at::kFloat);
  const at::Tensor lse = at::empty({p.N}, f32), out5 = at::empty({5}, f32), n_valid = at::empty({1}, y.options());
  if (chunks > 0 && p.x_dtype == LCE_F16) pre = at::empty({1}, f32);
  Workspace ws(bytes);
  void* const s = reinterpret_cast<void*>(stream);
  int rc = LCE_OK;
  const char* what = chunks > 0 ? "lce_forward_backward" : "lce_forward";
  {
    py::gil_scoped_release release;
    if (c.x != kInPlace) rc = copy_rows(c.x, x_in, p.N, p.H, x, p.ldx, s);
    if (rc == LCE_OK && c.w != kInPlace) rc = copy_rows(c.w, At, p.H, p.V, w, p.ldw, s);
    if (rc != LCE_OK) {
      what = "lce_pad_rows";
    } else if (chunks > 0) {
      const float* g = nullptr;
      if (pre.defined()) {
        rc = abi.stand_in((const int64_t*)y1.data_ptr(), p.N, ignore_index, (float*)pre.data_ptr(), s);
        g = (const float*)pre.data_ptr();
      } else {
        rc = abi.unit_gradient(&g);
      }
      if (rc == LCE_OK)
        rc = abi.forward_backward(&p, x.data_ptr(), w.data_ptr(), (const int64_t*)y1.data_ptr(), g, (float*)lse.data_ptr(),
                                  (float*)out5.data_ptr(), (int64_t*)n_valid.data_ptr(), ptr(dx), ptr(dw), ws.data.get(), bytes, s);
    } else {
      rc = abi.forward(&p, x.data_ptr(), w.data_ptr(), (const int64_t*)y1.data_ptr(), (float*)lse.data_ptr(), (float*)out5.data_ptr(),
                       (int64_t*)n_valid.data_ptr(), ws.data.get(), bytes, s);
    }
  }
  if (rc != LCE_OK) return py::make_tuple(rc, what);
  return py::make_tuple(out5, lse, n_valid, x, y1, w, p.w_layout, tensor_or_none(dx), tensor_or_none(dw), tensor_or_none(pre),
                        chunks > 0);
}

// The gradients by recomputing the logits, of what forward saved: (dx, dw), dense, dw as it is stored.  None: not handled.
py::object backward(const at::Tensor& x, const at::Tensor& y1, const at::Tensor& w, const at::Tensor& lse, const at::Tensor& n_valid,
                    const at::Tensor& g, int64_t ignore_index, double z_reg, double scale, int64_t n_chunk, bool need_dx, bool need_dw,
                    int pack, int layout, uintptr_t stream) {
  Call c;
  lce_problem& p = c.p;
  if (!(need_dx || need_dw) || w.dim() != 2) return py::none();
  if (!describe(x, layout == LCE_W_VH ? w.t() : w, true, c) || c.w != kInPlace || p.w_layout != layout) return py::none();
  for (const at::Tensor& t : {y1, lse, n_valid, g})
    if (!plain(t) || t.device() != x.device() || !t.is_contiguous()) return py::none();
  if (y1.scalar_type() != at::kLong || y1.numel() != p.N || lse.scalar_type() != at::kFloat || lse.numel() != p.N ||
      n_valid.scalar_type() != at::kLong || g.scalar_type() != at::kFloat || g.numel() != 1)
    return py::none();
  p.ignore_index = ignore_index;
  p.logit_scale = (float)scale;
  p.z_reg = (float)z_reg;
  p.n_chunk = n_chunk;
  p.pack_rows = pack;
  size_t bytes = 0;
  if (abi.check_problem(&p) != LCE_OK || abi.workspace_bytes(&p, nullptr, &bytes) != LCE_OK) return py::none();

  at::NoGradGuard no_grad;
  at::Tensor dx, dw;
  if (need_dx) dx = rows_of(p.N, p.H, p.lddx, x.options());
  if (need_dw) dw = rows_of(w.size(0), w.size(1), p.lddw, w.options());
  Workspace ws(bytes);
  int rc;
  {
    py::gil_scoped_release release;
    rc = abi.backward(&p, x.data_ptr(), w.data_ptr(), (const int64_t*)y1.data_ptr(), (const float*)lse.data_ptr(),
                      (const int64_t*)n_valid.data_ptr(), (const float*)g.data_ptr(), ptr(dx), ptr(dw), ws.data.get(), bytes,
                      reinterpret_cast<void*>(stream));
  }
  if (rc != LCE_OK) return py::make_tuple(rc, "lce_backward", py::none());
  if (need_dx) dx = dx.contiguous();
  if (need_dw) dw = dw.contiguous();
  return py::make_tuple(tensor_or_none(dx), tensor_or_none(dw));
}

}  // namespace

PYBIND11_MODULE(_lce_host, m) {
  m.def("bind", &bind);
  m.def("forward", &forward);
  m.def("backward", &backward);
}
