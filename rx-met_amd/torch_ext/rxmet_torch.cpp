// rxmet_torch.cpp — the autograd node of QuantizeDequantize's learnable min / max path in C++
// (module rxmet_torch, over librxmet.so's rxmet_qdq_forward_minmax / _backward_minmax).
//
// A training step of a small fake-quantised tensor is bound by the host: forward and backward of
// [64, 576] fp32, per channel, take 15 us of kernels and took 155 - 163 us through a Python
// autograd.Function with its bookkeeping.  This node makes the same allocations and launches
// without the interpreter: 67 us (bf16 [3001, 4099], per tensor: 156 -> 67 us for 62 us of
// kernels).  mi355x_qdq.py keeps the Python Function for what this one does not take: tensors that
// have to be copied first, tracing and tensor subclasses (_native_node there).
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <memory>
#include <stdexcept>
#include <string>

#include "rxmet_qdq.h"

namespace {

// The entry points of the librxmet.so that rxmet_lib.py has loaded (bind()): the module links to
// none by itself, so that one process never holds two copies of the library.
decltype(&rxmet_qdq_forward_minmax) forward_minmax = nullptr;
decltype(&rxmet_qdq_backward_minmax) backward_minmax = nullptr;
decltype(&rxmet_qdq_workspace_bytes_ex) workspace_bytes = nullptr;
const char *(*last_error)(void) = nullptr;

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Everything of a call that follows from shapes, types and options: made once per combination.
struct MinMaxPlan : torch::CustomClassHolder {
  rxmet_qdq_layout layout;
  rxmet_qdq_numerics numerics;
  at::ScalarType io;
  int64_t qmin, qmax, workspace;
  int32_t symmetric;
  float sym_offset, min_scale;
};

struct LibraryError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

void check(int rc, const char *what) {
  if (rc != 0)
    throw LibraryError(std::string(what) + " failed (" + std::to_string(rc) +
                       "): " + last_error());
}

rxmet_qdq_minmax_enc enc_of(const MinMaxPlan &p, const at::Tensor &mn, const at::Tensor &mx) {
  return {mn.const_data_ptr<float>(), mx.const_data_ptr<float>(), p.symmetric, p.sym_offset,
          p.min_scale, 0};
}

void check_tensors(const at::Tensor &x, const at::Tensor &mn, const at::Tensor &mx,
                   const MinMaxPlan &p) {
  const rxmet_qdq_layout &l = p.layout;
  const int64_t n = l.outer * l.C0 * l.mid * l.C1 * l.inner, c = l.C0 * l.C1;
  TORCH_CHECK(x.is_cuda() && mn.device() == x.device() && mx.device() == x.device() &&
                  x.scalar_type() == p.io && mn.scalar_type() == at::kFloat &&
                  mx.scalar_type() == at::kFloat && x.is_contiguous() && mn.is_contiguous() &&
                  mx.is_contiguous() && x.numel() == n && mn.numel() == c && mx.numel() == c,
              "qdq_minmax: the tensors do not match the plan");
}

void *stream_of(const at::Tensor &t) {
  return c10::hip::getCurrentHIPStream(t.get_device()).stream();
}

struct QdqMinMax : public torch::autograd::Function<QdqMinMax> {
  static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x, const at::Tensor &mn,
                            const at::Tensor &mx, const c10::intrusive_ptr<MinMaxPlan> &plan) {
    const c10::DeviceGuard guard(x.device());
    at::Tensor y = at::empty_like(x);
    const rxmet_qdq_minmax_enc enc = enc_of(*plan, mn, mx);
    check(forward_minmax(x.const_data_ptr(), y.mutable_data_ptr(), &plan->layout,
                         &plan->numerics, &enc, plan->qmin, plan->qmax, stream_of(x)),
          "rxmet_qdq_forward_minmax");
    ctx->save_for_backward({x, mn, mx});
    ctx->saved_data["plan"] = c10::IValue::make_capsule(plan);
    return y;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const at::Tensor &x = saved[0], &mn = saved[1], &mx = saved[2];
    const c10::intrusive_ptr<c10::intrusive_ptr_target> held = ctx->saved_data["plan"].toCapsule();
    const MinMaxPlan &p = *static_cast<MinMaxPlan *>(held.get());
    // unpack hooks may hand back other tensors than were packed
    check_tensors(x, mn, mx, p);
    const c10::DeviceGuard guard(x.device());
    const at::Tensor g = grads[0].to(x.scalar_type()).contiguous();
    const bool need_x = ctx->needs_input_grad(0), need_mn = ctx->needs_input_grad(1),
               need_mx = ctx->needs_input_grad(2), need_enc = need_mn || need_mx;
    at::Tensor dx = at::empty_like(x), d_min, d_max, ws;
    if (need_enc) {
      d_min = at::empty_like(mn);
      d_max = at::empty_like(mx);
      ws = at::empty({p.workspace}, x.options().dtype(at::kByte));
    }
    const rxmet_qdq_minmax_enc enc = enc_of(p, mn, mx);
    check(backward_minmax(
              x.const_data_ptr(), g.const_data_ptr(), dx.mutable_data_ptr(),
              need_enc ? d_min.mutable_data_ptr<float>() : nullptr,
              need_enc ? d_max.mutable_data_ptr<float>() : nullptr, &p.layout, &p.numerics, &enc,
              p.qmin, p.qmax, need_enc ? ws.mutable_data_ptr() : nullptr, stream_of(x)),
          "rxmet_qdq_backward_minmax");
    return {need_x ? dx : at::Tensor(), need_mn ? d_min : at::Tensor(),
            need_mx ? d_max : at::Tensor(), at::Tensor()};
  }
};

c10::intrusive_ptr<MinMaxPlan> make_plan(const std::vector<int64_t> &layout, int32_t io,
                                         int32_t internal, double shift, bool scalar_scale,
                                         int64_t qmin, int64_t qmax, bool symmetric,
                                         float sym_offset, float min_scale) {
  TORCH_CHECK(forward_minmax && last_error, "bind() comes first");
  TORCH_CHECK(layout.size() == 5 && io >= RXMET_QDQ_F32 && io <= RXMET_QDQ_F64,
              "a layout has five sizes, an io type four values");
  static constexpr at::ScalarType kIo[] = {at::kFloat, at::kHalf, at::kBFloat16, at::kDouble};
  auto p = c10::make_intrusive<MinMaxPlan>();
  p->layout = {layout[0], layout[1], layout[2], layout[3], layout[4]};
  p->numerics = {io, internal, shift, scalar_scale ? 1 : 0, 0};
  p->io = kIo[io];
  p->qmin = qmin;
  p->qmax = qmax;
  p->symmetric = symmetric ? 1 : 0;
  p->sym_offset = sym_offset;
  p->min_scale = min_scale;
  p->workspace = std::max<int64_t>(workspace_bytes(&p->layout, io), 16);
  return p;
}

at::Tensor qdq_minmax(const at::Tensor &x, const at::Tensor &mn, const at::Tensor &mx,
                      const c10::intrusive_ptr<MinMaxPlan> &plan) {
  check_tensors(x, mn, mx, *plan);
  return QdqMinMax::apply(x, mn, mx, plan);
}

void bind(uintptr_t forward, uintptr_t backward, uintptr_t workspace, uintptr_t error) {
  forward_minmax = reinterpret_cast<decltype(forward_minmax)>(forward);
  backward_minmax = reinterpret_cast<decltype(backward_minmax)>(backward);
  workspace_bytes = reinterpret_cast<decltype(workspace_bytes)>(workspace);
  last_error = reinterpret_cast<decltype(last_error)>(error);
}

}  // namespace

PYBIND11_MODULE(rxmet_torch, m) {
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const LibraryError &e) {
      py::set_error(py::module_::import("rxmet_lib").attr("RxmetError"), e.what());
    }
  });
  py::class_<MinMaxPlan, c10::intrusive_ptr<MinMaxPlan>>(m, "MinMaxPlan");
  m.def("bind", &bind);
  m.def("make_plan", &make_plan);
  m.def("qdq_minmax", &qdq_minmax);
}
