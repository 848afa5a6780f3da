// The calls whose host time is a large part of a small layer, as native code: the dynamic W8A8 Linear
// (quantization/kernels/scale_mm.py) and torch.ops._C.silu_and_mul on GPU tensors. They check what the Python code checks and
// leave every call that is not the ordinary one - another device, type, layout, a tensor subclass, wrong shapes - to it.
// A dense W8A8 MLP (two Linears around SiLU-mul) of 64 rows took 29.9 us of host time in Python, of 4 rows 24.5, most of it
// beside the launches (about 2.5 us each, five and three); here 24.3 and 21.2.
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>
#include <torch/library.h>

#include "kmoe.h"

namespace py = pybind11;

namespace {

py::object* g_silu_python = nullptr;  // the operator's Python body (kept for the life of the process)
py::object* g_check = nullptr;        // status code -> exception

void check(int rc) {
  if (rc != KMOE_OK) (*g_check)(rc);
}

bool activations(const at::Tensor& t, int* dtype) {
  const auto type = t.scalar_type();
  *dtype = type == at::kHalf ? KMOE_DT_F16 : KMOE_DT_BF16;
  return t.is_cuda() && (type == at::kBFloat16 || type == at::kHalf) && t.is_contiguous();
}

// The argument block of one Linear with everything but the batch; a call is one or two launches on the current stream, a
// scratch buffer of the allocator's (ordered by that stream, the graph's own while one is captured) and the output.
class Linear {
 public:
  Linear(uintptr_t w, uintptr_t w_max, int n, int k, int w_layout, int device, int max_rows)
      : device_(static_cast<c10::DeviceIndex>(device)), max_rows_(max_rows) {
    args_ = kmoe_linear_i8_args{};
    args_.w = reinterpret_cast<const int8_t*>(w);
    args_.w_max = reinterpret_cast<const float*>(w_max);
    args_.n = n;
    args_.k = k;
    args_.ld_x = k;
    args_.ldy = n;
    args_.w_layout = w_layout;
  }

  // None: a call for the Python code
  py::object operator()(py::handle object) const {
    if (!THPVariable_CheckExact(object.ptr())) return py::none();
    const at::Tensor& x = THPVariable_Unpack(object.ptr());
    int dtype;
    if (x.dim() != 2 || x.size(1) != args_.k || x.size(0) < 1 || x.size(0) > max_rows_ || !activations(x, &dtype) ||
        x.device().index() != device_ || c10::hip::current_device() != device_)
      return py::none();
    const int64_t rows = x.size(0);
    kmoe_linear_i8_args a = args_;  // a copy: threads may share the object
    at::Tensor y = at::empty({rows, args_.n}, x.options().requires_grad(false));
    const int64_t need = (rows * args_.k + 255) / 256 * 256 + 4 * rows;
    at::Tensor scratch = at::empty({need}, x.options().dtype(at::kByte).requires_grad(false));
    a.x = static_cast<const uint16_t*>(x.const_data_ptr());
    a.rows = static_cast<int32_t>(rows);
    a.y = static_cast<uint16_t*>(y.mutable_data_ptr());
    a.act_dtype = dtype;
    a.scratch = scratch.mutable_data_ptr();
    a.scratch_bytes = static_cast<size_t>(need);
    int rc;
    {
      py::gil_scoped_release nothing_of_python;
      rc = kmoe_linear_i8(&a, c10::hip::getCurrentHIPStream(device_).stream());
    }
    check(rc);
    return py::reinterpret_steal<py::object>(THPVariable_Wrap(std::move(y)));
  }

 private:
  kmoe_linear_i8_args args_;
  c10::DeviceIndex device_;
  int64_t max_rows_;
};

void silu_and_mul(at::Tensor out, const at::Tensor& x, int64_t axis, bool turn) {
  int dtype, dtype_out;
  const int64_t two_d = x.dim() > 0 ? x.size(-1) : 0;
  const int64_t rows = two_d > 0 ? x.numel() / two_d : 0;
  int rc = KMOE_OK;
  if (activations(x, &dtype) && activations(out, &dtype_out) && dtype == dtype_out && two_d > 0 && two_d % 2 == 0 &&
      out.numel() == rows * (two_d / 2) && rows < (1ll << 31) && two_d < (1ll << 31)) {
    rc = kmoe_silu_and_mul_dt(static_cast<const uint16_t*>(x.const_data_ptr()), two_d, static_cast<int>(rows), static_cast<int>(two_d / 2),
                              static_cast<uint16_t*>(out.mutable_data_ptr()), two_d / 2, dtype, c10::hip::getCurrentHIPStream().stream());
    if (rc != KMOE_OK) {
      py::gil_scoped_acquire python;
      check(rc);
    }
  } else {
    py::gil_scoped_acquire python;
    (*g_silu_python)(out, x, axis, turn);
  }
  if (!out.is_inference()) out.unsafeGetTensorImpl()->bump_version();  // written, unseen by autograd
}

}  // namespace

TORCH_LIBRARY_IMPL(_C, CUDA, m) { m.impl("silu_and_mul", silu_and_mul); }

PYBIND11_MODULE(kmoe_torch, m) {
  py::class_<Linear>(m, "Linear")
      .def(py::init<uintptr_t, uintptr_t, int, int, int, int, int>())
      .def("__call__", &Linear::operator());
  m.def("install", [](py::object check_status, py::object silu_python) {
    g_check = new py::object(std::move(check_status));
    g_silu_python = new py::object(std::move(silu_python));
  });
}
