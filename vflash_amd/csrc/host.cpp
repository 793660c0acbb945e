// The host side of the two W8A8 linears that users call most, natively: checks,
// allocations and launches of one call without a round trip through Python for
// each of them.
//
// A 17 x 5120 x 5120 linear keeps the GPU busy for 11 us, while the Python wrappers
// of its two kernels (argument checks, four allocations, two ctypes calls) take 24 us
// of host time; here it takes 10.  The adapter linear: 16 us of GPU time at 256 x 1536
// x 4608, 34 us of host time in the wrappers, 11 here.  Each function here takes
// the tensors of a call, and either runs the whole of it on the tensor's current
// stream or returns None without having enqueued anything that the caller sees:
// every other layout, type, device or error goes on to the Python wrappers, which
// decide and report as before.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

#include "../../include/vflash_amd.h"

namespace {

// The tensor behind a plain torch.Tensor or torch.nn.Parameter, else null.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}

bool gfx950(c10::DeviceIndex index) {
  const char* arch = at::cuda::getDeviceProperties(index)->gcnArchName;
  return std::strncmp(arch, "gfx950", 6) == 0 && (arch[6] == 0 || arch[6] == ':');
}

// The operands of a W8A8 linear in the layout the kernels take without a copy.
struct Linear {
  const at::Tensor *x, *w, *sw, *b;
  int64_t m, n, k, m_pad;
};

bool linear_ok(PyObject* const* a, Linear& l) {
  l.x = plain(a[0]);
  l.w = plain(a[1]);
  l.sw = plain(a[2]);
  l.b = a[3] == Py_None ? nullptr : plain(a[3]);
  if (!l.x || !l.w || !l.sw || (a[3] != Py_None && !l.b)) return false;
  if (l.x->scalar_type() != at::kBFloat16 || l.w->scalar_type() != at::kFloat8_e4m3fn ||
      l.sw->scalar_type() != at::kFloat)
    return false;
  if (l.x->dim() < 1 || l.w->dim() != 2 || !l.x->is_contiguous() || !l.sw->is_contiguous()) return false;
  l.n = l.w->size(0);
  l.k = l.w->size(1);
  if (l.n < 1 || l.k < 16 || l.k % 16 || l.x->size(-1) != l.k || l.x->numel() == 0) return false;
  if (l.w->stride(1) != 1 || l.sw->dim() != 2 || l.sw->size(0) != l.n || l.sw->size(1) != 1) return false;
  const c10::Device d = l.x->device();
  if (l.w->device() != d || l.sw->device() != d) return false;
  if (l.b && (l.b->dim() != 1 || l.b->size(0) != l.n || l.b->scalar_type() != at::kBFloat16 ||
              l.b->device() != d || !l.b->is_contiguous()))
    return false;
  l.m = l.x->numel() / l.k;
  l.m_pad = (l.m + 15) / 16 * 16;
  return gfx950(d.index());
}

// Other Python threads run while this one allocates and launches.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

at::Tensor output(const Linear& l) {
  c10::SmallVector<int64_t, 5> shape(l.x->sizes().begin(), l.x->sizes().end());
  shape.back() = l.n;
  return at::empty(shape, l.x->options().requires_grad(false));
}

// w8a8_linear(value, weight, scale, bias): quantize the rows, then the GEMM.
PyObject* w8a8_linear(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Linear l;
  if (nargs != 4 || !linear_ok(a, l)) Py_RETURN_NONE;
  at::Tensor out;
  int status;
  {
    const NoGil nogil;
    // Two allocations: with the scales right behind the codes (a whole number of
    // megabytes away) the 4096x3072x3072 linear took 43.8 us instead of 42.9.
    const at::Tensor code_rows = at::empty({l.m_pad, l.k}, l.x->options().dtype(at::kByte));
    const at::Tensor row_scales = at::empty({l.m_pad}, l.x->options().dtype(at::kFloat));
    out = output(l);
    uint8_t* codes = static_cast<uint8_t*>(code_rows.data_ptr());
    float* scales = static_cast<float*>(row_scales.data_ptr());
    void* stream = c10::hip::getCurrentHIPStream(l.x->device().index()).stream();
    status = vflash_quantize_rows_e4m3(l.x->data_ptr(), l.m, l.k, l.k, codes, scales, l.m_pad, stream);
    if (status == VFLASH_OK)
      status = vflash_fp8_linear(codes, scales, l.k, l.w->data_ptr(),
                                 static_cast<float*>(l.sw->data_ptr()), l.w->stride(0), l.m, l.n, l.k,
                                 l.b ? l.b->data_ptr() : nullptr, out.data_ptr(), l.n, stream);
  }
  if (status != VFLASH_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// w8a8_linear_lora(value, weight, scale, bias, down, up, scaling, strength): codes
// and t = bf16(x . down^T) in one launch, then the GEMM with the merged adapter.
PyObject* w8a8_linear_lora(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Linear l;
  if (nargs != 8 || !linear_ok(a, l)) Py_RETURN_NONE;
  const at::Tensor *down = plain(a[4]), *up = plain(a[5]);
  if (!down || !up || down->dim() != 2 || up->dim() != 2) Py_RETURN_NONE;
  const int64_t rank = down->size(0), ldt = (rank + 15) / 16 * 16;
  // Ranks that are a multiple of 8 need no padding of the rows of `up`.
  if (rank < 8 || rank > 128 || rank % 8 || down->size(1) != l.k || up->size(0) != l.n ||
      up->size(1) != rank)
    Py_RETURN_NONE;
  if (down->scalar_type() != at::kBFloat16 || up->scalar_type() != at::kBFloat16 ||
      !down->is_contiguous() || !up->is_contiguous() || down->device() != l.x->device() ||
      up->device() != l.x->device())
    Py_RETURN_NONE;
  const double scaling = PyFloat_AsDouble(a[6]), strength = PyFloat_AsDouble(a[7]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  at::Tensor out;
  int status;
  {
    const NoGil nogil;
    const at::Tensor code_rows = at::empty({l.m_pad, l.k}, l.x->options().dtype(at::kByte));
    const at::Tensor row_scales = at::empty({l.m_pad}, l.x->options().dtype(at::kFloat));
    const at::Tensor t_rows = at::empty({l.m, ldt}, l.x->options());
    out = output(l);
    uint8_t* codes = static_cast<uint8_t*>(code_rows.data_ptr());
    float* scales = static_cast<float*>(row_scales.data_ptr());
    void* t = t_rows.data_ptr();
    void* stream = c10::hip::getCurrentHIPStream(l.x->device().index()).stream();
    status = vflash_quantize_rows_lora_e4m3(l.x->data_ptr(), l.m, l.k, l.k, codes, scales, l.m_pad,
                                            down->data_ptr(), rank, t, ldt, stream);
    if (status == VFLASH_OK)
      status = vflash_fp8_linear_lora(codes, scales, l.k, l.w->data_ptr(),
                                      static_cast<float*>(l.sw->data_ptr()), l.w->stride(0), l.m, l.n,
                                      l.k, l.b ? l.b->data_ptr() : nullptr, t, ldt, up->data_ptr(),
                                      rank, rank, (float)scaling, (float)strength, out.data_ptr(), l.n,
                                      stream);
  }
  if (status != VFLASH_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"w8a8_linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(w8a8_linear)),
     METH_FASTCALL, nullptr},
    {"w8a8_linear_lora", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(w8a8_linear_lora)),
     METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&kModule); }
