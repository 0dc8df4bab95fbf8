// Shared by the translation units of the torch extension (torch_*.cpp; host code only).
//
// Every operator here serves the plain, valid case and DECLINES anything else by returning nullopt / None (wrong
// shapes, dtypes that need a conversion first, CPU tensors): the Python host side then runs its own path, which does
// the conversions and raises the reference's errors.  Both paths end in the same kernels.
#pragma once
#include <torch/extension.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "mamba_hip.h"

namespace mamba_ext {

using OptTensor = std::optional<at::Tensor>;
using TensorList = std::vector<OptTensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

inline int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MAMBA_F32;
    case at::kBFloat16: return MAMBA_BF16;
    case at::kHalf: return MAMBA_F16;
    default: return -1;
  }
}
inline int dtype_code(const at::Tensor &t) { return dtype_code(t.scalar_type()); }

inline bool on_device(const at::Tensor &t, const c10::Device &dev) { return t.is_cuda() && t.device() == dev; }
inline bool on_device(const OptTensor &t, const c10::Device &dev) { return !t.has_value() || on_device(*t, dev); }

inline void *stream_of(const c10::Device &dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

inline void check_rc(int rc, const char *what) {
  TORCH_CHECK(rc == MAMBA_OK, what, " failed: ", mamba_hip_strerror(rc), " (code ", rc, ")");
}

inline void *ptr(const OptTensor &t) { return t ? t->data_ptr() : nullptr; }

template <typename F> bool holds(const F &f, const at::Tensor &t) { return t.defined() && f(t); }
template <typename F> bool holds(const F &f, const OptTensor &t) { return t && holds(f, *t); }

// Whether autograd has to record a call: gradients are enabled and one of the tensors wants them.
template <typename... Args> bool records(const Args &...args) {
  auto wants = [](const at::Tensor &t) { return t.requires_grad(); };
  return at::GradMode::is_enabled() && (holds(wants, args) || ...);
}
// Whether a call is one for the Python autograd functions.  torch refuses them under a functorch transform, and with a
// forward-mode gradient on one of the tensors (with and without reverse-mode gradients; the kernels would drop it).  A jit
// trace records them as nodes to be run again; a call it does not see leaves its results in the trace as constants.
template <typename... Args> bool python_call(const Args &...args) {
  auto tangent = [](const at::Tensor &t) { return t._fw_grad(0).defined(); };
  return c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer) || (holds(tangent, args) || ...);
}

inline OptTensor opt(const at::Tensor &t) { return t.defined() ? OptTensor(t) : std::nullopt; }
inline at::Tensor tensor_or_none(const OptTensor &t) { return t ? *t : at::Tensor(); }

// The deterministic mode as mamba_amd/utils/determinism.py defines it; `set_deterministic_override` mirrors that
// module's explicit setting (-1: none).
bool deterministic();
void set_deterministic_override(int value);

// ---- convolution (torch_norm_conv.cpp)
// x, out, dout, dx: (batch, dim, seqlen) views with unit stride along the positions or the channels.
bool conv_params_ok(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &seq_idx);
void conv_fwd(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &seq_idx, bool silu,
              const at::Tensor &out);
// -> (dweight, dbias) in the parameters' dtype (and shape); dx is written
std::tuple<at::Tensor, OptTensor> conv_bwd(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias,
                                           const at::Tensor &dout, const OptTensor &seq_idx, bool silu, const at::Tensor &dx);

// The same on memory by strides (batch, channel, position) of `like`'s dtype and device; weight (dim, [1,] width).
struct ConvRows {
  const void *p;
  int64_t bs, cs, ls;
};
void conv_fwd(const at::Tensor &like, int64_t batch, int64_t dim, int64_t L, const ConvRows &x, const at::Tensor &weight,
              const OptTensor &bias, const OptTensor &seq_idx, bool silu, const ConvRows &out);
std::tuple<at::Tensor, OptTensor> conv_bwd(const at::Tensor &like, int64_t batch, int64_t dim, int64_t L, const ConvRows &x,
                                           const at::Tensor &weight, const OptTensor &bias, const ConvRows &dout,
                                           const OptTensor &seq_idx, bool silu, const ConvRows &dx);

// ---- gated norm (torch_norm_conv.cpp): x, z, dy, out (rows, dim), unit channel stride
struct GatedNorm {
  int64_t group_size;
  double eps;
  bool norm_before_gate, is_rms;
};
bool gated_norm_ok(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &z, const GatedNorm &o);
std::tuple<at::Tensor, OptTensor, at::Tensor> gated_norm_fwd(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias,
                                                            const OptTensor &z, const GatedNorm &o);  // out, mean, rstd
std::tuple<at::Tensor, at::Tensor, OptTensor, OptTensor> gated_norm_bwd(const at::Tensor &dy, const at::Tensor &x,
                                                                       const at::Tensor &weight, const OptTensor &bias,
                                                                       const OptTensor &mean, const at::Tensor &rstd,
                                                                       const OptTensor &z, const OptTensor &dz_out,
                                                                       const GatedNorm &o);  // dx, dweight, dbias, dz

// ---- matrix products (torch_gemm.cpp)
struct Mat {  // one operand: element (row, k) at p[row * rs + k * ks], one of the strides 1; rows are those of the result, or its columns
  const void *p;
  int64_t rs, ks;
};
// Products D = A B^T of operands of `type` on raw memory.  Those that the own kernels suit (mamba_gemm_suits: short ones, and large
// ones that the BLAS library splits badly) are collected and leave with run(), or once there are four, in an order of their own; the
// others leave at once.  So the products of two run() calls must not depend on each other, no result is there before run(), and
// the operands stay until then.
class Products {
 public:
  Products(const at::TensorOptions &options, at::ScalarType type) : options_(options), type_(type) {}
  Products &add(void *D, at::ScalarType d_type, int64_t ldd, int64_t M, int64_t N, int64_t K, Mat A, Mat B, bool accumulate = false,
                const void *bias = nullptr);
  void run();

 private:
  at::TensorOptions options_;
  at::ScalarType type_;
  MambaGemm g_[4];
  int count_ = 0;
};
void bind_norm_conv(pybind11::module_ &m);
void bind_scan(pybind11::module_ &m);
void bind_ssd(pybind11::module_ &m);

}  // namespace mamba_ext
