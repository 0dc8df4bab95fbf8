// The norms and the causal convolution on at::Tensor: argument checks, allocation, launch through the C ABI, and their
// autograd nodes (the roles of mamba_ssm/ops/triton/layer_norm.py:728, layernorm_gated.py:338 and the causal_conv1d
// package's autograd function).  A norm of one decoded token takes ~3 us of GPU time: in Python + ctypes its call was
// ~30 us of host time.
#include "torch_common.h"

namespace mamba_ext {
namespace {

at::Tensor rows_of(const at::Tensor &t) {
  if (t.dim() == 2 && t.stride(1) == 1) return t;  // (a view costs ~1 us, as much as a launch)
  const at::Tensor r = t.reshape({-1, t.size(-1)});
  return r.stride(1) == 1 ? r : r.contiguous();
}
at::Tensor shaped(const at::Tensor &t, at::IntArrayRef sizes) { return t.sizes() == sizes ? t : t.view(sizes); }
bool vector_ok(const at::Tensor &t, int64_t n) { return t.dim() == 1 && t.size(0) == n && t.is_contiguous(); }
bool params_ok(const at::Tensor &weight, const OptTensor &bias, int64_t n, const c10::Device &dev) {
  return on_device(weight, dev) && on_device(bias, dev) && dtype_code(weight) >= 0 && vector_ok(weight, n) &&
         (!bias || (bias->scalar_type() == weight.scalar_type() && vector_ok(*bias, n)));
}

// ------------------------------------------------------------------ residual-add norm
struct ResNorm {
  double eps;
  bool prenorm, is_rms;
  at::ScalarType stream;  // dtype of the residual stream
};

struct ResNormOut {
  at::Tensor y, sum;  // sum: undefined when no sum is written
  OptTensor mean;
  at::Tensor rstd;
};

ResNormOut res_norm_fwd(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &residual,
                        const ResNorm &o) {
  const int64_t M = x.size(0), N = x.size(1);
  const auto f32 = x.options().dtype(at::kFloat);
  ResNormOut r;
  r.y = at::empty({M, N}, x.options());
  if (residual || o.stream != x.scalar_type()) r.sum = at::empty({M, N}, x.options().dtype(o.stream));
  if (!o.is_rms) r.mean = at::empty({M}, f32);
  r.rstd = at::empty({M}, f32);
  if (M == 0) return r;
  NormResidualParams p{};
  p.rows = (int32_t)M, p.dim = (int32_t)N, p.dtype = dtype_code(x), p.res_dtype = dtype_code(o.stream);
  p.is_rms = o.is_rms, p.eps = (float)o.eps, p.weight_dtype = dtype_code(weight);
  p.x = x.data_ptr(), p.residual = ptr(residual), p.weight = weight.data_ptr(), p.bias = ptr(bias);
  p.out = r.y.data_ptr(), p.residual_out = r.sum.defined() ? r.sum.data_ptr() : nullptr;
  p.mean = r.mean ? r.mean->data_ptr<float>() : nullptr, p.rstd = r.rstd.data_ptr<float>();
  p.x_rs = x.stride(0), p.out_rs = N, p.residual_rs = residual ? residual->stride(0) : 0, p.residual_out_rs = N;
  c10::DeviceGuard guard(x.device());
  check_rc(norm_residual_fwd(&p, stream_of(x.device())), "norm_residual_fwd");
  return r;
}

struct ResNormFn : torch::autograd::Function<ResNormFn> {
  static variable_list forward(AutogradContext *ctx, const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias,
                               const OptTensor &residual, const ResNorm &o) {
    const at::Tensor x2 = rows_of(x);
    const OptTensor res2 = residual ? OptTensor(rows_of(*residual)) : std::nullopt;
    ResNormOut r = res_norm_fwd(x2, weight, bias, res2, o);
    ctx->save_for_backward({r.sum.defined() ? r.sum : x2, weight, tensor_or_none(bias), tensor_or_none(r.mean), r.rstd});
    ctx->set_materialize_grads(false);
    ctx->saved_data["has_residual"] = residual.has_value();
    ctx->saved_data["is_rms"] = o.is_rms;
    ctx->saved_data["eps"] = o.eps;
    ctx->saved_data["x_dtype"] = (int64_t)x.scalar_type();
    ctx->saved_data["shape"] = x.sizes().vec();
    variable_list out = {shaped(r.y, x.sizes())};
    if (o.prenorm) out.push_back(shaped(r.sum, x.sizes()));
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const at::Tensor &x = saved[0], &weight = saved[1], &rstd = saved[4];
    const OptTensor bias = opt(saved[2]), mean = opt(saved[3]);
    const bool has_residual = ctx->saved_data["has_residual"].toBool(), is_rms = ctx->saved_data["is_rms"].toBool();
    const auto x_dtype = (at::ScalarType)ctx->saved_data["x_dtype"].toInt();
    const std::vector<int64_t> shape = ctx->saved_data["shape"].toIntVector();
    const int64_t M = x.size(0), N = x.size(1);
    c10::DeviceGuard guard(x.device());
    at::Tensor dy = grads[0].defined() ? rows_of(grads[0]) : at::zeros({M, N}, x.options().dtype(x_dtype));
    if (dy.scalar_type() != x_dtype) dy = dy.to(x_dtype);
    OptTensor dres;
    if (grads.size() > 1 && grads[1].defined()) dres = rows_of(grads[1]).to(x.scalar_type());
    at::Tensor dx = at::empty({M, N}, x.options().dtype(x_dtype));
    at::Tensor dsum = has_residual && x_dtype != x.scalar_type() ? at::empty({M, N}, x.options()) : at::Tensor();
    std::vector<int64_t> sum_shape = bias ? std::vector<int64_t>{2, N} : std::vector<int64_t>{N};
    at::Tensor sums = M > 0 ? at::empty(sum_shape, weight.options()) : at::zeros(sum_shape, weight.options());
    if (M > 0) {
      NormResidualParams p{};
      p.rows = (int32_t)M, p.dim = (int32_t)N, p.dtype = dtype_code(x_dtype), p.res_dtype = dtype_code(x);
      p.is_rms = is_rms, p.eps = (float)ctx->saved_data["eps"].toDouble(), p.weight_dtype = dtype_code(weight);
      p.x = x.data_ptr(), p.weight = weight.data_ptr(), p.bias = ptr(bias);
      p.mean = mean ? mean->data_ptr<float>() : nullptr, p.rstd = rstd.data_ptr<float>();
      p.x_rs = x.stride(0);
      p.dy = dy.data_ptr(), p.dy_rs = dy.stride(0), p.dx = dx.data_ptr(), p.dx_rs = N;
      p.dresidual = ptr(dres), p.dresidual_rs = dres ? dres->stride(0) : 0;
      p.dresidual_in = dsum.defined() ? dsum.data_ptr() : nullptr, p.dresidual_in_rs = N;
      p.nparts = norm_residual_bwd_nparts(&p);
      at::Tensor parts = at::empty({bias ? 2 : 1, p.nparts, N}, x.options().dtype(at::kFloat));
      char *out = static_cast<char *>(sums.data_ptr());
      p.dweight = out, p.dw_part = parts.data_ptr<float>();
      if (bias) p.dbias = out + N * sums.element_size(), p.db_part = p.dw_part + (int64_t)p.nparts * N;
      check_rc(norm_residual_bwd(&p, stream_of(x.device())), "norm_residual_bwd");
    }
    variable_list g(5);
    g[0] = shaped(dx, shape);
    g[1] = bias ? sums.select(0, 0) : sums;
    if (bias) g[2] = sums.select(0, 1);
    if (has_residual) g[3] = shaped(dsum.defined() ? dsum : dx, shape);
    return g;
  }
};

// layer_norm_fn / rms_norm_fn without x1, weight1, dropout and rowscale: out, or (out, sum) with prenorm; None = declined
pybind11::object norm_residual(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &residual,
                               double eps, bool prenorm, bool residual_in_fp32, bool is_rms) {
  const pybind11::object no = pybind11::none();
  if (!x.is_cuda() || x.dim() < 1 || dtype_code(x) < 0 || x.size(-1) <= 0 || python_call(x, weight, bias, residual)) return no;
  const c10::Device dev = x.device();
  const int64_t N = x.size(-1);
  if (!params_ok(weight, bias, N, dev) || N > 65536 / (int64_t)x.element_size() || !on_device(residual, dev)) return no;
  ResNorm o{eps, prenorm, is_rms, x.scalar_type()};
  if (residual) {
    if (residual->sizes() != x.sizes()) return no;
    o.stream = residual->scalar_type();
  } else if (residual_in_fp32) {
    o.stream = at::kFloat;
  }
  if (o.stream != x.scalar_type() && o.stream != at::kFloat) return no;
  if (!residual && o.stream == x.scalar_type() && prenorm) return no;  // the sum handed on is x itself
  if (x.numel() / N > INT32_MAX) return no;
  if (!records(x, weight, bias, residual)) {
    ResNormOut r = res_norm_fwd(rows_of(x), weight, bias, residual ? OptTensor(rows_of(*residual)) : std::nullopt, o);
    const at::Tensor y = shaped(r.y, x.sizes());
    return prenorm ? pybind11::object(pybind11::make_tuple(y, shaped(r.sum, x.sizes()))) : pybind11::cast(y);
  }
  variable_list r = ResNormFn::apply(x, weight, bias, residual, o);
  return prenorm ? pybind11::object(pybind11::make_tuple(r[0], r[1])) : pybind11::cast(r[0]);
}

// ------------------------------------------------------------------ gated norm
void fill_gated(NormGatedParams &p, const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &z,
                const GatedNorm &o) {
  p.rows = (int32_t)x.size(0), p.dim = (int32_t)x.size(1), p.group_size = (int32_t)o.group_size, p.dtype = dtype_code(x);
  p.is_rms = o.is_rms, p.norm_before_gate = o.norm_before_gate, p.eps = (float)o.eps, p.weight_dtype = dtype_code(weight);
  p.x = x.data_ptr(), p.z = ptr(z), p.weight = weight.data_ptr(), p.bias = ptr(bias);
  p.x_rs = x.stride(0), p.z_rs = z ? z->stride(0) : 0;
}

struct GatedNormFn : torch::autograd::Function<GatedNormFn> {
  static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias,
                            const OptTensor &z, const GatedNorm &o) {
    const at::Tensor x2 = rows_of(x);
    const OptTensor z2 = z ? OptTensor(rows_of(*z)) : std::nullopt;
    auto [y, mean, rstd] = gated_norm_fwd(x2, weight, bias, z2, o);
    ctx->save_for_backward({x2, weight, tensor_or_none(bias), tensor_or_none(mean), rstd, tensor_or_none(z2)});
    ctx->saved_data["o"] = std::vector<int64_t>{o.group_size, o.norm_before_gate, o.is_rms};
    ctx->saved_data["eps"] = o.eps;
    return shaped(y, x.sizes());
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> v = ctx->saved_data["o"].toIntVector();
    const GatedNorm o{v[0], ctx->saved_data["eps"].toDouble(), v[1] != 0, v[2] != 0};
    const at::Tensor dy = rows_of(grads[0]).to(s[0].scalar_type());
    auto [dx, dw, db, dz] = gated_norm_bwd(dy, s[0], s[1], opt(s[2]), opt(s[3]), s[4], opt(s[5]), std::nullopt, o);
    variable_list g(5);
    g[0] = shaped(dx, grads[0].sizes());
    g[1] = dw;
    if (db) g[2] = *db;
    if (dz) g[3] = shaped(*dz, grads[0].sizes());
    return g;
  }
};

// layernorm_gated.layernorm_fn / rmsnorm_fn; None = declined
OptTensor norm_gated(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &z, double eps,
                     std::optional<int64_t> group_size, bool norm_before_gate, bool is_rms) {
  if (!x.is_cuda() || x.dim() < 1 || x.size(-1) <= 0 || (z && z->sizes() != x.sizes()) || python_call(x, weight, bias, z))
    return std::nullopt;
  const GatedNorm o{group_size.value_or(x.size(-1)), eps, norm_before_gate, is_rms};
  if (!gated_norm_ok(x, weight, bias, z, o)) return std::nullopt;
  if (!records(x, weight, bias, z))
    return shaped(std::get<0>(gated_norm_fwd(rows_of(x), weight, bias, z ? OptTensor(rows_of(*z)) : std::nullopt, o)), x.sizes());
  return GatedNormFn::apply(x, weight, bias, z, o);
}

// ------------------------------------------------------------------ convolution
ConvRows rows_at(const at::Tensor &t) { return {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)}; }

void fill_conv(CausalConvParams &p, int dtype, int64_t batch, int64_t dim, int64_t L, const ConvRows &x, const at::Tensor &weight,
               const OptTensor &bias, const OptTensor &seq_idx, bool silu) {
  p.batch = (int32_t)batch, p.dim = (int32_t)dim, p.seqlen = (int32_t)L, p.width = (int32_t)weight.size(-1);
  p.dtype = dtype, p.silu = silu, p.weight_dtype = dtype_code(weight);
  p.x = x.p, p.weight = weight.data_ptr(), p.bias = ptr(bias);
  p.seq_idx = seq_idx ? seq_idx->data_ptr<int32_t>() : nullptr;
  p.x_bs = x.bs, p.x_cs = x.cs, p.x_ls = x.ls;
}

at::Tensor like_layout(const at::Tensor &x) {
  const int64_t b = x.size(0), d = x.size(1), L = x.size(2);
  return x.stride(2) == 1 ? at::empty({b, d, L}, x.options()) : at::empty({b, L, d}, x.options()).transpose(1, 2);
}
// a gradient in x's layout
at::Tensor in_layout(const at::Tensor &g, const at::Tensor &x) {
  if (x.stride(2) == 1) return g.stride(2) == 1 ? g : g.contiguous();
  return g.stride(1) == 1 ? g : g.transpose(1, 2).contiguous().transpose(1, 2);
}

struct ConvFn : torch::autograd::Function<ConvFn> {
  static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias,
                            const OptTensor &seq_idx, bool silu) {
    at::Tensor out = like_layout(x);
    conv_fwd(x, weight, bias, seq_idx, silu, out);
    ctx->save_for_backward({x, weight, tensor_or_none(bias), tensor_or_none(seq_idx)});
    ctx->saved_data["silu"] = silu;
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    at::Tensor dx = like_layout(s[0]);
    auto [dw, db] = conv_bwd(s[0], s[1], opt(s[2]), in_layout(grads[0], s[0]), opt(s[3]), ctx->saved_data["silu"].toBool(), dx);
    variable_list g(5);
    g[0] = dx, g[1] = dw;
    if (db) g[2] = *db;
    return g;
  }
};

// causal_conv1d_fn without the streaming arguments; None = declined
OptTensor causal_conv1d(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &seq_idx, bool silu) {
  if (!x.is_cuda() || x.dim() != 3 || (x.stride(2) != 1 && x.stride(1) != 1) || python_call(x, weight, bias)) return std::nullopt;
  if (!conv_params_ok(x, weight, bias, seq_idx)) return std::nullopt;
  if (records(x, weight, bias)) return ConvFn::apply(x, weight, bias, seq_idx, silu);
  at::Tensor out = like_layout(x);
  conv_fwd(x, weight, bias, seq_idx, silu, out);
  return out;
}

}  // namespace

bool gated_norm_ok(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &z, const GatedNorm &o) {
  const c10::Device dev = x.device();
  const int64_t N = x.size(-1);
  return dtype_code(x) >= 0 && params_ok(weight, bias, N, dev) && on_device(z, dev) &&
         (!z || z->scalar_type() == x.scalar_type()) && o.group_size > 0 && N % o.group_size == 0 &&
         o.group_size <= 65536 / (int64_t)x.element_size() && x.numel() / N <= INT32_MAX;
}

std::tuple<at::Tensor, OptTensor, at::Tensor> gated_norm_fwd(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias,
                                                            const OptTensor &z, const GatedNorm &o) {
  const int64_t M = x.size(0), N = x.size(1), ngroups = N / o.group_size;
  const auto f32 = x.options().dtype(at::kFloat);
  at::Tensor out = at::empty({M, N}, x.options()), rstd = at::empty({M, ngroups}, f32);
  OptTensor mean;
  if (!o.is_rms) mean = at::empty({M, ngroups}, f32);
  if (M > 0) {
    NormGatedParams p{};
    fill_gated(p, x, weight, bias, z, o);
    p.out = out.data_ptr(), p.out_rs = N, p.mean = mean ? mean->data_ptr<float>() : nullptr, p.rstd = rstd.data_ptr<float>();
    c10::DeviceGuard guard(x.device());
    check_rc(norm_gated_fwd(&p, stream_of(x.device())), "norm_gated_fwd");
  }
  return {out, mean, rstd};
}

std::tuple<at::Tensor, at::Tensor, OptTensor, OptTensor> gated_norm_bwd(const at::Tensor &dy, const at::Tensor &x,
                                                                       const at::Tensor &weight, const OptTensor &bias,
                                                                       const OptTensor &mean, const at::Tensor &rstd,
                                                                       const OptTensor &z, const OptTensor &dz_out,
                                                                       const GatedNorm &o) {
  const int64_t M = x.size(0), N = x.size(1);
  c10::DeviceGuard guard(x.device());
  at::Tensor dx = at::empty({M, N}, x.options());
  OptTensor dz;
  if (z) dz = dz_out ? *dz_out : at::empty({M, N}, x.options());
  const int64_t nb = bias ? 2 : 1;
  at::Tensor sums = M > 0 ? at::empty({nb, N}, weight.options()) : at::zeros({nb, N}, weight.options());
  if (M > 0) {
    NormGatedParams p{};
    fill_gated(p, x, weight, bias, z, o);
    p.mean = mean ? mean->data_ptr<float>() : nullptr, p.rstd = rstd.data_ptr<float>();
    p.dy = dy.data_ptr(), p.dy_rs = dy.stride(0), p.dx = dx.data_ptr(), p.dx_rs = N;
    p.dz = ptr(dz), p.dz_rs = dz ? dz->stride(0) : 0;
    p.nparts = norm_gated_bwd_nparts(&p);
    at::Tensor parts = at::empty({nb, p.nparts, N}, x.options().dtype(at::kFloat));
    char *out = static_cast<char *>(sums.data_ptr());
    p.dweight = out, p.dw_part = parts.data_ptr<float>();
    if (bias) p.dbias = out + N * sums.element_size(), p.db_part = p.dw_part + (int64_t)p.nparts * N;
    check_rc(norm_gated_bwd(&p, stream_of(x.device())), "norm_gated_bwd");
  }
  OptTensor db;
  if (bias) db = sums.select(0, 1);
  return {dx, sums.select(0, 0), db, dz};
}

bool conv_params_ok(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &seq_idx) {
  const c10::Device dev = x.device();
  if (x.dim() != 3 || dtype_code(x) < 0 || !on_device(weight, dev) || !on_device(bias, dev) || !on_device(seq_idx, dev)) return false;
  const int64_t batch = x.size(0), dim = x.size(1), L = x.size(2);
  if (batch <= 0 || dim <= 0 || L <= 0 || batch > 65535 || dim > 65535 || L > INT32_MAX) return false;
  if (weight.dim() != 2 || weight.size(0) != dim || weight.size(1) < 2 || weight.size(1) > 4 || dtype_code(weight) < 0 ||
      !weight.is_contiguous())
    return false;
  if (bias && (bias->scalar_type() != weight.scalar_type() || !vector_ok(*bias, dim))) return false;
  return !seq_idx || (seq_idx->scalar_type() == at::kInt && seq_idx->is_contiguous() && seq_idx->dim() == 2 &&
                      seq_idx->size(0) == batch && seq_idx->size(1) == L);
}

void conv_fwd(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias, const OptTensor &seq_idx, bool silu,
              const at::Tensor &out) {
  conv_fwd(x, x.size(0), x.size(1), x.size(2), rows_at(x), weight, bias, seq_idx, silu, rows_at(out));
}
void conv_fwd(const at::Tensor &like, int64_t batch, int64_t dim, int64_t L, const ConvRows &x, const at::Tensor &weight,
              const OptTensor &bias, const OptTensor &seq_idx, bool silu, const ConvRows &out) {
  CausalConvParams p{};
  fill_conv(p, dtype_code(like), batch, dim, L, x, weight, bias, seq_idx, silu);
  p.out = const_cast<void *>(out.p), p.out_bs = out.bs, p.out_cs = out.cs, p.out_ls = out.ls;
  c10::DeviceGuard guard(like.device());
  check_rc(::causal_conv1d_fwd(&p, stream_of(like.device())), "causal_conv1d_fwd");
}

std::tuple<at::Tensor, OptTensor> conv_bwd(const at::Tensor &x, const at::Tensor &weight, const OptTensor &bias,
                                           const at::Tensor &dout, const OptTensor &seq_idx, bool silu, const at::Tensor &dx) {
  return conv_bwd(x, x.size(0), x.size(1), x.size(2), rows_at(x), weight, bias, rows_at(dout), seq_idx, silu, rows_at(dx));
}
std::tuple<at::Tensor, OptTensor> conv_bwd(const at::Tensor &like, int64_t batch, int64_t dim, int64_t L, const ConvRows &x,
                                           const at::Tensor &weight, const OptTensor &bias, const ConvRows &dout,
                                           const OptTensor &seq_idx, bool silu, const ConvRows &dx) {
  c10::DeviceGuard guard(like.device());
  CausalConvParams p{};
  fill_conv(p, dtype_code(like), batch, dim, L, x, weight, bias, seq_idx, silu);
  at::Tensor dw = at::empty(weight.sizes(), weight.options());
  OptTensor db;
  if (bias) db = at::empty(bias->sizes(), bias->options());
  p.dout = dout.p, p.dx = const_cast<void *>(dx.p), p.dweight = dw.data_ptr(), p.dbias = ptr(db);
  p.dout_bs = dout.bs, p.dout_cs = dout.cs, p.dout_ls = dout.ls, p.dx_bs = dx.bs, p.dx_cs = dx.cs, p.dx_ls = dx.ls;
  const int nparts = causal_conv1d_bwd_nparts(&p);
  if (nparts <= 0) check_rc(nparts ? nparts : -1, "causal_conv1d_bwd_nparts");
  at::Tensor part = at::empty({nparts * dim * 5}, like.options().dtype(at::kFloat));
  p.dw_part = part.data_ptr<float>();
  check_rc(::causal_conv1d_bwd(&p, stream_of(like.device())), "causal_conv1d_bwd");
  return {dw, db};
}

void bind_norm_conv(pybind11::module_ &m) {
  namespace py = pybind11;
  m.def("norm_residual", &norm_residual, py::arg("x"), py::arg("weight"), py::arg("bias"), py::arg("residual"), py::arg("eps"),
        py::arg("prenorm"), py::arg("residual_in_fp32"), py::arg("is_rms"),
        "Norm of x + residual with autograd: out, or (out, sum) with prenorm; None when the arguments need the Python path.");
  m.def("norm_gated", &norm_gated, py::arg("x"), py::arg("weight"), py::arg("bias"), py::arg("z"), py::arg("eps"),
        py::arg("group_size"), py::arg("norm_before_gate"), py::arg("is_rms"),
        "Gated group norm with autograd: out, or None when the arguments need the Python path.");
  m.def("causal_conv1d", &causal_conv1d, py::arg("x"), py::arg("weight"), py::arg("bias"), py::arg("seq_idx"), py::arg("silu"),
        "Causal depthwise convolution with autograd: out, or None when the arguments need the Python path.");
}

}  // namespace mamba_ext
