// The Mamba-1 scan and mixer on at::Tensor (the role of the reference's own binding around its kernels,
// csrc/selective_scan/selective_scan.cpp:226-349, and of its autograd functions,
// mamba_ssm/ops/selective_scan_interface.py:34 and :196).
#include "torch_common.h"

namespace mamba_ext {
namespace {

bool rows_ok(const at::Tensor &t, int64_t b, int64_t d, int64_t l, at::ScalarType ty) {
  return t.dim() == 3 && t.size(0) == b && t.size(1) == d && t.size(2) == l && t.scalar_type() == ty && t.stride(2) == 1;
}

// Fills the fields the forward and backward calls share; false = decline.
bool fill_scan(MambaScanParams &p, const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A, const at::Tensor &B,
               const at::Tensor &C, const OptTensor &D, const OptTensor &z, const OptTensor &delta_bias,
               bool delta_softplus) {
  const c10::Device dev = u.device();
  if (!on_device(u, dev) || !on_device(delta, dev) || !on_device(A, dev) || !on_device(B, dev) || !on_device(C, dev) ||
      !on_device(D, dev) || !on_device(z, dev) || !on_device(delta_bias, dev))
    return false;
  const int code = dtype_code(u);
  if (code < 0 || u.dim() != 3 || A.dim() != 2 || A.scalar_type() != at::kFloat || !A.is_contiguous()) return false;
  const int64_t batch = u.size(0), dim = u.size(1), L = u.size(2), N = A.size(1);
  if (batch <= 0 || dim <= 0 || L <= 0 || N <= 0 || A.size(0) != dim || N > mamba_hip_query(MAMBA_Q_MAX_DSTATE)) return false;
  if (batch > INT32_MAX || dim > INT32_MAX || L > INT32_MAX) return false;
  if (!rows_ok(u, batch, dim, L, u.scalar_type()) || !rows_ok(delta, batch, dim, L, u.scalar_type())) return false;
  if (z && !rows_ok(*z, batch, dim, L, u.scalar_type())) return false;
  int64_t G = 1;
  for (const at::Tensor *t : {&B, &C})
    if (t->dim() == 4) G = t->size(1);
  for (const at::Tensor *t : {&B, &C}) {
    if (t->dim() == 2) {
      if (t->scalar_type() != at::kFloat || t->size(0) != dim || t->size(1) != N || !t->is_contiguous()) return false;
    } else if (t->dim() == 4) {
      if (t->scalar_type() != u.scalar_type() || t->stride(3) != 1 || t->size(0) != batch || t->size(1) != G ||
          t->size(2) != N || t->size(3) != L)
        return false;
    } else {
      return false;
    }
  }
  if (dim % G != 0) return false;
  auto vec_ok = [&](const OptTensor &t) {
    return !t || (t->scalar_type() == at::kFloat && t->dim() == 1 && t->size(0) == dim && t->stride(0) == 1);
  };
  if (!vec_ok(D) || !vec_ok(delta_bias)) return false;
  p.batch = (int32_t)batch, p.dim = (int32_t)dim, p.seqlen = (int32_t)L, p.dstate = (int32_t)N, p.ngroups = (int32_t)G;
  p.dtype = code, p.delta_softplus = delta_softplus ? 1 : 0, p.a_complex = 0;
  p.bc_const = (B.dim() == 2 ? 1 : 0) | (C.dim() == 2 ? 2 : 0);
  p.u = u.data_ptr(), p.delta = delta.data_ptr(), p.A = A.data_ptr(), p.B = B.data_ptr(), p.C = C.data_ptr();
  p.D = ptr(D), p.z = ptr(z), p.delta_bias = ptr(delta_bias);
  p.u_bs = u.stride(0), p.u_ds = u.stride(1), p.delta_bs = delta.stride(0), p.delta_ds = delta.stride(1);
  if (z) p.z_bs = z->stride(0), p.z_ds = z->stride(1);
  if (B.dim() == 4) p.B_bs = B.stride(0), p.B_gs = B.stride(1), p.B_ns = B.stride(2);
  if (C.dim() == 4) p.C_bs = C.stride(0), p.C_gs = C.stride(1), p.C_ns = C.stride(2);
  return true;
}

// The number of segments of the sequence and their workspace, where the problem is split.
at::Tensor split_sequence(MambaScanParams &p, const at::Tensor &u, bool backward) {
  p.nseg = std::max(1, mamba1_scan_segments(&p, backward ? 1 : 0));
  if (p.nseg == 1) return at::Tensor();
  at::Tensor ws = at::empty({(int64_t)p.batch * p.nseg * p.dim * (p.dstate + 2)}, u.options().dtype(at::kFloat));
  p.seg_ws = ws.data_ptr<float>();
  return ws;
}

// selective_scan_cuda.fwd (selective_scan.cpp:226) on filled parameters -> (out, ckpt); real A only.
std::tuple<at::Tensor, at::Tensor> scan_fwd(MambaScanParams &p, const at::Tensor &u, const at::Tensor &delta) {
  const c10::Device dev = u.device();
  c10::DeviceGuard guard(dev);
  const int64_t tile = mamba_hip_query(MAMBA_Q_SCAN_TILE), ntiles = (p.seqlen + tile - 1) / tile;
  at::Tensor out = at::empty_like(delta);
  at::Tensor ckpt = at::empty({p.batch, p.dim, ntiles, p.dstate}, u.options().dtype(at::kFloat));
  p.out = out.data_ptr(), p.out_bs = out.stride(0), p.out_ds = out.stride(1);
  p.ckpt = ckpt.data_ptr<float>();
  const at::Tensor ws = split_sequence(p, u, false);
  check_rc(mamba1_scan_fwd(&p, stream_of(dev)), "mamba1_scan_fwd");
  return {out, ckpt};
}

std::optional<std::tuple<at::Tensor, at::Tensor>> scan_fwd_fast(const at::Tensor &u, const at::Tensor &delta,
                                                                const at::Tensor &A, const at::Tensor &B,
                                                                const at::Tensor &C, const OptTensor &D,
                                                                const OptTensor &z, const OptTensor &delta_bias,
                                                                bool delta_softplus) {
  MambaScanParams p{};
  if (!fill_scan(p, u, delta, A, B, C, D, z, delta_bias, delta_softplus)) return std::nullopt;
  return scan_fwd(p, u, delta);
}

// selective_scan_cuda.bwd (selective_scan.cpp:338) on filled parameters
// -> [du, ddelta, dA, dB, dC, dD, ddelta_bias, dz, out_z].  dB_out / dC_out: where the gradients of per-position B / C
// are written, (batch, ngroups, dstate, seqlen) views with unit position stride (allocated here when absent).
TensorList scan_bwd(MambaScanParams &p, const at::Tensor &u, const at::Tensor &delta, const at::Tensor &B, const at::Tensor &C,
                    const OptTensor &D, const OptTensor &z, const OptTensor &delta_bias, const at::Tensor &dout,
                    const at::Tensor &ckpt, const OptTensor &dz_in, bool recompute_out_z, const OptTensor &dB_out,
                    const OptTensor &dC_out) {
  const c10::Device dev = u.device();
  const int64_t batch = p.batch, dim = p.dim, L = p.seqlen, N = p.dstate, G = p.ngroups;
  c10::DeviceGuard guard(dev);
  const auto f32 = u.options().dtype(at::kFloat);
  const at::Tensor ws = split_sequence(p, u, true);
  const int64_t nseg = p.nseg, nparts = mamba1_scan_bwd_nparts(&p);
  if (nparts <= 0) check_rc(nparts ? (int)nparts : -1, "mamba1_scan_bwd_nparts");
  at::Tensor du = at::empty_like(u), ddelta = at::empty_like(delta);
  auto operand = [&](const at::Tensor &t, const OptTensor &given, at::Tensor &part, OptTensor &grad, int64_t &bs, int64_t &gs,
                     int64_t &ns) {
    if (t.dim() == 2) {
      part = at::empty({batch * nseg, dim, N}, f32);
      return;
    }
    part = at::empty({batch, G, nparts, N, L}, f32);
    grad = given ? *given : at::empty({batch, G, N, L}, t.options());
    bs = grad->stride(0), gs = grad->stride(1), ns = grad->stride(2);
  };
  at::Tensor dB32, dC32;
  OptTensor dB, dC, dz, out_z;
  operand(B, dB_out, dB32, dB, p.dB_bs, p.dB_gs, p.dB_ns);
  operand(C, dC_out, dC32, dC, p.dC_bs, p.dC_gs, p.dC_ns);
  // dA, dD and ddelta_bias: the partials of every (batch, segment) and, behind them, their sums
  at::Tensor part = at::empty({(batch * nseg + 1) * dim * (N + 2)}, f32);
  float *base = part.data_ptr<float>();
  const int64_t rows = batch * nseg;
  p.dA_part = base, p.dD_part = base + rows * dim * N, p.ddelta_bias_part = p.dD_part + rows * dim;
  at::Tensor sums = part.narrow(0, rows * dim * (N + 2), dim * (N + 2));
  p.dA = base + rows * dim * (N + 2), p.dD = p.dA + dim * N, p.ddelta_bias = p.dD + dim;
  if (z) {
    dz = dz_in ? *dz_in : at::empty_like(*z);
    if (recompute_out_z) out_z = at::empty_like(u);
  }
  p.ckpt = ckpt.data_ptr<float>();
  p.dout = dout.data_ptr(), p.du = du.data_ptr(), p.ddelta = ddelta.data_ptr();
  p.dz = ptr(dz), p.out_z = ptr(out_z);
  p.dB32 = dB32.data_ptr<float>(), p.dC32 = dC32.data_ptr<float>();
  p.dB = ptr(dB), p.dC = ptr(dC);
  p.dout_bs = dout.stride(0), p.dout_ds = dout.stride(1), p.du_bs = du.stride(0), p.du_ds = du.stride(1);
  p.ddelta_bs = ddelta.stride(0), p.ddelta_ds = ddelta.stride(1);
  if (dz) p.dz_bs = dz->stride(0), p.dz_ds = dz->stride(1);
  if (out_z) p.outz_bs = out_z->stride(0), p.outz_ds = out_z->stride(1);
  check_rc(mamba1_scan_bwd(&p, stream_of(dev)), "mamba1_scan_bwd");
  TensorList r(9);
  r[0] = du, r[1] = ddelta, r[2] = sums.narrow(0, 0, dim * N).view({dim, N});
  r[3] = B.dim() == 2 ? OptTensor(dB32.sum(0)) : dB;
  r[4] = C.dim() == 2 ? OptTensor(dC32.sum(0)) : dC;
  if (D) r[5] = sums.narrow(0, dim * N, dim);
  if (delta_bias) r[6] = sums.narrow(0, dim * (N + 1), dim);
  r[7] = dz, r[8] = out_z;
  return r;
}

bool ckpt_ok(const at::Tensor &ckpt, const MambaScanParams &p) {
  const int64_t tile = mamba_hip_query(MAMBA_Q_SCAN_TILE), ntiles = (p.seqlen + tile - 1) / tile;
  return ckpt.scalar_type() == at::kFloat && ckpt.dim() == 4 && ckpt.size(0) == p.batch && ckpt.size(1) == p.dim &&
         ckpt.size(2) == ntiles && ckpt.size(3) == p.dstate && ckpt.is_contiguous();
}

std::optional<TensorList> scan_bwd_fast(const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A,
                                        const at::Tensor &B, const at::Tensor &C, const OptTensor &D, const OptTensor &z,
                                        const OptTensor &delta_bias, const at::Tensor &dout, const at::Tensor &ckpt,
                                        const OptTensor &dz_in, bool delta_softplus, bool recompute_out_z) {
  MambaScanParams p{};
  if (!fill_scan(p, u, delta, A, B, C, D, z, delta_bias, delta_softplus)) return std::nullopt;
  const c10::Device dev = u.device();
  if (!on_device(dout, dev) || !on_device(ckpt, dev) || !on_device(dz_in, dev)) return std::nullopt;
  if (!rows_ok(dout, p.batch, p.dim, p.seqlen, u.scalar_type())) return std::nullopt;
  if (dz_in && (!z || !rows_ok(*dz_in, p.batch, p.dim, p.seqlen, u.scalar_type()))) return std::nullopt;
  if (!ckpt_ok(ckpt, p)) return std::nullopt;
  return scan_bwd(p, u, delta, B, C, D, z, delta_bias, dout, ckpt, dz_in, recompute_out_z, std::nullopt, std::nullopt);
}

// ------------------------------------------------------------------ selective_scan_fn
struct ScanArgs {  // as the kernels take them: unit last strides, B / C with a group axis
  at::Tensor u, delta, A, B, C;
  OptTensor D, z, delta_bias;
};
at::Tensor unit_last(const at::Tensor &t) { return t.stride(-1) == 1 ? t : t.contiguous(); }
ScanArgs normalised(const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A, const at::Tensor &B, const at::Tensor &C,
                    const OptTensor &D, const OptTensor &z, const OptTensor &delta_bias) {
  auto bc = [](const at::Tensor &t) {
    const at::Tensor r = t.dim() == 2 ? t.contiguous() : unit_last(t);
    return r.dim() == 3 ? r.unsqueeze(1) : r;
  };
  ScanArgs a{unit_last(u), unit_last(delta), A.contiguous(), bc(B), bc(C), std::nullopt, std::nullopt, delta_bias};
  if (D) a.D = D->contiguous();
  if (z) a.z = unit_last(*z);
  return a;
}

struct ScanFn : torch::autograd::Function<ScanFn> {
  static variable_list forward(AutogradContext *ctx, const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A,
                               const at::Tensor &B, const at::Tensor &C, const OptTensor &D, const OptTensor &z,
                               const OptTensor &delta_bias, bool delta_softplus, bool return_last_state) {
    const ScanArgs a = normalised(u, delta, A, B, C, D, z, delta_bias);
    MambaScanParams p{};
    TORCH_CHECK(fill_scan(p, a.u, a.delta, a.A, a.B, a.C, a.D, a.z, a.delta_bias, delta_softplus), "selective_scan: arguments");
    auto [out, ckpt] = scan_fwd(p, a.u, a.delta);
    ctx->save_for_backward({a.u, a.delta, a.A, a.B, a.C, tensor_or_none(a.D), tensor_or_none(a.z), tensor_or_none(a.delta_bias), ckpt});
    ctx->saved_data["softplus"] = delta_softplus;
    ctx->saved_data["squeeze"] = std::vector<int64_t>{B.dim() == 3, C.dim() == 3};
    ctx->set_materialize_grads(false);
    variable_list r = {out};
    if (return_last_state) r.push_back(ckpt.select(2, ckpt.size(2) - 1));
    return r;
  }
  // (the gradient of the last state is not considered, as in the reference, selective_scan_interface.py:118-124)
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const OptTensor D = opt(s[5]), z = opt(s[6]), bias = opt(s[7]);
    c10::DeviceGuard guard(s[0].device());
    const at::Tensor dout = grads[0].defined() ? unit_last(grads[0]) : at::zeros(s[0].sizes(), s[0].options());
    MambaScanParams p{};
    TORCH_CHECK(fill_scan(p, s[0], s[1], s[2], s[3], s[4], D, z, bias, ctx->saved_data["softplus"].toBool()), "selective_scan: arguments");
    const TensorList r = scan_bwd(p, s[0], s[1], s[3], s[4], D, z, bias, dout, s[8], std::nullopt, false, std::nullopt, std::nullopt);
    const std::vector<int64_t> squeeze = ctx->saved_data["squeeze"].toIntVector();
    variable_list g(10);
    g[0] = *r[0], g[1] = *r[1], g[2] = *r[2];
    g[3] = squeeze[0] ? r[3]->squeeze(1) : *r[3];
    g[4] = squeeze[1] ? r[4]->squeeze(1) : *r[4];
    g[5] = tensor_or_none(r[5]), g[6] = tensor_or_none(r[7]), g[7] = tensor_or_none(r[6]);
    return g;
  }
};

// selective_scan_fn: out, or (out, last_state); None = declined
pybind11::object selective_scan(const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A, const at::Tensor &B,
                                const at::Tensor &C, const OptTensor &D, const OptTensor &z, const OptTensor &delta_bias,
                                bool delta_softplus, bool return_last_state) {
  const pybind11::object no = pybind11::none();
  if (!u.is_cuda() || u.dim() != 3 || delta.dim() != 3 || A.dim() != 2 || B.dim() < 2 || C.dim() < 2 || B.dim() > 4 || C.dim() > 4 ||
      (z && z->dim() != 3) || A.is_complex())
    return no;
  const ScanArgs a = normalised(u, delta, A, B, C, D, z, delta_bias);
  MambaScanParams p{};
  if (!fill_scan(p, a.u, a.delta, a.A, a.B, a.C, a.D, a.z, a.delta_bias, delta_softplus)) return no;
  if (!records(u, delta, A, B, C, D, z, delta_bias)) {
    auto [out, ckpt] = scan_fwd(p, a.u, a.delta);
    return return_last_state ? pybind11::object(pybind11::make_tuple(out, ckpt.select(2, ckpt.size(2) - 1))) : pybind11::cast(out);
  }
  variable_list r = ScanFn::apply(u, delta, A, B, C, D, z, delta_bias, delta_softplus, return_last_state);
  return return_last_state ? pybind11::object(pybind11::make_tuple(r[0], r[1])) : pybind11::cast(r[0]);
}

// ------------------------------------------------------------------ mamba_inner_fn
// conv1d + SiLU -> x_proj -> dt_proj -> scan -> out_proj (selective_scan_interface.py:196-383) for a real A and B, C
// and delta from x_proj.  Every (batch, dim, seqlen) intermediate lives in memory as (dim, batch, seqlen), so that the
// projections see (dim, batch * seqlen) matrices; x_proj's output is formed as (rank + 2 dstate, batch * seqlen), whose
// row blocks are delta's factor and the scan's B and C as they lie (no transposing copies, forward or backward).
at::Tensor channel_major(const at::Tensor &m, int64_t batch, int64_t L) {  // (dim, batch * L) -> its (batch, dim, L) view
  return m.view({m.size(0), batch, L}).permute({1, 0, 2});
}
at::Tensor bc_rows(const at::Tensor &x_dbl, int64_t row, int64_t n, int64_t batch, int64_t L) {
  return x_dbl.narrow(0, row, n).view({n, batch, L}).permute({1, 0, 2}).unsqueeze(1);
}


struct InnerFn : torch::autograd::Function<InnerFn> {
  static at::Tensor forward(AutogradContext *ctx, const at::Tensor &xz, const at::Tensor &conv_weight, const OptTensor &conv_bias,
                            const at::Tensor &x_proj, const at::Tensor &dt_proj, const at::Tensor &out_proj,
                            const OptTensor &out_bias, const at::Tensor &A, const OptTensor &D, const OptTensor &delta_bias,
                            bool delta_softplus, int64_t checkpoint_lvl, at::ScalarType compute) {
    const int64_t batch = xz.size(0), d = xz.size(1) / 2, L = xz.size(2), N = A.size(1), R = dt_proj.size(1);
    const at::Tensor conv_w = conv_weight.squeeze(1), Ac = A.contiguous();
    const at::Tensor xp = x_proj.to(compute), dp = dt_proj.to(compute), op = out_proj.to(compute);
    const at::Tensor x = xz.narrow(1, 0, d), z = xz.narrow(1, d, d);
    at::Tensor conv = at::empty({d, batch * L}, xz.options());
    conv_fwd(x, conv_w, conv_bias, std::nullopt, true, channel_major(conv, batch, L));
    const at::Tensor x_dbl = at::mm(xp, conv);                                 // (rank + 2 n, b l)
    const at::Tensor delta = at::mm(dp, x_dbl.narrow(0, 0, R));                // (dim, b l)
    MambaScanParams p{};
    const at::Tensor u3 = channel_major(conv, batch, L), d3 = channel_major(delta, batch, L);
    TORCH_CHECK(fill_scan(p, u3, d3, Ac, bc_rows(x_dbl, R, N, batch, L), bc_rows(x_dbl, R + N, N, batch, L), D, z, delta_bias,
                          delta_softplus),
                "mamba_inner_fn: arguments");
    auto [out_z, ckpt] = scan_fwd(p, u3, d3);  // out_z has delta's layout
    const bool keep = checkpoint_lvl == 0;     // else conv and delta are formed again in the backward pass
    ctx->save_for_backward({xz, conv_w, tensor_or_none(conv_bias), x_dbl, xp, dp, op, keep ? conv : at::Tensor(),
                            keep ? delta : at::Tensor(), Ac, tensor_or_none(D), tensor_or_none(delta_bias), ckpt});
    ctx->saved_data["softplus"] = delta_softplus;
    ctx->saved_data["out_bias"] = out_bias.has_value();
    const at::Tensor rows = out_z.permute({1, 0, 2}).reshape({d, batch * L}).t();
    return at::linear(rows, op, out_bias ? OptTensor(out_bias->to(compute)) : std::nullopt).view({batch, L, -1});
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &xz = s[0], &conv_w = s[1], &x_dbl = s[3], &xp = s[4], &dp = s[5], &op = s[6], &Ac = s[9], &ckpt = s[12];
    const OptTensor conv_bias = opt(s[2]), D = opt(s[10]), delta_bias = opt(s[11]);
    const int64_t batch = xz.size(0), d = xz.size(1) / 2, L = xz.size(2), N = Ac.size(1), R = dp.size(1);
    c10::DeviceGuard guard(xz.device());
    const at::Tensor x = xz.narrow(1, 0, d), z = xz.narrow(1, d, d);
    at::Tensor conv = s[7], delta = s[8];
    if (!conv.defined()) {
      conv = at::empty({d, batch * L}, xz.options());
      conv_fwd(x, conv_w, conv_bias, std::nullopt, true, channel_major(conv, batch, L));
      delta = at::mm(dp, x_dbl.narrow(0, 0, R));
    }
    at::Tensor dxz = at::empty_like(xz);
    const at::Tensor dx = dxz.narrow(1, 0, d), dz = dxz.narrow(1, d, d);
    const at::Tensor dout = grads[0].reshape({batch * L, -1}).to(op.scalar_type());      // (b l) x e
    const at::Tensor dy = at::mm(op.t(), dout.t());                                      // (dim, b l)
    at::Tensor dx_dbl = at::empty_like(x_dbl);
    MambaScanParams p{};
    const at::Tensor u3 = channel_major(conv, batch, L), d3 = channel_major(delta, batch, L);
    const at::Tensor B = bc_rows(x_dbl, R, N, batch, L), C = bc_rows(x_dbl, R + N, N, batch, L);
    TORCH_CHECK(fill_scan(p, u3, d3, Ac, B, C, D, z, delta_bias, ctx->saved_data["softplus"].toBool()), "mamba_inner_fn: arguments");
    const TensorList r = scan_bwd(p, u3, d3, B, C, D, z, delta_bias, channel_major(dy, batch, L), ckpt, dz, true,
                                  bc_rows(dx_dbl, R, N, batch, L), bc_rows(dx_dbl, R + N, N, batch, L));
    auto matrix = [&](const at::Tensor &t) { return t.permute({1, 0, 2}).reshape({d, batch * L}); };
    at::Tensor dconv = matrix(*r[0]);
    const at::Tensor ddelta = matrix(*r[1]), out_z = matrix(*r[8]);
    const at::Tensor dop = at::mm(dout.t(), out_z.t());
    const at::Tensor ddp = at::mm(ddelta, x_dbl.narrow(0, 0, R).t());
    at::Tensor dt_rows = dx_dbl.narrow(0, 0, R);
    at::mm_out(dt_rows, dp.t(), ddelta);
    const at::Tensor dxp = at::mm(dx_dbl, conv.t());
    dconv.addmm_(xp.t(), dx_dbl);  // the scan's own du buffer: the x_proj path is added in place
    auto [dcw, dcb] = conv_bwd(x, conv_w, conv_bias, channel_major(dconv, batch, L), std::nullopt, true, dx);
    variable_list g(13);
    g[0] = dxz, g[1] = dcw.unsqueeze(1), g[2] = tensor_or_none(dcb), g[3] = dxp, g[4] = ddp, g[5] = dop;
    if (ctx->saved_data["out_bias"].toBool()) g[6] = dout.sum(0);
    g[7] = *r[2], g[8] = tensor_or_none(r[5]), g[9] = tensor_or_none(r[6]);
    return g;
  }
};

// mamba_inner_fn; None = declined
OptTensor mamba_inner(const at::Tensor &xz_in, const at::Tensor &conv_weight, const OptTensor &conv_bias, const at::Tensor &x_proj,
                      const at::Tensor &dt_proj, const at::Tensor &out_proj, const OptTensor &out_bias, const at::Tensor &A,
                      const OptTensor &D, const OptTensor &delta_bias, bool delta_softplus, int64_t checkpoint_lvl) {
  if (!xz_in.is_cuda() || xz_in.dim() != 3 || xz_in.size(1) % 2 != 0 || conv_weight.dim() != 3 || conv_weight.size(1) != 1)
    return std::nullopt;
  const at::Tensor xz = unit_last(xz_in);
  const c10::Device dev = xz.device();
  const bool autocast = at::autocast::is_autocast_enabled(at::kCUDA);
  const at::ScalarType compute = autocast ? at::autocast::get_autocast_dtype(at::kCUDA) : xz.scalar_type();
  if (dtype_code(xz) < 0 || compute != xz.scalar_type()) return std::nullopt;
  const int64_t batch = xz.size(0), d = xz.size(1) / 2, L = xz.size(2);
  if (batch <= 0 || d <= 0 || L <= 0 || A.dim() != 2 || A.scalar_type() != at::kFloat || A.size(0) != d) return std::nullopt;
  const int64_t N = A.size(1), R = dt_proj.dim() == 2 ? dt_proj.size(1) : 0;
  auto matrix_ok = [&](const at::Tensor &t, int64_t rows, int64_t cols) {
    return on_device(t, dev) && t.dim() == 2 && (rows < 0 || t.size(0) == rows) && t.size(1) == cols &&
           (t.scalar_type() == compute || (autocast && t.is_floating_point()));
  };
  if (R <= 0 || !matrix_ok(x_proj, R + 2 * N, d) || !matrix_ok(dt_proj, d, R) || !matrix_ok(out_proj, -1, d)) return std::nullopt;
  if (out_bias && (!on_device(*out_bias, dev) || out_bias->dim() != 1 || out_bias->size(0) != out_proj.size(0) ||
                   !(out_bias->scalar_type() == compute || (autocast && out_bias->is_floating_point()))))
    return std::nullopt;
  if (!conv_params_ok(xz.narrow(1, 0, d), conv_weight.squeeze(1), conv_bias, std::nullopt)) return std::nullopt;
  auto vec_ok = [&](const OptTensor &t) {
    return !t || (on_device(*t, dev) && t->scalar_type() == at::kFloat && t->dim() == 1 && t->size(0) == d && t->is_contiguous());
  };
  if (!on_device(A, dev) || !vec_ok(D) || !vec_ok(delta_bias) || N > mamba_hip_query(MAMBA_Q_MAX_DSTATE)) return std::nullopt;
  c10::DeviceGuard guard(dev);
  return InnerFn::apply(xz, conv_weight, conv_bias, x_proj, dt_proj, out_proj, out_bias, A, D, delta_bias, delta_softplus,
                        checkpoint_lvl, compute);
}

}  // namespace

void bind_scan(pybind11::module_ &m) {
  namespace py = pybind11;
  m.def("scan_fwd", &scan_fwd_fast, py::arg("u"), py::arg("delta"), py::arg("A"), py::arg("B"), py::arg("C"), py::arg("D"),
        py::arg("z"), py::arg("delta_bias"), py::arg("delta_softplus"),
        "selective_scan_cuda.fwd: returns (out, ckpt), or None when the arguments need the Python path.");
  m.def("scan_bwd", &scan_bwd_fast, py::arg("u"), py::arg("delta"), py::arg("A"), py::arg("B"), py::arg("C"), py::arg("D"),
        py::arg("z"), py::arg("delta_bias"), py::arg("dout"), py::arg("ckpt"), py::arg("dz"), py::arg("delta_softplus"),
        py::arg("recompute_out_z"),
        "selective_scan_cuda.bwd: returns [du, ddelta, dA, dB, dC, dD, ddelta_bias, dz, out_z], or None.");
  m.def("selective_scan", &selective_scan, py::arg("u"), py::arg("delta"), py::arg("A"), py::arg("B"), py::arg("C"), py::arg("D"),
        py::arg("z"), py::arg("delta_bias"), py::arg("delta_softplus"), py::arg("return_last_state"),
        "selective_scan_fn with autograd: out or (out, last_state), or None when the arguments need the Python path.");
  m.def("mamba_inner", &mamba_inner, py::arg("xz"), py::arg("conv_weight"), py::arg("conv_bias"), py::arg("x_proj"),
        py::arg("dt_proj"), py::arg("out_proj"), py::arg("out_bias"), py::arg("A"), py::arg("D"), py::arg("delta_bias"),
        py::arg("delta_softplus"), py::arg("checkpoint_lvl"),
        "mamba_inner_fn with autograd, or None when the arguments need the Python path.");
}

}  // namespace mamba_ext
