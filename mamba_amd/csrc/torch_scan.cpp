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
    } else if (t->dim() == 3) {  // one group, without its axis
      if (G != 1 || t->scalar_type() != u.scalar_type() || t->stride(2) != 1 || t->size(0) != batch || t->size(1) != N || t->size(2) != L)
        return false;
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
  auto bc_strides = [](const at::Tensor &t, int64_t &bs, int64_t &gs, int64_t &ns) {
    if (t.dim() > 2) bs = t.stride(0), gs = t.dim() == 4 ? t.stride(1) : 0, ns = t.stride(t.dim() - 2);
  };
  bc_strides(B, p.B_bs, p.B_gs, p.B_ns);
  bc_strides(C, p.C_bs, p.C_gs, p.C_ns);
  return true;
}

// The forward call on filled parameters, p.out included -> ckpt.  One allocation holds the workspace of a sequence that
// goes in segments.
at::Tensor run_scan_fwd(MambaScanParams &p, const c10::Device &dev) {
  const auto f32 = at::TensorOptions().dtype(at::kFloat).device(dev);
  const int64_t tile = mamba_hip_query(MAMBA_Q_SCAN_TILE), ntiles = (p.seqlen + tile - 1) / tile;
  at::Tensor ckpt = at::empty({p.batch, p.dim, ntiles, p.dstate}, f32), ws;
  p.ckpt = ckpt.data_ptr<float>();
  p.nseg = std::max(1, mamba1_scan_segments(&p, 0));
  if (p.nseg > 1) {
    ws = at::empty({(int64_t)p.batch * p.nseg * p.dim * (p.dstate + 2)}, f32);
    p.seg_ws = ws.data_ptr<float>();
  }
  check_rc(mamba1_scan_fwd(&p, stream_of(dev)), "mamba1_scan_fwd");
  return ckpt;
}

// The backward call on filled parameters, the operands' gradients included (dB / dC of per-position B / C; constant
// ones come back as partials) -> the sums dA (dim, dstate), dD and ddelta_bias (dim) in one array, one after the other.
struct ScanSums {
  at::Tensor sums, dB_parts, dC_parts;
};
ScanSums run_scan_bwd(MambaScanParams &p, const c10::Device &dev) {
  const auto f32 = at::TensorOptions().dtype(at::kFloat).device(dev);
  const int64_t batch = p.batch, dim = p.dim, N = p.dstate;
  p.nseg = std::max(1, mamba1_scan_segments(&p, 1));
  const int64_t nseg = p.nseg, nparts = mamba1_scan_bwd_nparts(&p);
  if (nparts <= 0) check_rc(nparts ? (int)nparts : -1, "mamba1_scan_bwd_nparts");
  const int64_t rows = batch * nseg, bc = batch * p.ngroups * nparts * N * p.seqlen;
  auto padded = [](int64_t n) { return (n + 63) / 64 * 64; };
  const int64_t seg = nseg > 1 ? padded(rows * dim * (N + 2)) : 0, part = padded(rows * dim * (N + 2));
  ScanSums r;
  r.sums = at::empty({dim * (N + 2)}, f32);
  at::Tensor ws = at::empty({seg + part + 2 * padded(bc)}, f32);
  float *base = ws.data_ptr<float>();
  if (nseg > 1) p.seg_ws = base;
  base += seg;
  p.dA_part = base, p.dD_part = base + rows * dim * N, p.ddelta_bias_part = p.dD_part + rows * dim;
  p.dA = r.sums.data_ptr<float>(), p.dD = p.dA + dim * N, p.ddelta_bias = p.dD + dim;
  p.dB32 = base + part, p.dC32 = p.dB32 + padded(bc);
  if (p.bc_const & 1) r.dB_parts = at::empty({rows, dim, N}, f32), p.dB32 = r.dB_parts.data_ptr<float>();
  if (p.bc_const & 2) r.dC_parts = at::empty({rows, dim, N}, f32), p.dC32 = r.dC_parts.data_ptr<float>();
  check_rc(mamba1_scan_bwd(&p, stream_of(dev)), "mamba1_scan_bwd");
  return r;
}

// selective_scan_cuda.fwd (selective_scan.cpp:226) on filled parameters -> (out, ckpt); real A only.
std::tuple<at::Tensor, at::Tensor> scan_fwd(MambaScanParams &p, const at::Tensor &u, const at::Tensor &delta) {
  const c10::Device dev = u.device();
  c10::DeviceGuard guard(dev);
  at::Tensor out = at::empty_like(delta);
  p.out = out.data_ptr(), p.out_bs = out.stride(0), p.out_ds = out.stride(1);
  return {out, run_scan_fwd(p, dev)};
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
// -> [du, ddelta, dA, dB, dC, dD, ddelta_bias, dz, out_z].
TensorList scan_bwd(MambaScanParams &p, const at::Tensor &u, const at::Tensor &delta, const at::Tensor &B, const at::Tensor &C,
                    const OptTensor &D, const OptTensor &z, const OptTensor &delta_bias, const at::Tensor &dout,
                    const at::Tensor &ckpt, const OptTensor &dz_in, bool recompute_out_z) {
  const c10::Device dev = u.device();
  c10::DeviceGuard guard(dev);
  const int64_t dim = p.dim, N = p.dstate;
  at::Tensor du = at::empty_like(u), ddelta = at::empty_like(delta);
  OptTensor dB, dC, dz, out_z;
  if (B.dim() > 2) {
    dB = at::empty(B.sizes(), B.options());
    p.dB = ptr(dB), p.dB_ns = p.seqlen, p.dB_gs = N * p.dB_ns, p.dB_bs = p.ngroups * p.dB_gs;
  }
  if (C.dim() > 2) {
    dC = at::empty(C.sizes(), C.options());
    p.dC = ptr(dC), p.dC_ns = p.seqlen, p.dC_gs = N * p.dC_ns, p.dC_bs = p.ngroups * p.dC_gs;
  }
  if (z) {
    dz = dz_in ? *dz_in : at::empty_like(*z);
    if (recompute_out_z) out_z = at::empty_like(u);
  }
  p.ckpt = ckpt.data_ptr<float>();
  p.dout = dout.data_ptr(), p.du = du.data_ptr(), p.ddelta = ddelta.data_ptr();
  p.dz = ptr(dz), p.out_z = ptr(out_z);
  p.dout_bs = dout.stride(0), p.dout_ds = dout.stride(1), p.du_bs = du.stride(0), p.du_ds = du.stride(1);
  p.ddelta_bs = ddelta.stride(0), p.ddelta_ds = ddelta.stride(1);
  if (dz) p.dz_bs = dz->stride(0), p.dz_ds = dz->stride(1);
  if (out_z) p.outz_bs = out_z->stride(0), p.outz_ds = out_z->stride(1);
  const ScanSums q = run_scan_bwd(p, dev);
  TensorList r(9);
  r[0] = du, r[1] = ddelta, r[2] = q.sums.as_strided({dim, N}, {N, 1}, 0);
  r[3] = B.dim() == 2 ? OptTensor(q.dB_parts.sum(0)) : dB;
  r[4] = C.dim() == 2 ? OptTensor(q.dC_parts.sum(0)) : dC;
  if (D) r[5] = q.sums.as_strided({dim}, {1}, dim * N);
  if (delta_bias) r[6] = q.sums.as_strided({dim}, {1}, dim * (N + 1));
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
  return scan_bwd(p, u, delta, B, C, D, z, delta_bias, dout, ckpt, dz_in, recompute_out_z);
}

// ------------------------------------------------------------------ selective_scan_fn
struct ScanArgs {  // as the kernels take them: unit last strides
  at::Tensor u, delta, A, B, C;
  OptTensor D, z, delta_bias;
};
at::Tensor unit_last(const at::Tensor &t) { return t.stride(-1) == 1 ? t : t.contiguous(); }
ScanArgs normalised(const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A, const at::Tensor &B, const at::Tensor &C,
                    const OptTensor &D, const OptTensor &z, const OptTensor &delta_bias) {
  auto bc = [](const at::Tensor &t) { return t.dim() == 2 ? t.contiguous() : unit_last(t); };
  ScanArgs a{unit_last(u), unit_last(delta), A.contiguous(), bc(B), bc(C), std::nullopt, std::nullopt, delta_bias};
  if (D) a.D = D->contiguous();
  if (z) a.z = unit_last(*z);
  return a;
}

struct ScanFn : torch::autograd::Function<ScanFn> {
  // the gradients are those of the caller's tensors, the kernels and the backward pass take `a`
  static variable_list forward(AutogradContext *ctx, const at::Tensor &, const at::Tensor &, const at::Tensor &, const at::Tensor &,
                               const at::Tensor &, const OptTensor &, const OptTensor &, const OptTensor &, const ScanArgs &a,
                               bool delta_softplus, bool return_last_state) {
    MambaScanParams p{};
    TORCH_CHECK(fill_scan(p, a.u, a.delta, a.A, a.B, a.C, a.D, a.z, a.delta_bias, delta_softplus), "selective_scan: arguments");
    auto [out, ckpt] = scan_fwd(p, a.u, a.delta);
    ctx->save_for_backward({a.u, a.delta, a.A, a.B, a.C, tensor_or_none(a.D), tensor_or_none(a.z), tensor_or_none(a.delta_bias), ckpt});
    ctx->saved_data["softplus"] = delta_softplus;
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
    const TensorList r = scan_bwd(p, s[0], s[1], s[3], s[4], D, z, bias, dout, s[8], std::nullopt, false);
    variable_list g(11);
    g[0] = *r[0], g[1] = *r[1], g[2] = *r[2];
    g[3] = *r[3], g[4] = *r[4];
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
      (z && z->dim() != 3) || A.is_complex() || python_call(u, delta, A, B, C, D, z, delta_bias))
    return no;
  const ScanArgs a = [&] {
    at::AutoGradMode no_grad(false);  // copies are not the caller's tensors: the node below knows those
    return normalised(u, delta, A, B, C, D, z, delta_bias);
  }();
  MambaScanParams p{};
  if (!fill_scan(p, a.u, a.delta, a.A, a.B, a.C, a.D, a.z, a.delta_bias, delta_softplus)) return no;
  if (!records(u, delta, A, B, C, D, z, delta_bias)) {
    auto [out, ckpt] = scan_fwd(p, a.u, a.delta);
    return return_last_state ? pybind11::object(pybind11::make_tuple(out, ckpt.select(2, ckpt.size(2) - 1))) : pybind11::cast(out);
  }
  variable_list r = ScanFn::apply(u, delta, A, B, C, D, z, delta_bias, a, delta_softplus, return_last_state);
  return return_last_state ? pybind11::object(pybind11::make_tuple(r[0], r[1])) : pybind11::cast(r[0]);
}

// ------------------------------------------------------------------ mamba_inner_fn
// conv1d + SiLU -> x_proj -> dt_proj -> scan -> out_proj (selective_scan_interface.py:196-383) for a real A and B, C
// and delta from x_proj.  Every (batch, dim, seqlen) intermediate lies in memory as (dim, batch, seqlen), so that the
// projections see (dim, batch * seqlen) matrices; x_proj's output is formed as (rank + 2 dstate, batch * seqlen), whose
// row blocks are delta's factor and the scan's B and C as they lie (no transposing copies, forward or backward).  A
// short call takes little GPU time, so this works on pointers and strides, keeps what it saves in few allocations and
// hands products that do not depend on each other over together.
struct InnerDims {
  int64_t batch, d, L, N, R, E, rows, BL;  // E: out_proj's rows; rows = R + 2 N; BL = batch * L
};
int64_t aligned8(int64_t n) { return (n + 7) / 8 * 8; }

// the scan's operands inside xz, the activations (conv, delta) and x_dbl, all of one dtype
void fill_inner_scan(MambaScanParams &p, const InnerDims &q, const at::Tensor &xz, char *conv, char *delta, char *x_dbl,
                     const at::Tensor &A, const OptTensor &D, const OptTensor &delta_bias, bool delta_softplus) {
  const int64_t es = xz.element_size();
  p.batch = (int32_t)q.batch, p.dim = (int32_t)q.d, p.seqlen = (int32_t)q.L, p.dstate = (int32_t)q.N, p.ngroups = 1;
  p.dtype = dtype_code(xz), p.delta_softplus = delta_softplus ? 1 : 0;
  p.u = conv, p.u_bs = q.L, p.u_ds = q.BL;
  p.delta = delta, p.delta_bs = q.L, p.delta_ds = q.BL;
  p.z = static_cast<char *>(xz.data_ptr()) + q.d * xz.stride(1) * es, p.z_bs = xz.stride(0), p.z_ds = xz.stride(1);
  p.B = x_dbl + q.R * q.BL * es, p.B_bs = q.L, p.B_gs = 0, p.B_ns = q.BL;
  p.C = x_dbl + (q.R + q.N) * q.BL * es, p.C_bs = q.L, p.C_gs = 0, p.C_ns = q.BL;
  p.A = A.data_ptr(), p.D = ptr(D), p.delta_bias = ptr(delta_bias);
}

// conv (d, BL) and delta (d, BL) from xz and x_dbl; x_dbl is formed first when `with_x_dbl`
void inner_activations(const InnerDims &q, const at::Tensor &xz, const at::Tensor &conv_w, const OptTensor &conv_bias,
                       const void *xp, const void *dp, char *conv, char *delta, char *x_dbl, bool with_x_dbl) {
  const at::ScalarType ty = xz.scalar_type();
  conv_fwd(xz, q.batch, q.d, q.L, {xz.data_ptr(), xz.stride(0), xz.stride(1), 1}, conv_w, conv_bias, std::nullopt, true,
           {conv, q.L, q.BL, 1});
  Products m(xz.options(), ty);
  if (with_x_dbl) m.add(x_dbl, ty, q.BL, q.rows, q.BL, q.d, {xp, q.d, 1}, {conv, 1, q.BL}).run();
  m.add(delta, ty, q.BL, q.d, q.BL, q.R, {dp, q.R, 1}, {x_dbl, 1, q.BL}).run();
}

struct InnerFn : torch::autograd::Function<InnerFn> {
  static at::Tensor forward(AutogradContext *ctx, const at::Tensor &xz, const at::Tensor &conv_w, const OptTensor &conv_bias,
                            const at::Tensor &x_proj, const at::Tensor &dt_proj, const at::Tensor &out_proj,
                            const OptTensor &out_bias, const at::Tensor &A, const OptTensor &D, const OptTensor &delta_bias,
                            bool delta_softplus, int64_t checkpoint_lvl, at::ScalarType compute) {
    InnerDims q;
    q.batch = xz.size(0), q.d = xz.size(1) / 2, q.L = xz.size(2), q.N = A.size(1), q.R = dt_proj.size(1), q.E = out_proj.size(0);
    q.rows = q.R + 2 * q.N, q.BL = q.batch * q.L;
    const int64_t es = xz.element_size();
    const at::Tensor Ac = A.contiguous();
    // the weights in the compute dtype: three pieces of one array where they are converted
    const void *xp, *dp, *op;
    at::Tensor w, xpc, dpc, opc;
    if (compute == at::kBFloat16 && x_proj.scalar_type() == at::kFloat && dt_proj.scalar_type() == at::kFloat &&
        out_proj.scalar_type() == at::kFloat && x_proj.is_contiguous() && dt_proj.is_contiguous() && out_proj.is_contiguous()) {
      const int64_t nx = aligned8(q.rows * q.d), nd = aligned8(q.d * q.R), no = q.E * q.d;
      w = at::empty({nx + nd + no}, xz.options());
      char *base = static_cast<char *>(w.data_ptr());
      const MambaCast c[3] = {{x_proj.data_ptr<float>(), base, q.rows * q.d}, {dt_proj.data_ptr<float>(), base + 2 * nx, q.d * q.R},
                              {out_proj.data_ptr<float>(), base + 2 * (nx + nd), no}};
      check_rc(mamba_cast_bf16(c, 3, stream_of(xz.device())), "mamba_cast_bf16");
      xp = c[0].dst, dp = c[1].dst, op = c[2].dst;
    } else {
      xpc = x_proj.to(compute).contiguous(), dpc = dt_proj.to(compute).contiguous(), opc = out_proj.to(compute).contiguous();
      xp = xpc.data_ptr(), dp = dpc.data_ptr(), op = opc.data_ptr();
    }
    at::Tensor x_dbl = at::empty({q.rows, q.BL}, xz.options()), act = at::empty({2 * aligned8(q.d * q.BL)}, xz.options());
    at::Tensor out_z = at::empty({q.d, q.BL}, xz.options()), out = at::empty({q.batch, q.L, q.E}, xz.options());
    char *conv = static_cast<char *>(act.data_ptr()), *delta = conv + aligned8(q.d * q.BL) * es;
    char *xd = static_cast<char *>(x_dbl.data_ptr());
    inner_activations(q, xz, conv_w, conv_bias, xp, dp, conv, delta, xd, true);
    MambaScanParams p{};
    fill_inner_scan(p, q, xz, conv, delta, xd, Ac, D, delta_bias, delta_softplus);
    p.out = out_z.data_ptr(), p.out_bs = q.L, p.out_ds = q.BL;
    const at::Tensor ckpt = run_scan_fwd(p, xz.device());
    const at::Tensor bias = out_bias ? out_bias->to(compute).contiguous() : at::Tensor();
    Products(xz.options(), compute)
        .add(out.data_ptr(), compute, q.E, q.BL, q.E, q.d, {out_z.data_ptr(), 1, q.BL}, {op, q.d, 1}, false, out_bias ? bias.data_ptr() : nullptr)
        .run();
    // with checkpoint_lvl 1 conv and delta are formed again in the backward pass
    ctx->save_for_backward({xz, conv_w, tensor_or_none(conv_bias), x_dbl, w, xpc, dpc, opc, checkpoint_lvl == 0 ? act : at::Tensor(),
                            Ac, tensor_or_none(D), tensor_or_none(delta_bias), ckpt});
    ctx->saved_data["o"] = std::vector<int64_t>{q.R, q.E, delta_softplus, out_bias.has_value(), (int64_t)x_proj.scalar_type(),
                                                (int64_t)dt_proj.scalar_type(), (int64_t)out_proj.scalar_type(),
                                                out_bias ? (int64_t)out_bias->scalar_type() : 0};
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> o = ctx->saved_data["o"].toIntVector();
    const at::Tensor &xz = s[0], &conv_w = s[1], &x_dbl = s[3], &w = s[4], &Ac = s[9], &ckpt = s[12];
    const OptTensor conv_bias = opt(s[2]), D = opt(s[10]), delta_bias = opt(s[11]);
    InnerDims q;
    q.batch = xz.size(0), q.d = xz.size(1) / 2, q.L = xz.size(2), q.N = Ac.size(1), q.R = o[0], q.E = o[1];
    q.rows = q.R + 2 * q.N, q.BL = q.batch * q.L;
    const int64_t es = xz.element_size(), part = aligned8(q.d * q.BL) * es, xs = xz.stride(1);
    const at::ScalarType ty = xz.scalar_type();
    c10::DeviceGuard guard(xz.device());
    const char *xp, *dp, *op;
    if (w.defined()) {
      xp = static_cast<const char *>(w.data_ptr()), dp = xp + 2 * aligned8(q.rows * q.d), op = dp + 2 * aligned8(q.d * q.R);
    } else {
      xp = static_cast<const char *>(s[5].data_ptr()), dp = static_cast<const char *>(s[6].data_ptr()), op = static_cast<const char *>(s[7].data_ptr());
    }
    char *xd = static_cast<char *>(x_dbl.data_ptr());
    at::Tensor act = s[8];
    if (!act.defined()) {
      act = at::empty({2 * aligned8(q.d * q.BL)}, xz.options());
      char *c = static_cast<char *>(act.data_ptr());
      inner_activations(q, xz, conv_w, conv_bias, xp, dp, c, c + part, xd, false);
    }
    char *conv = static_cast<char *>(act.data_ptr()), *delta = conv + part;
    at::Tensor dxz = at::empty_like(xz);  // in xz's layout
    if (dxz.stride(2) != 1) dxz = at::empty(xz.sizes(), xz.options());
    at::Tensor tmp = at::empty({4 * (part / es)}, xz.options());
    at::Tensor dx_dbl = at::empty({q.rows, q.BL}, xz.options());
    char *dy = static_cast<char *>(tmp.data_ptr()), *dconv = dy + part, *ddelta = dconv + part, *out_z = ddelta + part;
    char *dxd = static_cast<char *>(dx_dbl.data_ptr()), *dx = static_cast<char *>(dxz.data_ptr());
    const at::Tensor dout = grads[0].scalar_type() == ty && grads[0].is_contiguous() ? grads[0] : grads[0].to(ty).contiguous();  // (b l) x e
    const char *g_out = static_cast<const char *>(dout.data_ptr());
    Products m(xz.options(), ty);
    m.add(dy, ty, q.BL, q.d, q.BL, q.E, {op, 1, q.d}, {g_out, q.E, 1}).run();  // (dim, b l)
    MambaScanParams p{};
    fill_inner_scan(p, q, xz, conv, delta, xd, Ac, D, delta_bias, o[2] != 0);
    p.ckpt = ckpt.data_ptr<float>();
    p.dout = dy, p.dout_bs = q.L, p.dout_ds = q.BL, p.du = dconv, p.du_bs = q.L, p.du_ds = q.BL;
    p.ddelta = ddelta, p.ddelta_bs = q.L, p.ddelta_ds = q.BL, p.out_z = out_z, p.outz_bs = q.L, p.outz_ds = q.BL;
    p.dz = dx + q.d * dxz.stride(1) * es, p.dz_bs = dxz.stride(0), p.dz_ds = dxz.stride(1);
    p.dB = dxd + q.R * q.BL * es, p.dB_bs = q.L, p.dB_gs = 0, p.dB_ns = q.BL;
    p.dC = dxd + (q.R + q.N) * q.BL * es, p.dC_bs = q.L, p.dC_gs = 0, p.dC_ns = q.BL;
    const at::Tensor sums = run_scan_bwd(p, xz.device()).sums;
    // the weights' gradients in the weights' dtype
    auto like = [&](int64_t rows, int64_t cols, int64_t code) { return at::empty({rows, cols}, xz.options().dtype((at::ScalarType)code)); };
    auto direct = [&](int64_t code) { return (at::ScalarType)code == at::kFloat || (at::ScalarType)code == ty ? code : (int64_t)ty; };
    at::Tensor dxp = like(q.rows, q.d, direct(o[4])), ddp = like(q.d, q.R, direct(o[5])), dop = like(q.E, q.d, direct(o[6]));
    m.add(dop.data_ptr(), dop.scalar_type(), q.d, q.E, q.d, q.BL, {g_out, 1, q.E}, {out_z, q.BL, 1});
    m.add(ddp.data_ptr(), ddp.scalar_type(), q.R, q.d, q.R, q.BL, {ddelta, q.BL, 1}, {xd, q.BL, 1});
    m.add(dxd, ty, q.BL, q.R, q.BL, q.d, {dp, 1, q.R}, {ddelta, 1, q.BL}).run();
    m.add(dxp.data_ptr(), dxp.scalar_type(), q.d, q.rows, q.d, q.BL, {dxd, q.BL, 1}, {conv, q.BL, 1});
    m.add(dconv, ty, q.BL, q.d, q.BL, q.rows, {xp, 1, q.d}, {dxd, 1, q.BL}, true).run();  // added to the scan's own du
    auto [dcw, dcb] = conv_bwd(xz, q.batch, q.d, q.L, {xz.data_ptr(), xz.stride(0), xs, 1}, conv_w, conv_bias, {dconv, q.L, q.BL, 1},
                               std::nullopt, true, {dx, dxz.stride(0), dxz.stride(1), 1});
    variable_list g(13);
    g[0] = dxz, g[1] = dcw, g[2] = tensor_or_none(dcb), g[3] = dxp.to((at::ScalarType)o[4]), g[4] = ddp.to((at::ScalarType)o[5]);
    g[5] = dop.to((at::ScalarType)o[6]);
    if (o[3]) g[6] = dout.view({q.BL, q.E}).sum(0).to((at::ScalarType)o[7]);
    g[7] = sums.as_strided({q.d, q.N}, {q.N, 1}, 0);
    if (D) g[8] = sums.as_strided({q.d}, {1}, q.d * q.N);
    if (delta_bias) g[9] = sums.as_strided({q.d}, {1}, q.d * (q.N + 1));
    return g;
  }
};

// mamba_inner_fn; None = declined
OptTensor mamba_inner(const at::Tensor &xz_in, const at::Tensor &conv_weight, const OptTensor &conv_bias, const at::Tensor &x_proj,
                      const at::Tensor &dt_proj, const at::Tensor &out_proj, const OptTensor &out_bias, const at::Tensor &A,
                      const OptTensor &D, const OptTensor &delta_bias, bool delta_softplus, int64_t checkpoint_lvl) {
  if (!xz_in.is_cuda() || xz_in.dim() != 3 || xz_in.size(1) % 2 != 0 || conv_weight.dim() != 3 || conv_weight.size(1) != 1 ||
      python_call(xz_in, conv_weight, conv_bias, x_proj, dt_proj, out_proj, out_bias, A, D, delta_bias))
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
