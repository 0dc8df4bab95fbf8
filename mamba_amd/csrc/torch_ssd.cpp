// The Mamba-2 chunked scan and mixer on at::Tensor (the role of the reference's Python orchestration around its Triton
// launches, mamba_ssm/ops/triton/ssd_combined.py:343-395, :397-516, and of its autograd functions, :596 and :822).
#include "torch_common.h"

#include <limits>

namespace mamba_ext {
namespace {

// The checks of _prepare (mamba_amd/ops/triton/ssd_combined.py; reference ssd_combined.py:344-369) for operands that
// need no conversion, and the forward fields of SsdParams; false = decline.
struct SsdDims {
  int64_t batch, L, H, P, G, N, Q, nchunks;
  bool lp;
};
bool fill_ssd(SsdParams &p, SsdDims &d, const at::Tensor &x, const at::Tensor &dt, const at::Tensor &A, const at::Tensor &B,
              const at::Tensor &C, int64_t chunk_size, const OptTensor &D, const OptTensor &z, const OptTensor &dt_bias,
              const OptTensor &initial_states, const OptTensor &seq_idx, bool dt_softplus, double dt_min, double dt_max) {
  const c10::Device dev = x.device();
  if (!on_device(x, dev) || !on_device(dt, dev) || !on_device(A, dev) || !on_device(B, dev) || !on_device(C, dev) ||
      !on_device(D, dev) || !on_device(z, dev) || !on_device(dt_bias, dev) || !on_device(initial_states, dev) ||
      !on_device(seq_idx, dev))
    return false;
  const int code = dtype_code(x), dtc = dtype_code(dt);
  if (code < 0 || dtc < 0 || x.dim() != 4 || B.dim() != 4 || C.dim() != 4 || dt.dim() != 3 || A.dim() != 1) return false;
  d.batch = x.size(0), d.L = x.size(1), d.H = x.size(2), d.P = x.size(3), d.G = B.size(2), d.N = B.size(3), d.Q = chunk_size;
  if (d.batch <= 0 || d.L <= 0 || d.H <= 0 || d.G <= 0 || d.H % d.G != 0 || d.Q <= 0 || d.Q > 256) return false;
  if (d.N > mamba_hip_query(MAMBA_Q_SSD_MAX_DSTATE) || d.P > mamba_hip_query(MAMBA_Q_SSD_MAX_HEADDIM)) return false;
  if (B.size(0) != d.batch || B.size(1) != d.L || C.sizes() != B.sizes()) return false;
  if (dt.size(0) != d.batch || dt.size(1) != d.L || dt.size(2) != d.H || A.size(0) != d.H) return false;
  if (B.scalar_type() != x.scalar_type() || C.scalar_type() != x.scalar_type()) return false;
  if (x.stride(3) != 1 || B.stride(3) != 1 || C.stride(3) != 1) return false;
  if (A.scalar_type() != at::kFloat || !A.is_contiguous()) return false;
  if (z && (z->sizes() != x.sizes() || z->scalar_type() != x.scalar_type() || z->stride(3) != 1)) return false;
  if (D && (D->scalar_type() != at::kFloat || !D->is_contiguous() ||
            !((D->dim() == 1 && D->size(0) == d.H) || (D->dim() == 2 && D->size(0) == d.H && D->size(1) == d.P))))
    return false;
  if (dt_bias && (dt_bias->scalar_type() != at::kFloat || dt_bias->dim() != 1 || dt_bias->size(0) != d.H ||
                  !dt_bias->is_contiguous()))
    return false;
  if (initial_states && (initial_states->scalar_type() != at::kFloat || !initial_states->is_contiguous() ||
                         initial_states->dim() != 4 || initial_states->size(0) != d.batch ||
                         initial_states->size(1) != d.H || initial_states->size(2) != d.P || initial_states->size(3) != d.N))
    return false;
  if (seq_idx && (seq_idx->scalar_type() != at::kInt || !seq_idx->is_contiguous() || seq_idx->dim() != 2 ||
                  seq_idx->size(0) != d.batch || seq_idx->size(1) != d.L))
    return false;
  d.nchunks = (d.L + d.Q - 1) / d.Q;
  d.lp = x.scalar_type() == at::kBFloat16;
  p.batch = (int32_t)d.batch, p.seqlen = (int32_t)d.L, p.nheads = (int32_t)d.H, p.headdim = (int32_t)d.P;
  p.dstate = (int32_t)d.N, p.ngroups = (int32_t)d.G, p.chunk_size = (int32_t)d.Q, p.nchunks = (int32_t)d.nchunks;
  p.dtype = code, p.dt_dtype = dtc, p.dt_softplus = dt_softplus ? 1 : 0, p.D_has_hdim = (D && D->dim() == 2) ? 1 : 0;
  p.dt_min = (float)dt_min, p.dt_max = (float)std::min(dt_max, 3.0e38);
  p.x = x.data_ptr(), p.dt = dt.data_ptr(), p.A = A.data_ptr(), p.B = B.data_ptr(), p.C = C.data_ptr();
  p.D = D ? D->data_ptr() : nullptr, p.z = z ? z->data_ptr() : nullptr, p.dt_bias = dt_bias ? dt_bias->data_ptr() : nullptr;
  p.initial_states = initial_states ? initial_states->data_ptr<float>() : nullptr;
  p.seq_idx = seq_idx ? seq_idx->data_ptr<int32_t>() : nullptr;
  p.x_bs = x.stride(0), p.x_ls = x.stride(1), p.x_hs = x.stride(2);
  if (z) p.z_bs = z->stride(0), p.z_ls = z->stride(1), p.z_hs = z->stride(2);
  p.B_bs = B.stride(0), p.B_ls = B.stride(1), p.B_gs = B.stride(2);
  p.C_bs = C.stride(0), p.C_ls = C.stride(1), p.C_gs = C.stride(2);
  p.dt_bs = dt.stride(0), p.dt_ls = dt.stride(1), p.dt_hs = dt.stride(2);
  return true;
}

// The chunk length the kernels use for a call that names one of 64, 128 and 256: the scan's result is the same for each
// but for rounding, and they differ in cost.  A longer chunk writes and reads fewer chunk states (headdim x dstate per
// head) and, at 256, has the paired scan kernel; a shorter one has less of the quadratic part, the (chunk x chunk) tiles of
// dCB per group above all, which a call without gradients does not have, and more workgroups.  The named chunk stays unless
// another one was faster in about every call of its class.  W: the workgroups a chunk of 256 gives, one per head.
// Measured (64 / 128 / 256, us, bf16, headdim 64, gated; forward | forward + backward; g: groups, n: states):
//   1 x 777 x 24       g1 n128  W 96     27.2 / 21.6 / 26.1  |  90 / 89 / 117      few workgroups: not 256
//   1 x 4096 x 48      g8 n64   W 768    58.1 / 44.8 / 43.5  |  208 / 180 / 194    64 states, 8 groups: 256 without gradients,
//   2 x 7093 x 40      g8 n64   W 2240   181 / 124 / 116     |  567 / 473 / 481      128 with them,
//   1 x 32768 x 64     g8 n64   W 8192   571 / 422 / 367     |  1954 / 1619 / 1524   until the states outweigh the tiles
//   1 x 1531 x 80      g1 n64   W 480    38.9 / 32.8 / 32.5  |  162 / 153 / 160    1 group: the tiles weigh less
//   4 x 4096 x 16      g1 n64   W 1024   72 / 56 / 52        |  299 / 262 / 267
//   2 x 7093 x 40      g1 n128  W 2240   274 / 190 / 142     |  748 / 581 / 515    128 states: the states weigh twice
//   1 x 4039 x 72      g8 n128  W 1152   128 / 90 / 96       |  374 / 294 / 352    4.5 rounds of 256 CUs: half of one idle
//   1 x 32768 x 64     g8 n128  W 8192   898 / 590 / 484     |  2558 / 1931 / 1666
// Over 279 sizes (1 - 4 x 130 - 32768 x 16 - 80 heads, 1 and 8 groups, 64 and 128 states, gated or not) a call without
// gradients that names 64 / 128 / 256 takes 0.81 / 0.96 / 0.97 of the named chunk's time in the mean and 1.12 / 1.14 / 1.12
// at worst (calls of 25 - 45 us), one with gradients 0.89 / 1.00 / 0.97 and 1.02 / 1.16 / 1.05.  The lines were drawn
// before the kernels of chunks of 64 and 128 became faster: with gradients a named 128 that goes to 256 is the slower one
// at 128 states without a gate (1 x 19504 x 40, 8 groups: 770 against 663 us).  Operands in two halves, and sizes that the
// fused kernels do not take: 128, or a named 64 in a short call (80 sizes: 0.93 / 1.00 / 0.92).
int64_t kernel_chunk(int64_t named, int64_t batch, int64_t L, int64_t H, int64_t G, int64_t P, int64_t N, at::ScalarType type,
                     bool backward) {
  if (named != 64 && named != 128 && named != 256) return named;
  if (L <= 128) return L <= 64 ? 64 : 128;  // one chunk
  const int64_t W = batch * H * ((L + 255) / 256), at_most_128 = std::min<int64_t>(named, 128), at_least_128 = std::max<int64_t>(named, 128);
  const bool fused = (P == 32 || P == 64) && (N == 64 || N == 128);
  if (type != at::kBFloat16 || (!fused && N < 128)) {
    if (N >= 128 && G == 1 && W >= 8192) return at_least_128;
    return W < 384 ? at_most_128 : 128;
  }
  if (!backward) {
    if (W < 160) return W < 96 ? at_most_128 : 128;
    const int64_t W128 = batch * H * ((L + 127) / 128);
    if (W < 384 && (N < 128 || W128 * 5 < W * 9)) return 128;  // (with 128 states: much of the last chunk empty)
    return N >= 128 || W >= 768 ? 256 : at_least_128;
  }
  if (W < 384) return W < 256 ? at_most_128 : 128;
  const bool idle = W >= 768 && W < 2048 && (W + 255) / 256 * 256 * 10 >= W * 11;  // a tenth of 3 to 8 rounds
  if (N >= 128) return W >= (G == 1 ? 768 : 2048) ? 256 : idle ? 128 : at_least_128;
  return idle || W < (G == 1 ? 768 : 4096) ? 128 : at_least_128;
}

// Everything a forward or backward call of mamba_chunk_scan_combined takes, apart from its outputs.
struct SsdArgs {
  at::Tensor x, dt, A, B, C;
  int64_t chunk_size;
  OptTensor D, z, dt_bias, initial_states, seq_idx;
  bool dt_softplus;
  double dt_min, dt_max;
};
bool fill_ssd(SsdParams &p, SsdDims &d, const SsdArgs &a) {
  return fill_ssd(p, d, a.x, a.dt, a.A, a.B, a.C, a.chunk_size, a.D, a.z, a.dt_bias, a.initial_states, a.seq_idx, a.dt_softplus,
                  a.dt_min, a.dt_max);
}

// _mamba_chunk_scan_combined_fwd (ssd_combined.py:343) without cu_seqlens
// -> [out, out_x, dt_out, dA_cumsum, carried states, final_states]
TensorList ssd_fwd(SsdParams &p, const SsdDims &d, const SsdArgs &a, bool want_out_x) {
  const at::Tensor &x = a.x;
  const c10::Device dev = x.device();
  c10::DeviceGuard guard(dev);
  const auto f32 = x.options().dtype(at::kFloat);
  at::Tensor dt_out = at::empty({d.batch, d.H, d.nchunks, d.Q}, f32), dA_cumsum = at::empty({d.batch, d.H, d.nchunks, d.Q}, f32);
  at::Tensor states = at::empty({d.batch, d.nchunks, d.H, d.P, d.N}, f32);
  OptTensor states_lp;
  if (d.lp) states_lp = at::empty({d.batch, d.nchunks, d.H, d.P, d.N}, x.options());
  at::Tensor final_states = at::empty({d.batch, d.H, d.P, d.N}, f32);
  at::Tensor CB = at::empty({d.batch, d.nchunks, d.G, d.Q, d.Q}, f32);
  at::Tensor out = at::empty(x.sizes(), x.options());
  OptTensor out_x;
  if (a.z && want_out_x) out_x = at::empty(x.sizes(), x.options());
  p.dt_out = dt_out.data_ptr<float>(), p.dA_cumsum = dA_cumsum.data_ptr<float>(), p.states = states.data_ptr<float>();
  p.final_states = final_states.data_ptr<float>(), p.CB = CB.data_ptr<float>();
  p.states_lp = ptr(states_lp);
  p.out = out.data_ptr(), p.out_x = ptr(out_x);
  p.out_bs = out.stride(0), p.out_ls = out.stride(1), p.out_hs = out.stride(2);
  check_rc(ssd_combined_fwd(&p, stream_of(dev)), "ssd_combined_fwd");
  TensorList r(6);
  r[0] = out, r[1] = out_x, r[2] = dt_out, r[3] = dA_cumsum, r[4] = d.lp ? *states_lp : states, r[5] = final_states;
  return r;
}

// Where the caller wants gradients written (slices of wider buffers); allocated by the call when absent.
struct SsdGradOut {
  OptTensor dx, ddt, dB, dC;
};

// _mamba_chunk_scan_combined_bwd (ssd_combined.py:397) with the forward pass's dt_out / dA_cumsum / carried states
// kept, float atomics -> [dx, ddt, dA, dB, dC, dD, dz, ddt_bias, dinitial_states]
TensorList ssd_bwd(SsdParams &p, const SsdDims &d, const SsdArgs &a, const at::Tensor &dout, const at::Tensor &out,
                   const OptTensor &dfinal_states, const at::Tensor &dt_out, const at::Tensor &dA_cumsum,
                   const at::Tensor &carried, const SsdGradOut &to) {
  const at::Tensor &x = a.x;
  const c10::Device dev = x.device();
  c10::DeviceGuard guard(dev);
  const auto f32 = x.options().dtype(at::kFloat);
  at::Tensor dx = to.dx ? *to.dx : at::empty(x.sizes(), x.options());
  OptTensor dz, gbuf, dinit;
  if (a.z) dz = at::empty(x.sizes(), x.options()), gbuf = at::empty(x.sizes(), x.options());
  at::Tensor ddt = to.ddt ? *to.ddt : at::empty({d.batch, d.L, d.H}, a.dt.options());
  // one zeroed arena for the small accumulators the kernels add into; the three large ones (dCB, dB32, dC32) are
  // cleared below, and only where the library does not write them whole (ssd_bwd_overwrites)
  const int64_t nD = a.D ? a.D->numel() : 0, nHcQ = d.batch * d.H * d.nchunks * d.Q;
  const int64_t nCB = d.batch * d.nchunks * d.G * d.Q * d.Q, nBC = d.batch * d.L * d.G * d.N;
  const int64_t sizes[8] = {d.H, d.H, nD, nHcQ, nHcQ, nCB, nBC, nBC};  // the five small ones first
  int64_t total = 0, off[8];
  for (int i = 0; i < 8; ++i) {
    if (i >= 5) total = (total + 63) / 64 * 64;  // the large ones start on 256 bytes
    off[i] = total, total += sizes[i];
  }
  total = (total + 63) / 64 * 64;
  at::Tensor arena = at::empty({total}, f32);
  float *base = arena.data_ptr<float>();
  at::Tensor dstates = at::empty({d.batch, d.nchunks, d.H, d.P, d.N}, d.lp ? x.options() : f32);
  if (a.initial_states) dinit = at::empty({d.batch, d.H, d.P, d.N}, f32);
  p.dt_out = dt_out.data_ptr<float>(), p.dA_cumsum = dA_cumsum.data_ptr<float>();
  if (d.lp) p.states_lp = carried.data_ptr(); else p.states = carried.data_ptr<float>();
  if (a.z) p.out_x = out.data_ptr(); else p.out = out.data_ptr();
  p.out_bs = out.stride(0), p.out_ls = out.stride(1), p.out_hs = out.stride(2);
  p.dout = dout.data_ptr(), p.dfinal_states = dfinal_states ? dfinal_states->data_ptr<float>() : nullptr;
  p.dout_bs = dout.stride(0), p.dout_ls = dout.stride(1), p.dout_hs = dout.stride(2);
  p.dx = dx.data_ptr(), p.dz = ptr(dz), p.ddt = ddt.data_ptr(), p.gbuf = ptr(gbuf);
  p.dx_bs = dx.stride(0), p.dx_ls = dx.stride(1), p.dx_hs = dx.stride(2);
  p.ddt_bs = ddt.stride(0), p.ddt_ls = ddt.stride(1), p.ddt_hs = ddt.stride(2);
  p.dA = base + off[0], p.ddt_bias = base + off[1], p.dD = a.D ? base + off[2] : nullptr;
  p.ddA_cumsum = base + off[3], p.ddt_out = base + off[4];
  p.dCB = base + off[5], p.dB32 = base + off[6], p.dC32 = base + off[7];
  p.dinitial_states = dinit ? dinit->data_ptr<float>() : nullptr;
  if (d.lp) p.dstates_lp = dstates.data_ptr(); else p.dstates = dstates.data_ptr<float>();
  // dB / dC in the operands' dtype: written by the call's last stage
  at::Tensor dB = to.dB ? *to.dB : at::empty({d.batch, d.L, d.G, d.N}, a.B.options());
  at::Tensor dC = to.dC ? *to.dC : at::empty({d.batch, d.L, d.G, d.N}, a.C.options());
  p.dB = dB.data_ptr(), p.dC = dC.data_ptr();
  p.dB_bs = dB.stride(0), p.dB_ls = dB.stride(1), p.dB_gs = dB.stride(2);
  p.dC_bs = dC.stride(0), p.dC_ls = dC.stride(1), p.dC_gs = dC.stride(2);
  const int owned = ssd_bwd_overwrites(&p);
  void *stream = stream_of(dev);
  {
    int64_t at[3] = {0}, n[3] = {off[5]};
    int count = 1;
    if (!(owned & SSD_OVERWRITES_DCB)) at[count] = off[5], n[count++] = off[6] - off[5];
    if (!(owned & SSD_OVERWRITES_DBC)) at[count] = off[6], n[count++] = total - off[6];
    check_rc(ssd_clear(base, at, n, count, stream), "ssd_clear");
  }
  // CB: the fused forward never forms it; the backward kernels may not need it either
  at::Tensor CB;
  if (!(owned & SSD_BWD_FORMS_CB)) {
    CB = at::empty({d.batch, d.nchunks, d.G, d.Q, d.Q}, f32);
    p.CB = CB.data_ptr<float>();
    check_rc(ssd_bmm_chunk_fwd(&p, stream), "ssd_bmm_chunk_fwd");
  }
  check_rc(ssd_combined_bwd(&p, stream), "ssd_combined_bwd");
  TensorList r(9);
  r[0] = dx, r[1] = ddt, r[2] = arena.as_strided({d.H}, {1}, off[0]);
  r[3] = dB, r[4] = dC;
  if (a.D) r[5] = a.D->dim() == 2 ? arena.as_strided({d.H, d.P}, {d.P, 1}, off[2]) : arena.as_strided({d.H}, {1}, off[2]);
  r[6] = dz;
  if (a.dt_bias) r[7] = arena.as_strided({d.H}, {1}, off[1]);
  r[8] = dinit;
  return r;
}

// The same in the deterministic mode, whose integer sums the Python host side sets up.
TensorList ssd_bwd_deterministic(const SsdArgs &a, const at::Tensor &dout, const at::Tensor &out, const OptTensor &dfinal_states,
                                 const at::Tensor &dt_out, const at::Tensor &dA_cumsum, const at::Tensor &carried,
                                 const SsdGradOut &to) {
  namespace py = pybind11;
  using namespace py::literals;
  py::gil_scoped_acquire gil;
  at::AutoGradMode no_grad(false);
  const py::object f = py::module_::import("mamba_amd.ops.triton.ssd_combined").attr("_mamba_chunk_scan_combined_bwd");
  const py::object r = f(dout, a.x, a.dt, a.A, a.B, a.C, out, a.chunk_size, "D"_a = a.D, "z"_a = a.z, "dt_bias"_a = a.dt_bias,
                         "initial_states"_a = a.initial_states, "dfinal_states"_a = dfinal_states, "seq_idx"_a = a.seq_idx,
                         "dt_softplus"_a = a.dt_softplus, "dt_limit"_a = py::make_tuple(a.dt_min, a.dt_max),
                         "saved"_a = py::make_tuple(dt_out, dA_cumsum, carried), "dx"_a = to.dx, "ddt"_a = to.ddt,
                         "dB"_a = to.dB, "dC"_a = to.dC);
  return r.cast<TensorList>();
}

TensorList ssd_bwd_any(const SsdArgs &a, const at::Tensor &dout, const at::Tensor &out, const OptTensor &dfinal_states,
                       const at::Tensor &dt_out, const at::Tensor &dA_cumsum, const at::Tensor &carried, const SsdGradOut &to) {
  if (deterministic()) return ssd_bwd_deterministic(a, dout, out, dfinal_states, dt_out, dA_cumsum, carried, to);
  SsdParams p{};
  SsdDims d;
  TORCH_CHECK(fill_ssd(p, d, a), "mamba_chunk_scan_combined: arguments");
  return ssd_bwd(p, d, a, dout, out, dfinal_states, dt_out, dA_cumsum, carried, to);
}

std::optional<TensorList> ssd_fwd_fast(const at::Tensor &x, const at::Tensor &dt, const at::Tensor &A, const at::Tensor &B,
                                       const at::Tensor &C, int64_t chunk_size, const OptTensor &D, const OptTensor &z,
                                       const OptTensor &dt_bias, const OptTensor &initial_states, const OptTensor &seq_idx,
                                       bool dt_softplus, double dt_min, double dt_max, bool want_out_x) {
  SsdParams p{};
  SsdDims d;
  const SsdArgs a{x, dt, A, B, C, chunk_size, D, z, dt_bias, initial_states, seq_idx, dt_softplus, dt_min, dt_max};
  if (!fill_ssd(p, d, a)) return std::nullopt;
  return ssd_fwd(p, d, a, want_out_x);
}

std::optional<TensorList> ssd_bwd_fast(const at::Tensor &dout, const at::Tensor &x, const at::Tensor &dt, const at::Tensor &A,
                                       const at::Tensor &B, const at::Tensor &C, const at::Tensor &out, int64_t chunk_size,
                                       const OptTensor &D, const OptTensor &z, const OptTensor &dt_bias,
                                       const OptTensor &initial_states, const OptTensor &dfinal_states,
                                       const OptTensor &seq_idx, bool dt_softplus, double dt_min, double dt_max,
                                       const at::Tensor &dt_out, const at::Tensor &dA_cumsum, const at::Tensor &carried) {
  SsdParams p{};
  SsdDims d;
  const SsdArgs a{x, dt, A, B, C, chunk_size, D, z, dt_bias, initial_states, seq_idx, dt_softplus, dt_min, dt_max};
  if (!fill_ssd(p, d, a)) return std::nullopt;
  const c10::Device dev = x.device();
  if (!on_device(dout, dev) || !on_device(out, dev) || !on_device(dfinal_states, dev) || !on_device(dt_out, dev) ||
      !on_device(dA_cumsum, dev) || !on_device(carried, dev))
    return std::nullopt;
  auto like_x = [&](const at::Tensor &t) { return t.sizes() == x.sizes() && t.scalar_type() == x.scalar_type() && t.stride(3) == 1; };
  if (!like_x(dout) || !like_x(out)) return std::nullopt;
  const std::vector<int64_t> cs = {d.batch, d.H, d.nchunks, d.Q}, ss = {d.batch, d.nchunks, d.H, d.P, d.N};
  auto f32c = [](const at::Tensor &t, const std::vector<int64_t> &shape) {
    return t.scalar_type() == at::kFloat && t.is_contiguous() && t.sizes().vec() == shape;
  };
  if (!f32c(dt_out, cs) || !f32c(dA_cumsum, cs)) return std::nullopt;
  if (carried.sizes().vec() != ss || !carried.is_contiguous() ||
      carried.scalar_type() != (d.lp ? at::kBFloat16 : at::kFloat))
    return std::nullopt;
  if (dfinal_states && (!f32c(*dfinal_states, {d.batch, d.H, d.P, d.N}))) return std::nullopt;
  return ssd_bwd(p, d, a, dout, out, dfinal_states, dt_out, dA_cumsum, carried, {});
}

// ------------------------------------------------------------------ mamba_chunk_scan_combined
constexpr int SSD_NARGS = 11;  // the node's forward arguments

struct SsdOptions {
  int64_t chunk_size;
  bool dt_softplus, return_final;
  double dt_min, dt_max;
};

SsdArgs ssd_args(const variable_list &s, const SsdOptions &o) {  // from the saved tensors below
  return {s[1], s[2], s[4], s[5], s[6], o.chunk_size, opt(s[7]), opt(s[8]), opt(s[9]), opt(s[10]), opt(s[11]), o.dt_softplus, o.dt_min, o.dt_max};
}
void save_options(AutogradContext *ctx, const SsdOptions &o) {
  ctx->saved_data["o"] = std::vector<int64_t>{o.chunk_size, o.dt_softplus, o.return_final};
  ctx->saved_data["limit"] = std::vector<double>{o.dt_min, o.dt_max};
}
SsdOptions saved_options(AutogradContext *ctx) {
  const std::vector<int64_t> v = ctx->saved_data["o"].toIntVector();
  const std::vector<double> l = ctx->saved_data["limit"].toDoubleVector();
  return {v[0], v[1] != 0, v[2] != 0, l[0], l[1]};
}
at::Tensor unit_last(const at::Tensor &t) { return t.stride(-1) == 1 ? t : t.contiguous(); }

struct SsdFn : torch::autograd::Function<SsdFn> {
  static variable_list forward(AutogradContext *ctx, const at::Tensor &x, const at::Tensor &dt, const at::Tensor &A,
                               const at::Tensor &B, const at::Tensor &C, const OptTensor &D, const OptTensor &z,
                               const OptTensor &dt_bias, const OptTensor &initial_states, const OptTensor &seq_idx,
                               const SsdOptions &o) {
    const SsdArgs a{x, dt, A, B, C, o.chunk_size, D, z, dt_bias, initial_states, seq_idx, o.dt_softplus, o.dt_min, o.dt_max};
    SsdParams p{};
    SsdDims d;
    TORCH_CHECK(fill_ssd(p, d, a), "mamba_chunk_scan_combined: arguments");
    const TensorList r = ssd_fwd(p, d, a, true);
    // the fp32 dt, cumulative decay and chunk states of the forward pass stay alive for the backward pass instead of
    // being re-computed there as in the reference (ssd_combined.py:441-448)
    ctx->save_for_backward({z ? *r[1] : *r[0], x, dt, *r[3], A, B, C, tensor_or_none(D), tensor_or_none(z), tensor_or_none(dt_bias),
                            tensor_or_none(initial_states), tensor_or_none(seq_idx), *r[2], *r[4]});
    ctx->set_materialize_grads(false);
    save_options(ctx, o);
    variable_list out = {*r[0]};
    if (o.return_final) out.push_back(*r[5]);
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const SsdOptions o = saved_options(ctx);
    c10::DeviceGuard guard(s[1].device());
    at::Tensor dout = grads[0].defined() ? unit_last(grads[0]) : at::zeros(s[1].sizes(), s[1].options());
    if (dout.scalar_type() != s[1].scalar_type()) dout = dout.to(s[1].scalar_type());
    OptTensor dfinal;
    if (o.return_final && grads[1].defined()) dfinal = grads[1].to(at::kFloat).contiguous();
    const TensorList r = ssd_bwd_any(ssd_args(s, o), dout, s[0], dfinal, s[12], s[3], s[13], {});
    variable_list g(SSD_NARGS);
    g[0] = *r[0], g[1] = *r[1], g[2] = *r[2], g[3] = *r[3], g[4] = *r[4];
    g[5] = tensor_or_none(r[5]), g[6] = tensor_or_none(r[6]), g[7] = tensor_or_none(r[7]), g[8] = tensor_or_none(r[8]);
    return g;
  }
};

// mamba_chunk_scan_combined without varlen states: out, or (out, final_states); None = declined
pybind11::object chunk_scan(const at::Tensor &x, const at::Tensor &dt, const at::Tensor &A, const at::Tensor &B, const at::Tensor &C,
                            int64_t chunk_size, const OptTensor &D, const OptTensor &z, const OptTensor &dt_bias,
                            const OptTensor &initial_states, const OptTensor &seq_idx, bool dt_softplus, double dt_min,
                            double dt_max, bool return_final) {
  if (python_call(x, dt, A, B, C, D, z, dt_bias, initial_states)) return pybind11::none();
  const bool backward = records(x, dt, A, B, C, D, z, dt_bias, initial_states);
  if (x.dim() == 4 && B.dim() == 4)
    chunk_size = kernel_chunk(chunk_size, x.size(0), x.size(1), x.size(2), B.size(2), x.size(3), B.size(3), x.scalar_type(), backward);
  SsdParams p{};
  SsdDims d;
  const SsdArgs a{x, dt, A, B, C, chunk_size, D, z, dt_bias, initial_states, seq_idx, dt_softplus, dt_min, dt_max};
  if (!fill_ssd(p, d, a)) return pybind11::none();
  if (!backward) {
    const TensorList r = ssd_fwd(p, d, a, false);  // no gradient asked for: the pre-gate copy is not written
    return return_final ? pybind11::object(pybind11::make_tuple(*r[0], *r[5])) : pybind11::cast(*r[0]);
  }
  const SsdOptions o{chunk_size, dt_softplus, return_final, dt_min, dt_max};
  variable_list r = SsdFn::apply(x, dt, A, B, C, D, z, dt_bias, initial_states, seq_idx, o);
  return return_final ? pybind11::object(pybind11::make_tuple(r[0], r[1])) : pybind11::cast(r[0]);
}

// ------------------------------------------------------------------ mamba_split_conv1d_scan_combined
// The Mamba-2 block body as one node (ssd_combined.py:822) for d_nonssm = 0: the backward pass writes the gradients of
// z, xBC and dt straight into their slices of one dzxbcdt buffer, and the scan's dx, dB and dC into the slices of the
// buffer the convolution's backward pass reads.
struct BlockOptions {
  SsdOptions ssd;
  int64_t headdim, ngroups;
  double eps;
  bool silu, norm_before_gate;
};
constexpr int BLOCK_NARGS = 13;

// Slices of a (batch, seqlen, ...) tensor with unit last stride, from channel `at` on: as rows per (batch, position)
// (which follow one another, see split_conv_scan), as heads (batch, seqlen, n0, n1), as rows of a convolution
at::Tensor row_slice(const at::Tensor &t, int64_t at, int64_t n) {
  return t.as_strided({t.size(0) * t.size(1), n}, {t.stride(1), 1}, t.storage_offset() + at);
}
at::Tensor head_slice(const at::Tensor &t, int64_t at, int64_t n0, int64_t n1) {
  return t.as_strided({t.size(0), t.size(1), n0, n1}, {t.stride(0), t.stride(1), n1, 1}, t.storage_offset() + at);
}
at::Tensor step_slice(const at::Tensor &t, int64_t at, int64_t n) {
  return t.as_strided({t.size(0), t.size(1), n}, {t.stride(0), t.stride(1), 1}, t.storage_offset() + at);
}
ConvRows conv_rows(const at::Tensor &t, int64_t at) {
  return {static_cast<char *>(t.data_ptr()) + at * t.element_size(), t.stride(0), 1, t.stride(1)};
}

SsdArgs args_of(const at::Tensor &zxbcdt, const at::Tensor &xBC, const at::Tensor &A, const at::Tensor &D, bool gate,
                const at::Tensor &dt_bias, const OptTensor &initial_states, const OptTensor &seq_idx, int64_t H, int64_t P, int64_t G,
                int64_t N, const SsdOptions &o) {
  const int64_t dim = H * P;
  return {head_slice(xBC, 0, H, P), step_slice(zxbcdt, dim + xBC.size(2), H), A, head_slice(xBC, dim, G, N), head_slice(xBC, dim + G * N, G, N),
          o.chunk_size, D, gate ? OptTensor(head_slice(zxbcdt, 0, H, P)) : std::nullopt, dt_bias, initial_states, seq_idx, true, o.dt_min,
          o.dt_max};
}

struct BlockFn : torch::autograd::Function<BlockFn> {
  static variable_list forward(AutogradContext *ctx, const at::Tensor &zxbcdt, const at::Tensor &conv_weight, const OptTensor &conv_bias,
                               const at::Tensor &dt_bias, const at::Tensor &A, const at::Tensor &D, const OptTensor &initial_states,
                               const OptTensor &seq_idx, const OptTensor &norm_weight, const OptTensor &out_weight,
                               const OptTensor &out_bias, const BlockOptions &o, std::optional<at::ScalarType> autocast) {
    const int64_t H = D.size(0), P = o.headdim, G = o.ngroups, dim = H * P, batch = zxbcdt.size(0), L = zxbcdt.size(1);
    const at::Tensor &conv_w = conv_weight;
    const int64_t conv = conv_w.size(0), N = (conv - dim) / (2 * G);
    at::Tensor xBC = at::empty({batch, L, conv}, zxbcdt.options());
    conv_fwd(zxbcdt, batch, conv, L, conv_rows(zxbcdt, dim), conv_w, conv_bias, seq_idx, o.silu, conv_rows(xBC, 0));
    const bool gate_in_scan = !norm_weight;
    const SsdArgs a = args_of(zxbcdt, xBC, A, D, gate_in_scan, dt_bias, initial_states, seq_idx, H, P, G, N, o.ssd);
    SsdParams p{};
    SsdDims d;
    TORCH_CHECK(fill_ssd(p, d, a), "mamba_split_conv1d_scan_combined: arguments");
    const TensorList r = ssd_fwd(p, d, a, true);
    at::Tensor y = r[0]->view({batch * L, dim});
    OptTensor rstd;
    if (norm_weight) {
      // reads z where it lies inside zxbcdt (unit channel stride, row stride of the whole projection)
      auto [yn, mean, rs] = gated_norm_fwd(y, *norm_weight, std::nullopt, row_slice(zxbcdt, 0, dim), {dim / G, o.eps, o.norm_before_gate, true});
      y = yn, rstd = rs;
    }
    at::Tensor res, w;
    if (out_weight) {
      w = *out_weight;
      OptTensor bias = out_bias;
      if (autocast) {
        y = y.to(*autocast), w = w.to(*autocast);
        if (bias) bias = bias->to(*autocast);
      }
      y = y.contiguous(), w = w.contiguous();
      if (bias) bias = bias->contiguous();
      res = at::empty({batch, L, w.size(0)}, y.options());  // as it is returned: a view made here could not be written in place
      Products(y.options(), y.scalar_type())
          .add(res.data_ptr(), y.scalar_type(), w.size(0), batch * L, w.size(0), dim, {y.data_ptr(), dim, 1}, {w.data_ptr(), dim, 1}, false,
               bias ? bias->data_ptr() : nullptr)
          .run();
    }
    ctx->save_for_backward({zxbcdt, conv_w, tensor_or_none(conv_bias), xBC, gate_in_scan ? *r[1] : *r[0], *r[2], *r[3], *r[4], A, D,
                            dt_bias, tensor_or_none(initial_states), tensor_or_none(seq_idx), tensor_or_none(norm_weight),
                            tensor_or_none(rstd), w, out_weight ? y : at::Tensor()});
    ctx->set_materialize_grads(false);
    save_options(ctx, o.ssd);
    ctx->saved_data["b"] = std::vector<int64_t>{P, G, o.silu, o.norm_before_gate, 0, out_bias.has_value(), out_weight ? (int64_t)out_weight->scalar_type() : 0,
                                                out_bias ? (int64_t)out_bias->scalar_type() : 0};
    ctx->saved_data["eps"] = o.eps;
    variable_list out = {out_weight ? res : y.view({batch, L, dim})};
    if (o.ssd.return_final) out.push_back(*r[5]);
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const SsdOptions so = saved_options(ctx);
    const std::vector<int64_t> v = ctx->saved_data["b"].toIntVector();
    const at::Tensor &zxbcdt = s[0], &conv_w = s[1], &xBC = s[3], &scan_out = s[4], &D = s[9], &w = s[15], &y = s[16];
    const OptTensor conv_bias = opt(s[2]), norm_weight = opt(s[13]);
    const int64_t H = D.size(0), P = v[0], G = v[1], dim = H * P, batch = zxbcdt.size(0), L = zxbcdt.size(1), conv = conv_w.size(0);
    const int64_t N = (conv - dim) / (2 * G);
    c10::DeviceGuard guard(zxbcdt.device());
    at::Tensor dzxbcdt = at::empty(zxbcdt.sizes(), zxbcdt.options());
    variable_list g(BLOCK_NARGS);
    at::Tensor dy;
    if (w.defined()) {
      at::Tensor dout = grads[0].defined() ? grads[0].reshape({batch * L, -1}) : at::zeros({batch * L, w.size(0)}, w.options());
      dout = dout.to(w.scalar_type()).contiguous();
      const int64_t E = w.size(0);
      const at::ScalarType ty = w.scalar_type(), wt = (at::ScalarType)v[6];
      dy = at::empty({batch * L, dim}, w.options());
      at::Tensor dw = at::empty({E, dim}, w.options().dtype(wt == at::kFloat ? wt : ty));
      Products(w.options(), ty)
          .add(dy.data_ptr(), ty, dim, batch * L, dim, E, {dout.data_ptr(), E, 1}, {w.data_ptr(), 1, dim})
          .add(dw.data_ptr(), dw.scalar_type(), dim, E, dim, batch * L, {dout.data_ptr(), 1, E}, {y.data_ptr(), 1, dim})
          .run();
      g[9] = dw.to(wt);
      if (v[5]) g[10] = dout.sum(0).to((at::ScalarType)v[7]);
    } else {
      dy = grads[0].defined() ? unit_last(grads[0].reshape({batch * L, dim})) : at::zeros({batch * L, dim}, zxbcdt.options());
    }
    if (dy.scalar_type() != zxbcdt.scalar_type()) dy = dy.to(zxbcdt.scalar_type());
    if (norm_weight) {
      const GatedNorm o{dim / G, ctx->saved_data["eps"].toDouble(), v[3] != 0, true};
      auto [dx, dw, db, dz] = gated_norm_bwd(dy, scan_out.view({batch * L, dim}), *norm_weight, std::nullopt, std::nullopt, s[14],
                                             row_slice(zxbcdt, 0, dim), row_slice(dzxbcdt, 0, dim), o);
      dy = dx;
      g[8] = dw;
    }
    at::Tensor dxBC = at::empty(xBC.sizes(), xBC.options());
    const SsdArgs a = args_of(zxbcdt, xBC, s[8], D, !norm_weight, s[10], opt(s[11]), opt(s[12]), H, P, G, N, so);
    OptTensor dfinal;
    if (so.return_final && grads[1].defined()) dfinal = grads[1].to(at::kFloat).contiguous();
    const TensorList r = ssd_bwd_any(a, dy.view({batch, L, H, P}), scan_out, dfinal, s[5], s[6], s[7],
                                     {head_slice(dxBC, 0, H, P), step_slice(dzxbcdt, dim + conv, H), head_slice(dxBC, dim, G, N),
                                      head_slice(dxBC, dim + G * N, G, N)});
    if (!norm_weight) row_slice(dzxbcdt, 0, dim).copy_(r[6]->view({batch * L, dim}));
    // the convolution's backward kernel re-computes its pre-activation from xBC and writes into the xBC slice
    auto [dcw, dcb] = conv_bwd(zxbcdt, batch, conv, L, conv_rows(zxbcdt, dim), conv_w, conv_bias, conv_rows(dxBC, 0), opt(s[12]), v[2] != 0,
                               conv_rows(dzxbcdt, dim));
    g[0] = dzxbcdt, g[1] = dcw, g[2] = tensor_or_none(dcb), g[3] = *r[7], g[4] = *r[2], g[5] = *r[5];
    g[6] = tensor_or_none(r[8]);
    return g;
  }
};

// mamba_split_conv1d_scan_combined with d_nonssm = 0: out, or (out, final_states); None = declined
pybind11::object split_conv_scan(const at::Tensor &zxbcdt_in, const at::Tensor &conv_weight, const OptTensor &conv_bias,
                                 const at::Tensor &dt_bias, const at::Tensor &A, const at::Tensor &D, int64_t chunk_size,
                                 const OptTensor &initial_states, const OptTensor &seq_idx, double dt_min, double dt_max,
                                 bool return_final, bool silu, const OptTensor &norm_weight, double eps, const OptTensor &out_weight,
                                 const OptTensor &out_bias, std::optional<int64_t> headdim_in, int64_t G, bool norm_before_gate) {
  const pybind11::object no = pybind11::none();
  if (!zxbcdt_in.is_cuda() || zxbcdt_in.dim() != 3 || G <= 0 || (D.dim() != 1 && D.dim() != 2) || conv_weight.dim() < 2 ||
      (conv_weight.dim() == 3 && conv_weight.size(1) != 1) || conv_weight.dim() > 3)
    return no;
  if (python_call(zxbcdt_in, conv_weight, conv_bias, dt_bias, A, D, initial_states, norm_weight, out_weight, out_bias)) return no;
  if (D.dim() == 1 && !headdim_in) return no;
  // rows of (batch, seqlen) must follow one another: the norm walks them as one (rows, channels) matrix
  const bool rows = zxbcdt_in.stride(2) == 1 && (zxbcdt_in.size(0) == 1 || zxbcdt_in.stride(0) == zxbcdt_in.size(1) * zxbcdt_in.stride(1));
  const at::Tensor zxbcdt = rows ? zxbcdt_in : zxbcdt_in.contiguous();
  const c10::Device dev = zxbcdt.device();
  const int64_t H = D.size(0), P = D.dim() == 2 ? D.size(1) : *headdim_in, dim = H * P, conv = conv_weight.size(0);
  const int64_t batch = zxbcdt.size(0), L = zxbcdt.size(1);
  if (H <= 0 || P <= 0 || H % G != 0 || conv <= dim || (conv - dim) % (2 * G) != 0 || batch <= 0 || L <= 0) return no;
  const int64_t N = (conv - dim) / (2 * G);
  if (zxbcdt.size(2) != dim + conv + H || dt_bias.dim() != 1 || dt_bias.size(0) != H || A.dim() != 1 || A.size(0) != H) return no;
  chunk_size = kernel_chunk(chunk_size, batch, L, H, G, P, N, zxbcdt.scalar_type(),
                            records(zxbcdt, conv_weight, conv_bias, dt_bias, A, D, initial_states, norm_weight, out_weight, out_bias));
  const at::Tensor conv_w = conv_weight.dim() == 3 ? conv_weight.squeeze(1) : conv_weight;
  const at::Tensor xBC_in = zxbcdt.as_strided({batch, conv, L}, {zxbcdt.stride(0), 1, zxbcdt.stride(1)}, zxbcdt.storage_offset() + dim);
  if (!conv_params_ok(xBC_in, conv_w, conv_bias, seq_idx)) return no;
  // the scan's own checks, on operands of the right shapes and dtypes (x, B and C will be slices of a fresh buffer)
  SsdParams p{};
  SsdDims d;
  const SsdOptions so{chunk_size, true, return_final, dt_min, dt_max};
  SsdArgs a{head_slice(zxbcdt, dim, H, P), step_slice(zxbcdt, dim + conv, H), A, head_slice(zxbcdt, 2 * dim, G, N),
            head_slice(zxbcdt, 2 * dim + G * N, G, N), chunk_size, D, std::nullopt, dt_bias, initial_states, seq_idx, true, dt_min, dt_max};
  if (!norm_weight) a.z = head_slice(zxbcdt, 0, H, P);
  if (!fill_ssd(p, d, a)) return no;
  if (norm_weight &&
      !gated_norm_ok(row_slice(zxbcdt, 0, dim), *norm_weight, std::nullopt, std::nullopt, {dim / G, eps, norm_before_gate, true}))
    return no;
  std::optional<at::ScalarType> autocast;
  if (at::autocast::is_autocast_enabled(at::kCUDA)) autocast = at::autocast::get_autocast_dtype(at::kCUDA);
  if (out_weight) {
    const at::ScalarType want = autocast ? *autocast : zxbcdt.scalar_type();
    auto ok = [&](const at::Tensor &t) { return on_device(t, dev) && (t.scalar_type() == want || (autocast && t.is_floating_point())); };
    if (out_weight->dim() != 2 || out_weight->size(0) == 0 || out_weight->size(1) != dim || !ok(*out_weight)) return no;
    // (a bias that F.linear broadcasts or refuses is left to it)
    if (out_bias && (!ok(*out_bias) || out_bias->dim() != 1 || out_bias->size(0) != out_weight->size(0))) return no;
  } else if (out_bias) {
    return no;
  }
  c10::DeviceGuard guard(dev);
  const BlockOptions o{so, P, G, eps, silu, norm_before_gate};
  variable_list r = BlockFn::apply(zxbcdt, conv_weight, conv_bias, dt_bias, A, D, initial_states, seq_idx, norm_weight, out_weight,
                                   out_bias, o, autocast);
  return return_final ? pybind11::object(pybind11::make_tuple(r[0], r[1])) : pybind11::cast(r[0]);
}

}  // namespace

void bind_ssd(pybind11::module_ &m) {
  namespace py = pybind11;
  m.def("ssd_fwd", &ssd_fwd_fast, py::arg("x"), py::arg("dt"), py::arg("A"), py::arg("B"), py::arg("C"), py::arg("chunk_size"),
        py::arg("D"), py::arg("z"), py::arg("dt_bias"), py::arg("initial_states"), py::arg("seq_idx"), py::arg("dt_softplus"),
        py::arg("dt_min"), py::arg("dt_max"), py::arg("want_out_x"),
        "Forward of mamba_chunk_scan_combined: [out, out_x, dt_out, dA_cumsum, carried states, final_states], or None.");
  m.def("ssd_bwd", &ssd_bwd_fast, py::arg("dout"), py::arg("x"), py::arg("dt"), py::arg("A"), py::arg("B"), py::arg("C"),
        py::arg("out"), py::arg("chunk_size"), py::arg("D"), py::arg("z"), py::arg("dt_bias"), py::arg("initial_states"),
        py::arg("dfinal_states"), py::arg("seq_idx"), py::arg("dt_softplus"), py::arg("dt_min"), py::arg("dt_max"),
        py::arg("dt_out"), py::arg("dA_cumsum"), py::arg("carried"),
        "Backward of mamba_chunk_scan_combined with the forward pass's workspaces kept: [dx, ddt, dA, dB, dC, dD, dz, "
        "ddt_bias, dinitial_states], or None.");
  m.def("chunk_scan", &chunk_scan, py::arg("x"), py::arg("dt"), py::arg("A"), py::arg("B"), py::arg("C"), py::arg("chunk_size"),
        py::arg("D"), py::arg("z"), py::arg("dt_bias"), py::arg("initial_states"), py::arg("seq_idx"), py::arg("dt_softplus"),
        py::arg("dt_min"), py::arg("dt_max"), py::arg("return_final_states"),
        "mamba_chunk_scan_combined with autograd: out or (out, final_states), or None when the arguments need the Python path.");
  m.def("split_conv_scan", &split_conv_scan, py::arg("zxbcdt"), py::arg("conv_weight"), py::arg("conv_bias"), py::arg("dt_bias"),
        py::arg("A"), py::arg("D"), py::arg("chunk_size"), py::arg("initial_states"), py::arg("seq_idx"), py::arg("dt_min"),
        py::arg("dt_max"), py::arg("return_final_states"), py::arg("silu"), py::arg("norm_weight"), py::arg("eps"),
        py::arg("out_weight"), py::arg("out_bias"), py::arg("headdim"), py::arg("ngroups"), py::arg("norm_before_gate"),
        "mamba_split_conv1d_scan_combined with autograd, or None when the arguments need the Python path.");
}

}  // namespace mamba_ext
