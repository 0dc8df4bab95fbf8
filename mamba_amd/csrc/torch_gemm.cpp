// Matrix products of a mixer on raw operands: through the library's grouped kernels (mamba_gemm) where they suit, the others
// through the BLAS library.
#include "torch_common.h"

namespace mamba_ext {
namespace {

at::Tensor matrix(const void *p, int64_t rows, int64_t cols, int64_t rs, int64_t cs, const at::TensorOptions &o) {
  return at::from_blob(const_cast<void *>(p), {rows, cols}, {rs, cs}, o);
}

}  // namespace

Products &Products::add(void *D, at::ScalarType d_type, int64_t ldd, int64_t M, int64_t N, int64_t K, Mat A, Mat B, bool accumulate,
                        const void *bias) {
  MambaGemm g{};
  g.A = A.p, g.a_ms = A.rs, g.a_ks = A.ks, g.B = B.p, g.b_ns = B.rs, g.b_ks = B.ks, g.bias = bias, g.D = D, g.ldd = ldd;
  g.M = (int32_t)M, g.N = (int32_t)N, g.K = (int32_t)K, g.d_dtype = dtype_code(d_type), g.accumulate = accumulate;
  if (type_ == at::kBFloat16 && M <= INT32_MAX && N <= INT32_MAX && K <= INT32_MAX && mamba_gemm_suits(&g)) {
    if (count_ == 4) run();
    g_[count_++] = g;
    return *this;
  }
  const auto o = options_.dtype(type_);
  const at::Tensor a = matrix(A.p, M, K, A.rs, A.ks, o), b = matrix(B.p, K, N, B.ks, B.rs, o);
  at::Tensor d = matrix(D, M, N, ldd, 1, options_.dtype(d_type));
  TORCH_CHECK(!accumulate || (d_type == type_ && !bias), "Products: accumulate");
  if (accumulate) {
    at::addmm_out(d, d, a, b);
  } else if (bias) {
    const at::Tensor c = at::from_blob(const_cast<void *>(bias), {N}, o);
    if (d_type == type_) at::addmm_out(d, c, a, b);
    else d.copy_(at::addmm(c, a, b));
  } else if (d_type == type_) {
    at::mm_out(d, a, b);
  } else {
    d.copy_(at::mm(a, b));
  }
  return *this;
}

void Products::run() {
  if (!count_) return;
  const int64_t floats = mamba_gemm_plan(g_, count_);
  if (floats < 0) check_rc((int)floats, "mamba_gemm_plan");
  at::Tensor ws;
  if (floats) ws = at::empty({floats}, options_.dtype(at::kFloat));
  check_rc(mamba_gemm(g_, count_, floats ? ws.data_ptr<float>() : nullptr, stream_of(options_.device())), "mamba_gemm");
  count_ = 0;
}

}  // namespace mamba_ext
