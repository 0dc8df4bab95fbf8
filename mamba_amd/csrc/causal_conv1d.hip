// Depthwise causal 1-D convolution (kernel width 2..4) with optional SiLU, forward and backward, for
// gfx950.  It is the convolution in front of both scans (the reference calls the separate
// causal_conv1d package for it: mamba_ssm/ops/selective_scan_interface.py:224,
// mamba_ssm/ops/triton/ssd_combined.py:845); the arithmetic is
//   out[b, c, l] = act(bias[c] + sum_k w[c, k] x[b, c, l - (W-1) + k]),  x = 0 before the sequence,
// and with seq_idx a tap that reaches into another sequence of a packed row contributes nothing.
// Both memory layouts of the callers are served without a transpose:
//   * position-contiguous rows (batch, channel, position): a thread owns 8 consecutive positions of
//     one row (16-byte accesses) and reads the 3-position halo from the neighbouring chunk;
//   * channel-contiguous rows (batch, position, channel): a thread owns 8 consecutive channels and
//     walks a run of positions with the previous taps in registers, so every element is read once.
// The backward pass re-computes the pre-activation from x instead of storing it.
#include "common.hpp"

#include <type_traits>

namespace {

constexpr int MAXW = 4;

DEVI float dsilu(float pre) {  // d/dpre silu(pre)
  const float s = sigmoid_f(pre);
  return s * (1.f + pre * (1.f - s));
}
DEVI float silu_f(float v) { return v * sigmoid_f(v); }

// A workgroup's sums for channel c: taps (right-aligned as in load_taps) and bias.  Its own row `part` of dw_part
// where the caller gave that workspace; else float atomics into the shared sums, or -- p.det_scale set -- 64-bit
// integer atomics on terms scaled to a fixed point, whose result does not depend on the order of the adds (see
// SsdParams).
constexpr int NSUM = MAXW + 1;
DEVI void conv_sums_out(const CausalConvParams &p, int part, int c, const float (&dw)[MAXW], float db) {
  if (p.dw_part) {
    float *dst = p.dw_part + ((int64_t)part * p.dim + c) * NSUM;
#pragma unroll
    for (int k = 0; k < MAXW; ++k) dst[k] = dw[k];
    dst[MAXW] = db;
    return;
  }
  auto add = [&](void *sum, int64_t *shadow, int64_t idx, float v) {
    if (v == 0.f) return;
    if (p.det_scale) det_add(shadow, idx, v, p.det_scale[0]);
    else unsafeAtomicAdd(static_cast<float *>(sum) + idx, v);
  };
#pragma unroll
  for (int k = 0; k < MAXW; ++k) {
    const int j = k - (MAXW - p.width);
    if (j >= 0) add(p.dweight, p.det_dweight, (int64_t)c * p.width + j, dw[k]);
  }
  if (p.dbias) add(p.dbias, p.det_dbias, c, db);
}

// dweight / dbias: the rows of dw_part added up in order, written in the parameters' dtype.  One thread per (channel,
// tap or bias), eight rows in flight.
__global__ __launch_bounds__(256) void conv_reduce_kernel(const CausalConvParams p, int nparts) {
  const int i = blockIdx.x * 256 + threadIdx.x, row = p.dim * NSUM;
  if (i >= row) return;
  const int c = i / NSUM, k = i - c * NSUM;
  if (k == MAXW ? !p.dbias : k < MAXW - p.width) return;
  const float *src = p.dw_part + i;
  float acc = 0.f;
  int q = 0;
  for (; q + 8 <= nparts; q += 8) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = src[(int64_t)(q + j) * row];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc += v[j];
  }
  for (; q < nparts; ++q) acc += src[(int64_t)q * row];
  if (k == MAXW) st_param(p.dbias, p.weight_dtype, c, acc);
  else st_param(p.dweight, p.weight_dtype, (int64_t)c * p.width + k - (MAXW - p.width), acc);
}

// Taps of n channels c0 .. (n <= NCH; the last one again beyond), right-aligned in 4 slots: slot 3 multiplies x[l], slot
// 0 multiplies x[l - 3].  One switch over the dtype around all of the loads: a switch per value makes every load wait
// for the one before it.
template <int NCH> DEVI void load_taps(const CausalConvParams &p, int c0, int n, float (&w)[NCH][MAXW], float (&bias)[NCH]) {
  auto run = [&](auto *wt, auto *bt) {
    typedef std::remove_const_t<std::remove_pointer_t<decltype(wt)>> W;
    W wr[NCH][MAXW], br[NCH];
    const int lead = MAXW - p.width;
    if constexpr (NCH % 2 == 0) {
      if (lead == 0 && n == NCH) {  // whole rows of four: 8 taps per load
        Pack8<W> q[NCH / 2];
#pragma unroll
        for (int j = 0; j < NCH / 2; ++j) q[j].load_any(wt + (int64_t)(c0 + 2 * j) * MAXW);
#pragma unroll
        for (int e = 0; e < NCH; ++e) br[e] = bt ? bt[c0 + e] : W{};
#pragma unroll
        for (int j = 0; j < NCH / 2; ++j) {
          float v[8];
          q[j].unpack(v);
#pragma unroll
          for (int k = 0; k < 8; ++k) w[2 * j + (k >> 2)][k & 3] = v[k];
        }
#pragma unroll
        for (int e = 0; e < NCH; ++e) bias[e] = bt ? ld1<W>(&br[e]) : 0.f;
        return;
      }
    }
#pragma unroll
    for (int e = 0; e < NCH; ++e) {
      const int64_t c = c0 + min(e, n - 1);
#pragma unroll
      for (int k = 0; k < MAXW; ++k) wr[e][k] = wt[c * p.width + max(k - lead, 0)];
      br[e] = bt ? bt[c] : W{};
    }
#pragma unroll
    for (int e = 0; e < NCH; ++e) {
#pragma unroll
      for (int k = 0; k < MAXW; ++k) w[e][k] = k >= lead ? ld1<W>(&wr[e][k]) : 0.f;
      bias[e] = bt ? ld1<W>(&br[e]) : 0.f;
    }
  };
  switch (p.weight_dtype) {
    case MAMBA_BF16: run(static_cast<const bf16_t *>(p.weight), static_cast<const bf16_t *>(p.bias)); break;
    case MAMBA_F16: run(static_cast<const f16_t *>(p.weight), static_cast<const f16_t *>(p.bias)); break;
    default: run(static_cast<const float *>(p.weight), static_cast<const float *>(p.bias)); break;
  }
}

// ------------------------------------------------------------------ position-contiguous rows
// A workgroup of 256 threads is `tx` threads along the positions (8 each) by 256 / tx channels; the host picks tx, a
// power of two of 16 .. 256, so that short rows leave few threads without positions.
struct RowPos {
  int c, b, l0, tx, slot;
  bool live;
};
// WAVE: a wave lies inside one channel (tx >= 64), whose taps are then scalar loads
template <bool WAVE> DEVI RowPos row_position(const CausalConvParams &p, int txlog) {
  RowPos q;
  q.tx = 1 << txlog;
  q.slot = threadIdx.x >> txlog;
  if (WAVE) q.slot = __builtin_amdgcn_readfirstlane(q.slot);
  q.c = blockIdx.y * (256 >> txlog) + q.slot;
  q.b = blockIdx.z;
  q.l0 = (blockIdx.x * q.tx + (threadIdx.x & (q.tx - 1))) * 8;
  q.live = q.c < p.dim && q.l0 < p.seqlen;
  return q;
}

// How the rows are reached: element by element (L < 8), in 16-byte pieces of aligned rows of whole pieces, or in 16-byte
// pieces at any alignment with a ragged last piece.
constexpr int SCALAR = 0, ALIGNED = 1, ANY = 2;

// Positions l0 - 3 .. of a row, l0 a multiple of 8: the previous piece (for its last 3), this one and, NEXT, the
// following one, from positions that keep inside the row.  load() only requests them, so that a kernel can request
// every window it needs before it uses the first; window() puts them in place: element j is position l0 - 3 + j, 0
// outside [0, L).
template <typename T, int MODE, bool NEXT> struct RowWindow {
  static constexpr int NWIN = NEXT ? 19 : 11;
  Pack8<T> prev, cur, next;
  float s[NWIN];
  DEVI void load(const T *row, int l0, int L) {
    if constexpr (MODE == ALIGNED) {
      prev.load(row + max(l0 - 8, 0));
      cur.load(row + l0);
      if (NEXT) next.load(row + min(l0 + 8, L - 8));
    } else if constexpr (MODE == ANY) {
      prev.load_any(row + max(l0 - 8, 0));
      cur.load_any(row + min(l0, L - 8));
      if (NEXT) next.load_any(row + min(l0 + 8, L - 8));
    } else {
#pragma unroll
      for (int j = 0; j < NWIN; ++j) {
        const int l = l0 - 3 + j;
        s[j] = (l >= 0 && l < L) ? ld1<T>(row + l) : 0.f;
      }
    }
  }
  DEVI void window(int l0, int L, float (&win)[NWIN]) const {
    if constexpr (MODE == SCALAR) {
#pragma unroll
      for (int j = 0; j < NWIN; ++j) win[j] = s[j];
    } else {
      float a[8], c[8], n[8];
      prev.unpack(a);
      cur.unpack(c);
      if (MODE == ANY) row8_place(l0, L, c);
#pragma unroll
      for (int j = 0; j < 3; ++j) win[j] = l0 >= 8 ? a[5 + j] : 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) win[3 + j] = c[j];
      if constexpr (NEXT) {
        next.unpack(n);
        if (MODE == ANY) row8_place(l0 + 8, L, n);
#pragma unroll
        for (int j = 0; j < 8; ++j) win[11 + j] = l0 + 8 < L ? n[j] : 0.f;
      }
    }
  }
};
// 8 results at l0: 16 bytes, or element by element in the last piece of a ragged row
template <typename T, int MODE> DEVI void store_row8(T *row, int l0, int L, const float (&o)[8]) {
  if constexpr (MODE == ALIGNED) {
    st8<T>(row + l0, o);
  } else if (MODE == ANY && l0 + 8 <= L) {
    st8_any<T>(row + l0, o);
  } else {
    st8_guard<T, false>(row + l0, min(8, L - l0), o);
  }
}
template <int NWIN> DEVI void load_ids(const int32_t *seq, int l0, int L, int (&ids)[NWIN]) {
#pragma unroll
  for (int j = 0; j < NWIN; ++j) {
    const int l = l0 - 3 + j;
    ids[j] = (l >= 0 && l < L) ? seq[l] : -0x7fffffff;
  }
}

template <typename T, int MODE, bool WAVE> __global__ __launch_bounds__(256) void conv_rows_fwd_kernel(const CausalConvParams p, int txlog) {
  const RowPos q = row_position<WAVE>(p, txlog);
  if (!q.live) return;
  const int L = p.seqlen, c = q.c, b = q.b, l0 = q.l0;
  RowWindow<T, MODE, false> rx;
  rx.load(static_cast<const T *>(p.x) + b * p.x_bs + c * p.x_cs, l0, L);
  float wt[1][MAXW], bt[1];
  load_taps<1>(p, c, 1, wt, bt);
  const float(&w)[MAXW] = wt[0];
  const float bias = bt[0];
  float win[11];
  rx.window(l0, L, win);
  int ids[11];
  if (p.seq_idx) load_ids<11>(p.seq_idx + (int64_t)b * L, l0, L, ids);
  float o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float v = bias;
#pragma unroll
    for (int k = 0; k < MAXW; ++k) {
      float t = win[i + k];
      if (p.seq_idx && ids[i + k] != ids[i + 3]) t = 0.f;
      v = __builtin_fmaf(w[k], t, v);
    }
    o[i] = p.silu ? silu_f(v) : v;
  }
  store_row8<T, MODE>(static_cast<T *>(p.out) + b * p.out_bs + c * p.out_cs, l0, L, o);
}

// Sum over the tx threads of a channel: DPP adds inside rows of 16 lanes, then between the rows of a wave, then (tx >
// 64) between waves through LDS.  The channel's last thread of its first wave holds the result: returns whether this
// thread does.
DEVI bool channel_sum(float (&v)[NSUM], int tx, float (*red)[NSUM]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NSUM; ++k) {
    float x = row_sum_to_last(v[k]);
    if (tx >= 32) x += dpp_f<DPP_ROW_BCAST15, 0xa>(0.f, x);
    if (tx >= 64) x += dpp_f<DPP_ROW_BCAST31, 0xc>(0.f, x);
    v[k] = x;
  }
  if (tx <= 64) return (threadIdx.x & (tx - 1)) == (unsigned)tx - 1;
  if (lane == 63) {
#pragma unroll
    for (int k = 0; k < NSUM; ++k) red[wave][k] = v[k];
  }
  __syncthreads();
  const int waves = tx >> 6;
  if (lane != 63 || (wave & (waves - 1)) != 0) return false;
  for (int w = 1; w < waves; ++w) {
#pragma unroll
    for (int k = 0; k < NSUM; ++k) v[k] += red[wave + w][k];
  }
  return true;
}

template <typename T, int MODE, bool WAVE> __global__ __launch_bounds__(256) void conv_rows_bwd_kernel(const CausalConvParams p, int txlog) {
  __shared__ float red[4][NSUM];
  const RowPos q = row_position<WAVE>(p, txlog);
  const int L = p.seqlen, c = q.c, b = q.b, l0 = q.l0;
  float dw[MAXW] = {0.f, 0.f, 0.f, 0.f}, db = 0.f;
  if (q.live) {
    RowWindow<T, MODE, true> rx, rg;
    rx.load(static_cast<const T *>(p.x) + b * p.x_bs + c * p.x_cs, l0, L);
    rg.load(static_cast<const T *>(p.dout) + b * p.dout_bs + c * p.dout_cs, l0, L);
    float wt[1][MAXW], bt[1];
    load_taps<1>(p, c, 1, wt, bt);
    const float(&w)[MAXW] = wt[0];
    const float bias = bt[0];
    float xw[19], gw[19];  // x and dout at positions l0 - 3 .. l0 + 15 (dout's halo is not used)
    rx.window(l0, L, xw);
    rg.window(l0, L, gw);
    int ids[19];
    if (p.seq_idx) load_ids<19>(p.seq_idx + (int64_t)b * L, l0, L, ids);
    // gradient of the pre-activation at positions l0 .. l0 + 10 (own 8 and the 3 that still see them)
    float dpre[11];
#pragma unroll
    for (int j = 0; j < 11; ++j) {
      float v = bias;
#pragma unroll
      for (int k = 0; k < MAXW; ++k) {
        float t = xw[j + k];
        if (p.seq_idx && ids[j + k] != ids[j + 3]) t = 0.f;
        v = __builtin_fmaf(w[k], t, v);
      }
      const float g = gw[j + 3];
      dpre[j] = l0 + j < L ? (p.silu ? g * dsilu(v) : g) : 0.f;
    }
    float o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < MAXW; ++k) {  // x[l] enters out[l + 3 - k] through tap k
        float t = dpre[i + 3 - k];
        if (p.seq_idx && ids[i + 3 + 3 - k] != ids[i + 3]) t = 0.f;
        v = __builtin_fmaf(w[k], t, v);
      }
      o[i] = v;
#pragma unroll
      for (int k = 0; k < MAXW; ++k) {
        float t = xw[i + k];
        if (p.seq_idx && ids[i + k] != ids[i + 3]) t = 0.f;
        dw[k] = __builtin_fmaf(dpre[i], t, dw[k]);
      }
      db += dpre[i];
    }
    store_row8<T, MODE>(static_cast<T *>(p.dx) + b * p.dx_bs + c * p.dx_cs, l0, L, o);
  }
  float sums[NSUM] = {dw[0], dw[1], dw[2], dw[3], db};
  if (channel_sum(sums, q.tx, red) && c < p.dim) {
    const float taps[MAXW] = {sums[0], sums[1], sums[2], sums[3]};
    conv_sums_out(p, b * gridDim.x + blockIdx.x, c, taps, sums[MAXW]);
  }
}

// ------------------------------------------------------------------ channel-contiguous rows
constexpr int RUN = 32;   // positions per thread
constexpr int NRUN = 4;   // runs per workgroup (256 threads = 64 channel groups x 4 runs)

template <typename T, bool VEC> DEVI void load_ch8(const T *p, int nvalid, float (&o)[8]) {
  if constexpr (VEC) ld8<T>(p, o);
  else ld8_guard<T, false>(p, nvalid, 0.f, o);
}

template <typename T, bool VEC> __global__ __launch_bounds__(256) void conv_cl_fwd_kernel(const CausalConvParams p) {
  const int L = p.seqlen, b = blockIdx.z;
  const int cg = threadIdx.x & 63, run = threadIdx.x >> 6;
  const int c0 = (blockIdx.x * 64 + cg) * 8;
  if (c0 >= p.dim) return;
  const int nch = min(8, p.dim - c0);
  const int lbeg = (blockIdx.y * NRUN + run) * RUN, lend = min(lbeg + RUN, L);
  if (lbeg >= L) return;
  float w[8][MAXW], bias[8];
  load_taps<8>(p, c0, nch, w, bias);
  const T *xb = static_cast<const T *>(p.x) + b * p.x_bs + c0;
  T *ob = static_cast<T *>(p.out) + b * p.out_bs + c0;
  const int32_t *seq = p.seq_idx ? p.seq_idx + (int64_t)b * L : nullptr;
  float xw[3][8];  // x at l - 3, l - 2, l - 1
  int idw[3] = {-0x7fffffff, -0x7fffffff, -0x7fffffff};
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int l = lbeg - 3 + j;
#pragma unroll
    for (int e = 0; e < 8; ++e) xw[j][e] = 0.f;
    if (l >= 0) {
      load_ch8<T, VEC>(xb + (int64_t)l * p.x_ls, nch, xw[j]);
      if (seq) idw[j] = seq[l];
    }
  }
  for (int l4 = lbeg; l4 < lend; l4 += 4) {
    float xin[4][8];
    int idn[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // the loads of four positions first
      const int l = min(l4 + u, L - 1);
      load_ch8<T, VEC>(xb + (int64_t)l * p.x_ls, nch, xin[u]);
      idn[u] = seq ? seq[l] : 0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int l = l4 + u;
      if (l >= lend) break;
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = __builtin_fmaf(w[e][3], xin[u][e], bias[e]);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          float t = xw[j][e];
          if (seq && idw[j] != idn[u]) t = 0.f;
          v = __builtin_fmaf(w[e][j], t, v);
        }
        o[e] = p.silu ? silu_f(v) : v;
      }
      st8_guard<T, VEC>(ob + (int64_t)l * p.out_ls, nch, o);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        xw[0][e] = xw[1][e];
        xw[1][e] = xw[2][e];
        xw[2][e] = xin[u][e];
      }
      idw[0] = idw[1];
      idw[1] = idw[2];
      idw[2] = idn[u];
    }
  }
}

template <typename T, bool VEC> __global__ __launch_bounds__(256) void conv_cl_bwd_kernel(const CausalConvParams p) {
  __shared__ float red[NRUN - 1][64][8 * (MAXW + 1)];
  const int L = p.seqlen, b = blockIdx.z;
  const int cg = threadIdx.x & 63, run = threadIdx.x >> 6;
  const int c0 = (blockIdx.x * 64 + cg) * 8;
  const int nch = max(0, min(8, p.dim - c0));
  const int lbeg = (blockIdx.y * NRUN + run) * RUN, lend = min(lbeg + RUN, L);
  float dw[8][MAXW], db[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    db[e] = 0.f;
#pragma unroll
    for (int k = 0; k < MAXW; ++k) dw[e][k] = 0.f;
  }
  if (nch > 0 && lbeg < L) {
    float w[8][MAXW], bias[8];
    load_taps<8>(p, c0, nch, w, bias);
    const T *xb = static_cast<const T *>(p.x) + b * p.x_bs + c0;
    const T *gb = static_cast<const T *>(p.dout) + b * p.dout_bs + c0;
    T *dxb = static_cast<T *>(p.dx) + b * p.dx_bs + c0;
    const int32_t *seq = p.seq_idx ? p.seq_idx + (int64_t)b * L : nullptr;
    // Walk down from lend + 2: the first three steps only rebuild dpre at the positions after the run.
    const int ltop = min(lend + 2, L - 1);
    float xw[4][8];   // x at l - 3 .. l
    float dp[4][8];   // dpre at l .. l + 3
    int idx[7];       // sequence ids at l - 3 .. l + 3
#pragma unroll
    for (int j = 0; j < 7; ++j) {
      const int l = ltop - 3 + j;
      idx[j] = (seq && l >= 0 && l < L) ? seq[l] : -0x7fffffff;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int l = ltop - 3 + j;
#pragma unroll
      for (int e = 0; e < 8; ++e) xw[j][e] = dp[j][e] = 0.f;
      if (l >= 0) load_ch8<T, VEC>(xb + (int64_t)l * p.x_ls, nch, xw[j]);
    }
    for (int l4 = ltop; l4 >= lbeg; l4 -= 4) {
      // the loads of four steps first (dout at l4 .. l4 - 3, x at l4 - 4 .. l4 - 7): the stores of dx in
      // between would otherwise keep the compiler from moving them up
      float g4[4][8], x4[4][8];
      int id4[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int l = l4 - u;
        load_ch8<T, VEC>(gb + (int64_t)max(l, 0) * p.dout_ls, nch, g4[u]);
        load_ch8<T, VEC>(xb + (int64_t)max(l - 4, 0) * p.x_ls, nch, x4[u]);
        id4[u] = (seq && l - 4 >= 0) ? seq[l - 4] : -0x7fffffff;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int l = l4 - u;
        if (l < lbeg) break;
        // dpre at l
        float dcur[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float v = bias[e];
#pragma unroll
          for (int k = 0; k < MAXW; ++k) {
            float t = xw[k][e];
            if (seq && idx[k] != idx[3]) t = 0.f;
            v = __builtin_fmaf(w[e][k], t, v);
          }
          dcur[e] = p.silu ? g4[u][e] * dsilu(v) : g4[u][e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          dp[3][e] = dp[2][e];
          dp[2][e] = dp[1][e];
          dp[1][e] = dp[0][e];
          dp[0][e] = dcur[e];
        }
        if (l < lend) {
          float o[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            float v = 0.f;
#pragma unroll
            for (int k = 0; k < MAXW; ++k) {  // x[l] enters out[l + 3 - k] through tap k
              float t = dp[3 - k][e];
              if (seq && idx[3 + 3 - k] != idx[3]) t = 0.f;
              v = __builtin_fmaf(w[e][k], t, v);
            }
            o[e] = v;
#pragma unroll
            for (int k = 0; k < MAXW; ++k) {
              float t = xw[k][e];
              if (seq && idx[k] != idx[3]) t = 0.f;
              dw[e][k] = __builtin_fmaf(dcur[e], t, dw[e][k]);
            }
            db[e] += dcur[e];
          }
          st8_guard<T, VEC>(dxb + (int64_t)l * p.dx_ls, nch, o);
        }
        // slide both windows one position down
        const bool has = l - 4 >= 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          xw[3][e] = xw[2][e];
          xw[2][e] = xw[1][e];
          xw[1][e] = xw[0][e];
          xw[0][e] = has ? x4[u][e] : 0.f;
        }
#pragma unroll
        for (int j = 6; j > 0; --j) idx[j] = idx[j - 1];
        idx[0] = id4[u];
      }
    }
  }
  // the four runs of a channel group are summed in LDS, then leave once per channel and tap
  if (run > 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int k = 0; k < MAXW; ++k) red[run - 1][cg][e * (MAXW + 1) + k] = dw[e][k];
      red[run - 1][cg][e * (MAXW + 1) + MAXW] = db[e];
    }
  }
  __syncthreads();
  if (run == 0 && nch > 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (e >= nch) break;
      float taps[MAXW], v = db[e];
#pragma unroll
      for (int k = 0; k < MAXW; ++k) {
        taps[k] = dw[e][k];
#pragma unroll
        for (int r = 0; r < NRUN - 1; ++r) taps[k] += red[r][cg][e * (MAXW + 1) + k];
      }
#pragma unroll
      for (int r = 0; r < NRUN - 1; ++r) v += red[r][cg][e * (MAXW + 1) + MAXW];
      conv_sums_out(p, b * gridDim.y + blockIdx.y, c0 + e, taps, v);
    }
  }
}

// The backward pass with 4 channels per thread (rows whose 4-channel pieces are aligned: the VEC case).  The
// 8-channel kernel above keeps two windows, the taps and their gradients for 8 channels in 232 registers, two waves
// per SIMD; half the channels per thread is half the registers and twice the waves.  A thread's loads of the next
// four steps are requested, and kept in their storage format, before it works on the current four: memory and the
// SiLU re-computation overlap instead of alternating.
template <typename T> struct Raw4 {
  typedef u32x2 type;
};
template <> struct Raw4<float> {
  typedef u32x4 type;
};
template <typename T> DEVI void unpack4(const typename Raw4<T>::type &r, float (&o)[4]);
template <> DEVI void unpack4<bf16_t>(const u32x2 &r, float (&o)[4]) {
  o[0] = bf16_lo(r.x); o[1] = bf16_hi(r.x); o[2] = bf16_lo(r.y); o[3] = bf16_hi(r.y);
}
template <> DEVI void unpack4<f16_t>(const u32x2 &r, float (&o)[4]) {
  o[0] = f16_lo(r.x); o[1] = f16_hi(r.x); o[2] = f16_lo(r.y); o[3] = f16_hi(r.y);
}
template <> DEVI void unpack4<float>(const u32x4 &r, float (&o)[4]) {
  const f32x4 f = __builtin_bit_cast(f32x4, r);  // (the whole vector: a bit cast of one element of it is not one)
  o[0] = f.x; o[1] = f.y; o[2] = f.z; o[3] = f.w;
}
template <typename T> DEVI typename Raw4<T>::type pack4(const float (&v)[4]);
template <> DEVI u32x2 pack4<bf16_t>(const float (&v)[4]) { return u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])}; }
template <> DEVI u32x2 pack4<f16_t>(const float (&v)[4]) { return u32x2{pack_f16(v[0], v[1]), pack_f16(v[2], v[3])}; }
template <> DEVI u32x4 pack4<float>(const float (&v)[4]) {
  const f32x4 f = {v[0], v[1], v[2], v[3]};
  return __builtin_bit_cast(u32x4, f);
}

// The forward pass in the same form: 4 channels per thread, the next four positions requested before the current
// four are worked on.
// RUN: positions per thread, 32 where the grid fills the chip, 8 where it does not.  A short run is a chain of load
// latencies and little else, so all of its rows are requested before the taps, and nothing waits before that (with
// guarded single loads in front and the second four positions behind the first: 12.4 us for 2 x 1000 x 1792 in bf16).
template <typename T, int RUN> __global__ __launch_bounds__(256) void conv_cl_fwd4_kernel(const CausalConvParams p) {
  typedef typename Raw4<T>::type raw_t;
  constexpr int CPT = 4, AHEAD = RUN == 8 ? 2 : 1;  // groups of four positions in flight
  const int L = p.seqlen, b = blockIdx.z;
  const int cg = threadIdx.x & 63, run = threadIdx.x >> 6;
  const int c0 = (blockIdx.x * 64 + cg) * CPT;
  if (c0 >= p.dim) return;
  const int lbeg = (blockIdx.y * NRUN + run) * RUN, lend = min(lbeg + RUN, L);
  if (lbeg >= L) return;
  const T *xb = static_cast<const T *>(p.x) + b * p.x_bs + c0;
  T *ob = static_cast<T *>(p.out) + b * p.out_bs + c0;
  const int32_t *seq = p.seq_idx ? p.seq_idx + (int64_t)b * L : nullptr;
  raw_t xp[3], xn[AHEAD][4];
  int idw[3], idn[AHEAD][4];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int l = max(lbeg - 3 + j, 0);
    xp[j] = *reinterpret_cast<const raw_t *>(xb + (int64_t)l * p.x_ls);
    idw[j] = seq ? seq[l] : 0;
  }
  auto fetch = [&](int l4, raw_t(&x)[4], int(&id)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int l = min(l4 + u, L - 1);
      x[u] = *reinterpret_cast<const raw_t *>(xb + (int64_t)l * p.x_ls);
      id[u] = seq ? seq[l] : 0;
    }
  };
#pragma unroll
  for (int q = 0; q < AHEAD; ++q) fetch(lbeg + 4 * q, xn[q], idn[q]);
  float w[CPT][MAXW], bias[CPT];
  load_taps<CPT>(p, c0, CPT, w, bias);
  float xw[3][CPT];  // x at l - 3, l - 2, l - 1
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    unpack4<T>(xp[j], xw[j]);
    if (lbeg - 3 + j < 0) {
      idw[j] = -0x7fffffff;
#pragma unroll
      for (int e = 0; e < CPT; ++e) xw[j][e] = 0.f;
    }
  }
  auto use = [&](int l4, const raw_t(&x4)[4], const int(&id4)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int l = l4 + u;
      if (l >= lend) break;
      float xin[CPT], o[CPT];
      unpack4<T>(x4[u], xin);
#pragma unroll
      for (int e = 0; e < CPT; ++e) {
        float v = __builtin_fmaf(w[e][3], xin[e], bias[e]);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          float t = xw[j][e];
          if (seq && idw[j] != id4[u]) t = 0.f;
          v = __builtin_fmaf(w[e][j], t, v);
        }
        o[e] = p.silu ? silu_f(v) : v;
      }
      *reinterpret_cast<raw_t *>(ob + (int64_t)l * p.out_ls) = pack4<T>(o);
#pragma unroll
      for (int e = 0; e < CPT; ++e) {
        xw[0][e] = xw[1][e];
        xw[1][e] = xw[2][e];
        xw[2][e] = xin[e];
      }
      idw[0] = idw[1];
      idw[1] = idw[2];
      idw[2] = id4[u];
    }
  };
  if constexpr (RUN == 4 * AHEAD) {
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) use(lbeg + 4 * q, xn[q], idn[q]);
  } else {
    for (int l4 = lbeg; l4 < lend; l4 += 4) {
      raw_t x4[4];
      int id4[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) x4[u] = xn[0][u], id4[u] = idn[0][u];
      fetch(l4 + 4, xn[0], idn[0]);  // (past the run on the last turn: rows that exist, never used)
      use(l4, x4, id4);
    }
  }
}

// RUN: positions per thread.  A run costs a 6-position warm-up, the taps, and its share of the reduction of the
// filter gradients: long runs (128) where the grid still fills the chip, else 32, and 8 where even those leave compute
// units without work (the walk down a run is a serial chain: with few workgroups its length is the kernel's time).
// A run of 8 has all of its rows in flight at once (18.2 us for 2 x 1000 x 1792 in bf16 with one group of four ahead).
template <typename T, int RUN> __global__ __launch_bounds__(256) void conv_cl_bwd4_kernel(const CausalConvParams p) {
  typedef typename Raw4<T>::type raw_t;
  constexpr int CPT = 4, AHEAD = RUN == 8 ? 3 : 1;  // 8 positions and 3 behind them are three groups of four
  __shared__ float red[NRUN - 1][64][CPT * (MAXW + 1)];
  const int L = p.seqlen, b = blockIdx.z;
  const int cg = threadIdx.x & 63, run = threadIdx.x >> 6;
  const int c0 = (blockIdx.x * 64 + cg) * CPT;
  const bool live = c0 < p.dim;  // (dim is a multiple of 8 here: a thread has all of its 4 channels or none)
  const int lbeg = (blockIdx.y * NRUN + run) * RUN, lend = min(lbeg + RUN, L);
  float dw[CPT][MAXW], db[CPT];
#pragma unroll
  for (int e = 0; e < CPT; ++e) {
    db[e] = 0.f;
#pragma unroll
    for (int k = 0; k < MAXW; ++k) dw[e][k] = 0.f;
  }
  if (live && lbeg < L) {
    const T *xb = static_cast<const T *>(p.x) + b * p.x_bs + c0;
    const T *gb = static_cast<const T *>(p.dout) + b * p.dout_bs + c0;
    T *dxb = static_cast<T *>(p.dx) + b * p.dx_bs + c0;
    const int32_t *seq = p.seq_idx ? p.seq_idx + (int64_t)b * L : nullptr;
    // Walk down from lend + 2: the first three steps only rebuild dpre at the positions after the run.
    const int ltop = min(lend + 2, L - 1);
    // every load of the first AHEAD groups is issued before anything waits; masks come after the taps
    raw_t xp[4], gn[AHEAD][4], xn[AHEAD][4];
    int idp[7], idn[AHEAD][4];
#pragma unroll
    for (int j = 0; j < 7; ++j) idp[j] = seq ? seq[min(max(ltop - 3 + j, 0), L - 1)] : 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) xp[j] = *reinterpret_cast<const raw_t *>(xb + (int64_t)max(ltop - 3 + j, 0) * p.x_ls);
    // the loads of four steps: dout at l4 .. l4 - 3, x and the ids at l4 - 4 .. l4 - 7 (position 0 stands in below it)
    auto fetch = [&](int l4, raw_t(&g)[4], raw_t(&x)[4], int(&id)[4]) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int l = l4 - u;
        g[u] = *reinterpret_cast<const raw_t *>(gb + (int64_t)max(l, 0) * p.dout_ls);
        x[u] = *reinterpret_cast<const raw_t *>(xb + (int64_t)max(l - 4, 0) * p.x_ls);
        id[u] = seq ? seq[max(l - 4, 0)] : 0;
      }
    };
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) fetch(ltop - 4 * q, gn[q], xn[q], idn[q]);
    float w[CPT][MAXW], bias[CPT];
    load_taps<CPT>(p, c0, CPT, w, bias);
    float xw[4][CPT];  // x at l - 3 .. l
    float dp[4][CPT];  // dpre at l .. l + 3
    int idx[7];        // sequence ids at l - 3 .. l + 3
#pragma unroll
    for (int j = 0; j < 7; ++j) {
      const int l = ltop - 3 + j;
      idx[j] = l >= 0 && l < L ? idp[j] : -0x7fffffff;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unpack4<T>(xp[j], xw[j]);
#pragma unroll
      for (int e = 0; e < CPT; ++e) {
        dp[j][e] = 0.f;
        xw[j][e] = ltop - 3 + j >= 0 ? xw[j][e] : 0.f;
      }
    }
    auto use = [&](int l4, const raw_t(&g4)[4], const raw_t(&x4)[4], const int(&id4)[4]) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int l = l4 - u;
        if (l < lbeg) break;
        float gu[CPT], xu[CPT];
        unpack4<T>(g4[u], gu);
        unpack4<T>(x4[u], xu);
        // dpre at l
        float dcur[CPT];
#pragma unroll
        for (int e = 0; e < CPT; ++e) {
          float v = bias[e];
#pragma unroll
          for (int k = 0; k < MAXW; ++k) {
            float t = xw[k][e];
            if (seq && idx[k] != idx[3]) t = 0.f;
            v = __builtin_fmaf(w[e][k], t, v);
          }
          dcur[e] = p.silu ? gu[e] * dsilu(v) : gu[e];
        }
#pragma unroll
        for (int e = 0; e < CPT; ++e) {
          dp[3][e] = dp[2][e];
          dp[2][e] = dp[1][e];
          dp[1][e] = dp[0][e];
          dp[0][e] = dcur[e];
        }
        if (l < lend) {
          float o[CPT];
#pragma unroll
          for (int e = 0; e < CPT; ++e) {
            float v = 0.f;
#pragma unroll
            for (int k = 0; k < MAXW; ++k) {  // x[l] enters out[l + 3 - k] through tap k
              float t = dp[3 - k][e];
              if (seq && idx[3 + 3 - k] != idx[3]) t = 0.f;
              v = __builtin_fmaf(w[e][k], t, v);
            }
            o[e] = v;
#pragma unroll
            for (int k = 0; k < MAXW; ++k) {
              float t = xw[k][e];
              if (seq && idx[k] != idx[3]) t = 0.f;
              dw[e][k] = __builtin_fmaf(dcur[e], t, dw[e][k]);
            }
            db[e] += dcur[e];
          }
          *reinterpret_cast<raw_t *>(dxb + (int64_t)l * p.dx_ls) = pack4<T>(o);
        }
        // slide both windows one position down
        const bool has = l - 4 >= 0;
#pragma unroll
        for (int e = 0; e < CPT; ++e) {
          xw[3][e] = xw[2][e];
          xw[2][e] = xw[1][e];
          xw[1][e] = xw[0][e];
          xw[0][e] = has ? xu[e] : 0.f;
        }
#pragma unroll
        for (int j = 6; j > 0; --j) idx[j] = idx[j - 1];
        idx[0] = has ? id4[u] : -0x7fffffff;
      }
    };
    if constexpr (RUN == 8) {
#pragma unroll
      for (int q = 0; q < AHEAD; ++q) use(ltop - 4 * q, gn[q], xn[q], idn[q]);
    } else {
      for (int l4 = ltop; l4 >= lbeg; l4 -= 4) {
        raw_t g4[4], x4[4];
        int id4[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) g4[u] = gn[0][u], x4[u] = xn[0][u], id4[u] = idn[0][u];
        fetch(l4 - 4, gn[0], xn[0], idn[0]);  // (below the run on the last turn: rows that exist, never used)
        use(l4, g4, x4, id4);
      }
    }
  }
  // the four runs of a channel group are summed in LDS, then leave once per channel and tap
  if (run > 0) {
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
#pragma unroll
      for (int k = 0; k < MAXW; ++k) red[run - 1][cg][e * (MAXW + 1) + k] = dw[e][k];
      red[run - 1][cg][e * (MAXW + 1) + MAXW] = db[e];
    }
  }
  __syncthreads();
  if (run == 0 && live) {
#pragma unroll
    for (int e = 0; e < CPT; ++e) {
      float taps[MAXW], v = db[e];
#pragma unroll
      for (int k = 0; k < MAXW; ++k) {
        taps[k] = dw[e][k];
#pragma unroll
        for (int r = 0; r < NRUN - 1; ++r) taps[k] += red[r][cg][e * (MAXW + 1) + k];
      }
#pragma unroll
      for (int r = 0; r < NRUN - 1; ++r) v += red[r][cg][e * (MAXW + 1) + MAXW];
      conv_sums_out(p, b * gridDim.y + blockIdx.y, c0 + e, taps, v);
    }
  }
}

// ------------------------------------------------------------------ decode step
// One thread per (batch entry, channel): with xn = [conv_state, x] along the position axis,
//   out[t] = act(bias + sum_k w[k] xn[state_len + t - (W-1) + k]),  conv_state <- last state_len of xn
// (what the reference spells, for one new position and state_len = W, as roll + insert + dot:
// mamba_ssm/modules/mamba2.py:291-296).  The shift runs in place in ascending order, which is safe
// because every entry is written from a higher index of the same thread's own row.
template <typename T, typename S> __global__ __launch_bounds__(256) void conv_update_kernel(const CausalConvUpdateParams p) {
  const int c = blockIdx.x * 256 + threadIdx.x, b = blockIdx.y;
  if (c >= p.dim) return;
  const T *x = static_cast<const T *>(p.x) + b * p.x_bs + c * p.x_cs;
  T *out = static_cast<T *>(p.out) + b * p.out_bs + c * p.out_cs;
  const int slot = p.conv_state_indices ? p.conv_state_indices[b] : b;
  if (slot < 0 || slot >= p.state_rows) {  // padding entry of the batch: no state, zero output
    for (int t = 0; t < p.seqlen; ++t) st1<T>(out + t * p.out_ls, 0.f);
    return;
  }
  S *st = static_cast<S *>(p.conv_state) + slot * p.state_bs + c * p.state_cs;
  float w[MAXW], bias;
#pragma unroll
  for (int k = 0; k < MAXW; ++k) {
    const int j = k - (MAXW - p.width);
    w[k] = j >= 0 ? ld_param(p.weight, p.weight_dtype, (int64_t)c * p.width + j) : 0.f;
  }
  bias = p.bias ? ld_param(p.bias, p.weight_dtype, c) : 0.f;
  const int SL = p.state_len;
  float win[MAXW];  // win[0..2]: the three positions before the next output, win[3]: the new one
  if (p.cache_seqlens) {
    // circular buffer: position t of the sequence lives in slot t mod SL; taps the filter does not use stay 0
    const int len = p.cache_seqlens[b];
    auto slot_of = [&](int t) { return ((t % SL) + SL) % SL; };
#pragma unroll
    for (int i = 0; i < MAXW - 1; ++i)
      win[i] = i >= MAXW - p.width ? ld1<S>(st + slot_of(len - (MAXW - 1) + i) * p.state_ls) : 0.f;
    for (int t = 0; t < p.seqlen; ++t) st1<S>(st + slot_of(len + t) * p.state_ls, ld1<T>(x + t * p.x_ls));
  } else {
#pragma unroll
    for (int i = 0; i < MAXW - 1; ++i) {
      const int j = SL - (MAXW - 1) + i;
      win[i] = j >= 0 ? ld1<S>(st + j * p.state_ls) : 0.f;
    }
    for (int j = 0; j < SL; ++j) {
      const int src = j + p.seqlen;
      const float v = src < SL ? ld1<S>(st + src * p.state_ls) : ld1<T>(x + (src - SL) * p.x_ls);
      st1<S>(st + j * p.state_ls, v);
    }
  }
  for (int t = 0; t < p.seqlen; ++t) {
    win[3] = ld1<T>(x + t * p.x_ls);
    float v = bias;
#pragma unroll
    for (int k = 0; k < MAXW; ++k) v = __builtin_fmaf(w[k], win[k], v);
    st1<T>(out + t * p.out_ls, p.silu ? silu_f(v) : v);
    win[0] = win[1];
    win[1] = win[2];
    win[2] = win[3];
  }
}

// states[s, c, j] = x[cu_seqlens[s + 1] - state_len + j, c], zero where that position lies before
// the start of sequence s: the convolution state each sequence of a packed row leaves behind.
template <typename T> __global__ __launch_bounds__(256) void conv_varlen_states_kernel(const CausalConvVarlenParams p) {
  const int c = blockIdx.x * 256 + threadIdx.x, s = blockIdx.y;
  if (c >= p.dim) return;
  const int beg = p.cu_seqlens[s], end = p.cu_seqlens[s + 1];
  const T *x = static_cast<const T *>(p.x) + c * p.x_cs;
  T *o = static_cast<T *>(p.states) + s * p.states_bs + c * p.states_cs;
  for (int j = 0; j < p.state_len; ++j) {
    const int l = end - p.state_len + j;
    st1<T>(o + j * p.states_ls, l >= beg && l >= 0 && l < p.total ? ld1<T>(x + l * p.x_ls) : 0.f);
  }
}

// ------------------------------------------------------------------ launch
int check(const CausalConvParams *p, bool bwd) {
  if (!p || !p->x || !p->weight) return MAMBA_E_BADARG;
  if (p->batch <= 0 || p->dim <= 0 || p->seqlen <= 0) return MAMBA_E_BADARG;
  if (p->width < 2 || p->width > MAXW) return MAMBA_E_UNSUPPORTED;
  if (p->dtype != MAMBA_F32 && p->dtype != MAMBA_BF16 && p->dtype != MAMBA_F16) return MAMBA_E_BADARG;
  if (p->batch > 65535) return MAMBA_E_UNSUPPORTED;
  if (!bwd && !p->out) return MAMBA_E_BADARG;
  if (bwd && (!p->dout || !p->dx || !p->dweight)) return MAMBA_E_BADARG;
  if (p->weight_dtype < MAMBA_F32 || p->weight_dtype > MAMBA_F16) return MAMBA_E_BADARG;
  if (bwd && !p->dw_part && p->weight_dtype != MAMBA_F32) return MAMBA_E_BADARG;  // the atomic sums are fp32
  if (bwd && !p->dw_part && p->det_scale && (!p->det_dweight || (p->dbias && !p->det_dbias))) return MAMBA_E_BADARG;
  if (p->x_ls != 1 && p->x_cs != 1) return MAMBA_E_UNSUPPORTED;
  return MAMBA_OK;
}

bool al16(const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; }

// Which kernel serves a problem, on which grid.
struct Plan {
  bool rows, vec;        // vec: the channel-last kernels of 16-byte pieces
  int mode, txlog, run;  // rows: access and threads along the positions; channel-last: positions per thread
  dim3 grid;
  int nparts;      // rows of dw_part the backward kernel writes
};

int plan_conv(const CausalConvParams &p, bool bwd, Plan &q) {
  const int64_t m = p.dtype == MAMBA_F32 ? 4 : 8;
  q.rows = p.x_ls == 1 && (bwd ? p.dout_ls == 1 && p.dx_ls == 1 : p.out_ls == 1);
  if (q.rows) {
    auto al = [&](const void *ptr, int64_t a, int64_t b2) { return al16(ptr) && a % m == 0 && b2 % m == 0; };
    q.mode = p.seqlen % 8 == 0 && al(p.x, p.x_bs, p.x_cs) &&
                     (bwd ? al(p.dout, p.dout_bs, p.dout_cs) && al(p.dx, p.dx_bs, p.dx_cs) : al(p.out, p.out_bs, p.out_cs))
                 ? ALIGNED
                 : p.seqlen >= 8 ? ANY : SCALAR;
    // the widest split of the positions among the ones that leave the fewest threads idle
    const int units = (p.seqlen + 7) / 8;
    int best = -1;
    for (int t = 8; t >= 4; --t) {
      const int covered = (units + (1 << t) - 1) >> t << t;
      if (best < 0 || covered < best) best = covered, q.txlog = t;
    }
    const int per = 256 >> q.txlog;
    if ((p.dim + per - 1) / per > 65535) return MAMBA_E_UNSUPPORTED;
    q.grid = dim3(best >> q.txlog, (p.dim + per - 1) / per, p.batch);
    q.nparts = (int)q.grid.x * p.batch;
    return MAMBA_OK;
  }
  if (!(p.x_cs == 1 && (bwd ? p.dout_cs == 1 && p.dx_cs == 1 : p.out_cs == 1))) return MAMBA_E_UNSUPPORTED;
  auto ok = [&](const void *ptr, int64_t a, int64_t b2) { return al16(ptr) && a % m == 0 && b2 % m == 0; };
  q.vec = p.dim % 8 == 0 && ok(p.x, p.x_bs, p.x_ls) &&
          (bwd ? ok(p.dout, p.dout_bs, p.dout_ls) && ok(p.dx, p.dx_bs, p.dx_ls) : ok(p.out, p.out_bs, p.out_ls));
  const int xg = q.vec ? (p.dim + 255) / 256 : (p.dim + 511) / 512;
  auto yg = [&](int run) { return (p.seqlen + run * NRUN - 1) / (run * NRUN); };
  auto fills = [&](int run, int times) { return (int64_t)xg * yg(run) * p.batch >= times * (int64_t)cu_count(); };
  q.run = RUN;
  if (q.vec) {
    if (bwd && fills(128, 2)) q.run = 128;
    else if (!fills(RUN, bwd ? 1 : 2) && yg(8) <= 65535) q.run = 8;
  }
  if (yg(q.run) > 65535) return MAMBA_E_UNSUPPORTED;
  q.grid = dim3(xg, yg(q.run), p.batch);
  q.nparts = (int)q.grid.y * p.batch;
  return MAMBA_OK;
}

template <typename T> int launch_conv(const CausalConvParams &p, bool bwd, hipStream_t s) {
  Plan q{};
  const int rc = plan_conv(p, bwd, q);
  if (rc != MAMBA_OK) return rc;
  const dim3 block(256);
  if (q.rows) {
#define CONV_ROWS(MODE)                                                                                                     \
  if (q.txlog >= 6) {                                                                                                       \
    if (bwd) hipLaunchKernelGGL((conv_rows_bwd_kernel<T, MODE, true>), q.grid, block, 0, s, p, q.txlog);                    \
    else hipLaunchKernelGGL((conv_rows_fwd_kernel<T, MODE, true>), q.grid, block, 0, s, p, q.txlog);                        \
  } else {                                                                                                                  \
    if (bwd) hipLaunchKernelGGL((conv_rows_bwd_kernel<T, MODE, false>), q.grid, block, 0, s, p, q.txlog);                   \
    else hipLaunchKernelGGL((conv_rows_fwd_kernel<T, MODE, false>), q.grid, block, 0, s, p, q.txlog);                       \
  }
    if (q.mode == ALIGNED) CONV_ROWS(ALIGNED)
    else if (q.mode == ANY) CONV_ROWS(ANY)
    else CONV_ROWS(SCALAR)
#undef CONV_ROWS
  } else if (bwd) {
    if (!q.vec) hipLaunchKernelGGL((conv_cl_bwd_kernel<T, false>), q.grid, block, 0, s, p);
    else if (q.run == 128) hipLaunchKernelGGL((conv_cl_bwd4_kernel<T, 128>), q.grid, block, 0, s, p);
    else if (q.run == 8) hipLaunchKernelGGL((conv_cl_bwd4_kernel<T, 8>), q.grid, block, 0, s, p);
    else hipLaunchKernelGGL((conv_cl_bwd4_kernel<T, RUN>), q.grid, block, 0, s, p);
  } else {
    if (!q.vec) hipLaunchKernelGGL((conv_cl_fwd_kernel<T, false>), q.grid, block, 0, s, p);
    else if (q.run == 8) hipLaunchKernelGGL((conv_cl_fwd4_kernel<T, 8>), q.grid, block, 0, s, p);
    else hipLaunchKernelGGL((conv_cl_fwd4_kernel<T, RUN>), q.grid, block, 0, s, p);
  }
  if (bwd && p.dw_part)
    hipLaunchKernelGGL(conv_reduce_kernel, dim3((p.dim * NSUM + 255) / 256), block, 0, s, p, q.nparts);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}

int dispatch(const CausalConvParams *p, bool bwd, mamba_stream_t stream) {
  int rc = check(p, bwd);
  if (rc != MAMBA_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (p->dtype) {
    case MAMBA_F32: return launch_conv<float>(*p, bwd, s);
    case MAMBA_BF16: return launch_conv<bf16_t>(*p, bwd, s);
    default: return launch_conv<f16_t>(*p, bwd, s);
  }
}

template <typename T> int launch_update(const CausalConvUpdateParams &p, hipStream_t s) {
  dim3 grid((p.dim + 255) / 256, p.batch);
  switch (p.state_dtype) {
    case MAMBA_F32: hipLaunchKernelGGL((conv_update_kernel<T, float>), grid, dim3(256), 0, s, p); break;
    case MAMBA_BF16: hipLaunchKernelGGL((conv_update_kernel<T, bf16_t>), grid, dim3(256), 0, s, p); break;
    case MAMBA_F16: hipLaunchKernelGGL((conv_update_kernel<T, f16_t>), grid, dim3(256), 0, s, p); break;
    default: return MAMBA_E_BADARG;
  }
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}

}  // namespace

extern "C" int causal_conv1d_fwd(const CausalConvParams *p, mamba_stream_t stream) { return dispatch(p, false, stream); }
extern "C" int causal_conv1d_bwd(const CausalConvParams *p, mamba_stream_t stream) { return dispatch(p, true, stream); }

extern "C" int causal_conv1d_bwd_nparts(const CausalConvParams *p) {
  if (!p || p->batch <= 0 || p->dim <= 0 || p->seqlen <= 0 || p->batch > 65535) return MAMBA_E_BADARG;
  Plan q{};
  const int rc = plan_conv(*p, true, q);
  return rc == MAMBA_OK ? q.nparts : rc;
}

extern "C" int causal_conv1d_update(const CausalConvUpdateParams *p, mamba_stream_t stream) {
  if (!p || !p->x || !p->conv_state || !p->weight || !p->out) return MAMBA_E_BADARG;
  if (p->batch <= 0 || p->dim <= 0 || p->seqlen <= 0 || p->state_len < 0) return MAMBA_E_BADARG;
  if (p->width < 2 || p->width > MAXW) return MAMBA_E_UNSUPPORTED;
  if (p->state_len < p->width - 1 || p->state_rows <= 0) return MAMBA_E_BADARG;
  if (!p->conv_state_indices && p->state_rows < p->batch) return MAMBA_E_BADARG;
  if (p->batch > 65535) return MAMBA_E_UNSUPPORTED;
  if (p->weight_dtype < MAMBA_F32 || p->weight_dtype > MAMBA_F16) return MAMBA_E_BADARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (p->dtype) {
    case MAMBA_F32: return launch_update<float>(*p, s);
    case MAMBA_BF16: return launch_update<bf16_t>(*p, s);
    case MAMBA_F16: return launch_update<f16_t>(*p, s);
    default: return MAMBA_E_BADARG;
  }
}

extern "C" int causal_conv1d_varlen_states(const CausalConvVarlenParams *p, mamba_stream_t stream) {
  if (!p || !p->x || !p->cu_seqlens || !p->states) return MAMBA_E_BADARG;
  if (p->nseq <= 0 || p->dim <= 0 || p->total < 0 || p->state_len <= 0) return MAMBA_E_BADARG;
  if (p->nseq > 65535) return MAMBA_E_UNSUPPORTED;
  hipStream_t s = static_cast<hipStream_t>(stream);
  dim3 grid((p->dim + 255) / 256, p->nseq);
  switch (p->dtype) {
    case MAMBA_F32: hipLaunchKernelGGL((conv_varlen_states_kernel<float>), grid, dim3(256), 0, s, *p); break;
    case MAMBA_BF16: hipLaunchKernelGGL((conv_varlen_states_kernel<bf16_t>), grid, dim3(256), 0, s, *p); break;
    case MAMBA_F16: hipLaunchKernelGGL((conv_varlen_states_kernel<f16_t>), grid, dim3(256), 0, s, *p); break;
    default: return MAMBA_E_BADARG;
  }
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}
