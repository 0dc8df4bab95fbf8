// Mamba-2 SSD forward for gfx950: chunk_cumsum, chunk_state, state_passing,
// bmm (C B^T) and chunk_scan.  The three dense contractions run on bf16 MFMA
// through the block-GEMM core of ssd_common.hpp; the other two are small
// streaming kernels.
#include "ssd_common.hpp"

namespace {

// ------------------------------------------------------------ chunk_cumsum
// One workgroup per (batch, chunk, 4 heads); thread = position inside the chunk, so loads of
// dt (head-contiguous) are 4 consecutive elements per thread and the stores of dt_out / dA_cumsum
// (position-contiguous) are coalesced.  (The kernel is a chain of short latencies, so it wants many small
// workgroups: 15.5 us with 16 heads per workgroup at batch 4 x 16 chunks x 80 heads, 11.1 with 4, 10.2 with 2, when each load was waited for
// before the next; 8.9 with 4 heads' loads in flight together.)  dt -> (+bias, softplus, clamp), zero past the end of the
// sequence; dA_cumsum = running sum of dt * A over the chunk (wave DPP scan + cross-wave offsets).
constexpr int CS_HT = 4;

DEVI float wave_incl_sum(float x) {
  x += dpp_f<DPP_ROW_SHR + 1>(0.f, x);
  x += dpp_f<DPP_ROW_SHR + 2>(0.f, x);
  x += dpp_f<DPP_ROW_SHR + 4>(0.f, x);
  x += dpp_f<DPP_ROW_SHR + 8>(0.f, x);
  x += dpp_f<DPP_ROW_BCAST15, 0xa>(0.f, x);
  x += dpp_f<DPP_ROW_BCAST31, 0xc>(0.f, x);
  return x;
}

__global__ __launch_bounds__(256) void chunk_cumsum_fwd_kernel(const SsdParams p) {
  __shared__ float wtot[4][CS_HT];
  const int H = p.nheads, nc = p.nchunks, Q = p.chunk_size;
  const int l = threadIdx.x, lane = l & 63, wave = l >> 6;
  const int c = blockIdx.x, h0 = blockIdx.y * CS_HT, b = blockIdx.z;
  const int t = c * Q + l;
  const bool live = l < Q && t < p.seqlen;
  float dtv[CS_HT], cs[CS_HT], A[CS_HT], bias[CS_HT];
  // every load before the first use of any: the type is asked for once, heads and positions past the end repeat the last
  const float *const bp = static_cast<const float *>(p.dt_bias ? p.dt_bias : p.A);
#pragma unroll
  for (int i = 0; i < CS_HT; ++i) {
    const int h = min(h0 + i, H - 1);
    A[i] = static_cast<const float *>(p.A)[h];
    bias[i] = bp[h];
  }
  auto load = [&](auto type) {
    const auto *row = reinterpret_cast<const decltype(type) *>(p.dt) + b * p.dt_bs + (int64_t)min(t, p.seqlen - 1) * p.dt_ls;
#pragma unroll
    for (int i = 0; i < CS_HT; ++i) dtv[i] = ld1(row + min(h0 + i, H - 1) * p.dt_hs);
  };
  switch (p.dt_dtype) {
    case MAMBA_BF16: load(bf16_t{}); break;
    case MAMBA_F16: load(f16_t{}); break;
    default: load(float{}); break;
  }
#pragma unroll
  for (int i = 0; i < CS_HT; ++i) {
    float dt = dtv[i];
    if (p.dt_bias) dt += bias[i];
    if (p.dt_softplus) dt = softplus_f(dt);
    dt = live ? fminf(fmaxf(dt, p.dt_min), p.dt_max) : 0.f;
    dtv[i] = dt;
    cs[i] = wave_incl_sum(dt * A[i]);
    if (lane == 63) wtot[wave][i] = cs[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < CS_HT; ++i) {
    const int h = h0 + i;
    float off = 0.f;
    for (int w = 0; w < wave; ++w) off += wtot[w][i];
    if (h < H && l < Q) {
      const int64_t o = (((int64_t)b * H + h) * nc + c) * Q + l;
      p.dt_out[o] = dtv[i];
      p.dA_cumsum[o] = cs[i] + off;
    }
  }
}

DEVI bool seq_same(const int32_t *seq, int a, int b) { return seq[a] == seq[b]; }

// --------------------------------------------------------------- bmm (CB)
// CB[b, c, g, l, s] = sum_n C[l, n] B[s, n] for s-tiles at or below the l-tile,
// zeroed where seq_idx differs.
template <typename T, bool SPLIT> __global__ __launch_bounds__(256) void bmm_chunk_fwd_kernel(const SsdParams p) {
  __shared__ GemmLds lds;
  const int tid = threadIdx.x;
  const int Q = p.chunk_size, N = p.dstate, L = p.seqlen, G = p.ngroups;
  // blockIdx.x enumerates the lower-triangular tile pairs (mt >= nt)
  int mt = 0, rem = blockIdx.x;
  while (rem > mt) { rem -= mt + 1; ++mt; }
  const int nt = rem;
  const int c = blockIdx.y, b = blockIdx.z / G, g = blockIdx.z % G;
  const int t0 = c * Q;
  const int64_t Cb = b * p.C_bs + g * p.C_gs, Bb = b * p.B_bs + g * p.B_gs;
  GemmAcc acc;
  acc.zero();
  const int qlim = min(Q, L - t0);
  const T *Ca = static_cast<const T *>(p.C) + Cb + (int64_t)(t0 + mt * GB) * p.C_ls;
  const T *Ba = static_cast<const T *>(p.B) + Bb + (int64_t)(t0 + nt * GB) * p.B_ls;
  const bool va = rows_aligned16(Ca, p.C_ls), vb = rows_aligned16(Ba, p.B_ls);
  block_gemm_pipe<SPLIT>(
      acc, lds, 0, N,
      KcStager<SPLIT, T>(lds.ah, lds.al, Ca, p.C_ls, qlim - mt * GB, N, nullptr, nullptr, va, tid),
      KcStager<SPLIT, T>(lds.bh, lds.bl, Ba, p.B_ls, qlim - nt * GB, N, nullptr, nullptr, vb, tid),
      tid);
  float *CB = p.CB + (((int64_t)b * p.nchunks + c) * G + g) * Q * Q;
  const int32_t *seq = p.seq_idx ? p.seq_idx + (int64_t)b * L + t0 : nullptr;
  acc_foreach(acc, tid, [&](int m, int n, float v) {
    const int l = mt * GB + m, s = nt * GB + n;
    if (l < Q && s < Q) {
      float o = v;
      if (seq && (t0 + l >= L || t0 + s >= L || seq[l] != seq[s])) o = 0.f;
      CB[(int64_t)l * Q + s] = o;
    }
    return v;
  });
}

// The weights w_s = dt_s exp(a_last - a_s) of a chunk's positions in its last sequence, 0 for the others; w[] is 256
// long, entry per thread.  OWN: the chunk's steps and their running sums are formed here, by the arithmetic of
// chunk_cumsum_fwd_kernel, and stored when `store` says so (a launch of its own costs ~5 us, as much as a short
// sequence's whole chunk_state: see ssd_combined_fwd_one).
DEVI void chunk_weights(const SsdParams &p, int b, int h, int c, bool own, bool store, float *w, float *wtot) {
  const int Q = p.chunk_size, L = p.seqlen, H = p.nheads, t0 = c * Q, qlim = min(Q, L - t0), s = threadIdx.x;
  float *dA = p.dA_cumsum + (((int64_t)b * H + h) * p.nchunks + c) * Q;
  float *dt = p.dt_out + (((int64_t)b * H + h) * p.nchunks + c) * Q;
  float a, a_last, step;
  if (own) {
    const int lane = s & 63, wave = s >> 6;
    step = 0.f;
    if (s < qlim) {
      step = ld_dyn(p.dt, b * p.dt_bs + (int64_t)(t0 + s) * p.dt_ls + h * p.dt_hs, p.dt_dtype);
      if (p.dt_bias) step += static_cast<const float *>(p.dt_bias)[h];
      if (p.dt_softplus) step = softplus_f(step);
      step = fminf(fmaxf(step, p.dt_min), p.dt_max);
    }
    const float cs = wave_incl_sum(step * static_cast<const float *>(p.A)[h]);
    if (lane == 63) wtot[wave] = cs;
    lds_barrier();
    float off = 0.f;
    for (int i = 0; i < wave; ++i) off += wtot[i];
    a = cs + off;
    // (the positions past the chunk's end, if any, have no steps: the running sum at Q - 1 is the last wave's)
    if (s == Q - 1) wtot[4] = a;
    lds_barrier();
    a_last = wtot[4];
    if (store && s < Q) dt[s] = step, dA[s] = a;
  } else {
    const int i = min(s, Q - 1);
    a = dA[i], a_last = dA[Q - 1], step = dt[i];
  }
  bool ok = s < qlim;
  if (p.seq_idx) {
    const int32_t *seq = p.seq_idx + (int64_t)b * L + t0;
    const int last = seq[qlim - 1];
    ok = ok && last >= 0 && seq[min(s, qlim - 1)] == last;
  }
  w[s] = ok ? fast_exp(fminf(a_last - a, 0.f)) * step : 0.f;
}

// ------------------------------------------------------------ chunk_state
// states[b, c, h, p, n] = sum_s x[s, p] B[s, n] exp(a_last - a_s) dt_s over the
// positions s of the chunk that belong to the sequence of its last position.
template <typename T, bool SPLIT> __global__ __launch_bounds__(256) void chunk_state_fwd_kernel(const SsdParams p, int own_cumsum) {
  __shared__ GemmLds lds;
  __shared__ float w[256], wtot[5];
  const int tid = threadIdx.x;
  const int Q = p.chunk_size, N = p.dstate, L = p.seqlen, P = p.headdim, H = p.nheads;
  const int ntn = cdiv(N, GB);
  const Block3 blk = xcd_block_heads(H);  // the tiles of one (chunk, head) share its x / g rows: same L2
  const int pt = blk.x / ntn, nt = blk.x % ntn;
  const int c = blk.y, b = blk.z / H, h = blk.z % H;
  const int g = h / (H / p.ngroups);
  const int t0 = c * Q;
  const int qlim = min(Q, L - t0);
  chunk_weights(p, b, h, c, own_cumsum != 0, blk.x == 0, w, wtot);
  const int64_t xb = b * p.x_bs + h * p.x_hs, Bb = b * p.B_bs + g * p.B_gs;
  GemmAcc acc;
  acc.zero();
  // A = x^T (rows p, k = position), B = (B w)^T (rows n, k = position): both row-contiguous sources
  const T *xa = static_cast<const T *>(p.x) + xb + (int64_t)t0 * p.x_ls + pt * GB;
  const T *Ba = static_cast<const T *>(p.B) + Bb + (int64_t)t0 * p.B_ls + nt * GB;
  const bool va = rows_aligned16(xa, p.x_ls), vb = rows_aligned16(Ba, p.B_ls);
  block_gemm_pipe<SPLIT>(  // the first barrier inside publishes w
      acc, lds, 0, qlim,
      TrStager<SPLIT, T>(lds.ah, lds.al, xa, p.x_ls, P - pt * GB, qlim, nullptr, nullptr, va, tid),
      TrStager<SPLIT, T>(lds.bh, lds.bl, Ba, p.B_ls, N - nt * GB, qlim, w, nullptr, vb, tid),
      tid);
  float *st = p.states + (((int64_t)b * p.nchunks + c) * H + h) * P * N;
  acc_foreach(acc, tid, [&](int m, int n, float v) {
    const int pp = pt * GB + m, nn = nt * GB + n;
    if (pp < P && nn < N) st[(int64_t)pp * N + nn] = v;
    return v;
  });
}

// The same product with a 64 x 128 tile per workgroup, for whole 128-state blocks of aligned operands
// and chunks of whole k steps (the last one of any length: RAGGED).
template <typename T, bool SPLIT, int FORM>
__global__ __launch_bounds__(256, FORM == WIDE_DEEP ? (SPLIT ? 2 : 3) : 1) void chunk_state_fwd_wide_kernel(const SsdParams p, int own_cumsum) {
  constexpr bool RAGGED = FORM != WIDE_WHOLE;
  __shared__ GemmLdsWide<SPLIT> lds;
  __shared__ float w[256], wtot[5];
  const int tid = threadIdx.x;
  const int Q = p.chunk_size, N = p.dstate, L = p.seqlen, P = p.headdim, H = p.nheads;
  const int ntn = N / WB;
  const Block3 blk = xcd_block_heads(H);
  const int pt = blk.x / ntn, nt = blk.x % ntn;
  const int c = blk.y, b = blk.z / H, h = blk.z % H;
  const int g = h / (H / p.ngroups);
  const int t0 = c * Q;
  const int qlim = min(Q, L - t0);
  const T *xa = static_cast<const T *>(p.x) + b * p.x_bs + h * p.x_hs + (int64_t)t0 * p.x_ls + pt * GB;
  const T *Ba = static_cast<const T *>(p.B) + b * p.B_bs + g * p.B_gs + (int64_t)t0 * p.B_ls + nt * WB;
  GemmAccWide acc;
  acc.zero();
  WideTrStager<SPLIT, T, 64, RAGGED> sa(lds.ah, lds.al, xa, p.x_ls, P - pt * GB, nullptr, tid, qlim);
  WideTrStager<SPLIT, T, WB, RAGGED> sb(lds.bh, lds.bl, Ba, p.B_ls, WB, w, tid, qlim);
  const int k_end = round_to_step(qlim);
  auto weights = [&] { chunk_weights(p, b, h, c, own_cumsum != 0, blk.x == 0, w, wtot); };
  // the first barrier inside the product publishes w
  if constexpr (FORM == WIDE_DEEP) {
    WideDeep<SPLIT, WIDE_PF, decltype(sa), decltype(sb)> deep(sa, sb, k_end);
    weights();
    deep.run(acc, lds, tid);
  } else {
    weights();
    block_gemm_wide<SPLIT>(acc, lds, k_end, sa, sb, tid);
  }
  float *st = p.states + (((int64_t)b * p.nchunks + c) * H + h) * P * N;
  store_wide_rows(acc, lds, st + (int64_t)pt * GB * N + nt * WB, N, P - pt * GB, tid);
}

// ---------------------------------------------------- chunk_state_varlen
// Packed batch (batch 1): state at the last position of every sequence i = [cu[i], cu[i+1]).
// out[i, h, p, n] = sum_{k in the last chunk, k >= start} x[k, p] B[k, n] exp(a_end - a_k) dt_k
//                 + exp(a_end) states[c, h, p, n] if the sequence began before that chunk,
// with `states` the state entering each chunk.  Empty sequences give zeros.
template <typename T, bool SPLIT>
__global__ __launch_bounds__(256) void chunk_state_varlen_kernel(const SsdParams p, const int32_t *cu, float *out) {
  __shared__ GemmLds lds;
  __shared__ float w[256];
  const int tid = threadIdx.x;
  const int Q = p.chunk_size, N = p.dstate, P = p.headdim, H = p.nheads;
  const int ntn = cdiv(N, GB);
  const int pt = blockIdx.x / ntn, nt = blockIdx.x % ntn;
  const int i = blockIdx.y, h = blockIdx.z;
  const int g = h / (H / p.ngroups);
  const int start = cu[i], end = min(cu[i + 1], p.seqlen);
  float *dst = out + ((int64_t)i * H + h) * P * N;
  GemmAcc acc;
  acc.zero();
  if (end > start) {
    const int c = (end - 1) / Q, t0 = c * Q;
    const int kstart = max(start - t0, 0), kend = end - t0;
    const float *dA = p.dA_cumsum + ((int64_t)h * p.nchunks + c) * Q;
    const float *dt = p.dt_out + ((int64_t)h * p.nchunks + c) * Q;
    const float a_end = dA[kend - 1];
    for (int k = tid; k < Q; k += 256)
      w[k] = (k >= kstart && k < kend) ? fast_exp(fminf(a_end - dA[k], 0.f)) * dt[k] : 0.f;
    const T *xa = static_cast<const T *>(p.x) + h * p.x_hs + (int64_t)t0 * p.x_ls + pt * GB;
    const T *Ba = static_cast<const T *>(p.B) + g * p.B_gs + (int64_t)t0 * p.B_ls + nt * GB;
    const bool va = rows_aligned16(xa, p.x_ls), vb = rows_aligned16(Ba, p.B_ls);
    block_gemm_pipe<SPLIT>(  // the first barrier inside publishes w
        acc, lds, kstart / GK * GK, kend,
        TrStager<SPLIT, T>(lds.ah, lds.al, xa, p.x_ls, P - pt * GB, kend, nullptr, nullptr, va, tid),
        TrStager<SPLIT, T>(lds.bh, lds.bl, Ba, p.B_ls, N - nt * GB, kend, w, nullptr, vb, tid),
        tid);
    if (start < t0) {
      const carried_t<T> *Hc = carried_states<T>(p) + ((int64_t)c * H + h) * P * N;
      const float sc = fast_exp(a_end);
      acc_foreach(acc, tid, [&](int m, int n, float v) {
        const int pp = pt * GB + m, nn = nt * GB + n;
        return (pp < P && nn < N) ? __builtin_fmaf(sc, ld1<carried_t<T>>(Hc + (int64_t)pp * N + nn), v) : v;
      });
    }
  }
  acc_foreach(acc, tid, [&](int m, int n, float v) {
    const int pp = pt * GB + m, nn = nt * GB + n;
    if (pp < P && nn < N) dst[(int64_t)pp * N + nn] = v;
    return v;
  });
}

// ---------------------------------------------------------- state_passing
// In place over `states`: slot c receives the state ENTERING chunk c; the state
// after the last chunk goes to final_states.  A thread owns W consecutive elements of the
// (headdim x dstate) state; the chunk loop is a serial recurrence, so the local states of the
// next SP_PF chunks are always in flight (the compiler cannot hoist those loads over the in-place
// stores by itself).  TABLE: the per-chunk decay factors are put in LDS before the loop; read one by one inside
// it they are scalar loads, each waited for with everything else the scalar unit has in flight, and with few rows
// per chunk (one long packed batch) that wait was the time of a step.
constexpr int SP_PF = 4;
constexpr size_t SP_TABLE_BYTES = 32768;

template <int W> struct VecF;
template <> struct VecF<1> {
  float v[1];
  DEVI void load(const float *p) { v[0] = *p; }
  DEVI void store(float *p) const { *p = v[0]; }
};
template <> struct VecF<4> {
  float v[4];
  DEVI void load(const float *p) {
    const f32x4 t = *reinterpret_cast<const f32x4 *>(p);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
  }
  DEVI void store(float *p) const { *reinterpret_cast<f32x4 *>(p) = f32x4{v[0], v[1], v[2], v[3]}; }
};

// CT float: in place, slot c of `states` receives the state entering chunk c.  CT bf16_t: that state goes to
// states_lp in bf16 and `states` is only read.
template <int W, typename CT, bool TABLE> __global__ __launch_bounds__(256) void state_passing_fwd_kernel(const SsdParams p) {
  extern __shared__ float sp_decay[];
  const int PN = p.headdim * p.dstate, H = p.nheads, nc = p.nchunks, Q = p.chunk_size, L = p.seqlen;
  const int e = (blockIdx.x * 256 + threadIdx.x) * W;
  const int h = blockIdx.y, b = blockIdx.z;
  const float *dA = p.dA_cumsum + ((int64_t)b * H + h) * nc * Q;
  const int32_t *seq = p.seq_idx ? p.seq_idx + (int64_t)b * L : nullptr;
  auto decay_of = [&](int c) {  // carried-state factor of chunk c: 0 across a sequence boundary
    float scale = fast_exp(dA[c * Q + Q - 1]);
    if (seq) {
      const int seq_new = seq[min((c + 1) * Q, L) - 1], seq_prev = c > 0 ? seq[c * Q - 1] : 0;
      if (seq_new != seq_prev) scale = 0.f;
    }
    return scale;
  };
  if constexpr (TABLE) {
    for (int c = threadIdx.x; c < nc; c += 256) sp_decay[c] = decay_of(c);
    lds_barrier();
  }
  if (e >= PN) return;
  auto decay = [&](int c) { return TABLE ? sp_decay[c] : decay_of(c); };
  VecF<W> s;
#pragma unroll
  for (int i = 0; i < W; ++i) s.v[i] = 0.f;
  if (p.initial_states) s.load(p.initial_states + ((int64_t)b * H + h) * PN + e);
  auto slot = [&](int c) { return p.states + (((int64_t)b * nc + c) * H + h) * PN + e; };
  VecF<W> local[SP_PF];
  float scale[SP_PF];
#pragma unroll
  for (int j = 0; j < SP_PF; ++j) {
    local[j].load(slot(min(j, nc - 1)));
    scale[j] = decay(min(j, nc - 1));
  }
  // one chunk, its local state in slot j of the prefetch; `more`: request chunk c + SP_PF into the slot
  auto step = [&](int c, int j, bool more) {
    if constexpr (std::is_same_v<CT, float>) {
      s.store(slot(c));
    } else {
      CT *o = static_cast<CT *>(p.states_lp) + (((int64_t)b * nc + c) * H + h) * PN + e;
      if constexpr (W == 4) {
        *reinterpret_cast<u32x2 *>(o) = u32x2{pack_bf16(s.v[0], s.v[1]), pack_bf16(s.v[2], s.v[3])};
      } else {
        st1<CT>(o, s.v[0]);
      }
    }
    const VecF<W> loc = local[j];
    const float sc = scale[j];
    if (more) {  // past the last chunk the loads repeat it and nobody uses them: no branch, so no register copies
                 // (which would wait for the loads in flight) where the paths meet
      const int cn = min(c + SP_PF, nc - 1);
      local[j].load(slot(cn));
      scale[j] = decay(cn);
    }
#pragma unroll
    for (int i = 0; i < W; ++i) s.v[i] = __builtin_fmaf(sc, s.v[i], loc.v[i]);
  };
  // whole groups of SP_PF chunks without a branch inside, then the chunks left over from what the slots hold
  int c0 = 0;
  for (; c0 + SP_PF <= nc; c0 += SP_PF) {
#pragma unroll
    for (int j = 0; j < SP_PF; ++j) step(c0 + j, j, true);
  }
#pragma unroll
  for (int j = 0; j < SP_PF - 1; ++j)
    if (c0 + j < nc) step(c0 + j, j, false);
  s.store(p.final_states + ((int64_t)b * H + h) * PN + e);
}

// ------------------------------------------- chunk states and state passing in one pass
// bf16, headdim 64, 128 states, chunks of Q = 64 NS positions that tile the sequence: four waves per (batch, head) walk the
// sequence once, HH heads of a group to a workgroup.  Per chunk they write the state ENTERING the chunk (bf16, what the scan and
// the backward pass read), form the chunk's own state S_c (128 states x 64, k = position) and carry H <- decay_c H + S_c in
// fp32 registers; after the last chunk H is final_states.  The fp32 states of the chunks never exist in memory (4 x 4096
// positions, 80 heads: 168 MB written and read again), and the recurrence over the chunks costs no pass of its own.
// What bounds it is the rate at which a CU takes in rows (30 - 40 GB/s of x and B, whether they pass through registers or not
// and however many are in flight: a walk without its products takes 2.2 - 2.6 us per chunk of 256, two of them on a CU twice
// that).  So rows go to LDS as they are, by asynchronous loads that are two or three stages of 64 positions ahead in a ring of
// stages, and two walks on one CU share those of B (HH = 2).  A wave owns 32 states: it multiplies its columns of B with
// the weights of their positions as it reads them (nobody reads them twice), and all four read x.  States leave as 16 bytes a
// lane (as 8 the same walk took 81 us where it takes 71).  The weights of chunk c + 1 are formed while chunk c is multiplied.
// No branch surrounds a load or store of the walk: past the end the last stage comes once more, and each wait counts what was
// issued behind the rows that it is for.  Rows through registers, the weighted ones written to LDS (before) / this, 80 heads
// x 4096 positions: batch 2 59 / 47 us, batch 3 64 / 48, batch 4 91 / 71, batch 8 169 / 152; 128 heads in 8 groups x 2 x 32768
// 451 / 423.
template <int HH, int NS, bool HAS_SEQ> __global__ __launch_bounds__(256 * HH, 2) void chunk_state_passing_fwd_kernel(const SsdParams p) {
  constexpr int NW = 4 * HH, KS = 64, Q = KS * NS, P = 64, N = 128, XH = KS * P * 2, XB = HH * XH, SB = XB + KS * N * 2, RING = HH == 1 ? 3 : 4, AHEAD = RING - 1;
  constexpr int LOADS = SB / 1024 / NW, STORES = 4, TABLE = HAS_SEQ ? 5 : 3;  // of a wave: per stage; per chunk
  constexpr auto behind = [](int st) {
    int n = (AHEAD - 1) * LOADS;
    for (int d = 1; d <= AHEAD; ++d) n += ((st - d + 4 * NS) % NS == NS - 1 ? STORES : 0) + (d < AHEAD && (st - d + 4 * NS) % NS == 0 ? TABLE : 0);
    return n;
  };
  typedef __attribute__((address_space(3))) i16x4_t *lds_tr;
  typedef __attribute__((address_space(3))) f32x4 *lds_f4;
  typedef short i16x8_t __attribute__((ext_vector_type(8)));
  __shared__ __align__(256) char ring[RING * SB];
  __shared__ __align__(16) float wtab[HH][2][Q];
  __shared__ __align__(256) float raw[NW][TABLE][64];  // a wave's entries of dA_cumsum, its last one, dt, the sequence and the last one
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, gq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), hd = wave >> 2, wn = wave & 3;
  const int L = p.seqlen, H = p.nheads, nc = p.nchunks;
  const int id = xcd_linear_block() * HH + hd;
  const int h = id % H, b = id / H;
  const int g = h / (H / p.ngroups);
  const float *dA = p.dA_cumsum + ((int64_t)b * H + h) * nc * Q;
  const float *dtp = p.dt_out + ((int64_t)b * H + h) * nc * Q;
  const int32_t *seq = HAS_SEQ ? p.seq_idx + (int64_t)b * L : nullptr;
  // w_s = dt_s exp(a_last - a_s) for the positions of the chunk's last sequence, else 0; entry min(tid, Q - 1).  The decay of a
  // carried state over the chunk is 0 across a sequence boundary.  What they are formed of comes the same way as the rows, for
  // the compiler would wait for loads of its own until nothing at all is in flight.
  const int pos = min(wn * 64 + lane, Q - 1);
  const uint32_t raw_at = lds_address(&raw[wave][0][0]), ts = pos * 4;
  float decay;
  int s_before = 0;
  auto table_request = [&](int c) {
    load_async4(dA + c * Q, ts, raw_at);
    load_async4(dA + c * Q, (Q - 1) * 4, raw_at + 256);
    load_async4(dtp + c * Q, ts, raw_at + 512);
    if (HAS_SEQ) {
      load_async4(seq + c * Q, ts, raw_at + 768);
      load_async4(seq + c * Q, (Q - 1) * 4, raw_at + 1024);
    }
  };
  auto table_write = [&](int c) {
    const float a = raw[wave][0][lane], a_last = raw[wave][1][lane], dt = raw[wave][2][lane];
    float v = fast_exp(fminf(a_last - a, 0.f)) * dt;
    decay = fast_exp(a_last);
    if constexpr (HAS_SEQ) {
      const int sid = __float_as_int(raw[wave][3][lane]), last = __float_as_int(raw[wave][4][lane]);
      v = last >= 0 && sid == last ? v : 0.f;
      decay = last == s_before ? decay : 0.f;
      s_before = last;
    }
    if (wn * 64 < Q) wtab[hd][c & 1][pos] = v;
  };

  // rows -> LDS, 16 bytes a lane: 8 rows of x or 4 of B per instruction.  Units of 32 bytes are permuted within a row, so that
  // the transposing reads of 16 rows meet in no bank.
  const char *x_at = (const char *)(static_cast<const bf16_t *>(p.x) + b * p.x_bs + h * p.x_hs) + (lane >> 3) * (2 * p.x_ls) +
                     ((lane & 7) ^ (lane >> 4) << 1) * 16;
  const char *B_at = (const char *)(static_cast<const bf16_t *>(p.B) + b * p.B_bs + g * p.B_gs) + (lane >> 4) * (2 * p.B_ls) +
                     ((lane & 15) ^ ((wave & 1) * 4 + (lane >> 4)) << 1) * 16;
  const uint32_t lds0 = lds_address(&ring[0]), lds_end = lds0 + RING * SB;
  auto request = [&](int pos, uint32_t lds) {
#pragma unroll
    for (int q = 0; q < KS / 32; ++q) load_async16(x_at + (pos + (q * 4 + wn) * 8) * (2 * p.x_ls), lds + hd * XH + (q * 4 + wn) * 1024);
#pragma unroll
    for (int q = 0; q < KS / 4 / NW; ++q) load_async16(B_at + (pos + (q * NW + wave) * 4) * (2 * p.B_ls), lds + XB + (q * NW + wave) * 1024);
  };
  table_request(0);
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) request(min(k * KS, L - KS), lds0 + k * SB);

  // H: rows (states) 32 wave + 16 tn + 4 gq + r, columns 16 pt + j
  f32x4 Hs[2][4], acc[2][4];
  const int64_t own = j * N + wn * 32 + gq * 4;  // (+ 16 tn, + 16 N pt)
#pragma unroll
  for (int tn = 0; tn < 2; ++tn)
#pragma unroll
    for (int pt = 0; pt < 4; ++pt) Hs[tn][pt] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (p.initial_states) {
    const float *init = p.initial_states + ((int64_t)b * H + h) * P * N + own;
#pragma unroll
    for (int tn = 0; tn < 2; ++tn)
#pragma unroll
      for (int pt = 0; pt < 4; ++pt)
#pragma unroll
        for (int r = 0; r < 4; ++r) Hs[tn][pt][r] = init[pt * 16 * N + tn * 16 + r];
  }
  async_done<0>();  // (the first AHEAD stages)
  table_write(0);

  GLOBAL_AS char *carried = (GLOBAL_AS char *)(static_cast<bf16_t *>(p.states_lp) + ((int64_t)b * nc * H + h) * P * N + j * N + wn * 32 + (gq & 1) * 16 + (gq & 2) * 4);
  const int rr = 4 * gq + (j >> 2);  // this lane's row of a patch, and its place in it
  const uint32_t xo = hd * XH + rr * 128 + (j & 3) * 8 + (rr >> 1 & 3) * 32, Bo = XB + rr * 256 + (j & 3) * 8 + ((rr & 7) ^ (wn * 2)) * 32;
  uint32_t here = lds0, there = lds0 + AHEAD * SB;
#pragma unroll 1
  for (int c = 0; c < nc; ++c) {
#pragma unroll
    for (int tn = 0; tn < 2; ++tn)
#pragma unroll
      for (int pt = 0; pt < 4; ++pt) acc[tn][pt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t w_at = lds_address(&wtab[hd][c & 1][4 * gq]);
    const float d = decay;
#pragma unroll
    for (int st = 0; st < NS; ++st) {
      // behind the rows of this stage are those of the AHEAD - 1 next, and what the chunks that ended and began meanwhile
      // stored and asked for (the first AHEAD stages wait for nothing: they are there)
      switch (st) {
        case 0: async_done<behind(0)>(); break;
        case 1: async_done<behind(1)>(); break;
        case 2: async_done<behind(2)>(); break;
        default: async_done<behind(3)>(); break;
      }
      lds_barrier();  // they are there in all waves, and nobody reads the stage before any more
      if (st == 0) table_request(min(c + 1, nc - 1));
      request(min(c * Q + (st + AHEAD) * KS, L - KS), there);
#pragma unroll
      for (int k = 0; k < KS; k += 32) {
        const f32x4 w0 = *(lds_f4)(uintptr_t)(w_at + (st * KS + k) * 4), w1 = *(lds_f4)(uintptr_t)(w_at + (st * KS + k + 16) * 4);
        auto patches = [&](uint32_t at, int row) {
          const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)at);
          const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)(at + 16 * row));
          return (i16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        bf16x8_t bw[2];
#pragma unroll
        for (int tn = 0; tn < 2; ++tn) {
          const u32x4 v = __builtin_bit_cast(u32x4, patches(here + (Bo ^ (tn * 32)) + k * 256, 256));
          bw[tn] = __builtin_bit_cast(bf16x8_t, u32x4{pack_bf16(bf16_lo(v.x) * w0[0], bf16_hi(v.x) * w0[1]), pack_bf16(bf16_lo(v.y) * w0[2], bf16_hi(v.y) * w0[3]),
                                                      pack_bf16(bf16_lo(v.z) * w1[0], bf16_hi(v.z) * w1[1]), pack_bf16(bf16_lo(v.w) * w1[2], bf16_hi(v.w) * w1[3])});
        }
#pragma unroll
        for (int pt = 0; pt < 4; ++pt) {
          const bf16x8_t xf = __builtin_bit_cast(bf16x8_t, patches(here + (xo ^ (pt * 32)) + k * 128, 128));
#pragma unroll
          for (int tn = 0; tn < 2; ++tn) acc[tn][pt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[tn], xf, acc[tn][pt], 0, 0, 0);
        }
      }
      here = here + SB == lds_end ? lds0 : here + SB;
      there = there + SB == lds_end ? lds0 : there + SB;
    }
    async_done<NS * LOADS>();
    table_write(c + 1);  // read from the next stage's barrier on; last read a chunk ago
    // 16 bytes a lane: the even rows of lanes take the values of two rows of the first tile, the odd ones those of the second
#pragma unroll
    for (int pt = 0; pt < 4; ++pt) {
      const f32x4 u = Hs[0][pt], v = Hs[1][pt];
      const auto lo = __builtin_amdgcn_permlane16_swap(pack_bf16(u[0], u[1]), pack_bf16(v[0], v[1]), false, false);
      const auto hi = __builtin_amdgcn_permlane16_swap(pack_bf16(u[2], u[3]), pack_bf16(v[2], v[3]), false, false);
      *(GLOBAL_AS u32x4 *)(carried + pt * (32 * N)) = u32x4{(uint32_t)lo[0], (uint32_t)hi[0], (uint32_t)lo[1], (uint32_t)hi[1]};
#pragma unroll
      for (int tn = 0; tn < 2; ++tn)
#pragma unroll
        for (int r = 0; r < 4; ++r) Hs[tn][pt][r] = Hs[tn][pt][r] * d + acc[tn][pt][r];
    }
    carried += (int64_t)H * P * N * 2;
  }
  async_done<0>();  // (the requests past the end)
  float *last = p.final_states + ((int64_t)b * H + h) * P * N + own;
#pragma unroll
  for (int pt = 0; pt < 4; ++pt)
#pragma unroll
    for (int tn = 0; tn < 2; ++tn) *reinterpret_cast<f32x4 *>(last + pt * 16 * N + tn * 16) = Hs[tn][pt];
}

// ------------------------------------------------------------- chunk_scan
// out[l, p] = exp(a_l) [seq_l == seq before the chunk] sum_n C[l, n] Hc[p, n]
//           + sum_{s <= l} CB[l, s] exp(a_l - a_s) dt_s x[s, p] + D x[l, p];   out *= silu(z)
// One 64 x 64 tile (l, p) per workgroup: both products run through the software-pipelined block core, the second one's
// A operand (CB with the decay and the step) weighted on its way to LDS.  (Element by element from the functors of the
// unpipelined core every k step waited for its own loads: 56 us for 339 positions of 32 heads in fp16, 78 us for 1408
// of 48.)
template <bool SPLIT> struct DecayStager : KcStager<SPLIT, float> {
  using Base = KcStager<SPLIT, float>;
  const float *a, *dt;  // of the chunk
  int l0;               // the tile's first position
  DEVI DecayStager(Base base, const float *a_, const float *dt_, int l0_) : Base(base), a(a_), dt(dt_), l0(l0_) {}
  template <bool FAST> DEVI void commit(int k0) {
    const int r = this->t >> 2, k8 = (this->t & 3) * 8, l = l0 + r;
    const bool ok = r < this->rows_valid && k0 + k8 < this->k_valid;
    float v[8];
    this->q.unpack(v);
    const float al = a[min(l, 255)];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = k0 + k8 + e, kc = min(k, 255);
      v[e] = k <= l ? v[e] * fast_exp(fminf(al - a[kc], 0.f)) * dt[kc] : 0.f;
    }
    put8<SPLIT>(this->hi, this->lo, tile_off(r, k8), v, ok);
  }
};
template <typename T, bool SPLIT> __global__ __launch_bounds__(256) void chunk_scan_fwd_kernel(const SsdParams p) {
  __shared__ GemmLds lds;
  __shared__ float a_s[256], dt_s[256], rscale[GB];
  const int tid = threadIdx.x;
  const int Q = p.chunk_size, N = p.dstate, L = p.seqlen, P = p.headdim, H = p.nheads, G = p.ngroups;
  const int ntp = cdiv(P, GB);
  const int mt = blockIdx.x / ntp, pt = blockIdx.x % ntp;
  const int c = blockIdx.y, b = blockIdx.z / H, h = blockIdx.z % H;
  const int g = h / (H / G);
  const int t0 = c * Q;
  const int qlim = min(Q, L - t0);
  if (mt * GB >= qlim) return;
  const float *dA = p.dA_cumsum + (((int64_t)b * H + h) * p.nchunks + c) * Q;
  const float *dt = p.dt_out + (((int64_t)b * H + h) * p.nchunks + c) * Q;
  const int32_t *seq = p.seq_idx ? p.seq_idx + (int64_t)b * L + t0 : nullptr;
  a_s[tid] = tid < Q ? dA[tid] : 0.f;
  dt_s[tid] = tid < Q ? dt[tid] : 0.f;
  if (tid < GB) {
    const int l = mt * GB + tid;
    float sc = 0.f;
    if (l < qlim) {
      bool ok = true;
      if (seq) {
        const int prev = c > 0 ? seq[-1] : 0;
        ok = seq[l] == prev;
      }
      if (ok) sc = fast_exp(dA[l]);
    }
    rscale[tid] = sc;
  }
  const int64_t xb = b * p.x_bs + h * p.x_hs, Cb = b * p.C_bs + g * p.C_gs;
  const carried_t<T> *Hc = carried_states<T>(p) + (((int64_t)b * p.nchunks + c) * H + h) * P * N;
  const float *CB = p.CB + (((int64_t)b * p.nchunks + c) * G + g) * Q * Q;
  GemmAcc acc;
  acc.zero();
  {  // carried state -> outputs: A = C rows (l, n), B = Hc rows (p, n)
    const T *Ca = static_cast<const T *>(p.C) + Cb + (int64_t)(t0 + mt * GB) * p.C_ls;
    const carried_t<T> *Ha = Hc + (int64_t)pt * GB * N;
    block_gemm_pipe<SPLIT>(  // the first barrier inside publishes the tables
        acc, lds, 0, N,
        KcStager<SPLIT, T>(lds.ah, lds.al, Ca, p.C_ls, qlim - mt * GB, N, nullptr, nullptr, rows_aligned16(Ca, p.C_ls), tid),
        KcStager<SPLIT, carried_t<T>>(lds.bh, lds.bl, Ha, N, P - pt * GB, N, nullptr, nullptr, rows_aligned16(Ha, N), tid),
        tid);
    acc_foreach(acc, tid, [&](int m, int n, float v) { return v * rscale[m]; });
  }
  {  // inside the chunk, causal: A = CB rows (l, s) weighted, B = x^T (p, s)
    const int kmax = min((mt + 1) * GB, qlim);
    const float *CBa = CB + (int64_t)mt * GB * Q;
    const T *xa = static_cast<const T *>(p.x) + xb + (int64_t)t0 * p.x_ls + pt * GB;
    // (CB's rows are readable to their end; past kmax x counts as 0)
    DecayStager<SPLIT> sa(KcStager<SPLIT, float>(lds.ah, lds.al, CBa, Q, qlim - mt * GB, Q, nullptr, nullptr, rows_aligned16(CBa, Q), tid),
                          a_s, dt_s, mt * GB);
    block_gemm_pipe<SPLIT>(
        acc, lds, 0, kmax, sa,
        TrStager<SPLIT, T>(lds.bh, lds.bl, xa, p.x_ls, P - pt * GB, kmax, nullptr, nullptr, rows_aligned16(xa, p.x_ls), tid), tid);
  }
  const float *Dp = static_cast<const float *>(p.D);
  acc_foreach(acc, tid, [&](int m, int n, float v) {
    const int l = mt * GB + m, pp = pt * GB + n;
    if (l >= qlim || pp >= P) return v;
    float o = v;
    if (Dp) {
      const float d = p.D_has_hdim ? Dp[h * P + pp] : Dp[h];
      o = __builtin_fmaf(d, ldg<T>(p.x, xb + (int64_t)(t0 + l) * p.x_ls + pp), o);
    }
    const int64_t oi = b * p.out_bs + (int64_t)(t0 + l) * p.out_ls + h * p.out_hs + pp;
    if (p.z) {
      if (p.out_x) stg<T>(p.out_x, oi, o);
      const float z = ldg<T>(p.z, b * p.z_bs + (int64_t)(t0 + l) * p.z_ls + h * p.z_hs + pp);
      o *= z * sigmoid_f(z);
    }
    stg<T>(p.out, oi, o);
    return v;
  });
}

// ------------------------------------------------------------------ launch
int check(const SsdParams *p) {
  if (!p || !p->x || !p->dt || !p->A || !p->B || !p->C) return MAMBA_E_BADARG;
  if (p->batch <= 0 || p->seqlen <= 0 || p->nheads <= 0 || p->headdim <= 0 || p->dstate <= 0 || p->ngroups <= 0 ||
      p->chunk_size <= 0)
    return MAMBA_E_BADARG;
  if (p->nheads % p->ngroups != 0) return MAMBA_E_BADARG;
  if (p->nchunks != (p->seqlen + p->chunk_size - 1) / p->chunk_size) return MAMBA_E_BADARG;
  if (p->chunk_size > 256 || p->dstate > 256 || p->headdim > 256) return MAMBA_E_UNSUPPORTED;
  if ((int64_t)p->batch * p->nheads > 65535 || p->nchunks > 65535) return MAMBA_E_UNSUPPORTED;
  if (p->dtype != MAMBA_F32 && p->dtype != MAMBA_BF16 && p->dtype != MAMBA_F16) return MAMBA_E_BADARG;
  if (p->dt_dtype != MAMBA_F32 && p->dt_dtype != MAMBA_BF16 && p->dt_dtype != MAMBA_F16) return MAMBA_E_BADARG;
  return MAMBA_OK;
}
int launched() { return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH; }

#define SSD_DISPATCH(KERNEL, GRID)                                                                   \
  switch (p->dtype) {                                                                                \
    case MAMBA_BF16: hipLaunchKernelGGL((KERNEL<bf16_t, false>), GRID, dim3(256), 0, s, *p); break;  \
    case MAMBA_F16: hipLaunchKernelGGL((KERNEL<f16_t, true>), GRID, dim3(256), 0, s, *p); break;     \
    default: hipLaunchKernelGGL((KERNEL<float, true>), GRID, dim3(256), 0, s, *p); break;            \
  }

}  // namespace

static int ssd_chunk_cumsum_fwd_one(const SsdParams *p, mamba_stream_t stream) {
  int rc = check(p);
  if (rc) return rc;
  if (!p->dt_out || !p->dA_cumsum) return MAMBA_E_BADARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  dim3 grid(p->nchunks, (p->nheads + CS_HT - 1) / CS_HT, p->batch);
  hipLaunchKernelGGL(chunk_cumsum_fwd_kernel, grid, dim3(256), 0, s, *p);
  return launched();
}

static int ssd_bmm_chunk_fwd_one(const SsdParams *p, mamba_stream_t stream) {
  int rc = check(p);
  if (rc) return rc;
  if (!p->CB) return MAMBA_E_BADARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int nt = (p->chunk_size + GB - 1) / GB;
  dim3 grid(nt * (nt + 1) / 2, p->nchunks, p->batch * p->ngroups);
  SSD_DISPATCH(bmm_chunk_fwd_kernel, grid)
  return launched();
}

static int ssd_chunk_state_fwd_with(const SsdParams *p, mamba_stream_t stream, int own_cumsum) {
  int rc = check(p);
  if (rc) return rc;
  if (!p->states || !p->dt_out || !p->dA_cumsum) return MAMBA_E_BADARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  {
    // whole 128-state blocks, 16-byte aligned x / B rows, headdim in whole groups of 8, whole k steps
    const bool wide = p->dstate % WB == 0 && p->headdim % 8 == 0 && whole_k_steps(p) &&
                      wide_operand_ok(p->x, p->dtype, p->x_bs, p->x_ls, p->x_hs) &&
                      wide_operand_ok(p->B, p->dtype, p->B_bs, p->B_ls, p->B_gs);
    if (wide) {
      dim3 grid(((p->headdim + GB - 1) / GB) * (p->dstate / WB), p->nchunks, p->batch * p->nheads);
      const int form = wide_form(p, (int64_t)grid.x * grid.y * grid.z);
      SSD_DISPATCH_FORM(chunk_state_fwd_wide_kernel, grid, form, *p, own_cumsum)
      return launched();
    }
  }
  dim3 grid(((p->headdim + GB - 1) / GB) * ((p->dstate + GB - 1) / GB), p->nchunks, p->batch * p->nheads);
  switch (p->dtype) {
    case MAMBA_BF16: hipLaunchKernelGGL((chunk_state_fwd_kernel<bf16_t, false>), grid, dim3(256), 0, s, *p, own_cumsum); break;
    case MAMBA_F16: hipLaunchKernelGGL((chunk_state_fwd_kernel<f16_t, true>), grid, dim3(256), 0, s, *p, own_cumsum); break;
    default: hipLaunchKernelGGL((chunk_state_fwd_kernel<float, true>), grid, dim3(256), 0, s, *p, own_cumsum); break;
  }
  return launched();
}
static int ssd_chunk_state_fwd_one(const SsdParams *p, mamba_stream_t stream) { return ssd_chunk_state_fwd_with(p, stream, 0); }

extern "C" int ssd_chunk_state_varlen(const SsdParams *p, const int32_t *cu_seqlens, int nseq, float *varlen_states,
                                      mamba_stream_t stream) {
  int rc = check(p);
  if (rc) return rc;
  if (!p->dt_out || !p->dA_cumsum || !cu_seqlens || !varlen_states) return MAMBA_E_BADARG;
  if (!(p->dtype == MAMBA_BF16 ? p->states_lp : (void *)p->states)) return MAMBA_E_BADARG;  // the carried states
  if (p->batch != 1 || nseq < 0 || nseq > 65535) return MAMBA_E_BADARG;
  if (nseq == 0) return MAMBA_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  dim3 grid(((p->headdim + GB - 1) / GB) * ((p->dstate + GB - 1) / GB), nseq, p->nheads);
  switch (p->dtype) {
    case MAMBA_BF16:
      hipLaunchKernelGGL((chunk_state_varlen_kernel<bf16_t, false>), grid, dim3(256), 0, s, *p, cu_seqlens, varlen_states);
      break;
    case MAMBA_F16:
      hipLaunchKernelGGL((chunk_state_varlen_kernel<f16_t, true>), grid, dim3(256), 0, s, *p, cu_seqlens, varlen_states);
      break;
    default:
      hipLaunchKernelGGL((chunk_state_varlen_kernel<float, true>), grid, dim3(256), 0, s, *p, cu_seqlens, varlen_states);
      break;
  }
  return launched();
}

static int ssd_state_passing_fwd_one(const SsdParams *p, mamba_stream_t stream) {
  int rc = check(p);
  if (rc) return rc;
  if (!p->states || !p->final_states || !p->dA_cumsum) return MAMBA_E_BADARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int PN = p->headdim * p->dstate;
  auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const bool lp = p->dtype == MAMBA_BF16;
  if (lp && !p->states_lp) return MAMBA_E_BADARG;
  const size_t tbytes = (size_t)p->nchunks * sizeof(float);
  const bool table = tbytes <= SP_TABLE_BYTES;
  if (PN % 4 == 0 && al16(p->states) && al16(p->final_states) && al16(p->initial_states) && al16(p->states_lp)) {
    dim3 grid((PN / 4 + 255) / 256, p->nheads, p->batch);
    if (table) {
      if (lp) hipLaunchKernelGGL((state_passing_fwd_kernel<4, bf16_t, true>), grid, dim3(256), tbytes, s, *p);
      else hipLaunchKernelGGL((state_passing_fwd_kernel<4, float, true>), grid, dim3(256), tbytes, s, *p);
    } else {
      if (lp) hipLaunchKernelGGL((state_passing_fwd_kernel<4, bf16_t, false>), grid, dim3(256), 0, s, *p);
      else hipLaunchKernelGGL((state_passing_fwd_kernel<4, float, false>), grid, dim3(256), 0, s, *p);
    }
  } else {
    dim3 grid((PN + 255) / 256, p->nheads, p->batch);
    if (lp) hipLaunchKernelGGL((state_passing_fwd_kernel<1, bf16_t, false>), grid, dim3(256), 0, s, *p);
    else hipLaunchKernelGGL((state_passing_fwd_kernel<1, float, false>), grid, dim3(256), 0, s, *p);
  }
  return launched();
}

static int ssd_chunk_scan_fwd_one(const SsdParams *p, mamba_stream_t stream) {
  int rc = check(p);
  if (rc) return rc;
  if (!p->CB || !p->out || !p->dt_out || !p->dA_cumsum) return MAMBA_E_BADARG;
  if (!(p->dtype == MAMBA_BF16 ? p->states_lp : (void *)p->states)) return MAMBA_E_BADARG;  // the carried states
  hipStream_t s = static_cast<hipStream_t>(stream);
  dim3 grid(((p->chunk_size + GB - 1) / GB) * ((p->headdim + GB - 1) / GB), p->nchunks, p->batch * p->nheads);
  SSD_DISPATCH(chunk_scan_fwd_kernel, grid)
  return launched();
}

// chunk_state + state_passing in one launch (chunk_state_passing_fwd_kernel): the shapes it is compiled for, whole
// chunks, 16-byte aligned operands.
static bool chunk_state_passing_shapes_ok(const SsdParams *p) {
  auto al16 = [](const void *q) { return q && (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  return p->dtype == MAMBA_BF16 && p->headdim == 64 && p->dstate == WB && (p->chunk_size == 256 || p->chunk_size == 128) &&
         p->seqlen % p->chunk_size == 0 && (int64_t)p->nheads * p->batch <= INT32_MAX / 256 &&
         al16(p->states_lp) && al16(p->final_states) && p->dt_out && p->dA_cumsum &&
         wide_operand_ok(p->x, p->dtype, p->x_bs, p->x_ls, p->x_hs) && wide_operand_ok(p->B, p->dtype, p->B_bs, p->B_ls, p->B_gs);
}
// The combined forward pass takes it where there are enough (batch, head) pairs for one workgroup each to keep the
// chip busy: a workgroup takes ~3 us per chunk of 256 whatever their number, the two-kernel path ~24 ns per (batch, head, chunk).
// Walk / two kernels: 128 pairs x 4096 positions 46.8 / 47.9 us, x 2048 in chunks of 128 33.2 / 36.2, x 16384 in 8 groups
// 198 / 199; 160 pairs x 4096 47 / 52, x 512 in chunks of 128 12.6 / 21; 176 pairs in 8 groups 48 / 67; 240 pairs 48 / 95; 320
// 71 / 128; 192 pairs x 262144 in chunks of 128 3960 / 8073; one packed row of 64 heads x 32768 positions 388 / 202.
// With fewer than three pairs to four CUs, only where the two kernels need a launch for the steps' sums as well (sums_in_states,
// below): the whole forward pass of 128 pairs x 2048 positions 70.2 / 69.8, x 512 in chunks of 128 27.2 / 27.9 with the walk.
static bool sums_in_states(const SsdParams *p) { return (int64_t)p->nchunks * p->batch * p->nheads <= 8 * (int64_t)cu_count(); }
static bool chunk_state_passing_pays(const SsdParams *p) {
  const int64_t pairs = (int64_t)p->batch * p->nheads, cus = cu_count();
  return chunk_state_passing_shapes_ok(p) && (pairs >= cus * 3 / 4 || (pairs >= cus / 2 && !sums_in_states(p)));
}
template <int HH, int NS> static void launch_state_walk(const SsdParams &p, hipStream_t s) {
  const dim3 grid((uint32_t)p.nheads * (uint32_t)p.batch / HH), block(256 * HH);
  if (p.seq_idx) hipLaunchKernelGGL((chunk_state_passing_fwd_kernel<HH, NS, true>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((chunk_state_passing_fwd_kernel<HH, NS, false>), grid, block, 0, s, p);
}
extern "C" int ssd_chunk_state_passing_fwd(const SsdParams *p, mamba_stream_t stream) {
  int rc = check(p);
  if (rc) return rc;
  if (!chunk_state_passing_shapes_ok(p)) return MAMBA_E_UNSUPPORTED;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // Two heads to a workgroup where more than half of the last round's workgroups (one of two heads, or two of one, to a CU) are
  // there: one CU then takes in 128 KB per chunk for two walks instead of 192.  Else CUs would idle that can have a walk each.
  // One head / two, 4096 positions, chunks of 256: 256 walks 49 / 61 us, 320 90 / 71, 384 105 / 83, 448 108 / 88, 512 111 / 95;
  // 560 145 / 156, 640 152 / 163; 768 173 / 166, 896 196 / 169, 1024 (8 groups) 220 / 195.
  const int64_t walks = (int64_t)p->nheads * p->batch, cus = cu_count(), left = walks % (2 * cus);
  const bool two = p->nheads / p->ngroups % 2 == 0 && walks > cus && (left == 0 || left >= cus);
  if (p->chunk_size == 256) two ? launch_state_walk<2, 4>(*p, s) : launch_state_walk<1, 4>(*p, s);
  else two ? launch_state_walk<2, 2>(*p, s) : launch_state_walk<1, 2>(*p, s);
  return launched();
}

static int ssd_combined_fwd_one(const SsdParams *p, mamba_stream_t stream) {
  int rc = check(p);
  if (rc) return rc;
  const bool walk = chunk_state_passing_pays(p);
  // The steps and their sums: a launch of their own where there is much to do, in the chunk_state kernel (whose workgroups
  // then read the strided steps of their chunk one by one) while that has no more than eight workgroups per CU: 1531 x 80
  // heads 6.6 + 12.9 us against 15.1, 2 x 1000 x 24 5.4 + 10.2 against 11.9.
  const bool merged = !walk && sums_in_states(p);
  if (!merged && (rc = ssd_chunk_cumsum_fwd(p, stream))) return rc;
  if (walk) {
    if ((rc = ssd_chunk_state_passing_fwd(p, stream))) return rc;
  } else {
    if ((rc = ssd_chunk_state_fwd_with(p, stream, merged))) return rc;
    if ((rc = ssd_state_passing_fwd(p, stream))) return rc;
  }
  if (ssd_chunk_scan_fwd_fused_supported(p)) return ssd_chunk_scan_fwd_fused(p, stream);
  if ((rc = ssd_bmm_chunk_fwd(p, stream))) return rc;
  return ssd_chunk_scan_fwd(p, stream);
}

// Public entry points: the whole problem in one go when one launch can index it, else in slices of batch rows.
extern "C" int ssd_chunk_cumsum_fwd(const SsdParams *p, mamba_stream_t stream) { return ssd_sliced(p, stream, ssd_chunk_cumsum_fwd_one); }
extern "C" int ssd_bmm_chunk_fwd(const SsdParams *p, mamba_stream_t stream) { return ssd_sliced(p, stream, ssd_bmm_chunk_fwd_one); }
extern "C" int ssd_chunk_state_fwd(const SsdParams *p, mamba_stream_t stream) { return ssd_sliced(p, stream, ssd_chunk_state_fwd_one); }
extern "C" int ssd_state_passing_fwd(const SsdParams *p, mamba_stream_t stream) { return ssd_sliced(p, stream, ssd_state_passing_fwd_one); }
extern "C" int ssd_chunk_scan_fwd(const SsdParams *p, mamba_stream_t stream) { return ssd_sliced(p, stream, ssd_chunk_scan_fwd_one); }
extern "C" int ssd_combined_fwd(const SsdParams *p, mamba_stream_t stream) { return ssd_sliced(p, stream, ssd_combined_fwd_one); }
