// SSD chunk_scan forward fused with the C B^T contraction (bf16, gfx950), the form that keeps S = C B^T of the group (reference
// mamba_ssm/ops/triton/ssd_chunk_scan.py:49 _chunk_scan_fwd_kernel, :1259 _chunk_scan_fwd; the mathematics of
// chunk_scan_fwd_fused_kernel in ssd_scan_fused.hip):
//     y[l, p] = sum_{s <= l, same sequence} S[s, l] dt_s exp(a_l - a_s) x[s, p] + exp(a_l) sum_n H[p, n] C[l, n]   (+ D x, gate)
// One workgroup of one wave per 16 positions l works through a list of heads of one group.  S is formed once, in fp32, with the
// mask on it, and each wave keeps its column of tiles in registers: it lies as the B operand of the product with X^T (k = s).  A
// head's x rows and state go to LDS with asynchronous loads under the head before, one barrier per head; z comes and the
// outputs leave as whole pieces of rows through a patch per wave.  Two workgroups share a CU (chunk 128).  The kernel itself at
// 2 x 4096, 40 heads in 8 groups, chunk 128, no gate: 52 us as the one-tile form, 34 here (5.0 TB/s).
#include "ssd_common.hpp"

namespace {

DEVI f32x4 mfma_bf16(bf16x8_t a, bf16x8_t b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// What a decay's exponent (base 2) may reach: an exponential that stays finite, for the zeros of S to be multiplied by.
constexpr float kGrowth = 126.f;

// A head as the asynchronous loads lay it down: whole rows without padding, their 16-byte pieces permuted within the row so
// that the reads of 16 rows (state) and the transposing reads of 8 rows (x) meet in no bank.
template <int PT, int NK, int QT> struct ScanHead {
  uint16_t x[16 * QT * 16 * PT];    // x rows of the chunk
  uint16_t h[16 * PT * 32 * NK];    // the state the chunk is entered with, rows p
};
template <int PT, int NK, int QT> struct __align__(256) ScanShared {
  ScanHead<PT, NK, QT> first;
  union {
    struct {
      ScanHead<PT, NK, QT> second;
      uint16_t patch[QT][16 * 32];   // epilogue: a wave's 16 rows x 32 columns
    };
    uint16_t b_rows[16 * QT * 32 * NK];  // prologue: the chunk's B rows
  };
  float a2[2][16 * QT], cs[2][16 * QT], dt[2][16 * QT], d[2][16 * PT];
  int seq[16 * QT];
};

template <int PT, int NK, int QT, bool GATED>
__global__ __launch_bounds__(64 * QT, QT == 4 && PT * NK == 16 ? 2 : 4) void chunk_scan_fwd_group_kernel(const SsdParams p, const int hb) {
  constexpr int P = 16 * PT, N = 32 * NK, Q = 16 * QT;
  constexpr int RP = P / 8, MP = N / 8;  // 16-byte pieces of an x row, of a state or B row
  // What every wave issues for a head of a full chunk behind its loads of the next one: its stores of the output.  The wait
  // for those loads counts on all of them.
  constexpr int STORES = PT / 2;
  __shared__ ScanShared<PT, NK, QT> shm;
  typedef __attribute__((address_space(3))) i16x4_t *lds_tr;
  typedef __attribute__((address_space(3))) bf16x8_t *lds_frag;
  typedef __attribute__((address_space(3))) u32x4 *lds_u4;
  typedef __attribute__((address_space(3))) u32x2 *lds_u2;
  typedef __attribute__((address_space(3))) f32x4 *lds_f4;
  typedef __attribute__((address_space(3))) float *lds_f1;
  typedef short i16x8_t __attribute__((ext_vector_type(8)));

  int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int j = lane & 15, g = lane >> 4;
  const int H = p.nheads, G = p.ngroups, L = p.seqlen;
  // the heads of a workgroup are `per` apart: workgroups in flight together touch neighbouring heads
  const int hpg = H / G, per = hpg / hb;
  const int grp = blockIdx.x / per, h_first = grp * hpg + blockIdx.x % per;
  const int c = blockIdx.y, b = blockIdx.z;
  const int lt = wave, first = lt & ~1;  // this wave's l tile; its s tiles, two at a time, from the pair that holds lt down
  const int t0 = c * Q;
  const int qlim = min(Q, L - t0);
  const bf16_t *Bg = static_cast<const bf16_t *>(p.B) + b * p.B_bs + grp * p.B_gs;
  const bf16_t *Cg = static_cast<const bf16_t *>(p.C) + b * p.C_bs + grp * p.C_gs;
  const float *Dp = static_cast<const float *>(p.D);
  int l_own = lt * 16 + j;  // the position this lane's column stands for

  // ---- memory -> LDS: a wave moves 64 pieces of 16 bytes at a time; rows past the end of the sequence re-read its last row
  auto swz_row = [](int r) { return N == 128 ? r & 15 : r >> 1 & 7; };          // B and state rows: pieces
  auto swz_x = [](int r) { return P == 64 ? r >> 1 & 3 : r >> 2 & 1; };         // x rows: units of 32 bytes
  constexpr int XI = RP / 4, MI = (P * MP / 64 + QT - 1) / QT, BI = MP / 4;     // instructions per wave
  static_assert(XI * QT * 64 == Q * RP && BI * QT * 64 == Q * MP, "whole instructions per wave");
  uint32_t x_off[XI], m_off[MI];
#pragma unroll
  for (int q = 0; q < XI; ++q) {
    const int id = (q * QT + wave) * 64 + lane, r = id / RP;
    x_off[q] = (uint32_t)min(r, qlim - 1) * (uint32_t)(2 * p.x_ls) + ((id % RP) ^ swz_x(r) << 1) * 16;
  }
#pragma unroll
  for (int q = 0; q < MI; ++q) {
    const int id = (q * QT + wave) * 64 + lane, r = id / MP;
    m_off[q] = r * (2 * N) + ((id % MP) ^ swz_row(r)) * 16;
  }
  constexpr uint32_t HS = Q * P * 2;  // bytes from a head's x rows to its state
  const uint32_t lds0 = lds_address(&shm.first), lds1 = lds_address(&shm.second);
  // a head's tensors: uniform pointers that move on by `per` heads, and 32-bit offsets from them
  typedef const GLOBAL_AS char *gptr;
  typedef GLOBAL_AS char *gwptr;
  const int64_t row0 = (((int64_t)b * H + h_first) * p.nchunks + c) * Q, row_step = (int64_t)per * p.nchunks * Q;
  gptr x_at_head = (gptr)(static_cast<const bf16_t *>(p.x) + b * p.x_bs + (int64_t)t0 * p.x_ls + h_first * p.x_hs);
  gptr h_at_head = (gptr)(static_cast<const bf16_t *>(p.states_lp) + (((int64_t)b * p.nchunks + c) * H + h_first) * P * N);
  gptr z_at_head = GATED ? (gptr)(static_cast<const bf16_t *>(p.z) + b * p.z_bs + h_first * p.z_hs + (int64_t)t0 * p.z_ls) : x_at_head;
  gptr a_at_head = (gptr)(p.dA_cumsum + row0), dt_at_head = (gptr)(p.dt_out + row0);
  gptr d_at_head = Dp ? (gptr)(Dp + (p.D_has_hdim ? h_first * P : h_first)) : a_at_head;  // any valid address without D
  const int64_t x_step = 2 * per * p.x_hs, h_step = (int64_t)per * P * N * 2, z_step = 2 * per * p.z_hs;
  const int64_t d_step = Dp ? (int64_t)per * 4 * (p.D_has_hdim ? P : 1) : 0;
  const int64_t o0 = b * p.out_bs + h_first * p.out_hs + (int64_t)(t0 + lt * 16) * p.out_ls, o_step = 2 * per * p.out_hs;
  gwptr o_at_head = (gwptr)(static_cast<bf16_t *>(p.out) + o0), ox_at_head = p.out_x ? (gwptr)(static_cast<bf16_t *>(p.out_x) + o0) : o_at_head;
  u32x4 zr[GATED ? PT / 2 : 1];  // z of the wave's 16 positions, 32 columns per load, as whole pieces of rows
  auto request_z = [&]() {
    const uint32_t z_off = (uint32_t)min(lt * 16 + (lane >> 2), qlim - 1) * (uint32_t)(2 * p.z_ls) + (lane & 3) * 16;
#pragma unroll
    for (int e = 0; e < PT / 2; ++e) zr[e] = *(const GLOBAL_AS u32x4 *)(z_at_head + z_off + e * 64);
  };
  float n_a, n_dt, n_d;
  auto request_scalars = [&]() {
    const uint32_t pos = (uint32_t)min(tid, Q - 1) * 4u;
    n_a = *(const GLOBAL_AS float *)(a_at_head + pos);
    n_dt = *(const GLOBAL_AS float *)(dt_at_head + pos);
    n_d = *(const GLOBAL_AS float *)(d_at_head + (Dp && p.D_has_hdim ? (uint32_t)min(tid, P - 1) * 4u : 0u));
  };
  auto request_head = [&](uint32_t lds) {
#pragma unroll
    for (int q = 0; q < XI; ++q) load_async16((const void *)x_at_head, x_off[q], lds + (q * QT + wave) * 1024);
#pragma unroll
    for (int q = 0; q < MI; ++q)
      if (P * MP / 64 % QT == 0 || q * QT + wave < P * MP / 64) load_async16((const void *)h_at_head, m_off[q], lds + HS + (q * QT + wave) * 1024);
  };

  // ---- prologue: S[s, l] = B_s . C_l for the group, kept in fp32 for all its heads; zero where l < s, where the sequences
  // differ and past the end of the sequence
  request_scalars();
  request_head(lds0);
#pragma unroll
  for (int q = 0; q < BI; ++q) {
    const int id = (q * QT + wave) * 64 + lane, r = id / MP;
    load_async16(Bg + (int64_t)t0 * p.B_ls, (uint32_t)min(r, qlim - 1) * (uint32_t)(2 * p.B_ls) + ((id % MP) ^ swz_row(r)) * 16, lds1 + (q * QT + wave) * 1024);
  }
  bf16x8_t Cf[NK];  // C rows of this wave's l tile: B operand of both contractions (col l = j, k = n)
#pragma unroll
  for (int kk = 0; kk < NK; ++kk)
    Cf[kk] = __builtin_bit_cast(bf16x8_t, *(const GLOBAL_AS u32x4 *)(Cg + (int64_t)(t0 + min(l_own, qlim - 1)) * p.C_ls + kk * 32 + g * 8));
  bool carried = l_own < qlim;  // the state entering the chunk belongs to the position's sequence
  if (tid < Q) {
    int id = tid < qlim ? 0 : -2;
    if (p.seq_idx && tid < qlim) id = p.seq_idx[(int64_t)b * L + t0 + tid];
    shm.seq[tid] = id;
  }
  const int before = p.seq_idx && c > 0 ? p.seq_idx[(int64_t)b * L + t0 - 1] : 0;
  async_done<0>();
  lds_barrier();
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) asm volatile("" : "+v"(Cf[kk]));  // (there: no wait for them inside the loop)
  const int lid = shm.seq[l_own];
  carried = carried && lid == before;
  auto row_piece = [&](int kk) { return j * (2 * N) + ((swz_row(j) ^ g ^ (kk * 4)) * 16); };  // of the rows 16 i + j, in bytes
  auto s_tile = [&](int st) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) v = mfma_bf16(*(lds_frag)(uintptr_t)(lds1 + st * (32 * N) + row_piece(kk)), Cf[kk], v);
    const int s0 = st * 16 + 4 * g;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = s0 + r <= l_own && shm.seq[s0 + r] == lid && s0 + r < qlim ? v[r] : 0.f;
    return v;
  };
  // (S[k], S[k + 1]: tiles first - k and the one after it)
  f32x4 S[QT];
#pragma unroll
  for (int k = 0; k < QT; k += 2)
#pragma unroll
    for (int i = 0; i < 2; ++i) S[k + i] = first >= k ? s_tile(first - k + i) : f32x4{0.f, 0.f, 0.f, 0.f};

  uint32_t here = lds0, there = lds1;  // the head at work and the place of the one after it
#pragma unroll 1
  for (int hh = 0; hh < hb; ++hh) {
    const int odd = hh & 1;
    // the thread's index passes through an empty asm once per head, so that what derives from it is computed where it is
    // used instead of being carried (or spilled) across the loop over the heads
    asm volatile("" : "+v"(tid));
    lane = tid & 63, j = lane & 15, g = lane >> 4, l_own = lt * 16 + j;
    // This head's operands are there once no more is in flight than what followed them, in order (or twice as many)
    if (qlim == Q) async_done<STORES>();
    else async_done<0>();
    if (qlim < Q) {  // x is zero past the end of the sequence
#pragma unroll
      for (int q = 0; q < XI; ++q) {
        const int id = (q * QT + wave) * 64 + lane;
        if (id / RP >= qlim) *(lds_u4)(uintptr_t)(here + id * 16) = u32x4{0u, 0u, 0u, 0u};
      }
    }
    if (tid < Q) {
      shm.a2[odd][tid] = n_a * kLog2e;
      shm.dt[odd][tid] = n_dt;
      shm.cs[odd][tid] = n_dt * fast_exp2(fminf((__shfl(n_a, lane | 15, 64) - n_a) * kLog2e, kGrowth));
    }
    if (tid < P) shm.d[odd][tid] = Dp ? n_d : 0.f;
    lds_barrier();  // this head is there, and nobody reads the one before it any more
    if (GATED) request_z();
    // (the scalars always, after the last head its own once more: the compiler, which does not see the asynchronous loads,
    // then counts the same loads behind z on either way, and its wait for z does not drain those of the next head)
    const bool more = hh + 1 < hb;
    x_at_head += x_step, h_at_head += h_step, z_at_head += z_step;
    a_at_head += more ? row_step * 4 : 0, dt_at_head += more ? row_step * 4 : 0, d_at_head += more ? d_step : 0;
    request_scalars();
    if (more) request_head(there);

    f32x4 acc[PT];
#pragma unroll
    for (int pt = 0; pt < PT; ++pt) acc[pt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float *a2 = shm.a2[odd];
    const float al2 = a2[l_own];
    // X^T fragment of p tile pt for two s tiles: lane (j, g) gets row p = 16 pt + j and the k slots of lane group g, which are
    // positions 4 g .. 4 g + 3 of the first tile, then of the second: the layout in which S lies
    const uint32_t x_at = here + (4 * g + (j >> 2)) * (2 * P) + (j & 3) * 8 + swz_x(4 * g + (j >> 2)) * 32 + first * (32 * P);
    const uint32_t cs_at = lds_address(&shm.cs[odd][4 * g]) + first * 64, a2_at = lds_address(a2) + first * 64, dt_at = lds_address(&shm.dt[odd][4 * g]) + first * 64;

    // ---- inside the chunk: two s tiles, first - k and the next, with S of both.  Below the diagonal the decay is exp(a_l -
    // a_end) (dt_s exp(a_end - a_s)) with a_end the last a of the 16 positions s; the pair that holds the diagonal takes the
    // exact one; S is zero above it.  Both exponents are <= 0 where all steps are >= 0.  With steps of either sign one of them
    // may not be, though their sum is: below the diagonal tile neither is cut at 0, as in the other forms of this scan
    const float below = lt & 1 ? kGrowth : 0.f;  // the pair's first tile: below the diagonal, or the diagonal one
    auto block = [&](const int k, const f32x4 (&Sk)[2], const bool diagonal) {
      float m[8];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t o = (i - k) * 64;
        if (diagonal) {
          const f32x4 as = *(lds_f4)(uintptr_t)(a2_at + 16 * g + o), dts = *(lds_f4)(uintptr_t)(dt_at + o);
#pragma unroll
          for (int r = 0; r < 4; ++r) m[4 * i + r] = Sk[i][r] * dts[r] * fast_exp2(fminf(al2 - as[r], i == 0 ? below : 0.f));
        } else {
          const f32x4 cs = *(lds_f4)(uintptr_t)(cs_at + o);
          const float rl = fast_exp2(fminf(al2 - *(lds_f1)(uintptr_t)(a2_at + o + 60), kGrowth));
#pragma unroll
          for (int r = 0; r < 4; ++r) m[4 * i + r] = Sk[i][r] * cs[r] * rl;
        }
      }
      const u32x4 mp = {pack_bf16(m[0], m[1]), pack_bf16(m[2], m[3]), pack_bf16(m[4], m[5]), pack_bf16(m[6], m[7])};
      const bf16x8_t Mf = __builtin_bit_cast(bf16x8_t, mp);
#pragma unroll
      for (int pt = 0; pt < PT; ++pt) {
        const uint32_t src = (x_at ^ (pt * 32)) - k * (32 * P);
        const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)src);
        const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)(src + 32 * P));
        acc[pt] = mfma_bf16(__builtin_bit_cast(bf16x8_t, (i16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)), Mf, acc[pt]);
      }
    };
#pragma unroll
    for (int k = 0; k < QT; k += 2)
      if (first >= k) block(k, {S[k], S[k + 1]}, k == 0);

    // ---- carried state: y += exp(a_l) sum_n H[p, n] C[l, n]
    {
      const float w = carried ? fast_exp2(al2) : 0.f;
#pragma unroll
      for (int pt = 0; pt < PT; ++pt) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk)
          v = mfma_bf16(*(lds_frag)(uintptr_t)(here + HS + pt * (32 * N) + row_piece(kk)), Cf[kk], v);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[pt][r] = __builtin_fmaf(v[r], w, acc[pt][r]);
      }
    }
    asm volatile("" : "+v"(n_a), "+v"(n_dt), "+v"(n_d));  // (waited for before the stores, not behind them)

    // ---- + D x, pre-gate copy, gate, 32 columns at a time through the wave's patch: 16 rows x 32 columns, 16-byte pieces
    // permuted with the row, between whole rows (lane = 4 row + piece) and the accumulator layout (row j, columns 16 k + 4 g ..)
    const int rr = lane >> 2, piece = lane & 3;
    const uint32_t y_at = lds_address(&shm.patch[wave][0]), y_row = y_at + rr * 64 + ((piece ^ (rr >> 1 & 3)) * 16);
    auto y_acc = [&](int k) { return y_at + j * 64 + (((2 * k + (g >> 1)) ^ (j >> 1 & 3)) * 16) + (g & 1) * 8; };
    auto wave_sync = [] {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const uint32_t own_at = here + l_own * (2 * P) + g * 8 + swz_x(l_own) * 32;
    const uint32_t o_off = (uint32_t)rr * (uint32_t)(2 * p.out_ls) + piece * 16;
    const bool stored = lt * 16 + rr < qlim;
#pragma unroll
    for (int e = 0; e < STORES; ++e) {
      u32x2 zl[2];
      if (GATED) {
        *(lds_u4)(uintptr_t)y_row = zr[e];
        wave_sync();
#pragma unroll
        for (int k = 0; k < 2; ++k) zl[k] = *(lds_u2)(uintptr_t)y_acc(k);
        wave_sync();
      }
      if (Dp) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int pt = 2 * e + k;
          const u32x2 xw = *(lds_u2)(uintptr_t)(own_at ^ (pt * 32));
          const f32x4 xf = {bf16_lo(xw.x), bf16_hi(xw.x), bf16_lo(xw.y), bf16_hi(xw.y)};
          const f32x4 D4 = *reinterpret_cast<const f32x4 *>(&shm.d[odd][p.D_has_hdim ? pt * 16 + 4 * g : 0]);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[pt][r] = __builtin_fmaf(D4[r], xf[r], acc[pt][r]);
        }
      }
      auto leave = [&](gwptr dst) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const f32x4 &v = acc[2 * e + k];
          *(lds_u2)(uintptr_t)y_acc(k) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
        }
        wave_sync();
        const u32x4 out = *(lds_u4)(uintptr_t)y_row;
        if (stored) *(GLOBAL_AS u32x4 *)(dst + o_off + e * 64) = out;
        wave_sync();
      };
      if (GATED) {
        if (p.out_x) leave(ox_at_head);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const float zf[4] = {bf16_lo(zl[k].x), bf16_hi(zl[k].x), bf16_lo(zl[k].y), bf16_hi(zl[k].y)};
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[2 * e + k][r] *= zf[r] * sigmoid_f(zf[r]);
        }
      }
      leave(o_at_head);
    }
    o_at_head += o_step, ox_at_head += o_step;
    const uint32_t t = here;
    here = there;
    there = t;
  }
}

template <int PT, int NK, bool GATED> int launch_q(const SsdParams &p, hipStream_t s) {
  const int hb = heads_per_workgroup(p);
  const dim3 grid(p.nheads / hb, p.nchunks, p.batch);
  switch (p.chunk_size) {
    case 128: hipLaunchKernelGGL((chunk_scan_fwd_group_kernel<PT, NK, 8, GATED>), grid, dim3(512), 0, s, p, hb); break;
    case 64:
      if constexpr (!GATED || PT * NK < 16) {  // (not served, below)
        hipLaunchKernelGGL((chunk_scan_fwd_group_kernel<PT, NK, 4, GATED>), grid, dim3(256), 0, s, p, hb);
        break;
      }
      return MAMBA_E_UNSUPPORTED;
    default: return MAMBA_E_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}
template <int PT, int NK> int launch_z(const SsdParams &p, hipStream_t s) {
  if constexpr (NK > 2) {
    if (p.z) return launch_q<PT, NK, true>(p, s);
  }
  return p.z ? MAMBA_E_UNSUPPORTED : launch_q<PT, NK, false>(p, s);  // (64 states with a gate: not served, below)
}

}  // namespace

// Whether this form serves a problem that ssd_chunk_scan_fwd_fused_supported accepts, and is the faster one: chunks of 64 and
// 128 (at 256 the two tiles per wave of ssd_scan_paired.hip take 310 us against 342, 32768 positions x 64 heads; 179 against 191,
// 4 x 4096 x 80), more workgroups than CUs (two of them share one; with fewer the one-tile form is 2 % faster), and not 64 states
// with a gate (185 us for a forward pass of 4 x 4096 x 48 heads against 201).  C B^T of the group pays by the heads of a list.
// The stage alone, 900 sizes (1 - 4 x 64 - 16384 x 8 - 96 heads in 1 - 8 groups), time of the one-tile form / of this one by the
// heads of a list, 1 | 2 | 3 | 4 and more:
//   chunk 128, headdim 64, 128 states      1.19 | 1.44 | 1.46 | 1.55;  with a gate 1.12 | 1.24 | 1.23 | 1.12
//   chunk 128, less than that              0.80 - 0.84 | 0.95 - 0.99 | 1.01 - 1.10 | 1.02 - 1.3
//   chunk 64, headdim 64, 128 states       0.82 | 0.92 | 1.02 | 1.06;  with a gate 0.83 | 0.94 | 1.00 | 0.99
//   chunk 64, less than that               0.93 | 1.02 - 1.06 | 1.04 - 1.10 | 1.01 - 1.2
// (Offsets in a chunk are 32-bit.)
bool ssd_scan_group_serves(const SsdParams &p) {
  if (p.chunk_size > 128 || (p.z && p.dstate <= 64) || !p.states_lp) return false;
  const int hb = heads_per_workgroup(p);
  if ((int64_t)p.nheads / hb * p.nchunks * p.batch <= cu_count()) return false;
  const bool full = p.headdim == 64 && p.dstate == 128;
  if (p.chunk_size > 64 ? !full && hb < 3 : full ? p.z || hb < 4 : hb < 2) return false;
  return near_rows(p.x_ls) && near_rows(p.B_ls) && near_rows(p.out_ls) && (!p.z || near_rows(p.z_ls));
}

int ssd_scan_group_launch(const SsdParams &p, hipStream_t s) {
  if (p.headdim == 64) return p.dstate == 128 ? launch_z<4, 4>(p, s) : launch_z<4, 2>(p, s);
  return p.dstate == 128 ? launch_z<2, 4>(p, s) : launch_z<2, 2>(p, s);
}
