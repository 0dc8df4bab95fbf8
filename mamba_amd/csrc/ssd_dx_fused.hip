// SSD backward, dx (and the ddt / chunk-state ddA terms that come with it), fused with the C B^T contraction, for
// bf16 on gfx950.  The mirror image of the fused forward scan (ssd_scan_fused.hip; reference
// mamba_ssm/ops/triton/ssd_combined.py:94 _chunk_scan_chunk_state_bwd_dx, which reads a stored CB):
//     acc[p, s]  = w_s sum_n dS[p, n] B[s, n]                                  (carried-state part, MFMA)
//                + sum_{l >= s, same sequence} g[l, p] exp(a_l - a_s) sum_n C[l, n] B[s, n]
//     dx[s, p]   = dt_s acc[p, s] + D_p g[s, p]
//     ddt_out[s] += <x_s, acc_s>;  ddA_cumsum[s] -= dt_s <x_s, state part>, the same sum added at the chunk's end.
// One workgroup of one wave per 16 positions; wave w owns the positions s of tile w.  S[l, s] = C_l . B_s is the same for
// every head of the group: the prologue forms it once, in fp32, with the mask on it, and each wave keeps its column of tiles
// (8 in registers; of a 256 position chunk the rest in LDS, as the lanes hold them).  S leaves its MFMA with 4 consecutive l
// per lane for one s, which is the B-operand layout of the causal product (k = l), so the weighted product never leaves
// registers and CB is not read.  A head's g rows and state gradient go to LDS with asynchronous loads while the head before
// is at work, one barrier per head.  Below the diagonal the decay is factored as exp(a_l - a_t) exp(a_t - a_s) with a_t the
// first a of the l tile (both exponents <= 0): one multiply per element and one exponential per lane and tile; the pair of
// tiles with the diagonal uses the exact form.  x comes and dx leaves as whole pieces of rows, through a patch per wave.
//
// What bounds it: memory, 4.4 TB/s (4 x 4096, 80 heads) and 4.6 (32768 positions, 64 heads in 8 groups) through g, x, the
// state gradients and dx at 128-byte rows (a bare pass in that order reaches 4.5 - 4.7); of the time, the causal products
// are 15 %.  Forming S for every head (544 of a head's 1088 MFMAs and 57 % of its LDS reads), g and the state gradient
// through registers between three barriers, and x in 8-byte pieces of 16 rows (a quarter of the time) cost: 16384
// positions, 128 heads, chunk 256: 338 -> 247 us; 4 x 4096, 80 heads, chunk 256: 186 -> 147; 2 x 4096, 40 heads, chunk 128:
// 57 -> 41. Lists of one head, for which the prologue does not pay, take ssd_dx_short.hip (short_lists, below).  Requesting
// x a head ahead is slower (263, 152), streaming stores too (266, 164).
#include "ssd_common.hpp"

namespace {

DEVI f32x4 mfma_bf16(bf16x8_t a, bf16x8_t b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// A head as the asynchronous loads lay it down: whole rows without padding, their 16-byte pieces permuted within the row so
// that the reads of 16 rows (state gradient) and the transposing reads of 8 rows (g) meet in no bank.
template <int PT, int NK, int QT> struct DxHead {
  uint16_t g[16 * QT * 16 * PT];     // g rows of the chunk
  uint16_t ds[16 * PT * 32 * NK];    // the gradient of the state the chunk hands on, rows p
};
template <int PT, int NK, int QT> struct __align__(256) DxShared {
  DxHead<PT, NK, QT> first;
  union {
    struct {
      DxHead<PT, NK, QT> second;
      uint16_t patch[QT][16 * 32];   // epilogue: a wave's 16 rows x 32 columns
    };
    uint16_t c_rows[16 * QT * 32 * NK];  // prologue: the chunk's C rows
  };
  f32x4 s_far[QT > 8 ? 40 : 1][64];  // S of the tiles that a wave's registers do not hold: 8 of waves 0 and 1, 6 of 2 and 3, ..
  float a2[2][16 * QT], el[2][16 * QT], d[2][16 * PT];
  f32x4 dd[2][QT / 4], da[2][QT / 4];  // a wave's shares of dD and of the chunk end's ddA
  int seq[16 * QT];
};

template <int PT, int NK, int QT, bool DET>
__global__ __launch_bounds__(64 * QT, QT == 4 && PT * NK == 16 ? 2 : 4) void bwd_dx_fused_kernel(const SsdParams p, const int hb, const int sum_dD) {
  constexpr int P = 16 * PT, N = 32 * NK, Q = 16 * QT, SR = QT > 8 ? 8 : QT;
  constexpr int RP = P / 8, MP = N / 8;  // 16-byte pieces of a g row, of a state or C row
  // What every wave issues for a head of a full chunk behind its loads of the next one, whatever the values: the two adds of
  // its positions and its stores of dx.  The wait for those loads counts on all of them.
  constexpr int ADDS = 2, STORES = PT / 2;
  __shared__ DxShared<PT, NK, QT> shm;
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
  const int lt = wave, first = lt & ~1;  // this wave's s tile; its l tiles, two at a time, from the pair that holds lt on
  const int t0 = c * Q;
  const int qlim = min(Q, L - t0);
  const bf16_t *Bg = static_cast<const bf16_t *>(p.B) + b * p.B_bs + grp * p.B_gs;
  const bf16_t *Cg = static_cast<const bf16_t *>(p.C) + b * p.C_bs + grp * p.C_gs;
  const float *Dp = static_cast<const float *>(p.D);
  const View4 gv = g_view(p);
  const float dsc = det_scale_of(p);
  int s_own = lt * 16 + j;                 // the position this lane's column stands for
  const int s_row = min(s_own, qlim - 1);  // its row in memory (positions past the end are never stored)

  // ---- memory -> LDS: a wave moves 64 pieces of 16 bytes at a time; rows past the end of the sequence re-read its last row
  auto swz_row = [](int r) { return N == 128 ? r & 15 : r >> 1 & 7; };          // C and state rows: pieces
  auto swz_g = [](int r) { return P == 64 ? r >> 1 & 3 : r >> 2 & 1; };         // g rows: units of 32 bytes
  constexpr int GI = RP / 4, MI = (P * MP / 64 + QT - 1) / QT, CI = MP / 4;     // instructions per wave
  static_assert(GI * QT * 64 == Q * RP && CI * QT * 64 == Q * MP, "whole instructions per wave");
  uint32_t g_off[GI], m_off[MI];
#pragma unroll
  for (int q = 0; q < GI; ++q) {
    const int id = (q * QT + wave) * 64 + lane, r = id / RP;
    g_off[q] = (uint32_t)min(r, qlim - 1) * (uint32_t)(2 * gv.ls) + ((id % RP) ^ swz_g(r) << 1) * 16;
  }
#pragma unroll
  for (int q = 0; q < MI; ++q) {
    const int id = (q * QT + wave) * 64 + lane, r = id / MP;
    m_off[q] = r * (2 * N) + ((id % MP) ^ swz_row(r)) * 16;
  }
  constexpr uint32_t DS = Q * P * 2;  // bytes from a head's g rows to its state gradient
  const uint32_t lds0 = lds_address(&shm.first), lds1 = lds_address(&shm.second);
  // a head's tensors: uniform pointers that move on by `per` heads, and 32-bit offsets from them
  typedef const GLOBAL_AS char *gptr;
  const int64_t row0 = (((int64_t)b * H + h_first) * p.nchunks + c) * Q, row_step = (int64_t)per * p.nchunks * Q;
  gptr g_at_head = (gptr)(static_cast<const bf16_t *>(gv.ptr) + b * gv.bs + (int64_t)t0 * gv.ls + h_first * gv.hs);
  gptr ds_at_head = (gptr)(static_cast<const bf16_t *>(p.dstates_lp) + (((int64_t)b * p.nchunks + c) * H + h_first) * P * N);
  gptr x_at_head = (gptr)(static_cast<const bf16_t *>(p.x) + b * p.x_bs + h_first * p.x_hs + (int64_t)t0 * p.x_ls);
  gptr a_at_head = (gptr)(p.dA_cumsum + row0), dt_at_head = (gptr)(p.dt_out + row0);
  gptr d_at_head = Dp ? (gptr)(Dp + (p.D_has_hdim ? h_first * P : h_first)) : a_at_head;  // any valid address without D
  const int64_t g_step = 2 * per * gv.hs, ds_step = (int64_t)per * P * N * 2, x_step = 2 * per * p.x_hs;
  const int64_t d_step = Dp ? (int64_t)per * 4 * (p.D_has_hdim ? P : 1) : 0;
  GLOBAL_AS char *dx_at_head = (GLOBAL_AS char *)(static_cast<bf16_t *>(p.dx) + b * p.dx_bs + h_first * p.dx_hs + (int64_t)(t0 + lt * 16) * p.dx_ls);
  const int64_t dx_step = 2 * per * p.dx_hs;
  // x of the wave's 16 positions, 32 columns per load, as whole pieces of rows
  u32x4 xr[PT / 2];
  auto request_x = [&]() {
    const uint32_t x_off = (uint32_t)min(lt * 16 + (lane >> 2), qlim - 1) * (uint32_t)(2 * p.x_ls) + (lane & 3) * 16;
#pragma unroll
    for (int e = 0; e < PT / 2; ++e) xr[e] = *(const GLOBAL_AS u32x4 *)(x_at_head + x_off + e * 64);
  };
  float n_a, n_dt, n_d;
  auto request_scalars = [&]() {
    n_a = *(const GLOBAL_AS float *)(a_at_head + (uint32_t)min(tid, Q - 1) * 4u);
    n_dt = *(const GLOBAL_AS float *)(dt_at_head + (uint32_t)s_own * 4u);
    n_d = *(const GLOBAL_AS float *)(d_at_head + (Dp && p.D_has_hdim ? (uint32_t)min(tid, P - 1) * 4u : 0u));
  };
  auto request_head = [&](uint32_t lds) {
#pragma unroll
    for (int q = 0; q < GI; ++q) load_async16((const void *)g_at_head, g_off[q], lds + (q * QT + wave) * 1024);
#pragma unroll
    for (int q = 0; q < MI; ++q)
      if (P * MP / 64 % QT == 0 || q * QT + wave < P * MP / 64) load_async16((const void *)ds_at_head, m_off[q], lds + DS + (q * QT + wave) * 1024);
  };

  // ---- prologue: S[l, s] = C_l . B_s for the group, kept in fp32 for all its heads; zero where l < s, where the sequences
  // differ and past the end of the sequence
  request_scalars();
  request_head(lds0);
#pragma unroll
  for (int q = 0; q < CI; ++q) {
    const int id = (q * QT + wave) * 64 + lane, r = id / MP;
    load_async16(Cg + (int64_t)t0 * p.C_ls, (uint32_t)min(r, qlim - 1) * (uint32_t)(2 * p.C_ls) + ((id % MP) ^ swz_row(r)) * 16, lds1 + (q * QT + wave) * 1024);
  }
  bf16x8_t Bf[NK];  // B rows of this wave's s tile: B operand of both contractions (col s = j, k = n)
#pragma unroll
  for (int kk = 0; kk < NK; ++kk)
    Bf[kk] = __builtin_bit_cast(bf16x8_t, *(const GLOBAL_AS u32x4 *)(Bg + (int64_t)(t0 + s_row) * p.B_ls + kk * 32 + g * 8));
  bool own_last = s_own < qlim;  // the position belongs to the last sequence of the chunk
  if (tid < Q) {
    int id = tid < qlim ? 0 : -2;
    if (p.seq_idx && tid < qlim) id = p.seq_idx[(int64_t)b * L + t0 + tid];
    shm.seq[tid] = id;
  }
  async_done<0>();
  lds_barrier();
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) asm volatile("" : "+v"(Bf[kk]));  // (there: no wait for them inside the loop)
  const int sid = shm.seq[s_own];
  if (p.seq_idx) own_last = own_last && sid >= 0 && sid == shm.seq[qlim - 1];
  auto row_piece = [&](int kk) { return j * (2 * N) + ((swz_row(j) ^ g ^ (kk * 4)) * 16); };  // of the rows 16 i + j, in bytes
  auto s_tile = [&](int ltp) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) v = mfma_bf16(*(lds_frag)(uintptr_t)(lds1 + ltp * (32 * N) + row_piece(kk)), Bf[kk], v);
    const int l0 = ltp * 16 + 4 * g;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = l0 + r >= s_own && shm.seq[l0 + r] == sid && l0 + r < qlim ? v[r] : 0.f;
    return v;
  };
  f32x4 S[SR], *const far = shm.s_far[QT > 8 ? (lt >> 1) * (18 - 2 * (lt >> 1)) + (lt & 1) * (8 - first) : 0];  // (waves 0 .. 7 only)
#pragma unroll
  for (int k = 0; k < SR; ++k) S[k] = first + k < QT ? s_tile(first + k) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int ltp = first + SR; ltp < QT; ++ltp) far[(ltp - first - SR) * 64 + lane] = s_tile(ltp);

  // the waves' shares of a head, in a fixed order (by the wave with the shortest walk)
  auto add_shares = [&](int which, int h) {
    float dd = 0.f, da = 0.f;
#pragma unroll
    for (int w = 0; w < QT / 4; ++w) {
      const f32x4 a = shm.da[which][w], d = shm.dd[which][w];
      da += a[0], da += a[1], da += a[2], da += a[3];
      dd += d[0], dd += d[1], dd += d[2], dd += d[3];
    }
    acc_add<DET ? 1 : 0>(p.ddA_cumsum, p.det_ddA_cumsum, chunk_off(p, b, h, c) + Q - 1, da, dsc);
    if (sum_dD) acc_add<DET ? 1 : 0>(p.dD, p.det_dD, h, dd, dsc);
  };

  uint32_t here = lds0, there = lds1;  // the head at work and the place of the one after it
#pragma unroll 1
  for (int hh = 0; hh < hb; ++hh) {
    const int h = h_first + hh * per, odd = hh & 1;
    // the thread's index passes through an empty asm once per head, so that what derives from it is computed where it is
    // used instead of being carried (or spilled) across the loop over the heads
    asm volatile("" : "+v"(tid));
    lane = tid & 63, j = lane & 15, g = lane >> 4, s_own = lt * 16 + j;
    // This head's operands are there once no more is in flight than what followed them, in order (more in some waves)
    if (qlim == Q && !DET) async_done<ADDS + STORES>();
    else async_done<0>();
    if (qlim < Q) {  // g is zero past the end of the sequence
#pragma unroll
      for (int q = 0; q < GI; ++q) {
        const int id = (q * QT + wave) * 64 + lane;
        if (id / RP >= qlim) *(lds_u4)(uintptr_t)(here + id * 16) = u32x4{0u, 0u, 0u, 0u};
      }
    }
    if (tid < Q) {
      shm.a2[odd][tid] = n_a * kLog2e;
      shm.el[odd][tid] = fast_exp(fminf(n_a - __shfl(n_a, lane & 48, 64), 0.f));
    }
    if (tid < P) shm.d[odd][tid] = Dp ? n_d : 0.f;
    const float dts = n_dt;
    lds_barrier();  // this head is there, and nobody reads the one before it any more
    if (wave == QT - 1 && lane == 0 && hh > 0) add_shares(odd ^ 1, h - per);
    request_x();
    // (the scalars always, after the last head its own once more: the compiler, which does not see the asynchronous loads,
    // then counts the same loads behind x on either way, and its wait for x does not drain those of the next head)
    const bool more = hh + 1 < hb;
    g_at_head += g_step, ds_at_head += ds_step, x_at_head += x_step;
    a_at_head += more ? row_step * 4 : 0, dt_at_head += more ? row_step * 4 : 0, d_at_head += more ? d_step : 0;
    request_scalars();
    if (more) request_head(there);

    f32x4 acc[PT];
#pragma unroll
    for (int pt = 0; pt < PT; ++pt) acc[pt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float *a2 = shm.a2[odd];
    const float as2 = a2[s_own];
    // G^T fragment of p tile pt for two l tiles: lane (j, g) gets row p = 16 pt + j and the k slots of lane group g,
    // which are positions 4 g .. 4 g + 3 of the first tile, then of the second: the layout in which S lies.
    // Each half is one transposing load of a 4 x 16 patch.
    const uint32_t g_at = here + (4 * g + (j >> 2)) * (2 * P) + (j & 3) * 8 + swz_g(4 * g + (j >> 2)) * 32 + first * (32 * P);
    const uint32_t el_at = lds_address(&shm.el[odd][4 * g]) + first * 64, a2_at = lds_address(a2) + first * 64;

    // ---- inside the chunk: two l tiles, first + k and the next, with S of both.  The pair that holds the diagonal takes the
    // exact decay, exp(a_l - a_s); S is zero above it
    auto block = [&](const int k, const f32x4 (&Sk)[2], const bool diagonal) {
      float m[8];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (diagonal) {
          const f32x4 al = *(lds_f4)(uintptr_t)(a2_at + 16 * g + (k + i) * 64);
#pragma unroll
          for (int r = 0; r < 4; ++r) m[4 * i + r] = Sk[i][r] * fast_exp2(fminf(al[r] - as2, 0.f));
        } else {
          const f32x4 el = *(lds_f4)(uintptr_t)(el_at + (k + i) * 64);
          const float cs = fast_exp2(fminf(*(lds_f1)(uintptr_t)(a2_at + (k + i) * 64) - as2, 0.f));
#pragma unroll
          for (int r = 0; r < 4; ++r) m[4 * i + r] = Sk[i][r] * el[r] * cs;
        }
      }
      const u32x4 mp = {pack_bf16(m[0], m[1]), pack_bf16(m[2], m[3]), pack_bf16(m[4], m[5]), pack_bf16(m[6], m[7])};
      const bf16x8_t Mf = __builtin_bit_cast(bf16x8_t, mp);
#pragma unroll
      for (int pt = 0; pt < PT; ++pt) {
        const uint32_t src = (g_at ^ (pt * 32)) + k * (32 * P);
        const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)src);
        const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)(src + 32 * P));
        acc[pt] = mfma_bf16(__builtin_bit_cast(bf16x8_t, (i16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)), Mf, acc[pt]);
      }
    };
#pragma unroll
    for (int k = 0; k < SR; k += 2)
      if (first + k < QT) block(k, {S[k], S[k + 1]}, k == 0);
    if constexpr (QT > 8) {
#pragma unroll 1
      for (int k = SR; first + k < QT; k += 2) block(k, {far[(k - SR) * 64 + lane], far[(k - SR + 1) * 64 + lane]}, false);
    }

    // The wave's patch: 16 rows x 32 columns, 16-byte pieces permuted with the row; between whole rows (lane = 4 row + piece)
    // and the accumulator layout (row j, columns 16 k + 4 g .. + 3)
    const int rr = lane >> 2, piece = lane & 3;
    const uint32_t y_at = lds_address(&shm.patch[wave][0]), y_row = y_at + rr * 64 + ((piece ^ (rr >> 1 & 3)) * 16);
    auto y_acc = [&](int k) { return y_at + j * 64 + (((2 * k + (g >> 1)) ^ (j >> 1 & 3)) * 16) + (g & 1) * 8; };
    auto wave_sync = [] {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    u32x2 xl[PT];  // x of this lane's column s in the accumulator layout: rows p = 16 pt + 4 g .. + 3
#pragma unroll
    for (int e = 0; e < PT / 2; ++e) {
      *(lds_u4)(uintptr_t)y_row = xr[e];
      wave_sync();
#pragma unroll
      for (int k = 0; k < 2; ++k) xl[2 * e + k] = *(lds_u2)(uintptr_t)y_acc(k);
      wave_sync();
    }

    // ---- carried-state part, and the products with x: q1 of that part, q2 of the whole
    float q1 = 0.f, q2 = 0.f;
    {
      const float w = own_last ? fast_exp2(fminf(a2[Q - 1] - as2, 0.f)) : 0.f;
#pragma unroll
      for (int pt = 0; pt < PT; ++pt) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk)
          v = mfma_bf16(*(lds_frag)(uintptr_t)(here + DS + pt * (32 * N) + row_piece(kk)), Bf[kk], v);
        const float xf[4] = {bf16_lo(xl[pt].x), bf16_hi(xl[pt].x), bf16_lo(xl[pt].y), bf16_hi(xl[pt].y)};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc[pt][r] = __builtin_fmaf(v[r], w, acc[pt][r]);
          q1 = __builtin_fmaf(xf[r], v[r], q1);
          q2 = __builtin_fmaf(xf[r], acc[pt][r], q2);
        }
      }
      q1 *= w;
      q1 += __shfl_xor(q1, 16, 64);
      q1 += __shfl_xor(q1, 32, 64);
      q2 += __shfl_xor(q2, 16, 64);
      q2 += __shfl_xor(q2, 32, 64);
    }
    asm volatile("" : "+v"(n_a), "+v"(n_dt), "+v"(n_d));  // (waited for before the adds and stores, not behind them)
    // ---- ddt and the chunk-state terms of ddA, from the accumulator layout
    {
      const int64_t row_off = (((int64_t)b * H + h) * p.nchunks + c) * Q;
      const bool live = g == 0 && s_own < qlim;
      if (live) {  // (ADDS, not left out where a value is 0)
        acc_add<DET ? 1 : 0>(p.ddt_out, p.det_ddt_out, row_off + s_own, q2, dsc);
        acc_add<DET ? 1 : 0>(p.ddA_cumsum, p.det_ddA_cumsum, row_off + s_own, -dts * q1, dsc);
      }
      const float e = wave_sum_to_last(live ? dts * q1 : 0.f);  // ... and + at the chunk end, one add for all waves
      if (lane == 63) reinterpret_cast<float *>(shm.da[odd])[wave] = e;
    }

    // ---- dx = dt acc + D g, 32 columns at a time through the wave's patch, so that they leave as 16-byte pieces of rows
    // (the accumulator layout itself holds 8-byte pieces); dD[h] += sum_{s, p} g[s, p] x[s, p] where it is wanted (a D per
    // head and no gate: g is dout)
    float dd = 0.f;
    const uint32_t own_at = here + s_own * (2 * P) + g * 8 + swz_g(s_own) * 32;
#pragma unroll
    for (int e = 0; e < STORES; ++e) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int pt = 2 * e + k;
        f32x4 v = acc[pt] * dts;
        if (Dp || sum_dD) {
          const u32x2 gw = *(lds_u2)(uintptr_t)(own_at ^ (pt * 32));
          const f32x4 gf = {bf16_lo(gw.x), bf16_hi(gw.x), bf16_lo(gw.y), bf16_hi(gw.y)};
          const f32x4 D4 = *reinterpret_cast<const f32x4 *>(&shm.d[odd][p.D_has_hdim ? pt * 16 + 4 * g : 0]);
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = __builtin_fmaf(D4[r], gf[r], v[r]);
          if (sum_dD) {
            dd = __builtin_fmaf(bf16_lo(xl[pt].x), gf[0], dd);
            dd = __builtin_fmaf(bf16_hi(xl[pt].x), gf[1], dd);
            dd = __builtin_fmaf(bf16_lo(xl[pt].y), gf[2], dd);
            dd = __builtin_fmaf(bf16_hi(xl[pt].y), gf[3], dd);
          }
        }
        *(lds_u2)(uintptr_t)y_acc(k) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
      }
      wave_sync();
      const u32x4 out = *(lds_u4)(uintptr_t)y_row;
      if (lt * 16 + rr < qlim)  // (STORES)
        *(GLOBAL_AS u32x4 *)(dx_at_head + (uint32_t)rr * (uint32_t)(2 * p.dx_ls) + piece * 16 + e * 64) = out;
      wave_sync();
    }
    if (sum_dD) {
      dd = wave_sum_to_last(dd);
      if (lane == 63) reinterpret_cast<float *>(shm.dd[odd])[wave] = dd;
    }
    dx_at_head += dx_step;
    const uint32_t t = here;
    here = there;
    there = t;
  }
  lds_barrier();
  if (wave == QT - 1 && lane == 0) add_shares((hb - 1) & 1, h_first + (hb - 1) * per);
}

template <int PT, int NK, bool DET> int launch_q(const SsdParams &p, hipStream_t s, int dd) {
  const int hb = heads_per_workgroup(p);
  dim3 grid(p.nheads / hb, p.nchunks, p.batch);
  switch (p.chunk_size) {
    case 256: hipLaunchKernelGGL((bwd_dx_fused_kernel<PT, NK, 16, DET>), grid, dim3(1024), 0, s, p, hb, dd); break;
    case 128: hipLaunchKernelGGL((bwd_dx_fused_kernel<PT, NK, 8, DET>), grid, dim3(512), 0, s, p, hb, dd); break;
    case 64: hipLaunchKernelGGL((bwd_dx_fused_kernel<PT, NK, 4, DET>), grid, dim3(256), 0, s, p, hb, dd); break;
    default: return MAMBA_E_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}
template <int PT, bool DET> int launch_n(const SsdParams &p, hipStream_t s, int dd) {
  switch (p.dstate) {
    case 64: return launch_q<PT, 2, DET>(p, s, dd);
    case 128: return launch_q<PT, 4, DET>(p, s, dd);
    default: return MAMBA_E_UNSUPPORTED;
  }
}
template <bool DET> int launch_p(const SsdParams &p, hipStream_t s, int dd) {
  return p.headdim == 64 ? launch_n<4, DET>(p, s, dd) : launch_n<2, DET>(p, s, dd);
}

bool supported(const SsdParams *p) {
  if (p->dtype != MAMBA_BF16 || !p->dstates_lp) return false;
  if (p->headdim != 32 && p->headdim != 64) return false;
  if (p->dstate != 64 && p->dstate != 128) return false;
  if (p->chunk_size != 64 && p->chunk_size != 128 && p->chunk_size != 256) return false;
  // 16-byte pieces of rows everywhere
  const void *gptr = p->z ? static_cast<const void *>(p->gbuf) : p->dout;
  if (!gptr) return false;
  if (!aligned(p->x, 16) || !aligned(p->B, 16) || !aligned(p->C, 16) || !aligned(p->dx, 16) || !aligned(gptr, 16) ||
      !aligned(p->dstates_lp, 16))
    return false;
  if (p->x_bs % 8 || p->x_ls % 8 || p->x_hs % 8 || p->B_bs % 8 || p->B_ls % 8 || p->B_gs % 8 || p->C_bs % 8 ||
      p->C_ls % 8 || p->C_gs % 8 || p->dx_bs % 8 || p->dx_ls % 8 || p->dx_hs % 8)
    return false;
  if (!p->z && (p->dout_bs % 8 || p->dout_ls % 8 || p->dout_hs % 8)) return false;
  if (p->batch > 65535 || p->nchunks > 65535) return false;
  return true;
}

// ssd_dx_short.hip takes lists in which forming C B^T once for all heads does not pay, and rows whose places in a chunk 32-bit
// offsets do not reach.  The stage alone, 700 sizes (1 - 4 x 64 - 16384 x 8 - 96 heads in 1 - 8 groups), time of the short form /
// of this one, few workgroups (up to the CUs) and many, by the heads of a list, 1 | 2 | 3 and more:
//   headdim 64, 128 states, chunk 64    few 0.88 | 1.02 | 1.2     many 0.76 | 0.90 | 0.93 (3 heads), 0.9 - 1.2
//                           chunk 128       0.83 | 0.95 | 1.07         1.22 | 1.33 | 1.28
//                           chunk 256       0.84 | 1.01 | 1.2          0.88 | 1.06 | 1.13
//   less than that,         chunk 64        0.86 - 0.89 | 1.01 | 1.2   0.91 - 0.97 | 1.02 - 1.05 | 1.03 - 1.12
//                           chunk 128       0.80 - 0.82 | 0.96 | 1.1   0.81 - 0.85 | 0.97 - 0.99 | 1.04 - 1.16
//                           chunk 256       0.73 - 0.82 | 0.91 - 0.98 | 1.0 - 1.3   0.76 - 0.86 | 0.93 - 1.03 | 1.04 - 1.3
bool short_lists(const SsdParams *p) {
  if (!near_rows(p->x_ls) || !near_rows(p->dx_ls) || !near_rows(p->C_ls) || !near_rows(p->z ? (int64_t)p->nheads * p->headdim : p->dout_ls)) return true;
  const int hb = heads_per_workgroup(*p), Q = p->chunk_size;
  const bool many = (int64_t)p->nheads / hb * p->nchunks * p->batch > cu_count(), full = p->headdim == 64 && p->dstate == 128;
  if (hb == 1) return !(full && Q == 128 && many);
  if (Q == 64) return hb <= 3 && full && many;
  return hb == 2 && !many && (Q == 128 || !full);
}

}  // namespace

bool ssd_bwd_dx_fused_supported(const SsdParams *p) { return supported(p); }

// With sum_dD the launch also adds the heads' <g, x> to dD (one D per head): the whole of dD where no gate stands
// between dout and g.
int ssd_bwd_dx_fused_launch(const SsdParams *p, hipStream_t stream, bool sum_dD) {
  if (!supported(p)) return MAMBA_E_UNSUPPORTED;
  if (sum_dD && (!p->dD || p->D_has_hdim || (p->det_scale && !p->det_dD))) return MAMBA_E_BADARG;
  if (short_lists(p)) return ssd_bwd_dx_short_launch(*p, stream, sum_dD);
  return p->det_scale ? launch_p<true>(*p, stream, sum_dD) : launch_p<false>(*p, stream, sum_dD);
}
