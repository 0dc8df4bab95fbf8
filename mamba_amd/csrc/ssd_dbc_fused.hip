// SSD backward, the chunk-state parts of dB and dC (and the ddA_cumsum rows that come with dC), for bf16 on gfx950
// (reference mamba_ssm/ops/triton/ssd_chunk_state.py:902 _chunk_state_bwd_db and ssd_chunk_scan.py:1451
// _chunk_scan_bwd_dC; the same sums as bwd_dB_state_wide_kernel / bwd_dC_state_wide_kernel in ssd_bwd.hip):
//     dB[s, n] += sum_{h in group} w_h[s] sum_p x[s, h, p] dS[h, p, n],   w_h[s] = dt_s exp(a_last - a_s), s in the
//                                                                          chunk's last sequence, else 0
//     dC[l, n] += sum_{h in group} v_h[l] sum_p g[l, h, p] H[h, p, n],    v_h[l] = exp(a_l), l in the sequence the
//                                                                          chunk was entered in, else 0
//     ddA_cumsum[h, l] += sum_n (v_h[l] sum_p g[l, h, p] H[h, p, n]) C[l, n]
// with dS the gradient of the state a chunk hands on and H the state it was entered with.  One launch does both: half
// of its workgroups take dC, half dB.  A workgroup of up to 8 waves takes 16 positions per wave of a chunk (a 256 position
// chunk is two workgroups) and a list of heads of one group.  A head's rows (x or g) and its P x N matrix go to LDS with
// asynchronous loads, the next head's while this one's are multiplied, with one barrier per head.  Wave w owns positions 16 w
// .. 16 w + 15 and keeps their sum over the heads in registers (fp32, N / 16 tiles); the per-position weight is applied to the
// fp32 product of each head, not to the bf16 operand.  The matrix is the B operand with k = p: its fragments come from
// transposing LDS reads.
//
// Where a workgroup's list is the whole group and the dCB stage has left its tiles in bf16, the sums start from the in-chunk
// products (FIN), in the same registers and as steps of the same pipeline, and leave as the finished dB / dC: the fp32 sums are
// neither written nor read, and the stage that added the products to them is gone.
//
// What bounds it: at 2 workgroups of 8 waves per CU (128 registers a wave) the loads alone take 85 % of the time without the
// in-chunk products, the products alone 80 %.  One workgroup of 16 waves per CU, with heads staged through registers, had
// every wave in the same phase and spent half its time in waits.  16384 positions, 128 heads in 8 groups, chunk 256, with the
// in-chunk products: 300 -> 256 us; 2 x 4096, 40 heads in 8 groups, chunk 128: 65 -> 44; without them, 4 x 4096, 80 heads in
// one group: 130 -> 127 (5 TB/s through the L2).
#include "ssd_common.hpp"

namespace {

DEVI f32x4 mfma_bf16(bf16x8_t a, bf16x8_t b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

constexpr int MAXHB = 40;  // heads per workgroup at most (dbc_heads_per_workgroup never picks more)

// One staged head, as the asynchronous loads lay it down: whole rows without padding, their 16-byte pieces permuted within the
// row so that neither the A operand's 16-byte reads nor the transposing reads of a half-wave meet in a bank.
template <int PT, int NK, int WV> struct DbcBuf {
  uint16_t Rs[16 * WV * 16 * PT];  // rows of x / g
  uint16_t Ms[16 * PT * 32 * NK];  // the matrix
};
constexpr int DDA_RING = 16;  // heads whose ddA_cumsum rows a wave keeps until it adds them

// LDS of a workgroup: two staged heads.
template <int PT, int NK, int WV> struct __align__(256) DbcShared {
  DbcBuf<PT, NK, WV> first;
  union {
    struct {
      DbcBuf<PT, NK, WV> second;
      float dda[WV][DDA_RING][16];
    };
    uint16_t c_patch[WV][16 * (64 + 16)];  // a wave's 16 rows x 64 columns, before the second head's time and after the last's
  };
};

// One of the two products for the workgroup's list of heads (list number `lb` of those of the launch).
// FIN: the list is the whole group and dCB lies finished as bf16 (ssd_dcb_chunk.hip, or the tile pairs' kernel): the sums
// start from the in-chunk products, dC[l] from sum_{s <= l} dCB[l, s] B[s] and dB[s] from sum_{l >= s} dCB[l, s] C[l], and
// leave as the finished dB / dC in the operands' type.
template <int PT, int NK, int QT, int WV, bool IS_C, bool DET, bool FIN>
DEVI void dbc_body(const SsdParams &p, const int hb, const int lb, const int c, const int b, const int r0, DbcShared<PT, NK, WV> &shm) {
  constexpr int P = 16 * PT, N = 32 * NK, Q = 16 * QT, R = 16 * WV, NTL = N / 16, KK = P / 32;
  typedef __attribute__((address_space(3))) i16x4_t *lds_ptr;
  typedef short i16x8_t __attribute__((ext_vector_type(8)));

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int H = p.nheads, G = p.ngroups, L = p.seqlen;
  // the heads of a workgroup are `per` apart: workgroups in flight together touch neighbouring heads
  const int hpg = H / G, per = hpg / hb;
  const int grp = lb / per, h_first = grp * hpg + lb % per;
  const int t0 = c * Q;
  const int qlim = min(Q, L - t0);  // r0 < qlim: rows r0 .. r0 + R - 1 of the chunk are the workgroup's
  const float dsc = det_scale_of(p);
  const View4 gv = g_view(p);
  const bf16_t *rows_base = IS_C ? static_cast<const bf16_t *>(gv.ptr) + b * gv.bs : static_cast<const bf16_t *>(p.x) + b * p.x_bs;
  const int64_t r_ls = IS_C ? gv.ls : p.x_ls, r_hs = IS_C ? gv.hs : p.x_hs;
  const bf16_t *mats = static_cast<const bf16_t *>(IS_C ? p.states_lp : p.dstates_lp) + ((int64_t)b * p.nchunks + c) * H * P * N;

  // which of this lane's positions l0 .. l0 + 3 take part: inside the sequence, and in the one the carried state belongs to
  const int l0 = r0 + wave * 16 + 4 * g;
  uint32_t rows_ok = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    bool ok = l0 + r < qlim;
    if (p.seq_idx) {
      const int32_t *seq = p.seq_idx + (int64_t)b * L + t0;
      const int mine = seq[min(l0 + r, qlim - 1)];
      if (IS_C) {
        ok = ok && mine == (c > 0 ? seq[-1] : 0);
      } else {
        const int last = seq[qlim - 1];
        ok = ok && last >= 0 && mine == last;
      }
    }
    rows_ok |= (uint32_t)ok << r;
  }

  // ---- a head on its way to LDS: a wave moves 64 pieces of 16 bytes at a time.  Rows past the end of the sequence re-read
  // its last row; their weight is zero
  constexpr int RP = P / 8, MP = N / 8;  // pieces of a row of x / g, of the matrix
  constexpr int RI = R * RP / 64 / WV, MI = (P * MP / 64 + WV - 1) / WV;
  static_assert(RI * WV * 64 == R * RP, "whole instructions per wave");
  uint32_t r_off[RI], m_off[MI];
  // matrix rows: 32-byte units, permuted by the bits of the row that a half-wave's transposing read spans
  auto swz_row = [](int r, int columns) { return columns == 128 ? (r & 3) | (r >> 3 & 1) << 2 : (r >> 1 & 1) | (r >> 3 & 1) << 1; };
#pragma unroll
  for (int q = 0; q < RI; ++q) {
    const int id = (q * WV + wave) * 64 + lane, r = id / RP, piece = (id % RP) ^ ((r * RP >> 4) & (RP - 1));
    r_off[q] = (uint32_t)min(r, qlim - 1 - r0) * (uint32_t)(2 * r_ls) + piece * 16;
  }
#pragma unroll
  for (int q = 0; q < MI; ++q) {
    const int id = (q * WV + wave) * 64 + lane, r = id / MP;
    m_off[q] = r * (2 * N) + ((id % MP) ^ swz_row(r, N) << 1) * 16;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)&shm.first;
  const uint32_t lds1 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)&shm.second;
  typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
  f32x4 n_a, n_dt;
  float n_last = 0.f;
  const bf16_t *rows0 = rows_base + (int64_t)(t0 + r0) * r_ls;
  auto request_head = [&](int h, uint32_t lds) {
    const float *dA = p.dA_cumsum + (((int64_t)b * H + h) * p.nchunks + c) * Q;
    n_a = *(const GLOBAL_AS f32x4_any *)(dA + l0);
    if (!IS_C) {
      n_last = *(const GLOBAL_AS float *)(dA + Q - 1);
      n_dt = *(const GLOBAL_AS f32x4_any *)(p.dt_out + (((int64_t)b * H + h) * p.nchunks + c) * Q + l0);
    }
    const bf16_t *rr = rows0 + h * r_hs, *mm = mats + (int64_t)h * P * N;
#pragma unroll
    for (int q = 0; q < RI; ++q) load_async16(rr, r_off[q], lds + (q * WV + wave) * 1024);
#pragma unroll
    for (int q = 0; q < MI; ++q)
      if (P * MP / 64 % WV == 0 || q * WV + wave < P * MP / 64) load_async16(mm, m_off[q], lds + R * P * 2 + (q * WV + wave) * 1024);
  };

  // A step of the in-chunk products travels as a head does, P positions of the chunk in the place of P channels: for dC the
  // workgroup's rows of dCB and P rows of B, for dB P rows of dCB (its columns are the workgroup's positions) and of C.
  const bf16_t *dcb = FIN ? reinterpret_cast<const bf16_t *>(p.dCB) + (((int64_t)b * p.nchunks + c) * G + grp) * Q * Q : nullptr;
  const bf16_t *other = IS_C ? static_cast<const bf16_t *>(p.B) + b * p.B_bs + grp * p.B_gs : static_cast<const bf16_t *>(p.C) + b * p.C_bs + grp * p.C_gs;
  const int64_t other_ls = IS_C ? p.B_ls : p.C_ls;
  auto request_step = [&](int k0, uint32_t lds) {
    const bf16_t *rr = IS_C ? dcb + (int64_t)r0 * Q + k0 : dcb + (int64_t)k0 * Q + r0, *mm = other + (int64_t)(t0 + k0) * other_ls;
#pragma unroll
    for (int q = 0; q < RI; ++q) {
      const int id = (q * WV + wave) * 64 + lane;
      uint32_t off;
      if (IS_C) off = (id / RP) * (2 * Q) + ((id % RP) ^ ((id / RP * RP >> 4) & (RP - 1))) * 16;
      else off = (id / (R / 8)) * (2 * Q) + ((id % (R / 8)) ^ swz_row(id / (R / 8), R) << 1) * 16;
      load_async16(rr, off, lds + (q * WV + wave) * 1024);
    }
#pragma unroll
    for (int q = 0; q < MI; ++q) {
      const int id = (q * WV + wave) * 64 + lane, r = id / MP;
      const uint32_t off = (uint32_t)min(r, qlim - 1 - k0) * (uint32_t)(2 * other_ls) + ((id % MP) ^ swz_row(r, N) << 1) * 16;
      if (P * MP / 64 % WV == 0 || q * WV + wave < P * MP / 64) load_async16(mm, off, lds + R * P * 2 + (q * WV + wave) * 1024);
    }
  };
  const int k_first = IS_C ? 0 : r0, k_end = FIN ? (IS_C ? min(qlim, r0 + R) : qlim) : k_first;

  if (FIN) request_step(k_first, lds0);
  else request_head(h_first, lds0);

  // C at this lane's accumulator positions (rows 16 wave + 4 g + r, columns 16 nt + j): the wave's 16 rows go to
  // LDS as they lie in memory and a transposing read hands lane (j, g) column
  // 16 nt + j of rows 4 g .. 4 g + 3, which is that layout; cr(nt, r) is then one half of a register.
  u32x2 crp[IS_C ? NTL : 1];
  if (IS_C) {
    constexpr int CPP = 64 + 16;  // pitch of the patch (bf16): 16 rows x 64 columns at a time
    uint16_t *Cw = shm.c_patch[wave];
    const bf16_t *Cg = static_cast<const bf16_t *>(p.C) + b * p.C_bs + grp * p.C_gs;
#pragma unroll
    for (int half = 0; half < N / 64; ++half) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {  // 16 rows x 8 pieces of 8 columns
        const int id = lane + q * 64, rr = id >> 3, c8 = id & 7;
        const u32x4 v = *(const GLOBAL_AS u32x4 *)(Cg + (int64_t)(t0 + min(r0 + wave * 16 + rr, qlim - 1)) * p.C_ls + half * 64 + c8 * 8);
        *reinterpret_cast<u32x4 *>(&Cw[rr * CPP + c8 * 8]) = v;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const i16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)&Cw[(4 * g + (j >> 2)) * CPP + t * 16 + 4 * (j & 3)]);
        crp[half * 4 + t] = __builtin_bit_cast(u32x2, v);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    lds_barrier();  // every wave has its C values before other rows go where the patches are
  }
  auto cr = [&](int nt, int r) {
    const uint32_t w = (r & 2) ? crp[nt].y : crp[nt].x;
    return (r & 1) ? bf16_hi(w) : bf16_lo(w);
  };

  f32x4 sum[NTL];
#pragma unroll
  for (int nt = 0; nt < NTL; ++nt) sum[nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // lane constants of the operands' reads (bytes into a staged head).  k slots of lane group g: p = 32 kk + 8 g .. + 7
  const uint32_t a_at = (wave * 16 + j) * (2 * P), a_swz = ((j * RP >> 4) & (RP - 1)) ^ g;
  const uint32_t m_at = R * P * 2 + (8 * g + (j >> 2)) * (2 * N) + (j & 3) * 8 + swz_row(8 * g + (j >> 2), N) * 32;
  auto frag_tr = [&](uint32_t at, int row_bytes) {  // k slots of a 16 column unit, rows row_bytes apart
    const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(uintptr_t)at);
    const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(uintptr_t)(at + 4 * row_bytes));
    return __builtin_bit_cast(bf16x8_t, (i16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  uint32_t here = lds0, there = lds1;  // the head (or step) to work on, and the place of the one after it
  auto swap = [&]() { const uint32_t t = here; here = there; there = t; };

  if (FIN) {
    const uint32_t t_at = (8 * g + (j >> 2)) * (2 * R) + (j & 3) * 8 + ((wave ^ swz_row(8 * g + (j >> 2), R)) * 32);
#pragma unroll 1
    for (int k0 = k_first; k0 < k_end; k0 += P, swap()) {
      async_done<0>();
      lds_barrier();
      if (k0 + P < k_end) request_step(k0 + P, there);
      else request_head(h_first, there);
      // dCB is lower triangular, as whole tiles of 64 x 64: the others hold nothing
      const int mine = (r0 + wave * 16) >> 6;
      if (IS_C ? (k0 >> 6) > mine : (k0 >> 6) < mine) continue;
      bf16x8_t af[KK];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        if (IS_C) {
          af[kk] = *(__attribute__((address_space(3))) bf16x8_t *)(uintptr_t)(here + a_at + ((a_swz ^ (kk * 4)) * 16));
        } else {
          af[kk] = frag_tr(here + t_at + kk * (64 * R), 2 * R);
          if (k0 + P > qlim) {  // nothing comes from rows past the end of the sequence
            u32x4 v = __builtin_bit_cast(u32x4, af[kk]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int left = qlim - (k0 + kk * 32 + 8 * g + 2 * i);
              v[i] = left >= 2 ? v[i] : left == 1 ? v[i] & 0xffffu : 0u;
            }
            af[kk] = __builtin_bit_cast(bf16x8_t, v);
          }
        }
      }
#pragma unroll
      for (int nt = 0; nt < NTL; ++nt)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) sum[nt] = mfma_bf16(af[kk], frag_tr(((here + m_at) ^ (nt * 32)) + kk * (64 * N), 2 * N), sum[nt]);
    }
  }
  float(*const dda)[16] = shm.dda[wave];
#pragma unroll 1
  for (int hh = 0; hh < hb; ++hh, swap()) {
    async_done<0>();
    lds_barrier();  // this head is there, and nobody reads the one before it any more
    float wv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float w = IS_C ? fast_exp(n_a[r]) : fast_exp(fminf(n_last - n_a[r], 0.f)) * n_dt[r];
      wv[r] = (rows_ok >> r & 1) ? w : 0.f;
    }
    if (hh + 1 < hb) request_head(h_first + (hh + 1) * per, there);
    // (formed per head: carried across the loop, the addresses and the C values in fp32 do not fit the registers)
    uint32_t head = here + m_at;
    asm volatile("" : "+v"(head));
    if (IS_C) {
#pragma unroll
      for (int nt = 0; nt < NTL; ++nt) asm volatile("" : "+v"(crp[nt].x), "+v"(crp[nt].y));
    }
    f32x4 acc[NTL];
#pragma unroll
    for (int nt = 0; nt < NTL; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8_t af[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      af[kk] = *(__attribute__((address_space(3))) bf16x8_t *)(uintptr_t)(here + a_at + ((a_swz ^ (kk * 4)) * 16));
#pragma unroll
    for (int nt = 0; nt < NTL; ++nt) {
      const uint32_t m = head ^ (nt * 32);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) acc[nt] = mfma_bf16(af[kk], frag_tr(m + kk * (64 * N), 2 * N), acc[nt]);
    }
    if (IS_C) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float rs = 0.f;
#pragma unroll
        for (int nt = 0; nt < NTL; ++nt) rs = __builtin_fmaf(acc[nt][r], cr(nt, r), rs);
        rs *= wv[r];
        rs += dpp_f<DPP_ROW_SHR + 1>(0.f, rs);
        rs += dpp_f<DPP_ROW_SHR + 2>(0.f, rs);
        rs += dpp_f<DPP_ROW_SHR + 4>(0.f, rs);
        rs += dpp_f<DPP_ROW_SHR + 8>(0.f, rs);
        if (j == 15) dda[hh % DDA_RING][4 * g + r] = rs;
      }
    }
#pragma unroll
    for (int nt = 0; nt < NTL; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[nt][r] = __builtin_fmaf(acc[nt][r], wv[r], sum[nt][r]);

    // the wave's own rows of ddA_cumsum, whole rows of 16 positions at a time
    if (IS_C && (hh % DDA_RING == DDA_RING - 1 || hh == hb - 1)) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const int h0 = hh - hh % DDA_RING, l = r0 + wave * 16 + j;
      for (int k = g; h0 + k <= hh; k += 4) {
        const float d = dda[k][j];
        if (l < qlim && d != 0.f)
          acc_add<DET ? 1 : 0>(p.ddA_cumsum, p.det_ddA_cumsum, chunk_off(p, b, h_first + (h0 + k) * per, c) + l, d, dsc);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }

  if constexpr (FIN) {
    // ---- the finished sums leave in the operands' type, as whole 16-byte pieces of rows through a patch per wave
    constexpr int CPP = 64 + 16;
    lds_barrier();
    uint16_t *Cw = shm.c_patch[wave];
    bf16_t *dst = static_cast<bf16_t *>(IS_C ? p.dC : p.dB) + (IS_C ? b * p.dC_bs + grp * p.dC_gs : b * p.dB_bs + grp * p.dB_gs);
    const int64_t ls = IS_C ? p.dC_ls : p.dB_ls;
#pragma unroll
    for (int half = 0; half < N / 64; ++half) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) Cw[(4 * g + r) * CPP + t * 16 + j] = (uint16_t)f32_to_bf16_bits(sum[half * 4 + t][r]);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int q = 0; q < 2; ++q) {  // 16 rows x 8 pieces of 8 columns
        const int id = lane + q * 64, rr = id >> 3, c8 = id & 7;
        const u32x4 v = *reinterpret_cast<const u32x4 *>(&Cw[rr * CPP + c8 * 8]);
        if (r0 + wave * 16 + rr < qlim) *(GLOBAL_AS u32x4 *)(dst + (int64_t)(t0 + r0 + wave * 16 + rr) * ls + half * 64 + c8 * 8) = v;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  } else {
    // ---- the sums over this workgroup's heads join those of the others
    float *dst = IS_C ? p.dC32 : p.dB32;
    int64_t *shadow = IS_C ? p.det_dC : p.det_dB;
    // (the same adds as whole 128-byte lines of a row, through a patch per wave, measured no faster: 20 of a launch's
    // ~85 us go into these atomics, and it is their number that costs).  A workgroup that holds all heads of its group
    // is the only one to touch its rows of dB / dC, and the first of the backward pass to do so: it stores them, so
    // the caller need not clear them (ssd_bwd_overwrites reports this case).
    const bool alone = per == 1 && !DET;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int l = r0 + wave * 16 + 4 * g + r;
      if (l >= qlim) continue;
      const int64_t row = (((int64_t)b * L + t0 + l) * G + grp) * N + j;
      if (alone) {
#pragma unroll
        for (int nt = 0; nt < NTL; ++nt) dst[row + nt * 16] = sum[nt][r];
      } else {
#pragma unroll
        for (int nt = 0; nt < NTL; ++nt) acc_add<DET ? 1 : 0>(dst, shadow, row + nt * 16, sum[nt][r], dsc);
      }
    }
  }
}

// Both products in one launch: the first half of the workgroups along x takes dC, the second dB, each for one list
// of heads.  With lists twice as long as a launch per product would use to fill the chip there are half as many
// lists to add up with atomics, the two prologues run side by side, and the whole chip is busy to the end.
// (128 registers a wave; with 4 waves, 64 channels and 128 states LDS holds three workgroups)
template <int PT, int NK, int QT, int WV, bool DET, bool FIN>
__global__ __launch_bounds__(64 * WV, WV == 4 && PT * NK == 16 ? 3 : 4) void bwd_dbc_fused_kernel(const SsdParams p, const int hb) {
  __shared__ DbcShared<PT, NK, WV> shm;
  constexpr int PARTS = QT / WV;
  // the parts of a chunk are eight workgroups apart: on one XCD, whose L2 hands the second one the heads' matrices
  const int nlists = p.nheads / hb, id = blockIdx.y * gridDim.x + blockIdx.x, part = (id >> 3) % PARTS;
  const int unit = (id >> 3) / PARTS * 8 + (id & 7), x = unit % (2 * nlists), tile = unit / (2 * nlists);
  const int c = tile % p.nchunks, b = tile / p.nchunks, r0 = part * 16 * WV;
  if (b >= p.batch || c * 16 * QT + r0 >= p.seqlen) return;
  if (x < nlists) dbc_body<PT, NK, QT, WV, true, DET, FIN>(p, hb, x, c, b, r0, shm);
  else dbc_body<PT, NK, QT, WV, false, DET, FIN>(p, hb, x - nlists, c, b, r0, shm);
}

// Heads per workgroup for that launch: a divisor of the heads per group, MAXHB at most, by the same estimate as
// heads_per_workgroup with a fixed cost of 8 heads for the prologue and the final adds.  Both terms were measured on an earlier
// form, one workgroup of up to 16 waves per CU and chunk; this one has two or three on a CU, and two for a chunk of 256, so
// that the estimate is an order of the candidates rather than their times.
inline int dbc_heads_per_workgroup(const SsdParams &p) {
  const int hpg = p.nheads / p.ngroups, cus = cu_count();
  const int64_t tiles = (int64_t)p.nchunks * p.batch;
  int best = 1;
  double best_cost = 1e30;
  for (int hb = 1; hb <= MAXHB && hb <= hpg; ++hb) {
    if (hpg % hb) continue;
    const int64_t wgs = 2 * tiles * (p.nheads / hb);
    const double cost = (double)((wgs + cus - 1) / cus) * (8.0 + hb);
    if (cost < best_cost - 1e-9) best = hb, best_cost = cost;
  }
  return best;
}

template <int PT, int NK, bool DET, bool FIN> int launch_q(const SsdParams &p, hipStream_t s) {
  const int hb = FIN ? p.nheads / p.ngroups : dbc_heads_per_workgroup(p);
  // eight workgroups per part of a chunk side by side, a multiple of that where the other dimension would not hold the rest
  const int64_t units = 2 * (int64_t)(p.nheads / hb) * p.nchunks * p.batch, k = (units + 8 * 65535 - 1) / (8 * 65535);
  const int x = 8 * (int)k, y = (int)((units + x - 1) / x);
  switch (p.chunk_size) {
    case 256: hipLaunchKernelGGL((bwd_dbc_fused_kernel<PT, NK, 16, 8, DET, FIN>), dim3(2 * x, y), dim3(512), 0, s, p, hb); break;
    case 128: hipLaunchKernelGGL((bwd_dbc_fused_kernel<PT, NK, 8, 8, DET, FIN>), dim3(x, y), dim3(512), 0, s, p, hb); break;
    case 64: hipLaunchKernelGGL((bwd_dbc_fused_kernel<PT, NK, 4, 4, DET, FIN>), dim3(x, y), dim3(256), 0, s, p, hb); break;
    default: return MAMBA_E_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}
template <bool DET, bool FIN> int launch_pn(const SsdParams &p, hipStream_t s) {
  if (p.headdim == 64) return p.dstate == 128 ? launch_q<4, 4, DET, FIN>(p, s) : launch_q<4, 2, DET, FIN>(p, s);
  return p.dstate == 128 ? launch_q<2, 4, DET, FIN>(p, s) : launch_q<2, 2, DET, FIN>(p, s);
}

bool supported(const SsdParams *p) {
  if (p->dtype != MAMBA_BF16 || !p->dstates_lp || !p->states_lp) return false;
  if (p->headdim != 32 && p->headdim != 64) return false;
  if (p->dstate != 64 && p->dstate != 128) return false;
  if (p->chunk_size != 64 && p->chunk_size != 128 && p->chunk_size != 256) return false;
  // 16-byte pieces of the x and g rows
  const void *gptr = p->z ? static_cast<const void *>(p->gbuf) : p->dout;
  if (!gptr || !p->dB32 || !p->dC32 || !p->ddA_cumsum) return false;
  if (!aligned(p->x, 16) || !aligned(gptr, 16) || !aligned(p->dstates_lp, 16) || !aligned(p->states_lp, 16)) return false;
  if (p->x_bs % 8 || p->x_ls % 8 || p->x_hs % 8) return false;
  if (!p->z && (p->dout_bs % 8 || p->dout_ls % 8 || p->dout_hs % 8)) return false;
  if (!near_rows(p->x_ls) || (!p->z && !near_rows(p->dout_ls)) || (p->z && !near_rows((int64_t)p->nheads * p->headdim))) return false;
  if (p->batch > 65535 || p->nchunks > 65535) return false;
  return true;
}

}  // namespace

// True when ssd_bwd_dbc_fused_launch runs for this problem with one workgroup per (chunk, group): that workgroup
// stores its rows of dB32 / dC32.
bool ssd_bwd_dbc_fused_owns(const SsdParams *p) {
  if (p->det_scale || !supported(p)) return false;
  const int hb = dbc_heads_per_workgroup(*p);
  return hb == p->nheads / p->ngroups && 2 * (p->nheads / hb) <= 65535;
}

int ssd_bwd_dbc_fused_launch(const SsdParams *p, hipStream_t stream) {
  if (!supported(p)) return MAMBA_E_UNSUPPORTED;
  if (2 * (p->nheads / dbc_heads_per_workgroup(*p)) > 65535) return MAMBA_E_UNSUPPORTED;
  return p->det_scale ? launch_pn<true, false>(*p, stream) : launch_pn<false, false>(*p, stream);
}

// Whether ssd_bwd_dbc_finish_launch can follow a dCB stage that has left this problem's tiles as bf16: one workgroup per
// (chunk, group), 16-byte rows of B and C and of their gradients.
bool ssd_bwd_dbc_finishes(const SsdParams *p) {
  auto rows16 = [](const void *q, int64_t bs, int64_t ls, int64_t gs) { return q && aligned(q, 16) && bs % 8 == 0 && ls % 8 == 0 && gs % 8 == 0; };
  return ssd_bwd_dbc_fused_owns(p) && rows16(p->B, p->B_bs, p->B_ls, p->B_gs) && rows16(p->C, p->C_bs, p->C_ls, p->C_gs) &&
         near_rows(p->B_ls) && near_rows(p->C_ls) && rows16(p->dB, p->dB_bs, p->dB_ls, p->dB_gs) && rows16(p->dC, p->dC_bs, p->dC_ls, p->dC_gs) && aligned(p->dCB, 16);
}
int ssd_bwd_dbc_finish_launch(const SsdParams *p, hipStream_t stream) { return launch_pn<false, true>(*p, stream); }
