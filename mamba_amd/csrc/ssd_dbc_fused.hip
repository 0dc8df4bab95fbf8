// SSD backward, the chunk-state parts of dB and dC (and the ddA_cumsum rows that come with dC), for bf16 on gfx950
// (reference mamba_ssm/ops/triton/ssd_chunk_state.py:902 _chunk_state_bwd_db and ssd_chunk_scan.py:1451
// _chunk_scan_bwd_dC; the same sums as bwd_dB_state_wide_kernel / bwd_dC_state_wide_kernel in ssd_bwd.hip):
//     dB[s, n] += sum_{h in group} w_h[s] sum_p x[s, h, p] dS[h, p, n],   w_h[s] = dt_s exp(a_last - a_s), s in the
//                                                                          chunk's last sequence, else 0
//     dC[l, n] += sum_{h in group} v_h[l] sum_p g[l, h, p] H[h, p, n],    v_h[l] = exp(a_l), l in the sequence the
//                                                                          chunk was entered in, else 0
//     ddA_cumsum[h, l] += sum_n (v_h[l] sum_p g[l, h, p] H[h, p, n]) C[l, n]
// with dS the gradient of the state a chunk hands on and H the state it was entered with.  One launch does both: half
// of its workgroups take dC, half dB.  One workgroup of one wave
// per 16 positions works through a list of heads of one (batch, chunk, group): a head's rows (x or g, as they lie in
// memory) and its P x N matrix are staged in LDS, two heads deep, so that a single barrier per head separates the
// waves' products from the next commit and the loads of the head after next are in flight meanwhile.  Wave w owns
// positions 16 w .. 16 w + 15 and keeps their sum over the heads in registers (fp32, N / 16 tiles); the per-position
// weight is applied to the fp32 product of each head, not to the bf16 operand.  The matrix is the B operand with
// k = p: its fragments come from transposing LDS reads.
//
// Where a workgroup's list is the whole group and the dCB stage has left its tiles in bf16, the sums start from the in-chunk
// products (FIN), in the same registers, and leave as the finished dB / dC: the fp32 sums are neither written nor read, and
// the stage that added the products to them is gone.  16384 positions, 128 heads in 8 groups, chunk 256: 300 us against 256
// here and 185 there; 2 x 4096, 40 heads in 8 groups, chunk 128: 65 against 60 and 41.
#include "ssd_common.hpp"

namespace {

DEVI f32x4 mfma_bf16(bf16x8_t a, bf16x8_t b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

constexpr int MAXHB = 40;  // heads per workgroup at most (dbc_heads_per_workgroup never picks more)

// LDS of one staged head: rows of x / g (pitch P + 8: 16-byte aligned pieces), the matrix (pitch N + 16: the
// transposing reads of a half-wave cover all 64 banks once), the weight per position.
template <int PT, int NK, int QT> struct DbcBuf {
  uint16_t Rs[16 * QT * (16 * PT + 8)];
  uint16_t Ms[16 * PT * (32 * NK + 16)];
  float w[16 * QT];
};

// LDS of a launch: the two staged heads, and what lies in their place before the first and after the last one.
template <int PT, int NK, int QT> union __align__(16) DbcShared {
  static constexpr int N = 32 * NK, Q = 16 * QT, BP = N + 16, DP = Q + 16;
  static constexpr int BR = 64;                   // rows of B staged at a time
  DbcBuf<PT, NK, QT> buf[2];
  uint16_t c_patch[QT][16 * (64 + 16)];          // a wave's 16 rows x 64 columns
  uint16_t b_rows[BR * BP];                      // dC: rows of B
  struct {
    uint16_t dcb[64 * DP], c_rows[64 * BP];      // dB: 64 rows of dCB and of C
  } l;
};

// One of the two products for the workgroup's list of heads (list number `lb` of those of the launch).
// FIN: the list is the whole group and dCB lies finished as bf16 (ssd_dcb_chunk.hip, or the tile pairs' kernel): the sums
// start from the in-chunk products, dC[l] from sum_{s <= l} dCB[l, s] B[s] and dB[s] from sum_{l >= s} dCB[l, s] C[l], and
// leave as the finished dB / dC in the operands' type.
template <int PT, int NK, int QT, bool IS_C, bool DET, bool FIN>
DEVI void dbc_body(const SsdParams &p, const int hb, const int lb, DbcShared<PT, NK, QT> &shm, float (*dda_s)[16 * QT]) {
  constexpr int P = 16 * PT, N = 32 * NK, Q = 16 * QT, NT = 64 * QT, NTL = N / 16, KK = P / 32;
  constexpr int XP = P + 8, BP = N + 16;
  using Buf = DbcBuf<PT, NK, QT>;
  Buf *const buf = shm.buf;
  typedef __attribute__((address_space(3))) i16x4_t *lds_ptr;
  typedef short i16x8_t __attribute__((ext_vector_type(8)));

  int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int j = lane & 15, g = lane >> 4;
  const int H = p.nheads, G = p.ngroups, L = p.seqlen;
  // the heads of a workgroup are `per` apart: workgroups in flight together touch neighbouring heads
  const int hpg = H / G, per = hpg / hb;
  const int grp = lb / per, h_first = grp * hpg + lb % per;
  const int c = blockIdx.y, b = blockIdx.z;
  const int t0 = c * Q;
  const int qlim = min(Q, L - t0);
  const float dsc = det_scale_of(p);
  const View4 gv = g_view(p);
  const bf16_t *rows_base = IS_C ? static_cast<const bf16_t *>(gv.ptr) + b * gv.bs : static_cast<const bf16_t *>(p.x) + b * p.x_bs;
  const int64_t r_ls = IS_C ? gv.ls : p.x_ls, r_hs = IS_C ? gv.hs : p.x_hs;
  const bf16_t *mats = static_cast<const bf16_t *>(IS_C ? p.states_lp : p.dstates_lp) + ((int64_t)b * p.nchunks + c) * H * P * N;

  // position tid takes part: inside the sequence, and in the sequence the carried state belongs to
  bool row_ok = false;
  if (tid < Q) {
    row_ok = tid < qlim;
    if (p.seq_idx && row_ok) {
      const int32_t *seq = p.seq_idx + (int64_t)b * L + t0;
      if (IS_C) {
        row_ok = seq[tid] == (c > 0 ? seq[-1] : 0);
      } else {
        const int last = seq[qlim - 1];
        row_ok = last >= 0 && seq[tid] == last;
      }
    }
  }

  // ---- global -> registers -> LDS in 16-byte pieces, no branch around a load (rows past the end of the sequence
  // re-read its last row; their weight is zero)
  constexpr int GCH = Q * P / 8 / NT;
  static_assert(GCH * NT * 8 == Q * P, "whole pieces per thread");
  constexpr int HCH = (P * N / 8 + NT - 1) / NT;
  static_assert(NT >= Q, "one position per thread");
  u32x4 rregs[GCH], mregs[HCH];
  float sc_a = 0.f, sc_alast = 0.f, sc_dt = 0.f;
  auto load_head = [&](int h) {
    const bf16_t *rr = rows_base + h * r_hs;
#pragma unroll
    for (int q = 0; q < GCH; ++q) {
      const int id = tid + q * NT, r = id / (P / 8), c8 = id % (P / 8);
      rregs[q] = *(const GLOBAL_AS u32x4 *)(rr + (int64_t)(t0 + min(r, qlim - 1)) * r_ls + c8 * 8);
    }
    const bf16_t *mm = mats + (int64_t)h * P * N;
#pragma unroll
    for (int q = 0; q < HCH; ++q) mregs[q] = *(const GLOBAL_AS u32x4 *)(mm + (int64_t)min(tid + q * NT, P * N / 8 - 1) * 8);
    const float *dA = p.dA_cumsum + (((int64_t)b * H + h) * p.nchunks + c) * Q;
    const int pos = min(tid, Q - 1);
    sc_a = *(const GLOBAL_AS float *)(dA + pos);
    if (!IS_C) {
      sc_alast = *(const GLOBAL_AS float *)(dA + Q - 1);
      sc_dt = *(const GLOBAL_AS float *)(p.dt_out + (((int64_t)b * H + h) * p.nchunks + c) * Q + pos);
    }
  };
  auto commit_head = [&](Buf &B) {
#pragma unroll
    for (int q = 0; q < GCH; ++q) {
      const int id = tid + q * NT, r = id / (P / 8), c8 = id % (P / 8);
      *reinterpret_cast<u32x4 *>(&B.Rs[r * XP + c8 * 8]) = rregs[q];
    }
#pragma unroll
    for (int q = 0; q < HCH; ++q) {
      const int id = tid + q * NT, pp = id / (N / 8), c8 = id % (N / 8);
      if (id < P * N / 8) *reinterpret_cast<u32x4 *>(&B.Ms[pp * BP + c8 * 8]) = mregs[q];
    }
    if (tid < Q) {
      const float wv = IS_C ? fast_exp(sc_a) : fast_exp(fminf(sc_alast - sc_a, 0.f)) * sc_dt;
      B.w[tid] = row_ok ? wv : 0.f;
    }
  };

  load_head(h_first);

  // C at this lane's accumulator positions (rows 16 wave + 4 g + r, columns 16 nt + j): the wave's 16 rows go to
  // LDS as they lie in memory (the staging buffers are still empty) and a transposing read hands lane (j, g) column
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
        const u32x4 v = *(const GLOBAL_AS u32x4 *)(Cg + (int64_t)(t0 + min(wave * 16 + rr, qlim - 1)) * p.C_ls + half * 64 + c8 * 8);
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
    lds_barrier();  // every wave has its C values before the first head is committed over the patches
  }
  auto cr = [&](int nt, int r) {
    const uint32_t w = (r & 2) ? crp[nt].y : crp[nt].x;
    return (r & 1) ? bf16_hi(w) : bf16_lo(w);
  };

  f32x4 sum[NTL];
#pragma unroll
  for (int nt = 0; nt < NTL; ++nt) sum[nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  if constexpr (FIN) {
    // k slots of lane group g, in either operand: positions 4 g .. + 3 of 32, then 16 further on
    auto frag_tr = [&](const uint16_t *rows, int pitch, int k0, int col0) {
      const uint16_t *src = &rows[(k0 + 4 * g + (j >> 2)) * pitch + col0 + 4 * (j & 3)];
      const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)src), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(src + 16 * pitch));
      return __builtin_bit_cast(bf16x8_t, (i16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    const bf16_t *dcb = reinterpret_cast<const bf16_t *>(p.dCB) + (((int64_t)b * p.nchunks + c) * G + grp) * Q * Q;
    // Rows of B (C), ROWS at a time, go through registers into LDS: the next ones are requested before the products of the
    // ones that lie there.  Zeros past the end of the sequence (0 times what lies there would be no zero).
    constexpr int ROWS = IS_C ? DbcShared<PT, NK, QT>::BR : 64, RC = (ROWS * (N / 8) + NT - 1) / NT;
    u32x4 rows[RC];
    const bf16_t *src = IS_C ? static_cast<const bf16_t *>(p.B) + b * p.B_bs + grp * p.B_gs : static_cast<const bf16_t *>(p.C) + b * p.C_bs + grp * p.C_gs;
    const int64_t src_ls = IS_C ? p.B_ls : p.C_ls;
    auto piece = [&](int q) { return min(tid + q * NT, ROWS * (N / 8) - 1); };
    auto request_rows = [&](int r0) {
#pragma unroll
      for (int q = 0; q < RC; ++q)
        rows[q] = *(const GLOBAL_AS u32x4 *)(src + (int64_t)(t0 + min(r0 + piece(q) / (N / 8), qlim - 1)) * src_ls + piece(q) % (N / 8) * 8);
    };
    auto commit_rows = [&](uint16_t *dst, int r0) {
#pragma unroll
      for (int q = 0; q < RC; ++q) {
        const int r = piece(q) / (N / 8), c8 = piece(q) % (N / 8);
        const bool live = r0 + r < qlim;
        const u32x4 v = {live ? rows[q].x : 0u, live ? rows[q].y : 0u, live ? rows[q].z : 0u, live ? rows[q].w : 0u};
        *reinterpret_cast<u32x4 *>(&dst[r * BP + c8 * 8]) = v;
      }
    };
    if constexpr (IS_C) {
      constexpr int KB = ROWS / 32;
      const bf16_t *row = dcb + (int64_t)(wave * 16 + j) * Q + 4 * g;
      u32x2 a[KB][2];  // the wave's rows of dCB: the A operand as it lies in memory
      auto request = [&](int s0) {
        request_rows(s0);
#pragma unroll
        for (int kk = 0; kk < KB; ++kk) {  // (nothing is read past the 32 positions that hold the wave's last row)
          const uint32_t k0 = min(s0 + kk * 32, wave * 16 & ~31);
          a[kk][0] = *(const GLOBAL_AS u32x2 *)(row + k0);
          a[kk][1] = *(const GLOBAL_AS u32x2 *)(row + k0 + 16);
        }
      };
      request(0);
#pragma unroll 1
      for (int s0 = 0; s0 < qlim; s0 += ROWS) {
        lds_barrier();
        commit_rows(shm.b_rows, s0);
        bf16x8_t af[KB];
#pragma unroll
        for (int kk = 0; kk < KB; ++kk) af[kk] = __builtin_bit_cast(bf16x8_t, u32x4{a[kk][0].x, a[kk][0].y, a[kk][1].x, a[kk][1].y});
        lds_barrier();
        if (s0 + ROWS < qlim) request(s0 + ROWS);
        // (up to the 32 positions that hold the wave's last row: dCB is zero above the diagonal there)
#pragma unroll
        for (int kk = 0; kk < KB; ++kk)
          if (s0 + kk * 32 < wave * 16 + 16) {
#pragma unroll
            for (int nt = 0; nt < NTL; ++nt) sum[nt] = mfma_bf16(af[kk], frag_tr(shm.b_rows, BP, kk * 32, nt * 16), sum[nt]);
          }
      }
    } else {
      constexpr int DP = DbcShared<PT, NK, QT>::DP, RD = 64 * (Q / 8) / NT;
      static_assert(RD * NT == 64 * (Q / 8), "whole pieces per thread");
      u32x4 drows[RD];
      auto request = [&](int l0) {
        request_rows(l0);
#pragma unroll
        for (int q = 0; q < RD; ++q)  // (the tiles above the diagonal are nothing's, and neither read nor used)
          drows[q] = *(const GLOBAL_AS u32x4 *)(dcb + (int64_t)(l0 + (tid + q * NT) / (Q / 8)) * Q + min((tid + q * NT) % (Q / 8) * 8, l0 + 56));
      };
      request(0);
#pragma unroll 1
      for (int l0 = 0; l0 < qlim; l0 += 64) {
        lds_barrier();
        commit_rows(shm.l.c_rows, l0);
#pragma unroll
        for (int q = 0; q < RD; ++q)
          *reinterpret_cast<u32x4 *>(&shm.l.dcb[(tid + q * NT) / (Q / 8) * DP + (tid + q * NT) % (Q / 8) * 8]) = drows[q];
        lds_barrier();
        if (l0 + 64 < qlim) request(l0 + 64);
        if (l0 + 64 > wave * 16) {
#pragma unroll
          for (int k0 = 0; k0 < 64; k0 += 32) {
            const bf16x8_t a = frag_tr(shm.l.dcb, DP, k0, wave * 16);
#pragma unroll
            for (int nt = 0; nt < NTL; ++nt) sum[nt] = mfma_bf16(a, frag_tr(shm.l.c_rows, BP, k0, nt * 16), sum[nt]);
          }
        }
      }
    }
    lds_barrier();  // the first head goes where these rows are
  }

  commit_head(buf[0]);
  load_head(h_first + min(1, hb - 1) * per);
  lds_barrier();

#pragma unroll 1
  for (int hh = 0; hh < hb; ++hh) {
    // the thread's indices pass through an empty asm once per head, so that the addresses derived from them are
    // computed where they are used instead of being carried (or spilled) across the loop over the heads
    asm volatile("" : "+v"(tid), "+v"(lane), "+v"(j), "+v"(g));
    Buf &B = buf[hh & 1];
    f32x4 acc[NTL];
#pragma unroll
    for (int nt = 0; nt < NTL; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      // k slots of lane group g: p = 32 kk + 4 g .. + 3, then 16 further on (both operands alike)
      const uint16_t *ar = &B.Rs[(wave * 16 + j) * XP + kk * 32 + 4 * g];
      const u32x2 a_lo = *reinterpret_cast<const u32x2 *>(ar), a_hi = *reinterpret_cast<const u32x2 *>(ar + 16);
      const bf16x8_t af = __builtin_bit_cast(bf16x8_t, u32x4{a_lo.x, a_lo.y, a_hi.x, a_hi.y});
#pragma unroll
      for (int nt = 0; nt < NTL; ++nt) {
        const uint16_t *src = &B.Ms[(kk * 32 + 4 * g + (j >> 2)) * BP + nt * 16 + 4 * (j & 3)];
        const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)src);
        const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(src + 16 * BP));
        const bf16x8_t bfr = __builtin_bit_cast(bf16x8_t, (i16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        acc[nt] = mfma_bf16(af, bfr, acc[nt]);
      }
    }
    const f32x4 wv = *reinterpret_cast<const f32x4 *>(&B.w[wave * 16 + 4 * g]);
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
        if (j == 15) dda_s[hh][wave * 16 + 4 * g + r] = rs;
      }
    }
#pragma unroll
    for (int nt = 0; nt < NTL; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[nt][r] = __builtin_fmaf(acc[nt][r], wv[r], sum[nt][r]);

    // the next head's operands go to the other buffer (last read one head ago, before the barrier that ended that
    // head); the loads of the head after it follow, then the one barrier of this head
    commit_head(buf[(hh + 1) & 1]);
    load_head(h_first + min(hh + 2, hb - 1) * per);
    lds_barrier();
  }

  if constexpr (FIN) {
    // ---- the finished sums leave in the operands' type, as whole 16-byte pieces of rows through a patch per wave (the
    // staged heads are dead: the last commit went there before the last barrier, and nobody reads it)
    constexpr int CPP = 64 + 16;
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
        if (wave * 16 + rr < qlim) *(GLOBAL_AS u32x4 *)(dst + (int64_t)(t0 + wave * 16 + rr) * ls + half * 64 + c8 * 8) = v;
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
      const int l = wave * 16 + 4 * g + r;
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
  if (IS_C) {
    for (int idx = tid; idx < hb * Q; idx += NT) {
      const int hh = idx / Q, l = idx % Q;
      const float d = dda_s[hh][l];
      if (l < qlim && d != 0.f)
        acc_add<DET ? 1 : 0>(p.ddA_cumsum, p.det_ddA_cumsum, chunk_off(p, b, h_first + hh * per, c) + l, d, dsc);
    }
  }
}

// Both products in one launch: the first half of the workgroups along x takes dC, the second dB, each for one list
// of heads.  With lists twice as long as a launch per product would use to fill the chip there are half as many
// lists to add up with atomics, the two prologues run side by side, and the whole chip is busy to the end.
template <int PT, int NK, int QT, bool DET, bool FIN>
__global__ __launch_bounds__(64 * QT) void bwd_dbc_fused_kernel(const SsdParams p, const int hb) {
  __shared__ DbcShared<PT, NK, QT> shm;
  __shared__ float dda_s[MAXHB][16 * QT];  // the heads' ddA_cumsum rows of the dC product, flushed at the end
  const int nlists = gridDim.x / 2;
  if ((int)blockIdx.x < nlists) dbc_body<PT, NK, QT, true, DET, FIN>(p, hb, blockIdx.x, shm, dda_s);
  else dbc_body<PT, NK, QT, false, DET, FIN>(p, hb, blockIdx.x - nlists, shm, dda_s);
}

// Heads per workgroup for that launch: a divisor of the heads per group, MAXHB at most, by the same estimate as
// heads_per_workgroup with the fixed cost these kernels measure (prologue and final adds: about 8 heads' worth).
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
  dim3 grid(2 * (p.nheads / hb), p.nchunks, p.batch);
  switch (p.chunk_size) {
    case 256: hipLaunchKernelGGL((bwd_dbc_fused_kernel<PT, NK, 16, DET, FIN>), grid, dim3(1024), 0, s, p, hb); break;
    case 128: hipLaunchKernelGGL((bwd_dbc_fused_kernel<PT, NK, 8, DET, FIN>), grid, dim3(512), 0, s, p, hb); break;
    case 64: hipLaunchKernelGGL((bwd_dbc_fused_kernel<PT, NK, 4, DET, FIN>), grid, dim3(256), 0, s, p, hb); break;
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
         rows16(p->dB, p->dB_bs, p->dB_ls, p->dB_gs) && rows16(p->dC, p->dC_bs, p->dC_ls, p->dC_gs) && aligned(p->dCB, 16);
}
int ssd_bwd_dbc_finish_launch(const SsdParams *p, hipStream_t stream) { return launch_pn<false, true>(*p, stream); }
