// SSD backward, the gradient of the chunk's C B^T and the in-chunk share of ddA_cumsum, for bf16 on gfx950 (reference
// mamba_ssm/ops/triton/ssd_chunk_scan.py:1524 _chunk_scan_bwd_dcb and :1638 _chunk_scan_bwd_ddAcs_stable; the same sums as
// bwd_dcb_rows_kernel in ssd_bwd.hip, which works a 64 x 64 tile pair per workgroup):
//     dCB[l, s] = sum_{h in group} (sum_p g[l, h, p] x[s, h, p]) dt_s exp(a_l - a_s),     s <= l in one sequence
//     ddA_cumsum[h, l] += sum_s w[l, s] - sum_l' w[l', l],   w = (the head's term of dCB) * (C B^T)
// One workgroup holds the whole lower triangle of one (batch, chunk, group): its QT (QT + 1) / 2 blocks of 16 x 16 are
// dealt to QT / 2 waves as QT + 1 blocks each, wave w taking rows of tiles w and QT - 1 - w, and a block's sum over the
// heads and its value of C B^T stay in registers (2 x 4 per lane and block: 136 of the 256 that two waves per SIMD have at
// QT = 16).  So a head's g and x rows are read once, where the tile pairs of a chunk of 256 read them 2.5 times (the L2
// serves most of that, but each reading is a wait of its own), and a head takes one barrier for the whole chunk: its
// operands lie two heads deep in LDS.
// What bounds it: the waves' own instructions (4 batch rows x 4096 positions x 80 heads x 64, 20 heads per workgroup: some
// wave of a SIMD issues in 83 % of the cycles, ~1000 instructions per head and wave, 20 vector ones per block for the four
// weights of a lane; the matrix cores are busy in 10 %, the LDS in 28 %).  5 us per head there, 3.5 TB/s; within a backward
// pass 172 -> 119 us, with the launch that formed C B^T gone as well (9 us); 32768 positions x 64 heads in 8 groups: 298 ->
// 208 (4.1 TB/s).  Tried and not kept: column sums added with LDS atomics (172 us); ddA_cumsum stored instead of added with
// atomics, both operands requested at the start of a head instead of one in each half (122 - 130); factors selected instead
// of the one branch where a wave passes from its long to its short row (119 against 118).
#include "ssd_common.hpp"

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// What a decay's exponent (base 2) may reach: an exponential that stays finite, for the zeros of a masked C B^T to be
// multiplied by.
constexpr float kGrowth = 126.f;

DEVI f32x4 mfma_bf16(bf16x8_t a, bf16x8_t b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// x + y folded: lanes 0 - 31 get the sum of x over the two halves of the wave, lanes 32 - 63 that of y
DEVI float fold32(float x, float y) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y), false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
// the same for neighbouring rows of 16 lanes: even rows get the sums of x over a pair of rows, odd rows those of y
DEVI float fold16(float x, float y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y), false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}

// FORM_CB: no CB buffer, the workgroup forms its blocks of C B^T itself, with the loop that forms the heads' products.
// lp: this workgroup holds all heads of its group (nsplit 1), and the next stage takes the finished blocks as bf16 (what
// its MFMA operand would round them to anyway): they are stored as bf16, packed at the start of the dCB buffer.
template <int PT, int QT, bool FORM_CB>
__global__ __launch_bounds__(32 * QT) void bwd_dcb_chunk_kernel(const SsdParams p, const int lp, const int nsplit) {
  constexpr int P = 16 * PT, Q = 16 * QT, NW = QT / 2, NT = 64 * NW, NBK = QT + 1;
  constexpr int PC = P / 8, KS = P / 32, NP = Q * PC / NT;  // 16-byte pieces of a row; k slices; pieces per thread and operand
  static_assert(NP * NT == Q * PC && NT >= Q, "whole pieces and one position per thread");
  // A head's operands, two heads deep.  Rows lie unpadded, their pieces exchanged so that the 16 rows of a fragment read
  // cover the 64 banks once.
  struct Buf {
    uint16_t g[Q * P], x[Q * P];  // rows of g (C while C B^T is formed) and of x (B)
    float el[Q];                  // exp(a_l - a at the first position of l's tile)
    float a2[Q];                  // a log2 e
    f32x2 col[Q];                 // a_s log2 e, dt_s
  };
  __shared__ __align__(16) Buf buf[2];
  // A head's ddA_cumsum shares: the row sums by position, and a wave's column sums as its long row's columns followed by
  // its short row's.
  __shared__ float rowp[2][Q], colp[2][NW * NBK * 16];

  int tid = threadIdx.x, lane = tid & 63, i = lane & 15, gq = lane >> 4;
  int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int L = p.seqlen, H = p.nheads, G = p.ngroups, hpg = H / G;
  const int g = blockIdx.x / nsplit, hs = blockIdx.x % nsplit, c = blockIdx.y, b = blockIdx.z;
  const int nh = (hpg - hs + nsplit - 1) / nsplit, h0 = g * hpg + hs;  // the list's heads lie nsplit apart
  const int t0 = c * Q, qlim = min(Q, L - t0);

  // Blocks of this wave, whose rows of tiles are the short one w and the long one QT - 1 - w: k < NW the long row's first
  // NW columns; NW .. QT - 2 the rest of it, then the short row's columns (which of the two depends on the wave: a block's
  // data are reached by address and its factors selected, there is no branch); QT - 1 the long row's diagonal, QT the
  // short row's.
  auto is_long = [&](int k) { return k < NW || k == QT - 1 || (k < QT && k < QT - 1 - wave); };
  auto row_tile = [&](int k) { return is_long(k) ? QT - 1 - wave : wave; };
  auto col_tile = [&](int k) { return k < NW ? k : k >= QT - 1 ? row_tile(k) : k - (is_long(k) ? 0 : QT - 1 - wave); };

  // A thread's pieces of one operand (rows past the end of the sequence re-read its last row; what they produce is
  // masked): at the same places of every head's rows.
  typedef const GLOBAL_AS char *gptr;
  auto fetch = [&](u32x4(&dst)[NP], const bf16_t *base, int64_t ls) {
    const gptr src = (gptr)(base + (int64_t)t0 * ls);
    const uint32_t r = (uint32_t)tid / PC, c8 = (uint32_t)tid % PC;
#pragma unroll
    for (int q = 0; q < NP; ++q)
      dst[q] = *(const GLOBAL_AS u32x4 *)(src + (min(r + q * (NT / PC), (uint32_t)qlim - 1u) * (uint32_t)ls + c8 * 8u) * 2u);
  };
  auto swizzled = [&](uint32_t r, uint32_t c8) { return r * P + (c8 ^ (r / (16 / PC) % PC)) * 8; };
  static_assert(NT / PC % 16 == 0, "a thread's pieces lie at one place of the exchange");
  auto commit = [&](uint16_t *dst, const u32x4(&src)[NP]) {
    uint16_t *to = dst + swizzled((uint32_t)tid / PC, (uint32_t)tid % PC);
#pragma unroll
    for (int q = 0; q < NP; ++q) *reinterpret_cast<u32x4 *>(to + q * (NT / PC) * P) = src[q];
  };
  const View4 gv = g_view(p);
  u32x4 piece[NP];
  auto fetch_g = [&](int hl) { fetch(piece, static_cast<const bf16_t *>(gv.ptr) + b * gv.bs + (h0 + hl * nsplit) * gv.hs, gv.ls); };
  auto fetch_x = [&](int hl) { fetch(piece, static_cast<const bf16_t *>(p.x) + b * p.x_bs + (h0 + hl * nsplit) * p.x_hs, p.x_ls); };
  float sc_a = 0.f, sc_ref = 0.f, sc_dt = 0.f;
  auto fetch_scalars = [&](int hl) {
    const float *dA = chunk_row(p.dA_cumsum, p, b, h0 + hl * nsplit, c), *dt = chunk_row(p.dt_out, p, b, h0 + hl * nsplit, c);
    const int pos = min(tid, Q - 1);
    sc_a = *(const GLOBAL_AS float *)(dA + pos);
    sc_ref = *(const GLOBAL_AS float *)(dA + (pos & ~15));
    sc_dt = *(const GLOBAL_AS float *)(dt + pos);
  };
  auto commit_scalars = [&](Buf &to) {
    const int pos = min(tid, Q - 1);  // (the threads past the chunk write its last position's values once more)
    to.el[pos] = fast_exp2(fminf((sc_a - sc_ref) * kLog2e, kGrowth));
    to.a2[pos] = sc_a * kLog2e;
    to.col[pos] = f32x2{sc_a * kLog2e, sc_dt};
  };

  // The products of the wave's blocks in turn on a staged pair of operands, each handed to f(k, product, the block's
  // column data); mid() runs after half of them.  A block's fragments are requested two blocks ahead and its MFMAs issued
  // one ahead, so that neither is waited for; nothing else moves across a block's end, which bounds the registers.
  struct Frag {
    bf16x8_t row[KS], col[KS];
  };
  const int frag0 = (int)swizzled(i, gq);  // (the k slices differ in the exchanged bits alone)
  auto load_frag = [&](const Buf &at, int k, Frag &o, bool rows) {
    // (uniform offsets: scalar registers)
    const int ro = __builtin_amdgcn_readfirstlane(row_tile(k) * (16 * P)), co = __builtin_amdgcn_readfirstlane(col_tile(k) * (16 * P));
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      const int at8 = frag0 ^ (kk * 32);
      if (rows) o.row[kk] = *reinterpret_cast<const bf16x8_t *>(&at.g[ro + at8]);
      o.col[kk] = *reinterpret_cast<const bf16x8_t *>(&at.x[co + at8]);
    }
    return at.col[__builtin_amdgcn_readfirstlane(col_tile(k) * 16) + i];
  };
  auto products = [&](const Buf &at, auto init, auto f, auto mid) {
    Frag fr;
    f32x2 sc = load_frag(at, 0, fr, true);
    f32x4 v = init(0);
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) v = mfma_bf16(fr.row[kk], fr.col[kk], v);
    f32x2 sc1 = load_frag(at, 1, fr, 1 >= NW);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < NBK; ++k) {
      f32x4 v1 = {0.f, 0.f, 0.f, 0.f};
      f32x2 sc2 = {0.f, 0.f};
      if (k < QT) {
        v1 = init(k + 1);
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) v1 = mfma_bf16(fr.row[kk], fr.col[kk], v1);
      }
      if (k + 1 < QT) sc2 = load_frag(at, k + 2, fr, k + 2 >= NW);
      f(k, v, sc);
      v = v1, sc = sc1, sc1 = sc2;
      __builtin_amdgcn_sched_barrier(0);
      if (k == NBK / 2) {
        mid();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  // Sequence ids of the chunk's positions, in a buffer that is free when they are needed; a row past the end of the
  // sequence belongs to none of the columns before it.
  int *seq_s = reinterpret_cast<int *>(buf[1].x);
  auto write_seq = [&]() {
    if (tid < Q) seq_s[tid] = tid >= qlim ? INT32_MIN + tid : p.seq_idx ? p.seq_idx[(int64_t)b * L + t0 + tid] : 0;
  };
  // The elements of block k that take part keep their value, the others (s > l, another sequence, past the end) get 0.
  auto mask = [&](int k, f32x4 v) {
    const i32x4 sl = *reinterpret_cast<const i32x4 *>(&seq_s[row_tile(k) * 16 + gq * 4]);
    const int ss = seq_s[col_tile(k) * 16 + i];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = sl[r] == ss && (k < QT - 1 || gq * 4 + r >= i) ? v[r] : 0.f;
    return v;
  };

  f32x4 sum[NBK], cb[NBK];
#pragma unroll
  for (int k = 0; k < NBK; ++k) sum[k] = cb[k] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch_scalars(0);
  if constexpr (FORM_CB) {
    const bf16_t *Cg = static_cast<const bf16_t *>(p.C) + b * p.C_bs + g * p.C_gs, *Bg = static_cast<const bf16_t *>(p.B) + b * p.B_bs + g * p.B_gs;
#pragma unroll 1
    for (int n0 = 0; n0 < p.dstate; n0 += P) {
      u32x4 bp[NP];
      fetch(piece, Cg + n0, p.C_ls);
      fetch(bp, Bg + n0, p.B_ls);
      lds_barrier();
      commit(buf[0].g, piece);
      commit(buf[0].x, bp);
      lds_barrier();
      products(buf[0], [&](int k) { return cb[k]; }, [&](int k, const f32x4 &v, const f32x2 &) { cb[k] = v; }, [] {});
    }
  } else {
    const float *CB = p.CB + (((int64_t)b * p.nchunks + c) * G + g) * Q * Q;
#pragma unroll
    for (int k = 0; k < NBK; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) cb[k][r] = CB[(row_tile(k) * 16 + gq * 4 + r) * Q + col_tile(k) * 16 + i];
  }
  write_seq();
  fetch_g(0);
  lds_barrier();
#pragma unroll
  for (int k = 0; k < NBK; ++k) {
    cb[k] = mask(k, cb[k]);
    __builtin_amdgcn_sched_barrier(0);
  }
  commit(buf[0].g, piece);
  fetch_x(0);
  commit(buf[0].x, piece);
  commit_scalars(buf[0]);
  lds_barrier();

  // a head's ddA_cumsum share of position tid, once every wave has left its row and column sums
  auto combine = [&](int hl) {
    if (tid < Q) {
      const float *const cp = colp[hl & 1];
      const int st = tid >> 4, sts = min(st, NW - 1);
      float d = rowp[hl & 1][tid];
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float v = cp[w * NBK * 16 + tid], u = cp[(w * NBK + QT - w + sts) * 16 + (tid & 15)];
        d -= st < QT - w ? v : 0.f;  // (the waves whose long row, whose short row has column tile st)
        d -= st <= w ? u : 0.f;
      }
      acc_add<0>(p.ddA_cumsum, nullptr, chunk_off(p, b, h0 + hl * nsplit, c) + tid, d, 0.f);
    }
  };

#pragma unroll 1
  for (int hl = 0; hl < nh; ++hl) {
    // the thread's indices are new values to the compiler in every head: addresses derived from them are computed where
    // they are used instead of being carried across the loop
    asm volatile("" : "+v"(tid), "+v"(lane), "+v"(i), "+v"(gq), "+s"(wave));
    wave = __builtin_amdgcn_readfirstlane(wave);  // (uniform again to the compiler)
    const Buf &at = buf[hl & 1];
    Buf &to = buf[(hl & 1) ^ 1];
    const int next = min(hl + 1, nh - 1);  // (the last head's own rows again rather than a branch)
    if (hl > 0) combine(hl - 1);
    fetch_g(next);
    fetch_scalars(next);

    // Below the diagonal the decay is taken apart at the first position of l's tile, exp(a_l - a_ref) * exp(a_ref - a_s):
    // one exponential per column and block.  (Both exponents are <= 0 where all steps are >= 0.  With steps of either sign
    // one may be above, though their sum is not: neither is cut at 0.)  rs: sums over the blocks of a row of tiles below the
    // diagonal, without the row's factor el; they join those of the short (a) and the long row (b) where the row ends.
    f32x4 rs = {0.f, 0.f, 0.f, 0.f}, rsa = rs, rsb = rs, el = *reinterpret_cast<const f32x4 *>(&at.el[(QT - 1 - wave) * 16 + gq * 4]);
    float ref = readlane_f(at.a2[(QT - 1 - wave) * 16], 0);
    float cs[4] = {0.f, 0.f, 0.f, 0.f};
    float *const cp = colp[hl & 1] + wave * (NBK * 16);
    products(
        at, [&](int) { return f32x4{0.f, 0.f, 0.f, 0.f}; },
        [&](int k, const f32x4 &v, const f32x2 &col) {
          float csum = 0.f;
          if (k >= QT - 1) {
            // the diagonal: the exact decay, s <= l
            const f32x4 a_l = *reinterpret_cast<const f32x4 *>(&at.a2[row_tile(k) * 16 + gq * 4]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float e = v[r] * col.y * fast_exp2(fminf(a_l[r] - col.x, 0.f));
              const float d = gq * 4 + r >= i ? e : 0.f, w = d * cb[k][r];
              sum[k][r] += d;
              csum += w;
              if (k == QT) rsa[r] += w;
              else rsb[r] += w;
            }
          } else {
            const float f = col.y * fast_exp2(fminf(ref - col.x, kGrowth));
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float t = v[r] * f, w = t * cb[k][r];
              sum[k][r] = __builtin_fmaf(t, el[r], sum[k][r]);
              csum = __builtin_fmaf(w, el[r], csum);
              rs[r] += w;
            }
            // (formed here, not behind the branch below)
            asm volatile("" : "+v"(sum[k]), "+v"(csum));
            if (k >= NW - 1 && k == QT - 2 - wave) {  // the long row ends here; the short one follows
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                rsb[r] = rs[r] * el[r];
                rs[r] = 0.f;
              }
              el = *reinterpret_cast<const f32x4 *>(&at.el[wave * 16 + gq * 4]);
              ref = readlane_f(at.a2[wave * 16], 0);
            }
            if (k == QT - 2) {
#pragma unroll
              for (int r = 0; r < 4; ++r) rsa[r] = rs[r] * el[r];
            }
          }
          // column sums over the four lane groups, four blocks at a time
          cs[k & 3] = csum;
          if (k == QT) {
            const float h = fold32(csum, csum), t = fold16(h, h);
            cp[k * 16 + i] = t;  // (the same in the four lane groups)
          } else if ((k & 3) == 3) {
            // groups of 16 lanes: block k - 3, k - 1, k - 2, k
            int slot = (k & ~3) + (gq & 1) * 2 + (gq >> 1);
            // the long row's diagonal stands before the short row's columns
            if (k >= NW) slot = slot < QT - 1 - wave ? slot : slot == QT - 1 ? QT - 1 - wave : slot + 1;
            cp[slot * 16 + i] = fold16(fold32(cs[0], cs[1]), fold32(cs[2], cs[3]));
          }
        },
        [&] {
          commit(to.g, piece);
          commit_scalars(to);
          fetch_x(next);
        });
    // The eight row sums (four of each row of tiles) over the 16 lanes of a row, by halving: a lane keeps half of its sums
    // and hands the other half to a lane that keeps those, until it has one row's.
    float h4[4], h2[2];
#pragma unroll
    for (int r = 0; r < 4; ++r) h4[r] = (i & 8 ? rsb[r] : rsa[r]) + dpp_f<0x128>(0.f, i & 8 ? rsa[r] : rsb[r]);  // row_ror:8
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float keep = i & 4 ? h4[k + 2] : h4[k], give = i & 4 ? h4[k] : h4[k + 2];
      h2[k] = keep + dpp_f<0x141>(0.f, give);  // row_half_mirror: a lane of the other four
    }
    float h1 = (i & 2 ? h2[1] : h2[0]) + dpp_f<0x4e>(0.f, i & 2 ? h2[0] : h2[1]);  // quad_perm [2, 3, 0, 1]
    h1 += dpp_f<0xb1>(0.f, h1);                                                    // quad_perm [1, 0, 3, 2]
    rowp[hl & 1][(i & 8 ? QT - 1 - wave : wave) * 16 + gq * 4 + ((i >> 1) & 3)] = h1;  // (two lanes, one value)
    commit(to.x, piece);
    // the one barrier of a head: its operands were last read before it, the next head's and its sums are there after it
    lds_barrier();
  }
  combine(nh - 1);
  write_seq();  // (the last commits went to either buffer before the barrier; nobody reads them)
  lds_barrier();

  // One list per group: the workgroup owns the triangle and stores it as whole 64 x 64 tiles, zeros included, so the
  // caller need not clear dCB (the next stage reads those tiles only).  Else several add into it, and it starts zeroed.
  const int64_t out = (((int64_t)b * p.nchunks + c) * G + g) * Q * Q;
  auto store = [&](int lt, int st, const f32x4 &v) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t at = out + (lt * 16 + gq * 4 + r) * Q + st * 16 + i;
      if (lp) st1<bf16_t>(reinterpret_cast<bf16_t *>(p.dCB) + at, v[r]);
      else p.dCB[at] = v[r];
    }
  };
#pragma unroll
  for (int k = 0; k < NBK; ++k) {
    const f32x4 v = mask(k, sum[k]);
    if (nsplit == 1) {
      store(row_tile(k), col_tile(k), v);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (v[r] != 0.f)
          acc_add<0>(p.dCB, nullptr, out + (row_tile(k) * 16 + gq * 4 + r) * Q + col_tile(k) * 16 + i, v[r], 0.f);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (nsplit == 1) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int lt : {wave, QT - 1 - wave})
      for (int st = lt + 1; st <= (lt | 3); ++st) store(lt, st, zero);
  }
}

template <int PT, int QT> int launch_q(const SsdParams &p, bool lp, int nsplit, hipStream_t s) {
  const dim3 grid(p.ngroups * nsplit, p.nchunks, p.batch);
  if (p.CB) hipLaunchKernelGGL((bwd_dcb_chunk_kernel<PT, QT, false>), grid, dim3(32 * QT), 0, s, p, lp ? 1 : 0, nsplit);
  else hipLaunchKernelGGL((bwd_dcb_chunk_kernel<PT, QT, true>), grid, dim3(32 * QT), 0, s, p, lp ? 1 : 0, nsplit);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}
template <int PT> int launch_p(const SsdParams &p, bool lp, int nsplit, hipStream_t s) {
  switch (p.chunk_size) {
    case 256: return launch_q<PT, 16>(p, lp, nsplit, s);
    case 128: return launch_q<PT, 8>(p, lp, nsplit, s);
    case 64: return launch_q<PT, 4>(p, lp, nsplit, s);
    default: return MAMBA_E_UNSUPPORTED;
  }
}

}  // namespace

int ssd_bwd_dcb_chunk_launch(const SsdParams *p, bool lp, int nsplit, hipStream_t s) {
  if (nsplit < 1 || nsplit > p->nheads / p->ngroups) return MAMBA_E_UNSUPPORTED;
  return p->headdim == 64 ? launch_p<4>(*p, lp, nsplit, s) : launch_p<2>(*p, lp, nsplit, s);
}
