// Mamba-1 selective scan, forward, with the lanes along the states instead of along the sequence (gfx950, wave64;
// reference csrc/selective_scan/selective_scan_fwd_kernel.cuh, the same outputs as scan_fwd_kernel in mamba1_scan.hip).
//
// A wave holds 8 channels, 8 lanes each, two of the 16 states per lane, and walks the positions one after the other: a
// (position, channel, state) costs the exponent, its exponential, the input term, the recurrence and the output term, with
// no second pass over the positions and no scan across lanes.  What the lanes along the sequence need for those, 4.5 of
// their 10.5 vector instructions, is replaced by the sum of the output terms over a channel's 8 lanes: seven DPP adds for
// four positions at a time, each add halving the positions that a lane goes on with (bank masks), 0.9 per element.
//   * 64 positions at a time: a lane loads 8 positions of one channel's rows (16 bytes), forms step and step * u and
//     leaves them in LDS; the scan reads them back as 8 lanes' common operands, four positions per 16 bytes, and puts the
//     outputs in their place, from where the lane that wrote them adds D u, applies the gate and stores 16 bytes.  All of
//     that stays inside a wave.  The B and C rows are staged once for the workgroup's four waves, as the
//     (B, B, C, C) a lane reads per position.
//   * state after every 128 positions to `ckpt`, as the other kernel writes it.
// What bounds it: vector issue.  8 x 5120 channels x 4096 positions, bf16: 660 us (806 for the lanes along the sequence),
// 8.0 vector instructions per element, 1.4 of them transcendental; the vector pipe executes in 99 % of the busy time, LDS
// in 48 %.  Five waves per SIMD (96 registers): a single one leaves half of the issue slots empty (7.3 us per 128
// positions where five take 20.9).  Measured and not kept: the sum over the lanes as fp32 matrix products with ones (959
// us: the matrix and the vector pipe share the issue); the next positions' operands read ahead at four waves per SIMD (682).
//
// With few channels the walk itself is what a call waits for, and a wave alone on its SIMD issues an instruction in four
// clocks.  Then a lane takes one state (SPL 1: 16 lanes and 4 channels of a wave, 16 channels of a workgroup, 128 positions at
// a time): twice the waves at nearly half the instructions each, 4.8 us per 128 positions instead of 7.3, 6.5 with two of the
// half as large workgroups on a CU.  More of them per CU issue more in all than two states per lane do (fwd_cost).
#include "mamba1_scan.hpp"

namespace {

constexpr int SWAVES = 4;
constexpr int BCP = 32;                // floats of a position's B and C values
// SPL states per lane (2: 8 lanes and 8 channels of a wave; 1: 16 lanes, 4 channels), ST positions of a step of the workgroup
template <int SPL> struct Serial {
  static constexpr int lanes = 16 / SPL, channels = 64 / lanes, ST = 512 / channels;
  static constexpr int XP = 2 * ST + 4;  // LDS pitch of a channel's (step, step * u) pairs
};
static_assert(Serial<2>::channels * SWAVES == PASS_CH && TILE % Serial<1>::ST == 0 && NB16 == 16, "the geometry of the other scan kernels");

DEVI int bc_at(int t) { return t * BCP + (t >> 3) * BCP; }  // (a spare row after every 8: the writers' banks)

// States n .. n + NS - 1 entering this workgroup's segment, as seg_state_in has them one by one.  What eight segments left is
// requested together, and nothing that was loaded before (A) is waited for ahead of it: a segment after the other is a memory
// latency for each (1 x 1536 channels x 777 positions in seven segments, one state per lane as well: 24.3 -> 22.8 us).
constexpr int SEG_BATCH = 8;
template <int NS> DEVI void seg_states_in(const MambaScanParams &p, const Geo &q, int d, int n, const float (&A)[NS], float (&h)[NS]) {
#pragma unroll
  for (int e = 0; e < NS; ++e) h[e] = 0.f;
  for (int s0 = 0; s0 < q.seg; s0 += SEG_BATCH) {
    float sums[SEG_BATCH], v[SEG_BATCH][NS], A2[NS];
#pragma unroll
    for (int k = 0; k < SEG_BATCH; ++k) {
      if (s0 + k >= q.seg) break;
      const int64_t row = seg_row(p, q.b, s0 + k, d);
      sums[k] = seg_sums(p)[row];
#pragma unroll
      for (int e = 0; e < NS; ++e) v[k][e] = p.seg_ws[row * p.dstate + n + e];
    }
#pragma unroll
    for (int e = 0; e < NS; ++e) {
      A2[e] = A[e];
      asm volatile("" : "+v"(A2[e]));  // (here, not ahead of the loop)
      A2[e] *= kLog2e;
    }
#pragma unroll
    for (int k = 0; k < SEG_BATCH; ++k) {
      if (s0 + k >= q.seg) break;
#pragma unroll
      for (int e = 0; e < NS; ++e) h[e] = __builtin_fmaf(fast_exp2(A2[e] * sums[k]), h[e], v[k][e]);
    }
  }
}

// AHEAD: the next four positions' operands are read ahead of the four at work, where a SIMD has few waves.
template <typename T, int MODE, int SPL, bool AHEAD>
__global__ __launch_bounds__(64 * SWAVES, AHEAD ? 4 : 5) void scan_fwd_serial_kernel(const MambaScanParams p) {
  constexpr int ST = Serial<SPL>::ST, SCH = Serial<SPL>::channels, XP = Serial<SPL>::XP, PC = ST / 8;
  __shared__ __align__(16) float xs[SWAVES][SCH * XP], bcs[(ST + PC) * BCP];
  const int L = p.seqlen, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Geo q = geometry<SCH * SWAVES>(p, 1);
  const int b = q.b, d0 = q.g * q.Dg + q.cb * (SCH * SWAVES) + wave * SCH;
  // scan, two states per lane: lane = (channel pair: row of 16 lanes, bank of 4, channel of the pair, state half): states s2 and
  // s2 + 1; one: lane = (channel: row, state)
  const int bank = (lane >> 2) & 3, ch = SPL == 2 ? (lane >> 4) * 2 + ((lane >> 1) & 1) : lane >> 4;
  const int s2 = SPL == 2 ? 2 * (bank * 2 + (lane & 1)) : lane & 15;
  // rows: lane = (channel cu, piece of 8 positions)
  const int cu = lane / PC, piece = lane % PC;
  const bool valid = d0 + cu < q.dend;
  const int du_ = min(d0 + cu, q.dend - 1), ds = min(d0 + ch, q.dend - 1);
  const T *urow = (const T *)p.u + b * p.u_bs + du_ * p.u_ds;
  const T *drow = (const T *)p.delta + b * p.delta_bs + du_ * p.delta_ds;
  const T *zrow = p.z ? (const T *)p.z + b * p.z_bs + du_ * p.z_ds : urow;
  const float bias = p.delta_bias ? ((const float *)p.delta_bias)[du_] : 0.f;
  const float Dd = p.D ? ((const float *)p.D)[du_] : 0.f;
  // staging of B and C: thread = (state, operand, piece), with 16 pieces two of them
  const int sn = tid & 15, which = (tid >> 4) & 1, sp = tid >> 5;
  const T *brow = which ? (const T *)p.C + b * p.C_bs + q.g * p.C_gs + sn * p.C_ns : (const T *)p.B + b * p.B_bs + q.g * p.B_gs + sn * p.B_ns;
  // a position's values as a lane reads them: (B, B, C, C) or (B, C)
  float *const bdst = bcs + bc_at(sp * 8) + (SPL == 2 ? (sn >> 1) * 4 + which * 2 + (sn & 1) : sn * 2 + which);

  float A[SPL], h[SPL];
#pragma unroll
  for (int e = 0; e < SPL; ++e) A[e] = ((const float *)p.A)[(int64_t)ds * 16 + s2 + e];
  float *const xrow = &xs[wave][cu * XP + piece * 16];        // this lane's 8 positions as a producer
  float *const srow = &xs[wave][ch * XP];                     // its channel as a consumer
  const float *const brd = bcs + 2 * s2;

  const int tfirst = q.tile0 * TILE, tlast = min(L, q.tile1 * TILE);
  auto place = [&](float (&v)[8], int t0, int tl) {
    if constexpr (MODE == ROWS_ANY) {
      if (t0 + ST > L) row8_place(tl, L, v);
    }
  };
  Pack8<T> nu, nd, nb[PC / 8];
  auto request = [&](int t0) {
    load_items<T, MODE>(nu, urow, t0 + piece * 8, L, 8);
    load_items<T, MODE>(nd, drow, t0 + piece * 8, L, 8);
#pragma unroll
    for (int k = 0; k < PC / 8; ++k) load_items<T, MODE>(nb[k], brow, t0 + (sp + 8 * k) * 8, L, 8);
  };
  if constexpr (AHEAD) {
    request(tfirst);
    seg_states_in<SPL>(p, q, ds, s2, A, h);
#pragma unroll
    for (int e = 0; e < SPL; ++e) A[e] *= kLog2e;
  } else {  // (other waves have work meanwhile, and the registers are few)
#pragma unroll
    for (int e = 0; e < SPL; ++e) {
      A[e] *= kLog2e;
      h[e] = seg_state_in(p, q, ds, s2 + e, A[e]);
    }
    request(tfirst);
  }
  for (int t0 = tfirst; t0 < tlast; t0 += ST) {
    const int tl = t0 + piece * 8, nvalid = min(max(L - tl, 0), 8);
    Pack8<T> ku = nu, kz;
    {
      float u[8], dl[8];
      nu.unpack(u);
      nd.unpack(dl);
      place(u, t0, tl);
      place(dl, t0, tl);
#pragma unroll
      for (int i = 0; i < 8; ++i) dl[i] += bias;
      if (p.delta_softplus) {
#pragma unroll
        for (int i = 0; i < 8; ++i) dl[i] = softplus_f(dl[i]);
      }
      if (t0 + ST > L) {  // positions past the end leave the state as it is
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          dl[i] = i < nvalid ? dl[i] : 0.f;
          u[i] = i < nvalid ? u[i] : 0.f;
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) u[i] *= dl[i];
      f32x4 *const dst = reinterpret_cast<f32x4 *>(xrow);
      dst[0] = f32x4{dl[0], dl[1], dl[2], dl[3]};
      dst[1] = f32x4{u[0], u[1], u[2], u[3]};
      dst[2] = f32x4{dl[4], dl[5], dl[6], dl[7]};
      dst[3] = f32x4{u[4], u[5], u[6], u[7]};
    }
    lds_barrier();  // the positions before have been read
#pragma unroll
    for (int k = 0; k < PC / 8; ++k) {
      float v[8];
      nb[k].unpack(v);
      const int ts = t0 + (sp + 8 * k) * 8;
      if (t0 + ST > L) {
        place(v, t0, ts);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = ts + i < L ? v[i] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) bdst[(72 * k + i) * BCP] = v[i];
    }
    lds_barrier();
    request(min(t0 + ST, tlast - 1) / ST * ST);
    load_items<T, MODE>(kz, zrow, tl, L, 8);

    float *const put = srow + ((bank & 1) << 1 | bank >> 1);
    // four positions, 4 k to 4 k + 3: their operands, and their outputs summed over the lanes of a channel
    typedef float bc_t __attribute__((ext_vector_type(2 * SPL)));
    struct Four {
      f32x4 dl, dx;
      bc_t bc[4];
    };
    auto read = [&](Four &o, const float *at, const float *bp) {
      o.dl = *reinterpret_cast<const f32x4 *>(at), o.dx = *reinterpret_cast<const f32x4 *>(at + 4);
#pragma unroll
      for (int t = 0; t < 4; ++t) o.bc[t] = *reinterpret_cast<const bc_t *>(bp + t * BCP);
    };
    auto walk = [&](const Four &o) {
      float y[4];
      if constexpr (AHEAD) {  // the exponentials first, then the chain
        float decay[4][SPL], x[4][SPL];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int e = 0; e < SPL; ++e) decay[t][e] = fast_exp2(o.dl[t] * A[e]), x[t][e] = o.dx[t] * o.bc[t][e];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int e = 0; e < SPL; ++e) {
            h[e] = __builtin_fmaf(decay[t][e], h[e], x[t][e]);
            y[t] = e ? __builtin_fmaf(h[e], o.bc[t][SPL + e], y[t]) : h[e] * o.bc[t][SPL];
          }
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
          for (int e = 0; e < SPL; ++e) h[e] = __builtin_fmaf(fast_exp2(o.dl[t] * A[e]), h[e], o.dx[t] * o.bc[t][e]);
          y[t] = __builtin_fmaf(h[SPL - 1], o.bc[t][2 * SPL - 1], h[0] * o.bc[t][SPL]);
        }
      }
      float r, w, v;
      asm volatile("s_nop 1\n\t"
                   "v_add_f32_dpp %0, %3, %3 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
                   "v_add_f32_dpp %1, %5, %5 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
                   "v_add_f32_dpp %0, %4, %4 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
                   "v_add_f32_dpp %1, %6, %6 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
                   "s_nop 0\n\t"
                   "v_add_f32_dpp %2, %0, %0 row_ror:12 row_mask:0xf bank_mask:0x5\n\t"
                   "v_add_f32_dpp %2, %1, %1 row_ror:4 row_mask:0xf bank_mask:0xa\n\t"
                   "s_nop 1\n\t"
                   "v_add_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
                   : "=&v"(r), "=&v"(w), "=&v"(v)
                   : "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]));
      if constexpr (SPL == 1) asm volatile("s_nop 1\n\tv_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t" : "+v"(v));
      return v;
    };
    if constexpr (AHEAD) {
      Four even, odd;
      const float *at = srow, *bp = brd;
      float *to = put;
      read(even, at, bp);
#pragma unroll 1
      for (int g8 = 0; g8 < ST / 8; ++g8) {
        read(odd, at + 8, bp + 4 * BCP);
        __builtin_amdgcn_sched_barrier(0);
        to[0] = walk(even);
        __builtin_amdgcn_sched_barrier(0);
        const int on = g8 + 1 < ST / 8 ? 1 : 0;  // (the last four again at the end)
        at += 16 * on, bp += 9 * on * BCP;
        read(even, at, bp);
        __builtin_amdgcn_sched_barrier(0);
        to[8] = walk(odd);
        __builtin_amdgcn_sched_barrier(0);
        to += 16;
      }
    } else {
      const float *at = srow, *bp = brd;
      float *to = put;
#pragma unroll 1
      for (int g8 = 0; g8 < ST / 8; ++g8) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          Four o;
          read(o, at + half * 8, bp + half * 4 * BCP);
          to[half * 8] = walk(o);
        }
        at += 16, to += 16;
        bp += 9 * BCP;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    {
      const f32x4 lo = *reinterpret_cast<const f32x4 *>(xrow), hi = *reinterpret_cast<const f32x4 *>(xrow + 8);
      float y[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w}, u[8];
      ku.unpack(u);
      place(u, t0, tl);
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = __builtin_fmaf(Dd, u[i], y[i]);
      if (p.z) {
        float z[8];
        kz.unpack(z);
        place(z, t0, tl);
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] *= z[i] * sigmoid_f(z[i]);
      }
      T *const orow = (T *)p.out + b * p.out_bs + du_ * p.out_ds + tl;
      if constexpr (MODE == ROWS_ANY) {
        if (valid && nvalid >= KI) st8_any<T>(orow, y);
        else if (valid && nvalid > 0) st8_guard<T, false>(orow, nvalid, y);
      } else {
        st8_guard<T, true>(orow, valid ? nvalid : 0, y);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (((t0 + ST) % TILE == 0 || t0 + ST >= L) && d0 + ch < q.dend) {
      float *ck = p.ckpt + (((int64_t)b * p.dim + ds) * q.ntiles + t0 / TILE) * 16 + s2;
      if constexpr (SPL == 2) {
        typedef f32x2 f32x2_a4 __attribute__((aligned(4)));
        *reinterpret_cast<f32x2_a4 *>(ck) = f32x2{h[0], h[1]};
      } else {
        *ck = h[0];
      }
    }
  }
}

template <typename T, int MODE, int SPL> void launch_s(const MambaScanParams &p, hipStream_t s) {
  constexpr int WCH = Serial<SPL>::channels * SWAVES;
  const dim3 grid(p.ngroups * ((p.dim / p.ngroups + WCH - 1) / WCH), p.batch, p.nseg > 1 ? p.nseg : 1), block(64 * SWAVES);
  // one state per lane is for calls that leave a SIMD few waves; with two, up to two workgroups per CU (39.3 -> 38.2 us at 4 x 1024 x
  // 1024 in four segments; five per CU 660 -> 682 at 8 x 5120 x 4096)
  if (SPL == 1 || (int64_t)grid.x * grid.y * grid.z <= 2 * cu_count()) hipLaunchKernelGGL((scan_fwd_serial_kernel<T, MODE, SPL, true>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((scan_fwd_serial_kernel<T, MODE, SPL, SPL == 1>), grid, block, 0, s, p);
}
template <typename T> int launch_t(const MambaScanParams &p, int spl, int mode, hipStream_t s) {
  if (mode == ROWS_ALIGNED) spl == 1 ? launch_s<T, ROWS_ALIGNED, 1>(p, s) : launch_s<T, ROWS_ALIGNED, 2>(p, s);
  else spl == 1 ? launch_s<T, ROWS_ANY, 1>(p, s) : launch_s<T, ROWS_ANY, 2>(p, s);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}

}  // namespace

int mamba1_fwd_serial_launch(const MambaScanParams &p, int spl, int mode, hipStream_t s) {
  switch (p.dtype) {
    case MAMBA_F32: return launch_t<float>(p, spl, mode, s);
    case MAMBA_BF16: return launch_t<bf16_t>(p, spl, mode, s);
    default: return launch_t<f16_t>(p, spl, mode, s);
  }
}
