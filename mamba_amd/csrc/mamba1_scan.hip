// Mamba-1 selective scan, forward and backward, for gfx950 (wave64).
//
// Work decomposition
//   * a wave owns 4 channels of one (batch, group) at a time, one per DPP row of 16 lanes; the 16
//     lanes of a row hold 16 consecutive 8-step segments of the sequence, i.e. one 128-step tile
//     per pass.  A lane loads its 8 items of u/delta/z with one 16-byte access.  Every cross-lane
//     step of the scans then stays inside a DPP row (row_shr / row_shl), which is the cheap kind.
//   * the 8 waves of a workgroup walk the tiles together and share the B and C rows of the tile,
//     staged once per tile in LDS as fp32; a backward workgroup takes several passes of 32 channels
//     over a tile.
//   * per state n: an 8-step in-register recurrence per lane, a row scan of the (decay, value)
//     pairs across the 16 lanes, and a carry from the previous tile kept in LDS.
//   * the state after every tile is written to `ckpt`; the backward pass walks the tiles in
//     reverse, restarts each tile from ckpt, and runs the adjoint recurrence with a reversed row
//     scan.  dB/dC are summed over the channels of the workgroup in LDS (waves take turns on
//     disjoint state rows; LDS float atomics are far too slow for this), written once per tile as
//     one partial per workgroup, and summed over the workgroups in a fixed order by a second
//     kernel: no float atomics anywhere, so every gradient repeats bit for bit.
#include "mamba1_scan.hpp"

#include <stdlib.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

size_t mamba1_bwd_mx_lds(int passes, int np);                                                       // mamba1_scan_bwd_mx.hip
int mamba1_bwd_mx_launch(const MambaScanParams &p, int passes, bool vec, hipStream_t stream);  // likewise
size_t mamba1_bwd_k4_lds(int passes);                                                          // mamba1_scan_bwd_k4.hip
bool mamba1_bwd_k4_serves(const MambaScanParams &p);                                           // likewise
int mamba1_fwd_serial_launch(const MambaScanParams &p, int spl, int mode, hipStream_t s);       // mamba1_scan_serial.hip
int mamba1_bwd_k4_launch(const MambaScanParams &p, int pa, int pb, int nparts, hipStream_t stream);  // likewise

namespace {

// ------------------------------------------------------------------ segments of the sequence
// With few (batch, channel) rows the chip is filled by cutting the sequence into p.nseg segments (p.seg_ws).  A
// segment's part of the recurrence is a (decay, value) pair per (channel, state), as a lane's and a tile's are: the
// value is formed by scan_seg_kernel, the decay is exp(A * sum of the segment's steps), and the scan kernels compose the
// pairs of the segments before theirs when they start.  The adjoint is handled the same way from the other end.  seg_ws:
// values (batch, nseg, dim, N), then the sums of the steps (batch, nseg, dim; backward: without the first one), then the
// first steps (batch, nseg, dim; backward only).
// Adjoint at the first position of the segment after this workgroup's, and the decay of that position
DEVI float seg_adjoint_in(const MambaScanParams &p, const Geo &q, int d, int n, float A2, float &decay) {
  float g = 0.f;
  decay = 0.f;
  for (int s = q.nseg - 1; s > q.seg; --s) {
    const int64_t row = seg_row(p, q.b, s, d);
    // from the first position of segment s + 1 back to that of segment s; `decay` is the former's
    g = __builtin_fmaf(fast_exp2(A2 * seg_sums(p)[row]) * decay, g, p.seg_ws[row * p.dstate + n]);
    decay = fast_exp2(A2 * seg_firsts(p)[row]);
  }
  return g;
}

// What every segment adds.  Forward: the state after the segment from a zero state, sum over t of
// exp(A (steps after t)) B_t step_t u_t.  Backward: the adjoint at the segment's first position from a zero adjoint
// behind it, sum over t of exp(A (steps after the first position up to t)) C_t dy_t.  Either way a lane runs its 8
// steps from zero and weights the result with one exponential of the steps between it and the segment's end (start):
// no scan across lanes and no carry, only one sum over the 16 lanes of a row at the end.  The steps between are summed as
// such, never as a difference of longer sums: every exponent then has the sign of A, so that no factor can overflow where
// the recurrence itself does not, and a large step elsewhere in the tile costs them no bits.  Where it runs the chip is
// short of waves and a segment short of tiles, so latency bounds it: no LDS and no barrier (a lane reads its 8 items of
// the B or C rows itself, the same 256 bytes for the four rows of every wave, from the caches), a group of states'
// items requested ahead, workgroups of four independent waves.
constexpr int SEG_THREADS = 256, SEG_CH = SEG_THREADS / 64 * ROWS;
template <typename T, int MODE, int BC, bool BWD>
__global__ __launch_bounds__(SEG_THREADS, BWD || sizeof(T) == 4 ? 3 : 4) void scan_seg_kernel(const MambaScanParams p) {
  constexpr bool CONST_BC = BWD ? (BC & 2) != 0 : (BC & 1) != 0;  // the operand is one value per channel and state
  constexpr int NG = sizeof(T) == 4 ? 2 : 4;                      // states whose items are requested together
  const int N = p.dstate, L = p.seqlen;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & (RL - 1);
  const int Dg = p.dim / p.ngroups, cblocks = (Dg + SEG_CH - 1) / SEG_CH;
  const int g = blockIdx.x / cblocks, b = blockIdx.y;
  const int seg = blockIdx.z + (BWD ? 1 : 0);  // backward: segment 0 sends its adjoint nowhere
  const int all = (L + TILE - 1) / TILE, per = tiles_per_segment(all, p.nseg);
  const int tile0 = seg * per, tile1 = min(all, tile0 + per), ntiles = tile1 - tile0;
  const int dend = (g + 1) * Dg, dw = g * Dg + (int)(blockIdx.x % cblocks) * SEG_CH + (tid >> 4);
  const bool valid = dw < dend;
  const int d = min(dw, dend - 1);
  const T *urow = BWD ? (const T *)p.dout + b * p.dout_bs + d * p.dout_ds : (const T *)p.u + b * p.u_bs + d * p.u_ds;
  const T *drow = (const T *)p.delta + b * p.delta_bs + d * p.delta_ds;
  const bool gated = BWD && p.z;
  const T *zrow = gated ? (const T *)p.z + b * p.z_bs + d * p.z_ds : drow;
  const float bias = p.delta_bias ? ((const float *)p.delta_bias)[d] : 0.f;
  const int64_t row = seg_row(p, b, seg, d);
  const T *Sg = BWD ? (const T *)p.C + b * p.C_bs + g * p.C_gs : (const T *)p.B + b * p.B_bs + g * p.B_gs;
  const int64_t S_ns = BWD ? p.C_ns : p.B_ns;
  auto tile_of = [&](int k) { return BWD ? tile0 + k : tile1 - 1 - k; };
  if (BWD && MODE == ROWS_ANY && L - tile0 * TILE < KI) {
    // A last segment of fewer positions than a lane has items: 8 items from L - 8 on would reach into the segment before,
    // whose values must not count even as zero times an infinity.  A lane takes a state, position by position.
    const int t0 = tile0 * TILE;
    auto step = [&](int t) {
      const float v = ld1<T>(drow + t) + bias;
      return p.delta_softplus ? softplus_f(v) : v;
    };
    float run = 0.f;
    for (int t = t0 + 1; t < L; ++t) run += step(t);
    for (int n = c; n < N; n += RL) {
      const float A2 = ((const float *)p.A)[(int64_t)d * N + n] * kLog2e;
      float acc = 0.f;
      for (int t = L - 1; t >= t0; --t) {
        float x = ld1<T>(urow + t);
        if (gated) {
          const float z = ld1<T>(zrow + t);
          x *= z * sigmoid_f(z);
        }
        const float v = CONST_BC ? ((const float *)p.C)[(int64_t)d * N + n] : ld1<T>(Sg + n * S_ns + t);
        acc = t + 1 < L ? __builtin_fmaf(fast_exp2(step(t + 1) * A2), acc, x * v) : x * v;
      }
      if (valid) p.seg_ws[row * N + n] = acc;
    }
    if (c == 0 && valid) {
      seg_sums(p)[row] = run;
      seg_firsts(p)[row] = step(t0);
    }
    return;
  }
  for (int n0 = 0; n0 < N; n0 += NB16) {
    float acc[NB16], A2[NB16];
#pragma unroll
    for (int n = 0; n < NB16; ++n) acc[n] = 0.f;
    Pack8<T> ku, kd, kz, ks[2][NG];
    auto fetch_rows = [&](int k) {
      const int tl = tile_of(k) * TILE + c * KI;
      load_items<T, MODE>(ku, urow, tl, L, KI);
      load_items<T, MODE>(kd, drow, tl, L, KI);
      if (BWD) load_items<T, MODE>(kz, zrow, tl, L, KI);
    };
    auto fetch_states = [&](Pack8<T>(&dst)[NG], int k, int n) {
      if (CONST_BC) return;
#pragma unroll
      for (int s = 0; s < NG; ++s)
        load_items<T, MODE>(dst[s], Sg + (int64_t)min(n0 + n + s, N - 1) * S_ns, tile_of(k) * TILE + c * KI, L, KI);
    };
    float run = 0.f, first = 0.f;  // steps of the tiles already taken; backward: without the segment's first step, `first`
    fetch_rows(0);
    fetch_states(ks[0], 0, 0);
    // (requested behind the first tile's items, all at once: ahead of them, they are a latency of their own, 31.1 -> 27.8 us
    // at 2 x 1536 channels x 2048 positions in fp32, 27.0 -> 25.6 in bf16)
#pragma unroll
    for (int n = 0; n < NB16; ++n) A2[n] = ((const float *)p.A)[(int64_t)d * N + min(n0 + n, N - 1)];
#pragma unroll
    for (int n = 0; n < NB16; ++n) A2[n] = n0 + n < N ? A2[n] * kLog2e : 0.f;
    for (int k = 0; k < ntiles; ++k) {
      // A lane in a ragged row's last piece reads 8 items from L - 8 on like the other rows' lanes, and leaves out the
      // ones before its own, which are the lane before's (nothing has to be moved into place: the order is what counts).
      const int tl = tile_of(k) * TILE + c * KI, shift = tl - min(tl, L - KI);
      float x[8], dl[8], z[8], dsum = 0.f, own = 0.f;  // own: the first step of the lane's own (backward)
      ku.unpack(x);
      kd.unpack(dl);
      if (BWD) kz.unpack(z);
      const int kn = min(k + 1, ntiles - 1);  // (the last tile again at the end)
      fetch_rows(kn);
      if (gated) {
#pragma unroll
        for (int i = 0; i < KI; ++i) x[i] *= z[i] * sigmoid_f(z[i]);
      }
#pragma unroll
      for (int i = 0; i < KI; ++i) {
        float v = dl[i] + bias;
        if (p.delta_softplus) v = softplus_f(v);
        x[i] = i >= shift ? x[i] : 0.f;
        if constexpr (BWD) {  // the decays behind the lane's first position
          own = i == shift ? v : own;
          dl[i] = i > shift ? v : 0.f;
        } else {
          dl[i] = i >= shift ? v : 0.f;
          x[i] *= dl[i];
        }
        dsum += dl[i];
      }
      if (BWD && k == 0) {
        first = __shfl(own, lane & ~(RL - 1), 64);
        own = c == 0 ? 0.f : own;
      }
      dsum += own;
      // Steps of the row's lanes from this one on (backward: up to this one), and of those behind (before) it.
      constexpr int STEP = BWD ? DPP_ROW_SHR : DPP_ROW_SHL;
      float incl = dsum;
      incl += dpp_f<STEP + 1>(0.f, incl);
      incl += dpp_f<STEP + 2>(0.f, incl);
      incl += dpp_f<STEP + 4>(0.f, incl);
      incl += dpp_f<STEP + 8>(0.f, incl);
      const float away = run + dpp_f<STEP + 1>(0.f, incl) + own;
      run += __shfl(incl, BWD ? lane | (RL - 1) : lane & ~(RL - 1), 64);
#pragma unroll
      for (int n = 0; n < NB16; n += NG) {
        const int cur = (n / NG) & 1;
        if (n + NG < NB16) fetch_states(ks[cur ^ 1], k, n + NG);
        else fetch_states(ks[cur ^ 1], kn, 0);
#pragma unroll
        for (int s = 0; s < NG; ++s) {
          float v[8];
          if constexpr (CONST_BC) {
            load_bc<1>(v, nullptr, BWD ? p.C : p.B, d, N, n0 + n + s, n + s, c);
          } else {
            ks[cur][s].unpack(v);
          }
          // (x is zero past the end and A2 for padded states, whose sums are not stored)
          float h;
          if constexpr (BWD) {
            h = x[KI - 1] * v[KI - 1];
#pragma unroll
            for (int i = KI - 2; i >= 0; --i) h = __builtin_fmaf(fast_exp2(dl[i + 1] * A2[n + s]), h, x[i] * v[i]);
          } else {
            h = x[0] * v[0];
#pragma unroll
            for (int i = 1; i < KI; ++i) h = __builtin_fmaf(fast_exp2(dl[i] * A2[n + s]), h, x[i] * v[i]);
          }
          acc[n + s] = __builtin_fmaf(fast_exp2(away * A2[n + s]), h, acc[n + s]);
        }
      }
    }
#pragma unroll
    for (int n = 0; n < NB16; ++n) {
      const float v = row_sum_to_last(acc[n]);
      if (c == RL - 1 && valid && n0 + n < N) p.seg_ws[row * N + n0 + n] = v;
    }
    if (c == RL - 1 && valid && n0 == 0) {
      seg_sums(p)[row] = run;
      if (BWD) seg_firsts(p)[row] = first;
    }
  }
}

// ------------------------------------------------------------------ forward
// BC: bit 0 = B is an input-independent (dim, dstate) fp32 matrix, bit 1 = C likewise
// (selective_scan_fwd_kernel.cuh:74 kIsVariableB / kIsVariableC false).
// HALF: a checkpoint every 64 positions instead of every 128 (the state entering lane 8 of a row is the state after
// the tile's first 64 positions): ckpt is then (batch, dim, ceil(L / 64), N).  For the backward kernel that walks
// 64-position tiles (mamba1_scan_bwd_k4.hip).
template <typename T, int MODE, int BC, bool HALF>
__global__ __launch_bounds__(NTHREADS, 4) void scan_fwd_kernel(const MambaScanParams p, const int passes) {
  extern __shared__ __align__(16) float smem[];
  const int N = p.dstate, L = p.seqlen;
  const int NBLK = (N + NB16 - 1) / NB16, NP = NBLK * NB16;
  float *Bs = smem;
  float *Cs = Bs + BC_FLOATS;
  float *A2s = Cs + BC_FLOATS;                 // [passes * PASS_CH][NP]  A * log2(e)
  float *hcar = A2s + passes * PASS_CH * NP;   // [passes * PASS_CH][NP]  state carried across tiles
  float *hmid = hcar + passes * PASS_CH * NP;  // [passes * PASS_CH][NP]  state after the tile's first half (HALF)

  const int tid = threadIdx.x, lane = tid & 63, c = lane & (RL - 1), rsel = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Geo q = geometry(p, passes);
  const int b = q.b;
  const int chl = wave * ROWS + rsel;  // this lane's channel within a pass
  const T *Bg = (const T *)p.B + b * p.B_bs + q.g * p.B_gs;
  const T *Cg = (const T *)p.C + b * p.C_bs + q.g * p.C_gs;
  const float *Ag = (const float *)p.A;
  const int d0 = q.g * q.Dg + q.cb * passes * PASS_CH;  // first channel of the workgroup

  for (int i = tid; i < passes * PASS_CH * NP; i += NTHREADS) {
    const int ch = i / NP, n = i % NP, d = d0 + ch;
    const float A2 = (d < q.dend && n < N) ? Ag[(int64_t)d * N + n] * kLog2e : 0.f;
    A2s[i] = A2;
    hcar[i] = (d < q.dend && n < N) ? seg_state_in(p, q, d, n, A2) : 0.f;
  }
  lds_barrier();

  for (int tile = q.tile0; tile < q.tile1; ++tile) {
    const int t0 = tile * TILE, tl = t0 + c * KI;
    for (int r = 0; r < passes; ++r) {
      if (d0 + r * PASS_CH >= q.dend) break;  // the whole pass lies past the group (the same in every wave)
      const int chw = r * PASS_CH + chl;
      const bool valid = d0 + chw < q.dend;
      const int d = min(d0 + chw, q.dend - 1);
      const int nvalid = valid ? min(max(L - tl, 0), KI) : 0;
      float u[8], dl[8], du[8], y[8], dsum = 0.f;
      Pack8<T> ku, kd, kz;  // raw rows: every load is issued before the first conversion
      kz.zero();
      load_items<T, MODE>(ku, (const T *)p.u + b * p.u_bs + d * p.u_ds, tl, L, nvalid);
      load_items<T, MODE>(kd, (const T *)p.delta + b * p.delta_bs + d * p.delta_ds, tl, L, nvalid);
      if (p.z) load_items<T, MODE>(kz, (const T *)p.z + b * p.z_bs + d * p.z_ds, tl, L, nvalid);
      const float bias = p.delta_bias ? ((const float *)p.delta_bias)[d] : 0.f;
      ku.unpack(u);
      kd.unpack(dl);
      place_items<MODE>(u, t0, tl, L);
      place_items<MODE>(dl, t0, tl, L);
#pragma unroll
      for (int i = 0; i < KI; ++i) {
        float x = dl[i] + bias;
        if (p.delta_softplus) x = softplus_f(x);
        dl[i] = (i < nvalid) ? x : 0.f;
        u[i] = (i < nvalid) ? u[i] : 0.f;
        du[i] = dl[i] * u[i];
        y[i] = 0.f;
      }
#pragma unroll
      for (int i = 0; i < KI; ++i) dsum += dl[i];
      for (int nb = 0; nb < NBLK; ++nb) {
        if (BC != 3 && (NBLK > 1 || r == 0)) {
          lds_barrier();
          stage_bc<T, MODE, BC>(Bs, Cs, Bg, p.B_ns, Cg, p.C_ns, nb * NB16, N, t0, L, tid);
          lds_barrier();
        }
        const float *A2row = A2s + chw * NP + nb * NB16;
        float *hrow = hcar + chw * NP + nb * NB16;
        float *mrow = hmid + chw * NP + nb * NB16;
        const int nmax = min(NB16, N - nb * NB16);
        // two states per iteration: their row scans are interleaved (padded rows are inert:
        // A = 0, B = C = 0)
        for (int n = 0; n < nmax; n += 2) {
          // Pass 1 runs the lane's 8 steps from a zero state to get the lane's (decay, value) pair;
          // the decay over the lane is one exp of the summed delta instead of 7 products. Pass 2
          // reruns the 8 steps from the state the row scan gives this lane.
          float a[2][8], bb[2][8], Cv[2][8], hc[2];
          float sa[2], sb[2];
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const float A2 = A2row[n + s];
            hc[s] = hrow[n + s];
            float Bv[8];
            load_bc<BC & 1>(Bv, Bs, p.B, d, N, nb * NB16 + n + s, n + s, c);
            load_bc<BC & 2>(Cv[s], Cs, p.C, d, N, nb * NB16 + n + s, n + s, c);
            sa[s] = fast_exp2(dsum * A2);
#pragma unroll
            for (int i = 0; i < KI; ++i) {
              a[s][i] = fast_exp2(dl[i] * A2);
              bb[s][i] = du[i] * Bv[i];
            }
            float hl = bb[s][0];
#pragma unroll
            for (int i = 1; i < KI; ++i) hl = __builtin_fmaf(a[s][i], hl, bb[s][i]);
            sb[s] = hl;
          }
          row_scan_fwd2(sa[0], sb[0], sa[1], sb[1]);
          const float hend[2] = {__builtin_fmaf(sa[0], hc[0], sb[0]), __builtin_fmaf(sa[1], hc[1], sb[1])};
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            float h = dpp_f<DPP_ROW_SHR + 1>(hc[s], hend[s]);  // state entering this lane
            if (c == RL - 1) hrow[n + s] = hend[s];            // state after the tile
            if constexpr (HALF) {
              if (c == RL / 2) mrow[n + s] = h;                // state after the tile's first half
            }
#pragma unroll
            for (int i = 0; i < KI; ++i) {
              h = __builtin_fmaf(a[s][i], h, bb[s][i]);
              y[i] = __builtin_fmaf(h, Cv[s][i], y[i]);
            }
          }
        }
      }
      if (p.D) {
        const float Dd = ((const float *)p.D)[d];
#pragma unroll
        for (int i = 0; i < KI; ++i) y[i] = __builtin_fmaf(Dd, u[i], y[i]);
      }
      if (p.z) {
        float z[8];
        kz.unpack(z);
        place_items<MODE>(z, t0, tl, L);
#pragma unroll
        for (int i = 0; i < KI; ++i) y[i] *= z[i] * sigmoid_f(z[i]);
      }
      T *const orow = (T *)p.out + b * p.out_bs + d * p.out_ds + tl;
      if constexpr (MODE == ROWS_ANY) {
        if (nvalid >= KI) st8_any<T>(orow, y);
        st8_tail<T, MODE>(orow, true, t0, L, nvalid, y);
      } else {
        st8_guard<T, MODE == ROWS_ALIGNED>(orow, nvalid, y);
      }
      if (valid) {  // a row's own lanes wrote its slots of hcar: no other wave touches them
        const float *hfin = hcar + chw * NP;
        if constexpr (HALF) {
          const int nhalf = (L + TILE / 2 - 1) / (TILE / 2);
          float *ck = p.ckpt + (((int64_t)b * p.dim + d) * nhalf + 2 * tile) * N;
          const float *hm = hmid + chw * NP;
          for (int n = c; n < N; n += RL) ck[n] = hm[n];
          if (2 * tile + 1 < nhalf)
            for (int n = c; n < N; n += RL) ck[N + n] = hfin[n];
        } else {
          float *ck = p.ckpt + (((int64_t)b * p.dim + d) * q.ntiles + tile) * N;
          for (int n = c; n < N; n += RL) ck[n] = hfin[n];
        }
      }
    }
  }
}

// ----------------------------------------------------------------- backward

// `passes` passes of PASS_CH channels per tile; the dB / dC sums of all of them leave once per tile as
// partial number (workgroup's place in its group), or after every pass and block when the states come
// in blocks of 16 (the host side then asks for one pass).
// CKH: the checkpoints come every 64 positions (see scan_fwd_kernel): the state entering tile t is slot 2 t - 1.
template <typename T, int MODE, int BC, bool CKH>
__global__ __launch_bounds__(NTHREADS) void scan_bwd_kernel(const MambaScanParams p, const int passes) {
  constexpr bool ck_half = CKH;
  extern __shared__ __align__(16) float smem[];
  const int N = p.dstate, L = p.seqlen;
  const int NBLK = (N + NB16 - 1) / NB16, NP = NBLK * NB16;
  const int WCH = passes * PASS_CH;
  float *Bs = smem;
  float *Cs = Bs + BC_FLOATS;
  float *dBs = Cs + BC_FLOATS;        // fp32 sums over the workgroup's channels: [n][half][lane][4]
  float *dCs = dBs + ACC_FLOATS;
  float *hcar = dCs + ACC_FLOATS;     // [PASS_CH][NP] state entering the tile (from ckpt), per pass
  float *A1s = hcar + PASS_CH * NP;   // [WCH][NP] A
  float *gcar = A1s + WCH * NP;       // adjoint at the first position of the following tile
  float *anx = gcar + WCH * NP;       // decay at the first position of the following tile
  float *dAacc = anx + WCH * NP;      // [WCH][NP]
  float *dDacc = dAacc + WCH * NP;    // [WCH]
  float *dbacc = dDacc + WCH;         // [WCH]
  BwdRow<T> *rows = reinterpret_cast<BwdRow<T> *>(dbacc + WCH);  // [WCH]
  float *dBcacc = reinterpret_cast<float *>(rows + WCH);  // [WCH][NP] gradients of input-independent B / C (BC != 0)
  float *dCcacc = dBcacc + WCH * NP;
  static_assert(sizeof(BwdRow<T>) == 80, "the host side sizes the LDS table with 80 bytes per channel");

  const int tid = threadIdx.x, lane = tid & 63, c = lane & (RL - 1), rsel = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Geo q = geometry(p, passes);
  const int b = q.b;
  const int chl = wave * ROWS + rsel;
  const int d0 = q.g * q.Dg + q.cb * WCH;
  const int ntiles = q.ntiles;
  const bool has_z = p.z != nullptr;
  T *const spare = reinterpret_cast<T *>(bwd_spare + tid * 8);  // where this thread's unwanted row stores go

  const T *Bg = (const T *)p.B + b * p.B_bs + q.g * p.B_gs;
  const T *Cg = (const T *)p.C + b * p.C_bs + q.g * p.C_gs;
  const float *Ag = (const float *)p.A;
  // partials of this workgroup: (batch, ngroups, nparts, dstate, seqlen), nparts = cblocks (x passes when NBLK > 1)
  const int per_wg = NBLK > 1 ? passes : 1;
  const int64_t part0 = ((int64_t)b * p.ngroups + q.g) * (q.cblocks * per_wg) + (int64_t)q.cb * per_wg;

  for (int i = tid; i < WCH * NP; i += NTHREADS) {
    const int ch = i / NP, n = i % NP, d = d0 + ch;
    const float A1 = (d < q.dend && n < N) ? Ag[(int64_t)d * N + n] : 0.f;
    A1s[i] = A1;
    float a_next = 0.f;
    gcar[i] = (d < q.dend && n < N) ? seg_adjoint_in(p, q, d, n, A1 * kLog2e, a_next) : 0.f;
    anx[i] = a_next;
    dAacc[i] = 0.f;
    if constexpr (BC != 0) {
      dBcacc[i] = 0.f;
      dCcacc[i] = 0.f;
    }
  }
  for (int i = tid; i < WCH; i += NTHREADS) {
    dDacc[i] = 0.f;
    dbacc[i] = 0.f;
    const int d = min(d0 + i, q.dend - 1);  // channels past the group stand on its last one; their lanes are masked
    BwdRow<T> w;
    w.u = (const T *)p.u + b * p.u_bs + d * p.u_ds;
    w.delta = (const T *)p.delta + b * p.delta_bs + d * p.delta_ds;
    w.dout = (const T *)p.dout + b * p.dout_bs + d * p.dout_ds;
    w.z = has_z ? (const T *)p.z + b * p.z_bs + d * p.z_ds : w.u;  // without z the u row stands in, read and unused
    w.du = (T *)p.du + b * p.du_bs + d * p.du_ds;
    w.ddelta = (T *)p.ddelta + b * p.ddelta_bs + d * p.ddelta_ds;
    w.dz = has_z ? (T *)p.dz + b * p.dz_bs + d * p.dz_ds : nullptr;
    w.out_z = (has_z && p.out_z) ? (T *)p.out_z + b * p.outz_bs + d * p.outz_ds : nullptr;
    w.ckpt = p.ckpt + ((int64_t)b * p.dim + d) * (ck_half ? (L + TILE / 2 - 1) / (TILE / 2) : ntiles) * N;
    w.D = p.D ? ((const float *)p.D)[d] : 0.f;
    w.bias = p.delta_bias ? ((const float *)p.delta_bias)[d] : 0.f;
    rows[i] = w;
  }
  lds_barrier();

  constexpr int NPP = NB16 / NWAVES;  // state rows per wave and phase (see the state loop)
  constexpr int NPH = NB16 / NPP;
  static_assert(NPP == 2 && NPH == NWAVES, "two states per step, one row slot per wave and phase");
  // The rows of the next (tile, pass) are fetched while the current one is computed.
  struct Rows {
    Pack8<T> u, delta, dout, z;
    float ck;  // checkpointed state n = c entering the tile (when the padded state count is 16)
  };
  auto fetch_rows = [&](Rows &k, int tile, int r) {
    const BwdRow<T> &w = rows[r * PASS_CH + chl];
    const int tl = tile * TILE + c * KI;
    const int nvalid = min(max(L - tl, 0), KI);
    // No branch around any of these loads (the checkpoint of tile 0 stands in where there is none to read, the u
    // row where there is no z): with the same memory operations on every path through a step the compiler counts
    // those in flight exactly, and a wait for these rows leaves the younger stores of the step before draining.
    k.ck = *(const GLOBAL_AS float *)(w.ckpt + (int64_t)max(ck_half ? 2 * tile - 1 : tile - 1, 0) * N + min(c, N - 1));
    load_items<T, MODE>(k.u, w.u, tl, L, nvalid);
    load_items<T, MODE>(k.delta, w.delta, tl, L, nvalid);
    load_items<T, MODE>(k.dout, w.dout, tl, L, nvalid);
    load_items<T, MODE>(k.z, w.z, tl, L, nvalid);
  };
  int npass = 0;  // passes that hold at least one channel of the group (the same in every wave)
  while (npass < passes && d0 + npass * PASS_CH < q.dend) ++npass;
  Rows nxt;
  fetch_rows(nxt, q.tile1 - 1, 0);

  for (int tile = q.tile1 - 1; tile >= q.tile0; --tile) {
    const int t0 = tile * TILE, tl = t0 + c * KI;
    for (int r = 0; r < npass; ++r) {
      const int chw = r * PASS_CH + chl;
      const bool valid = d0 + chw < q.dend;
      const int d = min(d0 + chw, q.dend - 1);
      const int nvalid = valid ? min(max(L - tl, 0), KI) : 0;
      float u[8], dl[8], du[8], dy[8], acc[8], dd[8], y[8], dsum = 0.f, dtail = 0.f;
      const float Dd = rows[chw].D, bias = rows[chw].bias;
      {
        // The rows requested during the previous step are unpacked where they were loaded, and only then are the
        // next step's rows requested into the same registers: nothing of them has to be copied (a copy held
        // across the loop's back edge went through scratch memory).  The epilogue reads z and dout again.
        nxt.u.unpack(u);
        nxt.delta.unpack(dl);
        nxt.dout.unpack(dy);
        place_items<MODE>(u, t0, tl, L);
        place_items<MODE>(dl, t0, tl, L);
        place_items<MODE>(dy, t0, tl, L);
#pragma unroll
        for (int i = 0; i < KI; ++i) {  // lanes past the end read a clamped position: mask them
          u[i] = (i < nvalid) ? u[i] : 0.f;
          dy[i] = (i < nvalid) ? dy[i] : 0.f;
        }
        if (has_z) {
          float z[8];
          nxt.z.unpack(z);
          place_items<MODE>(z, t0, tl, L);
#pragma unroll
          for (int i = 0; i < KI; ++i) dy[i] *= z[i] * sigmoid_f(z[i]);
        }
#pragma unroll
        for (int i = 0; i < KI; ++i) {
          float x = dl[i] + bias;
          if (p.delta_softplus) x = softplus_f(x);
          dl[i] = (i < nvalid) ? x : 0.f;
          du[i] = dl[i] * u[i];
          acc[i] = 0.f;
          dd[i] = 0.f;
          y[i] = 0.f;
        }
#pragma unroll
        for (int i = 1; i < KI; ++i) dtail += dl[i];
        dsum = dtail + dl[0];
        // state entering this tile (a row's own lanes write and read its slots)
        if (NBLK == 1) {
          hcar[chl * NP + c] = (c < N && tile > 0) ? nxt.ck : 0.f;
        } else {
          for (int n = c; n < NP; n += RL) {
            float v = 0.f;
            if (tile > 0 && n < N)
              v = *(const GLOBAL_AS float *)(rows[chw].ckpt + (int64_t)(ck_half ? 2 * tile - 1 : tile - 1) * N + n);
            hcar[chl * NP + n] = v;
          }
        }
        {  // the very last step fetches tile 0 once more rather than branch around the loads
          const bool more = r + 1 < npass;
          fetch_rows(nxt, more ? tile : max(tile - 1, 0), more ? r + 1 : 0);
        }
      }
      for (int nb = 0; nb < NBLK; ++nb) {
        if (BC != 3 && (NBLK > 1 || r == 0)) {
          lds_barrier();
          stage_bc<T, MODE, BC>(Bs, Cs, Bg, p.B_ns, Cg, p.C_ns, nb * NB16, N, t0, L, tid);
          for (int i = tid * 4; i < 2 * ACC_FLOATS; i += NTHREADS * 4)  // dBs and dCs are adjacent
            *reinterpret_cast<f32x4 *>(dBs + i) = f32x4{0.f, 0.f, 0.f, 0.f};
          lds_barrier();
        }
        {
          // The 8 waves add their channels' dB/dC terms into the shared LDS sums without atomics: between
          // two workgroup barriers every wave adds into another pair of state rows, and the 4 channels of a
          // wave have their own slots of a row.  A phase has two halves, the states and adjoints of the pair
          // (vector ALU work) and the sums (LDS traffic).  Waves 4-7 meet the barrier at the end of a phase;
          // waves 0-3 meet the same barrier between their two halves, so they run half a phase behind and
          // the two waves of a SIMD are never in the same half: one computes while the other waits for LDS.
          // Between barriers j and j + 1 waves 0-3 add the sums of phase j into rows (w + j) % 8 * 2, + 1 and
          // waves 4-7 those of phase j + 1 into rows (w + j) % 8 * 2, + 1 (their rows run one phase behind):
          // eight different pairs.
          const bool early = wave < NWAVES / 2;
          const int slot_shift = early ? 0 : NPH - 1;
          const float *A1row = A1s + chw * NP + nb * NB16;
          const float *hrow = hcar + chl * NP + nb * NB16;
          float *grow = gcar + chw * NP + nb * NB16;
          float *arow = anx + chw * NP + nb * NB16;
          float *dArow = dAacc + chw * NP + nb * NB16;
          // the LDS operands of a phase's two states: A, the carries, the B and C rows
          struct Operands {
            float A1[2], hc[2], gc[2], an[2], Bv[2][8], Cv[2][8];
          };
          auto fetch_operands = [&](Operands &o, int ph) {
            const int n = ((wave + ph + slot_shift) % NPH) * NPP;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
              o.A1[s] = A1row[n + s];
              o.hc[s] = hrow[n + s];
              o.gc[s] = grow[n + s];
              o.an[s] = arow[n + s];
              load_bc<BC & 1>(o.Bv[s], Bs, p.B, d, N, nb * NB16 + n + s, n + s, c);
              load_bc<BC & 2>(o.Cv[s], Cs, p.C, d, N, nb * NB16 + n + s, n + s, c);
            }
          };
          Operands ops;
          fetch_operands(ops, 0);
          // The loop's place in its 64-byte lines, which else moves with any change to the code above: most of its
          // instructions take 8 bytes, and vector issue bounds it.  8 x 5120 x 4096 bf16, forward + backward, with 0 - 7
          // words behind the boundary: 3229 3186 3218 3196 3229 3210 3250 3221 us.
          asm volatile(".p2align 6\n\ts_nop 0");
          for (int ph = 0; ph < NPH; ++ph) {
            const int n = ((wave + ph + slot_shift) % NPH) * NPP;
            constexpr bool active = true;  // padded states run on zeros (A = B = C = 0)
            float A1[2], gc[2], an[2];
            float Cv[2][8], a[2][8], bb[2][8], h[2][8];
            float gfirst[2], a_next_lane[2];
            if (active) {
              // Forward states: pass 1 runs the lane's 8 steps from zero for the lane's (decay, value)
              // pair, the decay being one exp of the summed delta; pass 2 reruns them from the state
              // the row scan gives this lane. The adjoint is handled the same way in reverse.
              float hc[2], sa[2], sb[2], hend[2];
#pragma unroll
              for (int s = 0; s < 2; ++s) {
                A1[s] = ops.A1[s];
                hc[s] = ops.hc[s];
                gc[s] = ops.gc[s];
                an[s] = ops.an[s];
                const float A2 = A1[s] * kLog2e;
#pragma unroll
                for (int i = 0; i < KI; ++i) {
                  Cv[s][i] = ops.Cv[s][i];
                  a[s][i] = fast_exp2(dl[i] * A2);
                  bb[s][i] = du[i] * ops.Bv[s][i];
                }
                sa[s] = fast_exp2(dsum * A2);
                float hl = bb[s][0];
#pragma unroll
                for (int i = 1; i < KI; ++i) hl = __builtin_fmaf(a[s][i], hl, bb[s][i]);
                sb[s] = hl;
              }
              row_scan_fwd2(sa[0], sb[0], sa[1], sb[1]);
#pragma unroll
              for (int s = 0; s < 2; ++s) hend[s] = __builtin_fmaf(sa[s], hc[s], sb[s]);
              float ra[2], rb[2];
#pragma unroll
              for (int s = 0; s < 2; ++s) {
                float hp = dpp_f<DPP_ROW_SHR + 1>(hc[s], hend[s]);
#pragma unroll
                for (int i = 0; i < KI; ++i) {
                  hp = __builtin_fmaf(a[s][i], hp, bb[s][i]);
                  h[s][i] = hp;  // true states
                }
                if (has_z) {
#pragma unroll
                  for (int i = 0; i < KI; ++i) y[i] = __builtin_fmaf(h[s][i], Cv[s][i], y[i]);
                }
                // adjoint recurrence g[t] = dy[t] C[t] + a[t+1] g[t+1]; Cv becomes dy * C
                a_next_lane[s] = dpp_f<DPP_ROW_SHL + 1>(an[s], a[s][0]);
#pragma unroll
                for (int i = 0; i < KI; ++i) Cv[s][i] *= dy[i];
                float gl = Cv[s][KI - 1];
#pragma unroll
                for (int i = KI - 2; i >= 0; --i) gl = __builtin_fmaf(a[s][i + 1], gl, Cv[s][i]);
                ra[s] = fast_exp2(dtail * (A1[s] * kLog2e)) * a_next_lane[s];
                rb[s] = gl;
              }
              row_scan_rev2(ra[0], rb[0], ra[1], rb[1]);
#pragma unroll
              for (int s = 0; s < 2; ++s) gfirst[s] = __builtin_fmaf(ra[s], gc[s], rb[s]);
            }
            if (early) lds_barrier();  // the early waves meet the others here, between the two halves
            if (active) {
#pragma unroll
              for (int s = 0; s < 2; ++s) {
                const float gx = dpp_f<DPP_ROW_SHL + 1>(gc[s], gfirst[s]);  // adjoint at the next lane's first item
                if (c == 0) {
                  grow[n + s] = gfirst[s];
                  arow[n + s] = a[s][0];
                }
                float dAp = 0.f, dBp = 0.f, dCp = 0.f;
                float sB[8], sC[8], Bv[8];
                load_bc<BC & 1>(Bv, Bs, p.B, d, N, nb * NB16 + n + s, n + s, c);
                if constexpr (!(BC & 1)) lds_ld8<4 * 64>(dBs + (n + s) * ACC_PITCH, lane, sB);
                if constexpr (!(BC & 2)) lds_ld8<4 * 64>(dCs + (n + s) * ACC_PITCH, lane, sC);
                float gi = gx, an_i = a_next_lane[s];
#pragma unroll
                for (int i = KI - 1; i >= 0; --i) {
                  gi = __builtin_fmaf(an_i, gi, Cv[s][i]);
                  an_i = a[s][i];
                  if constexpr (BC & 2) dCp = __builtin_fmaf(dy[i], h[s][i], dCp);
                  else sC[i] = __builtin_fmaf(dy[i], h[s][i], sC[i]);
                  if constexpr (BC & 1) dBp = __builtin_fmaf(gi, du[i], dBp);
                  else sB[i] = __builtin_fmaf(gi, du[i], sB[i]);
                  acc[i] = __builtin_fmaf(gi, Bv[i], acc[i]);
                  const float w = gi * (h[s][i] - bb[s][i]);  // g * a * h[t-1]
                  dd[i] = __builtin_fmaf(A1[s], w, dd[i]);
                  dAp = __builtin_fmaf(dl[i], w, dAp);
                }
                if constexpr (!(BC & 1)) lds_st8<4 * 64>(dBs + (n + s) * ACC_PITCH, lane, sB);
                if constexpr (!(BC & 2)) lds_st8<4 * 64>(dCs + (n + s) * ACC_PITCH, lane, sC);
                dAp = row_sum_to_last(dAp);
                if (c == RL - 1) dArow[n + s] += dAp;  // the slot belongs to this row alone
                if constexpr (BC & 1) {
                  dBp = row_sum_to_last(dBp);
                  if (c == RL - 1) dBcacc[chw * NP + nb * NB16 + n + s] += dBp;
                }
                if constexpr (BC & 2) {
                  dCp = row_sum_to_last(dCp);
                  if (c == RL - 1) dCcacc[chw * NP + nb * NB16 + n + s] += dCp;
                }
              }
            }
            if (ph + 1 < NPH) fetch_operands(ops, ph + 1);
            if (!early) lds_barrier();
          }
        }
        if (BC != 3 && (NBLK > 1 || r == npass - 1)) {
          lds_barrier();  // waves 0-3 add their last sums after the last barrier of the phases
          // One partial per workgroup: the sum over the 4 channel slots of every (state, position), written
          // with plain stores (positions past the end and padded states are skipped).
          const int n0 = nb * NB16;
          const int64_t part = part0 + (NBLK > 1 ? r : 0);
          constexpr int FIRST = (BC & 1) ? NB16 * TILE / 4 : 0, LAST = (BC & 2) ? NB16 * TILE / 4 : 2 * NB16 * TILE / 4;
          for (int o = FIRST + tid; o < LAST; o += NTHREADS) {
            const int which = o >> 9, n = (o >> 5) & 15, q4 = o & 31;  // positions 4 q4 .. 4 q4 + 3 of state n
            const float *src = (which ? dCs : dBs) + n * ACC_PITCH + (q4 & 1) * 256 + (q4 >> 1) * 4;
            f32x4 v = *reinterpret_cast<const f32x4 *>(src);
#pragma unroll
            for (int k = 1; k < ROWS; ++k) {
              const f32x4 w = *reinterpret_cast<const f32x4 *>(src + k * RL * 4);
              v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w;
            }
            const int t = t0 + 4 * q4;
            if (n0 + n >= N || t >= L) continue;
            float *dst = (which ? p.dC32 : p.dB32) + (part * N + n0 + n) * L + t;
            if (MODE == ROWS_ALIGNED || (MODE == ROWS_ANY && t + 3 < L)) {
              *(GLOBAL_AS f32x4_a4 *)dst = v;
            } else {
              dst[0] = v.x;
              if (t + 1 < L) dst[1] = v.y;
              if (t + 2 < L) dst[2] = v.z;
              if (t + 3 < L) dst[3] = v.w;
            }
          }
        }
      }
      {
        float o[8];
        const BwdRow<T> w = rows[chw];
        Pack8<T> z_k, dout_k;  // read again here rather than held through the state loop: they come from the caches
        load_items<T, MODE>(z_k, w.z, tl, L, nvalid);
        load_items<T, MODE>(dout_k, w.dout, tl, L, nvalid);
        float dbs = 0.f, dDs = 0.f;
#pragma unroll
        for (int i = 0; i < KI; ++i) o[i] = __builtin_fmaf(dl[i], acc[i], Dd * dy[i]);
        st8_or_spare_global<T, MODE>(w.du + tl, nvalid, true, spare, o);
        st8_tail<T, MODE>(w.du + tl, true, t0, L, nvalid, o);
#pragma unroll
        for (int i = 0; i < KI; ++i) {
          float gd = __builtin_fmaf(u[i], acc[i], dd[i]);
          if (p.delta_softplus) gd *= softplus_slope_f(dl[i]);
          gd = (i < nvalid) ? gd : 0.f;
          o[i] = gd;
          dbs += gd;
          dDs = __builtin_fmaf(dy[i], u[i], dDs);
        }
        st8_or_spare_global<T, MODE>(w.ddelta + tl, nvalid, true, spare, o);
        st8_tail<T, MODE>(w.ddelta + tl, true, t0, L, nvalid, o);
        float oz[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (has_z) {
          float z[8], dout[8];
          z_k.unpack(z);
          dout_k.unpack(dout);
          place_items<MODE>(z, t0, tl, L);
          place_items<MODE>(dout, t0, tl, L);
#pragma unroll
          for (int i = 0; i < KI; ++i) {
            const float yf = __builtin_fmaf(Dd, u[i], y[i]);
            const float s = sigmoid_f(z[i]);
            o[i] = dout[i] * yf * s * (1.f + z[i] * (1.f - s));
            oz[i] = yf * z[i] * s;
          }
        }
        st8_or_spare_global<T, MODE>(w.dz + tl, nvalid, has_z, spare, o);
        st8_or_spare_global<T, MODE>(w.out_z + tl, nvalid, w.out_z != nullptr, spare, oz);
        st8_tail<T, MODE>(w.dz + tl, has_z, t0, L, nvalid, o);
        st8_tail<T, MODE>(w.out_z + tl, w.out_z != nullptr, t0, L, nvalid, oz);
        dbs = row_sum_to_last(dbs);
        dDs = row_sum_to_last(dDs);
        if (c == RL - 1) {
          dbacc[chw] += dbs;
          dDacc[chw] += dDs;
        }
      }
    }
  }
  lds_barrier();
  // per-(batch, segment, channel) partial sums, reduced over batch and segments afterwards
  const int64_t bseg = (int64_t)b * q.nseg + q.seg;
  for (int i = tid; i < WCH * N; i += NTHREADS) {
    const int ch = i / N, n = i % N, d = d0 + ch;
    if (d >= q.dend) continue;
    p.dA_part[(bseg * p.dim + d) * N + n] = dAacc[ch * NP + n];
    if constexpr (BC & 1) p.dB32[(bseg * p.dim + d) * N + n] = dBcacc[ch * NP + n];
    if constexpr (BC & 2) p.dC32[(bseg * p.dim + d) * N + n] = dCcacc[ch * NP + n];
  }
  for (int ch = tid; ch < WCH; ch += NTHREADS) {
    const int d = d0 + ch;
    if (d >= q.dend) continue;
    p.dD_part[bseg * p.dim + d] = dDacc[ch];
    p.ddelta_bias_part[bseg * p.dim + d] = dbacc[ch];
  }
}

// The sums that leave the backward kernels as partials, in one launch, every sum in the order of its parts.  Workgroups
// [0, nbc) form dB / dC (dB first): a thread takes 4 consecutive positions of one (batch, group, state) row, four parts
// in flight.  The others form dA, dD and ddelta_bias: a thread per value, over batch x segments.
struct ReduceGeo {
  int nparts, nsum, nbc, per_row;  // partials of dB / dC; of the others; workgroups of dB / dC; quads of a row
  int64_t rows, row_len;           // rows of one operand (batch x groups x states) and its positions
};
template <typename T>
__global__ __launch_bounds__(256) void reduce_parts_kernel(const MambaScanParams p, const ReduceGeo r) {
  if ((int)blockIdx.x >= r.nbc) {
    const int64_t DN = (int64_t)p.dim * p.dstate * (p.a_complex ? 2 : 1), i = (int64_t)(blockIdx.x - r.nbc) * 256 + threadIdx.x;
    const float *src;
    float *dst;
    int64_t at = i, stride = p.dim;
    if (i < DN) {
      src = p.dA_part, dst = p.dA, stride = DN;
    } else if (i < DN + p.dim) {
      src = p.dD_part, dst = p.dD, at = i - DN;
    } else {
      src = p.ddelta_bias_part, dst = p.ddelta_bias, at = i - DN - p.dim;
      if (at >= p.dim) return;
    }
    if (!dst) return;
    float v = 0.f;
    for (int k = 0; k < r.nsum; ++k) v += src[k * stride + at];
    dst[at] = v;
    return;
  }
  const bool first_c = (p.bc_const & 1) != 0;  // dB is no per-position gradient: the workgroups belong to dC
  const int half = first_c || (p.bc_const & 2) ? r.nbc : r.nbc / 2;
  const bool is_c = first_c || (int)blockIdx.x >= half;
  const int64_t quad = (int64_t)(is_c && !first_c ? blockIdx.x - half : blockIdx.x) * 256 + threadIdx.x;
  if (quad >= r.rows * r.per_row) return;
  const int64_t row = quad / r.per_row;
  const int e = (int)(quad - row * r.per_row) * 4, len = (int)r.row_len;
  const int N = p.dstate, n = (int)(row % N);
  const int64_t bg = row / N, b = bg / p.ngroups, g = bg - b * p.ngroups;
  const float *src = (is_c ? p.dC32 : p.dB32) + (bg * r.nparts * N + n) * r.row_len + e;
  T *dst = static_cast<T *>(is_c ? p.dC : p.dB) + (is_c ? b * p.dC_bs + g * p.dC_gs + n * p.dC_ns : b * p.dB_bs + g * p.dB_gs + n * p.dB_ns) + e;
  const int64_t pitch = N * r.row_len;
  if (e + 4 <= len) {
    f32x4 v = *(const GLOBAL_AS f32x4_a4 *)src;
    int k = 1;
    for (; k + 4 <= r.nparts; k += 4) {
      f32x4 w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = *(const GLOBAL_AS f32x4_a4 *)(src + (k + j) * pitch);
#pragma unroll
      for (int j = 0; j < 4; ++j) v += w[j];
    }
    for (; k < r.nparts; ++k) v += *(const GLOBAL_AS f32x4_a4 *)(src + k * pitch);
    typedef u32x2 u32x2_a2 __attribute__((aligned(2)));
    if constexpr (DT<T>::id == MAMBA_F32) *(GLOBAL_AS f32x4_a4 *)dst = v;
    else if constexpr (DT<T>::id == MAMBA_BF16) *(GLOBAL_AS u32x2_a2 *)dst = u32x2{pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)};
    else *(GLOBAL_AS u32x2_a2 *)dst = u32x2{pack_f16(v.x, v.y), pack_f16(v.z, v.w)};
  } else {
    for (int i = 0; i < 4 && e + i < len; ++i) {
      float v = src[i];
      for (int k = 1; k < r.nparts; ++k) v += src[k * pitch + i];
      st1<T>(dst + i, v);
    }
  }
}

// ------------------------------------------------------------------ launch
inline bool aligned16(const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

inline size_t fwd_lds(int passes, int np, bool half) {
  return sizeof(float) * (2 * BC_FLOATS + (half ? 3 : 2) * passes * PASS_CH * np);
}
inline size_t bwd_lds(int passes, int np, int bc) {
  const int wch = passes * PASS_CH;
  return sizeof(float) * (2 * BC_FLOATS + 2 * ACC_FLOATS + PASS_CH * np + (bc ? 6 : 4) * wch * np + 2 * wch) +
         (size_t)wch * 80;  // + BwdRow per channel
}
constexpr size_t LDS_LIMIT = 160 * 1024;

int compute_units() {
  static int cus = 0;
  if (cus > 0) return cus;
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
    (void)hipGetLastError();
    return 256;  // not cached: asked again on the next call
  }
  cus = n;
  return n;
}

// Which backward kernel serves a problem.  The kernel with fp32 sums of dB / dC in LDS (below) serves every problem by
// default.  MAMBA_AMD_M1_BWD=mx in the environment (read once) sends bf16 rows with per-position B and C to the kernel
// whose dB / dC sums are formed by the matrix cores (mamba1_scan_bwd_mx.hip): measured 8 % slower at batch 8 x 5120
// channels x 4096 positions x 16 states, kept for comparisons.
// MAMBA_AMD_M1_BWD=k4 (read once): checkpoints every 64 positions from the forward kernel, and the backward kernel
// that walks 64-position tiles with 4 items per lane (mamba1_scan_bwd_k4.hip) where it serves the problem; the default
// backward kernel reads the denser checkpoints everywhere else.
bool k4_mode() {
  static const int want = [] {
    const char *e = getenv("MAMBA_AMD_M1_BWD");
    return (e && e[0] == 'k') ? 1 : 0;
  }();
  return want != 0;
}
int ckpt_tile(bool a_complex) { return a_complex ? TILE_COMPLEX : (k4_mode() ? TILE / 2 : TILE); }

bool use_mx(const MambaScanParams &p) {
  static const int want_mx = [] {
    const char *e = getenv("MAMBA_AMD_M1_BWD");
    return (e && e[0] == 'm') ? 1 : 0;
  }();
  return want_mx && p.dtype == MAMBA_BF16 && !(p.bc_const & 3) && !p.a_complex;
}

// Passes of PASS_CH channels a backward workgroup takes per tile.  More passes mean fewer, larger
// partials of dB / dC; the count is chosen so that the workgroups still fill whole rounds over the
// compute units (one workgroup per unit): the smallest rounds * passes wins, ties go to more passes.
int bwd_passes(const MambaScanParams &p, int64_t *cost_out = nullptr) {
  const int np = (p.dstate + NB16 - 1) / NB16 * NB16;
  const int Dg = p.dim / p.ngroups, cus = compute_units();
  const int64_t nseg = std::max(1, p.nseg);
  int best = 1;
  int64_t best_cost = -1;
  for (int r = 1; r <= MAX_PASSES; ++r) {
    if (r > 1 && np > NB16) break;  // states in blocks: the sums leave after every block
    if ((use_mx(p) ? mamba1_bwd_mx_lds(r, np) : bwd_lds(r, np, p.bc_const & 3)) > LDS_LIMIT) break;
    if (r > 1 && (r - 1) * PASS_CH >= Dg) break;
    const int64_t wgs = (int64_t)p.batch * nseg * p.ngroups * ((Dg + PASS_CH * r - 1) / (PASS_CH * r));
    const int64_t cost = (wgs + cus - 1) / cus * r;
    if (best_cost < 0 || cost <= best_cost) {
      best_cost = cost;
      best = r;
    }
  }
  if (cost_out) *cost_out = std::max<int64_t>(1, best_cost);
  return best;
}

// MAMBA_AMD_FWD_MIN_LDS (bytes): a measurement hook.  A workgroup of scan_fwd_kernel that asks for more LDS shares its CU with
// fewer others (160 KB per CU), which is how that kernel's speed against resident waves per SIMD is measured; where the
// hook is set, that kernel runs.
size_t fwd_min_lds() {
  static const size_t v = getenv("MAMBA_AMD_FWD_MIN_LDS") ? (size_t)atol(getenv("MAMBA_AMD_FWD_MIN_LDS")) : 0;
  return v;
}

// The forward kernel that serves a problem and its estimated time in us, for 16 states.  scan_fwd_serial_kernel
// (mamba1_scan_serial.hip) takes 16 states and per-position B and C.  With two states per lane up to five of its workgroups
// share a CU, and a tile (half tiles where the sequence ends in one) takes a round of them 7.3, 10.7, 14.1, 17.5, 20.9; with
// one, a workgroup has half as many channels and a tile takes 4.8, 6.5, 9.1, 11.6: 1 x 1536 x 256 15.1 -> 12.4 us, 8 x 1024 x
// 2048 117 -> 104, 2 x 4096 x 2048 117 -> 104, 1 x 768 x 4096 in segments 43 -> 36; from five of them on two states per lane stay
// (4 x 5120 x 512: 59 both ways).  scan_fwd_kernel: up to two per CU, 6.6 or 10.9, and a seventh more of that on rows with a
// ragged end.  Measured, 8 x 5120 channels x 4096 positions bf16: 806 -> 660 us; 8 x 2368 x 8086: 1235 -> 971; 7 x 3184 x 192: 35 -> 24;
// by these estimates it still takes ragged rows of a single tile on up to a workgroup per CU (2 x 3072 x 87).
bool serial_takes(const MambaScanParams &p) {
  return p.dstate == NB16 && !(p.bc_const & 3) && !p.a_complex && !k4_mode() && !fwd_min_lds() && p.seqlen >= KI;
}
struct FwdCost {
  int spl;  // states per lane of scan_fwd_serial_kernel, 0: scan_fwd_kernel
  double us;
};
FwdCost fwd_cost(const MambaScanParams &p, int nseg) {
  const int ntiles = (p.seqlen + TILE - 1) / TILE, Dg = p.dim / p.ngroups, cus = compute_units();
  const int64_t wgs = (int64_t)p.batch * p.ngroups * ((Dg + PASS_CH - 1) / PASS_CH) * nseg;
  const int per = (ntiles + nseg - 1) / nseg;
  if (!serial_takes(p)) {
    const double rounds = (double)((wgs + 2 * cus - 1) / (2 * cus));
    return {0, 6.4 * rounds * (wgs > cus ? 1.47 : 1.0) * ((p.dstate + NB16 - 1) / NB16) * per + 2.0 * rounds};
  }
  const double tiles = nseg > 1 ? (double)per : 0.5 * ((p.seqlen + TILE / 2 - 1) / (TILE / 2));
  const int64_t pairs = wgs / (2 * cus), odd = wgs - pairs * 2 * cus;
  const double round = (10.9 * (double)pairs + (odd > cus ? 10.9 : odd > 0 ? 6.6 : 0.0)) * (p.seqlen % KI ? 1.15 : 1.0);
  const FwdCost lanes{0, round * std::ceil(tiles) + 2.0 * (double)(pairs + (odd > 0))};
  const int64_t fives = wgs / (5 * cus), rest = (wgs - fives * 5 * cus + cus - 1) / cus;
  const FwdCost two{2, (20.9 * (double)fives + (rest ? 3.9 + 3.4 * (double)rest : 0.0)) * tiles + (p.seqlen % KI ? 3.4 : 2.0)};
  const int64_t halves = (int64_t)p.batch * p.ngroups * ((Dg + PASS_CH / 2 - 1) / (PASS_CH / 2)) * nseg;
  const int64_t fours = halves / (4 * cus), left = (halves - fours * 4 * cus + cus - 1) / cus;
  const FwdCost one{1, (11.6 * (double)fours + (left > 1 ? 1.4 + 2.55 * (double)left : 4.8 * (double)left)) * per + (p.seqlen % KI ? 3.4 : 2.0)};
  const FwdCost serial = one.us < two.us ? one : two;
  return serial.us < lanes.us ? serial : lanes;
}

// Segments of the sequence: the split with the least estimated time in us, for 16 states.  The terms were fitted to the
// times of 1 .. 32 segments (forward at 45 sizes: fwd_cost; backward at 13, batch 1 - 8, 768 - 5120 channels, 256 - 8192
// positions; within 10 % of almost all).  A tile of a round of backward workgroups (one per CU) takes 13 per pass and a
// third of that for what the passes share, a round's start and end 5.3.  The pass over the segments (all but one) takes 2.7
// (forward) or 4.5 (backward) a tile, twice that from four of its workgroups per CU on, and every segment 0.9 or 1.8 for
// its launch and for going through the segments before it; forward segments of a single tile, which a second launch and its wait for
// the first outweigh, no less than 3.5 together.  A split has to promise 1 % (forward) or 6 % (backward).  (Up to 128
// channels in all, smaller than any model's, scans are cut as before, 1 x 40 x 129 13.0 whole and 14.5 cut: the edges of segments
// are checked against the oracle at those sizes.)
// Forward scans that only scan_fwd_kernel takes (fwd_cost) keep the terms that were fitted to them: 6.4 a tile of a round of up
// to two workgroups per CU, half as much again where two share one, 3.0 for a tile of the pass over the segments, 6 % to
// promise.  (The terms for 16 states cut them too finely: 2 x 4160 x 1261, 4 states, 53 us whole and 70 in five segments; 2 x
// 1552 x 4029, 64 states, 420 us in five and 501 in 32.)
// Measured: 1536 channels x 777 positions of one sequence 35 -> 23 us forward, 133 -> 63 backward; 6 x 944 x 4251: 242 -> 181
// forward.  Forward, 1536 channels, whole and in segments: x 192 12.4 and 14.0 (two), x 256 12.3 and 13.7 (two), x 384 17.2, 19.8 (two) and
// 14.9 (three), x 777 35 and 32, 27, 28 and 23 (two, three, four, seven); 2 x 1536 x 257 18.2 and 21.3 (three).  (Asked of longer
// segments as well, the 3.5 cut 3 x 2880 x 1897 in fifteen instead of three: 151 for 140.)
constexpr int MAX_SEGMENTS = 32;
int scan_segments(const MambaScanParams &p, bool bwd) {
  const int ntiles = (p.seqlen + TILE - 1) / TILE, Dg = p.dim / p.ngroups, cus = compute_units();
  const int64_t rows = (int64_t)p.batch * p.ngroups;
  const int64_t seg_wgs = rows * ((Dg + SEG_CH - 1) / SEG_CH);
  if (p.a_complex || p.batch > 65535 || k4_mode() || use_mx(p)) return 1;
  const int blocks = (p.dstate + NB16 - 1) / NB16;
  const bool fine = !bwd && serial_takes(p), short_segments_cost = fine && (int64_t)p.batch * p.dim > 128;
  int best = 1;
  double best_cost = -1.0;
  for (int s = 1; s <= std::min(ntiles, MAX_SEGMENTS); ++s) {
    const int per = (ntiles + s - 1) / s;
    if (s > 1 && (s - 1) * per >= ntiles) continue;  // leaves the last segment empty
    double cost;
    if (bwd) {
      MambaScanParams q = p;
      q.nseg = s;
      int64_t rounds_passes = 1;
      const int r = bwd_passes(q, &rounds_passes);
      cost = 13.0 * (double)rounds_passes * (1.0 + 0.33 / r) * blocks * per + 5.3 * (double)rounds_passes / r;
    } else {
      cost = fwd_cost(p, s).us;
    }
    if (s > 1) {
      const double share = std::max(1.0, 0.52 * (double)((seg_wgs * (s - 1) + cus - 1) / cus));
      const double each = bwd ? 1.8 * s : short_segments_cost && per == 1 ? std::max(3.5, 0.9 * s) : 0.9 * s;
      cost = (fine ? 1.01 : 1.06) * (cost + (bwd ? 4.5 : fine ? 2.7 : 3.0) * share * blocks * per + each);
    }
    if (best_cost < 0 || cost < best_cost) best_cost = cost, best = s;
  }
  return best;
}

// The 4-items-per-lane backward kernel (k4 mode): two workgroups share a compute unit, so its workgroups may take
// pa and pb passes alternately (the long and the short one of a unit); pa == pb: all the same.  Chosen like
// bwd_passes: rounds of workgroups over the units' two places, times the mean passes of a round.
struct K4Plan {
  int pa, pb, nparts;
};
K4Plan k4_plan(const MambaScanParams &p) {
  const int Dg = p.dim / p.ngroups, cus = compute_units();
  static const int cand[6][2] = {{1, 1}, {2, 1}, {2, 2}, {3, 1}, {3, 2}, {3, 3}};
  K4Plan best{1, 1, 1};
  double best_cost = -1;
  for (const auto &c : cand) {
    const int pa = c[0], pb = c[1];
    if (mamba1_bwd_k4_lds(pa) > LDS_LIMIT / 2) continue;
    if (pa > 1 && (pa - 1) * PASS_CH >= Dg) continue;
    const int per = pa == pb ? (Dg + PASS_CH * pa - 1) / (PASS_CH * pa) : 2 * ((Dg + PASS_CH * (pa + pb) - 1) / (PASS_CH * (pa + pb)));
    const int64_t wgs = (int64_t)p.batch * p.ngroups * per;
    const double cost = (double)((wgs + 2 * cus - 1) / (2 * cus)) * 0.5 * (pa + pb);
    if (best_cost < 0 || cost <= best_cost) best_cost = cost, best = K4Plan{pa, pb, per};
  }
  return best;
}
bool use_k4(const MambaScanParams &p) { return k4_mode() && mamba1_bwd_k4_serves(p); }

int bwd_nparts(const MambaScanParams &p) {
  if (use_k4(p)) return k4_plan(p).nparts;
  const int Dg = p.dim / p.ngroups, r = bwd_passes(p);
  return (Dg + PASS_CH * r - 1) / (PASS_CH * r) * (p.dstate > NB16 ? r : 1);
}

// Raises a kernel's dynamic LDS limit to `lds` bytes on the current device, once: the largest size granted so far is
// remembered per (device, kernel), so that repeated launches (and launches under stream capture) make no runtime call.
}  // namespace

bool mamba1_allow_lds(const void *kernel, size_t lds) {
  static std::mutex mu;
  static std::map<std::pair<int, const void *>, size_t> granted;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  std::lock_guard<std::mutex> lock(mu);
  size_t &have = granted[{dev, kernel}];
  if (lds <= have) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  have = lds;
  return true;
}

namespace {

template <typename KernelT>
int launch(KernelT kernel, const MambaScanParams &p, int passes, size_t lds, hipStream_t stream) {
  const int Dg = p.dim / p.ngroups;
  const int cblocks = (Dg + PASS_CH * passes - 1) / (PASS_CH * passes);
  if (lds > LDS_LIMIT) return MAMBA_E_UNSUPPORTED;
  if (!mamba1_allow_lds(reinterpret_cast<const void *>(kernel), lds)) return MAMBA_E_LAUNCH;
  dim3 grid(p.ngroups * cblocks, p.batch, std::max(1, p.nseg)), block(NTHREADS);
  hipLaunchKernelGGL(kernel, grid, block, lds, stream, p, passes);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}

template <typename T, int BC, bool BWD> int launch_segments(const MambaScanParams &p, int mode, hipStream_t stream) {
  if (p.nseg <= 1) return MAMBA_OK;
  const int Dg = p.dim / p.ngroups;
  const dim3 grid(p.ngroups * ((Dg + SEG_CH - 1) / SEG_CH), p.batch, p.nseg - 1), block(SEG_THREADS);
  if (mode == ROWS_ALIGNED) hipLaunchKernelGGL((scan_seg_kernel<T, ROWS_ALIGNED, BC, BWD>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((scan_seg_kernel<T, ROWS_ANY, BC, BWD>), grid, block, 0, stream, p);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}

int check_common(const MambaScanParams *p) {
  if (!p || !p->u || !p->delta || !p->A || !p->B || !p->C || !p->ckpt) return MAMBA_E_BADARG;
  if (p->batch <= 0 || p->dim <= 0 || p->seqlen <= 0 || p->dstate <= 0 || p->ngroups <= 0) return MAMBA_E_BADARG;
  if (p->dim % p->ngroups != 0) return MAMBA_E_BADARG;
  if (p->dstate > MAX_DSTATE) return MAMBA_E_UNSUPPORTED;
  if (p->dtype != MAMBA_F32 && p->dtype != MAMBA_BF16 && p->dtype != MAMBA_F16) return MAMBA_E_BADARG;
  if (p->nseg > 1) {  // every segment holds at least one tile
    const int ntiles = (p->seqlen + TILE - 1) / TILE, per = (ntiles + p->nseg - 1) / p->nseg;
    if (!p->seg_ws || p->nseg > MAX_SEGMENTS || (p->nseg - 1) * per >= ntiles) return MAMBA_E_BADARG;
    if (p->a_complex || p->batch > 65535 || k4_mode() || use_mx(*p)) return MAMBA_E_UNSUPPORTED;
  }
  return MAMBA_OK;
}

// 16-byte accesses need every row start aligned and whole 8-item groups.
bool vec_ok(const MambaScanParams &p, bool bwd) {
  const int es = p.dtype == MAMBA_F32 ? 4 : 2;
  const int64_t m = 16 / es;
  auto ok = [&](const void *ptr, int64_t s0, int64_t s1) { return !ptr || (aligned16(ptr) && s0 % m == 0 && s1 % m == 0); };
  if (p.seqlen % 8 != 0) return false;
  bool v = ok(p.u, p.u_bs, p.u_ds) && ok(p.delta, p.delta_bs, p.delta_ds) && ok(p.z, p.z_bs, p.z_ds);
  if (!(p.bc_const & 1)) v = v && ok(p.B, p.B_bs, p.B_gs) && p.B_ns % m == 0;
  if (!(p.bc_const & 2)) v = v && ok(p.C, p.C_bs, p.C_gs) && p.C_ns % m == 0;
  if (!bwd) return v && ok(p.out, p.out_bs, p.out_ds);
  if (!(p.bc_const & 1)) v = v && aligned16(p.dB32);
  if (!(p.bc_const & 2)) v = v && aligned16(p.dC32);
  return v && ok(p.dout, p.dout_bs, p.dout_ds) && ok(p.du, p.du_bs, p.du_ds) &&
         ok(p.ddelta, p.ddelta_bs, p.ddelta_ds) && ok(p.dz, p.dz_bs, p.dz_ds) && ok(p.out_z, p.outz_bs, p.outz_ds);
}
int row_mode(const MambaScanParams &p, bool bwd) {
  return vec_ok(p, bwd) ? ROWS_ALIGNED : p.seqlen >= KI ? ROWS_ANY : ROWS_SCALAR;
}

// dB / dC of per-position operands and, where the caller wants the finished sums, dA, dD and ddelta_bias.  `which`: bit
// 0 the former, bit 1 the latter (a problem served in slices of batch rows adds those up once, at the end).
template <typename T> int reduce_sums(const MambaScanParams &p_in, int nparts, int which, hipStream_t stream) {
  MambaScanParams p = p_in;
  ReduceGeo r{};
  const int64_t cx = p.a_complex ? 2 : 1, G = p.ngroups, N = p.dstate;
  r.nparts = nparts, r.nsum = p.batch * std::max(1, p.nseg);
  r.row_len = p.seqlen * cx;
  r.rows = (int64_t)p.batch * G * N;
  r.per_row = (int)((r.row_len + 3) / 4);
  if (!(p.dB_bs | p.dB_gs | p.dB_ns)) p.dB_bs = G * N * r.row_len, p.dB_gs = N * r.row_len, p.dB_ns = r.row_len;
  if (!(p.dC_bs | p.dC_gs | p.dC_ns)) p.dC_bs = G * N * r.row_len, p.dC_gs = N * r.row_len, p.dC_ns = r.row_len;
  const int operands = (which & 1) ? ((p.bc_const & 1) ? 0 : 1) + ((p.bc_const & 2) ? 0 : 1) : 0;
  const int64_t each = (r.rows * r.per_row + 255) / 256, nbc = operands * each;
  int64_t sums = 0;
  if ((which & 2) && (p.dA || p.dD || p.ddelta_bias)) sums = ((int64_t)p.dim * (N * cx + 2) + 255) / 256;
  if (nbc + sums == 0) return MAMBA_OK;
  if (nbc + sums > 0x7fffffff) return MAMBA_E_UNSUPPORTED;
  r.nbc = (int)nbc;
  hipLaunchKernelGGL(reduce_parts_kernel<T>, dim3((unsigned)(nbc + sums)), dim3(256), 0, stream, p, r);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}
template <typename T> int reduce_dBC(const MambaScanParams &p, const MambaScanParams &plan, int nparts, hipStream_t stream) {
  return reduce_sums<T>(p, nparts, p.batch == plan.batch ? 3 : 1, stream);
}

// `plan`: the whole problem, of which p may be a slice of batch rows; it decides the passes per workgroup and with
// them the number of dB / dC partials, which must be the same for every slice.
template <typename T, bool BWD, int BC> int dispatch_bc(const MambaScanParams &p, const MambaScanParams &plan, hipStream_t stream) {
  const int np = (p.dstate + NB16 - 1) / NB16 * NB16;
  const int mode = row_mode(p, BWD);
  int rc = launch_segments<T, BC, BWD>(p, mode, stream);
  if (rc != MAMBA_OK) return rc;
  if (!BWD) {
    const bool half = k4_mode();
    const int spl = fwd_cost(p, std::max(1, p.nseg)).spl;
    if (spl) return mamba1_fwd_serial_launch(p, spl, mode, stream);
    const size_t lds = std::max(fwd_lds(1, np, half), fwd_min_lds());
    if (half)
      return mode == ROWS_ALIGNED ? launch(scan_fwd_kernel<T, ROWS_ALIGNED, BC, true>, p, 1, lds, stream)
                                  : launch(scan_fwd_kernel<T, ROWS_SCALAR, BC, true>, p, 1, lds, stream);
    switch (mode) {
      case ROWS_ALIGNED: return launch(scan_fwd_kernel<T, ROWS_ALIGNED, BC, false>, p, 1, lds, stream);
      case ROWS_ANY: return launch(scan_fwd_kernel<T, ROWS_ANY, BC, false>, p, 1, lds, stream);
      default: return launch(scan_fwd_kernel<T, ROWS_SCALAR, BC, false>, p, 1, lds, stream);
    }
  }
  if (use_k4(plan)) {
    const K4Plan k = k4_plan(plan);
    if (mode == ROWS_ALIGNED) {
      if constexpr (std::is_same_v<T, bf16_t> && BC == 0) {
        rc = mamba1_bwd_k4_launch(p, k.pa, k.pb, k.nparts, stream);
        return rc != MAMBA_OK ? rc : reduce_dBC<T>(p, plan, k.nparts, stream);
      }
    }
    // rows the 4-item kernel does not take (unaligned views): the default kernel with as many passes as a long and a
    // short workgroup together, whose partials are fewer than the workspace was sized for: the others are cleared
    const int64_t bytes = (int64_t)p.batch * p.ngroups * k.nparts * p.dstate * p.seqlen * 4;
    rc = mamba_hip_zero(p.dB32, bytes, stream);
    if (rc == MAMBA_OK) rc = mamba_hip_zero(p.dC32, bytes, stream);
    if (rc != MAMBA_OK) return rc;
    const int passes = k.pa == k.pb ? k.pa : k.pa + k.pb;
    rc = launch(scan_bwd_kernel<T, ROWS_SCALAR, BC, true>, p, passes, bwd_lds(passes, np, BC), stream);
    return rc != MAMBA_OK ? rc : reduce_dBC<T>(p, plan, k.nparts, stream);
  }
  const int passes = bwd_passes(plan);
  if (use_mx(p)) {
    rc = mamba1_bwd_mx_launch(p, passes, mode == ROWS_ALIGNED, stream);
    return rc != MAMBA_OK ? rc : reduce_dBC<T>(p, plan, bwd_nparts(plan), stream);
  }
  const size_t lds = bwd_lds(passes, np, BC);
  if (k4_mode())
    rc = mode == ROWS_ALIGNED ? launch(scan_bwd_kernel<T, ROWS_ALIGNED, BC, true>, p, passes, lds, stream)
                              : launch(scan_bwd_kernel<T, ROWS_SCALAR, BC, true>, p, passes, lds, stream);
  else if (mode == ROWS_ALIGNED) rc = launch(scan_bwd_kernel<T, ROWS_ALIGNED, BC, false>, p, passes, lds, stream);
  else if (mode == ROWS_ANY) rc = launch(scan_bwd_kernel<T, ROWS_ANY, BC, false>, p, passes, lds, stream);
  else rc = launch(scan_bwd_kernel<T, ROWS_SCALAR, BC, false>, p, passes, lds, stream);
  return rc != MAMBA_OK ? rc : reduce_dBC<T>(p, plan, bwd_nparts(plan), stream);
}

template <typename T, bool BWD> int dispatch(const MambaScanParams &p, const MambaScanParams &plan, hipStream_t stream) {
  switch (p.bc_const & 3) {
    case 0: return dispatch_bc<T, BWD, 0>(p, plan, stream);
    case 1: return dispatch_bc<T, BWD, 1>(p, plan, stream);
    case 2: return dispatch_bc<T, BWD, 2>(p, plan, stream);
    default: return dispatch_bc<T, BWD, 3>(p, plan, stream);
  }
}

// The grid's batch coordinate is 16 bits wide: a larger batch is served in slices of rows (rows are independent; every
// per-row pointer is advanced, the per-(batch, channel) partial sums included).
constexpr int MAX_GRID_BATCH = 65535;

MambaScanParams batch_slice(const MambaScanParams &p, int64_t b0, int nb, int nparts) {
  MambaScanParams q = p;
  q.batch = nb;
  const int64_t es = p.dtype == MAMBA_F32 ? 4 : 2, cx = p.a_complex ? 2 : 1;
  const int tile = ckpt_tile(p.a_complex);
  const int64_t ntiles = (p.seqlen + tile - 1) / tile, N = p.dstate, L = p.seqlen, G = p.ngroups, D = p.dim;
  auto adv = [&](auto *&ptr, int64_t elems, int64_t size) {
    if (ptr) ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(
                 reinterpret_cast<uintptr_t>(ptr) + (uintptr_t)(b0 * elems * size));
  };
  adv(q.u, p.u_bs, es), adv(q.delta, p.delta_bs, es), adv(q.z, p.z_bs, es), adv(q.out, p.out_bs, es);
  if (!(p.bc_const & 1)) adv(q.B, p.B_bs, es);
  if (!(p.bc_const & 2)) adv(q.C, p.C_bs, es);
  adv(q.ckpt, D * ntiles * N * cx, 4);
  adv(q.dout, p.dout_bs, es), adv(q.du, p.du_bs, es), adv(q.ddelta, p.ddelta_bs, es), adv(q.dz, p.dz_bs, es);
  adv(q.out_z, p.outz_bs, es);
  adv(q.dB32, (p.bc_const & 1) ? D * N * cx : G * nparts * N * L * cx, 4);
  adv(q.dC32, (p.bc_const & 2) ? D * N * cx : G * nparts * N * L * cx, 4);
  adv(q.dA_part, D * N * cx, 4), adv(q.dD_part, D, 4), adv(q.ddelta_bias_part, D, 4);
  adv(q.dB, (p.dB_bs | p.dB_gs | p.dB_ns) ? p.dB_bs : G * N * L * cx, es);
  adv(q.dC, (p.dC_bs | p.dC_gs | p.dC_ns) ? p.dC_bs : G * N * L * cx, es);
  adv(q.det_dB, G * N * L * cx, 8), adv(q.det_dC, G * N * L * cx, 8);
  return q;
}

}  // namespace

int mamba1_scan_complex(const MambaScanParams *p, hipStream_t s, bool bwd);  // mamba1_scan_complex.hip

int mamba1_scan_tile(bool a_complex) { return ckpt_tile(a_complex); }  // positions per checkpoint tile

namespace {
int scan_fwd_one(const MambaScanParams &p, hipStream_t s) {
  if (p.a_complex) return mamba1_scan_complex(&p, s, false);
  switch (p.dtype) {
    case MAMBA_F32: return dispatch<float, false>(p, p, s);
    case MAMBA_BF16: return dispatch<bf16_t, false>(p, p, s);
    default: return dispatch<f16_t, false>(p, p, s);
  }
}

int scan_bwd_one(const MambaScanParams &p, const MambaScanParams &plan, mamba_stream_t stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (p.a_complex) {
    // the complex kernels add their dB / dC terms into one fp32 copy with atomics: clear it, run, convert
    const int64_t bytes = (int64_t)p.batch * p.ngroups * p.dstate * 2 * p.seqlen * 4;
    int rc = MAMBA_OK;
    if (!(p.bc_const & 1)) rc = mamba_hip_zero(p.dB32, bytes, stream);
    if (rc == MAMBA_OK && !(p.bc_const & 2)) rc = mamba_hip_zero(p.dC32, bytes, stream);
    if (p.det_scale && ((!(p.bc_const & 1) && !p.det_dB) || (!(p.bc_const & 2) && !p.det_dC))) return MAMBA_E_BADARG;
    if (rc == MAMBA_OK) rc = mamba1_scan_complex(&p, s, true);
    if (rc == MAMBA_OK && p.det_scale) {  // the integer sums -> the fp32 sums the conversion below reads
      if (!(p.bc_const & 1)) rc = ssd_det_convert(p.det_dB, p.dB32, bytes / 4, p.det_scale, stream);
      if (rc == MAMBA_OK && !(p.bc_const & 2)) rc = ssd_det_convert(p.det_dC, p.dC32, bytes / 4, p.det_scale, stream);
    }
    if (rc != MAMBA_OK) return rc;
    switch (p.dtype) {
      case MAMBA_F32: return reduce_dBC<float>(p, plan, 1, s);
      case MAMBA_BF16: return reduce_dBC<bf16_t>(p, plan, 1, s);
      default: return reduce_dBC<f16_t>(p, plan, 1, s);
    }
  }
  switch (p.dtype) {
    case MAMBA_F32: return dispatch<float, true>(p, plan, s);
    case MAMBA_BF16: return dispatch<bf16_t, true>(p, plan, s);
    default: return dispatch<f16_t, true>(p, plan, s);
  }
}
}  // namespace

extern "C" int mamba1_scan_fwd(const MambaScanParams *p, mamba_stream_t stream) {
  int rc = check_common(p);
  if (rc != MAMBA_OK) return rc;
  if (!p->out) return MAMBA_E_BADARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  for (int64_t b0 = 0; b0 < p->batch; b0 += MAX_GRID_BATCH) {
    const int nb = (int)std::min<int64_t>(MAX_GRID_BATCH, p->batch - b0);
    rc = p->batch <= MAX_GRID_BATCH ? scan_fwd_one(*p, s) : scan_fwd_one(batch_slice(*p, b0, nb, 1), s);
    if (rc != MAMBA_OK) return rc;
  }
  return MAMBA_OK;
}

// ----------------------------------------------------- forward without a caller workspace
// The tile checkpoints of mamba1_scan_fwd_noalloc live in this array instead of a caller buffer.
// Host code never uses the array's name as an address: the device address is looked up once per
// device with hipGetSymbolAddress and kept in g_scratch_ptr.
constexpr int64_t SCRATCH_FLOATS = (int64_t)MAMBA_NOALLOC_SCRATCH_BYTES / 4;
constexpr int SCRATCH_MAX_DEVICES = 64;
static __device__ __align__(256) float scratch[SCRATCH_FLOATS];
static float *g_scratch_ptr[SCRATCH_MAX_DEVICES];  // per device, null until resolved

namespace {
// Device address of `scratch` on the current device (resolved on first use), or null on failure.
float *scratch_for_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SCRATCH_MAX_DEVICES) {
    (void)hipGetLastError();
    return nullptr;
  }
  float *ptr = __atomic_load_n(&g_scratch_ptr[dev], __ATOMIC_ACQUIRE);
  if (ptr) return ptr;
  if (hipGetSymbolAddress(reinterpret_cast<void **>(&ptr), HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
    (void)hipGetLastError();
    return nullptr;
  }
  __atomic_store_n(&g_scratch_ptr[dev], ptr, __ATOMIC_RELEASE);
  return ptr;
}

// last_state[b, d, :] = ckpt[b, d, ntiles - 1, :]; `width` floats per (b, d) row (dstate, or 2 * dstate
// for a complex state).
__global__ __launch_bounds__(256) void gather_last_state_kernel(const float *__restrict__ ckpt, float *__restrict__ last,
                                                                int64_t rows, int ntiles, int width) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= rows * width) return;
  const int64_t row = i / width;
  const int n = (int)(i - row * width);
  last[i] = ckpt[(row * ntiles + (ntiles - 1)) * width + n];
}
}  // namespace

extern "C" int mamba_hip_init(void) { return scratch_for_current_device() ? MAMBA_OK : MAMBA_E_LAUNCH; }

extern "C" int mamba1_scan_fwd_noalloc(const MambaScanParams *p, float *last_state, mamba_stream_t stream) {
  if (!p) return MAMBA_E_BADARG;
  if (p->batch <= 0 || p->dim <= 0 || p->seqlen <= 0 || p->dstate <= 0) return MAMBA_E_BADARG;
  const int tile = ckpt_tile(p->a_complex);
  const int ntiles = (p->seqlen + tile - 1) / tile;
  const int width = p->dstate * (p->a_complex ? 2 : 1);
  const int64_t rows = (int64_t)p->batch * p->dim;
  if (rows * ntiles > SCRATCH_FLOATS / width) return MAMBA_E_UNSUPPORTED;  // checkpoints beyond the fixed buffer
  float *ws = scratch_for_current_device();
  if (!ws) return MAMBA_E_LAUNCH;
  MambaScanParams q = *p;
  q.ckpt = ws;
  q.nseg = 0;
  const int rc = mamba1_scan_fwd(&q, stream);
  if (rc != MAMBA_OK || !last_state) return rc;
  const int64_t n = rows * width;
  if ((n + 255) / 256 > 0x7fffffff) return MAMBA_E_UNSUPPORTED;
  hipLaunchKernelGGL(gather_last_state_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), ws, last_state, rows, ntiles, width);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}

extern "C" int mamba1_scan_bwd_nparts(const MambaScanParams *p) {
  if (!p || p->batch <= 0 || p->dim <= 0 || p->seqlen <= 0 || p->dstate <= 0 || p->ngroups <= 0 ||
      p->dim % p->ngroups != 0)
    return MAMBA_E_BADARG;
  if (p->dstate > MAX_DSTATE) return MAMBA_E_UNSUPPORTED;
  return p->a_complex ? 1 : bwd_nparts(*p);
}

extern "C" int mamba1_scan_bwd(const MambaScanParams *p, mamba_stream_t stream) {
  int rc = check_common(p);
  if (rc != MAMBA_OK) return rc;
  if (!p->dout || !p->du || !p->ddelta || !p->dB32 || !p->dC32 || !p->dA_part || !p->dD_part || !p->ddelta_bias_part)
    return MAMBA_E_BADARG;
  if ((!(p->bc_const & 1) && !p->dB) || (!(p->bc_const & 2) && !p->dC)) return MAMBA_E_BADARG;
  if (p->z && !p->dz) return MAMBA_E_BADARG;
  const int nparts = p->a_complex ? 1 : bwd_nparts(*p);
  for (int64_t b0 = 0; b0 < p->batch; b0 += MAX_GRID_BATCH) {
    const int nb = (int)std::min<int64_t>(MAX_GRID_BATCH, p->batch - b0);
    rc = p->batch <= MAX_GRID_BATCH ? scan_bwd_one(*p, *p, stream) : scan_bwd_one(batch_slice(*p, b0, nb, nparts), *p, stream);
    if (rc != MAMBA_OK) return rc;
  }
  if (p->batch > MAX_GRID_BATCH) return reduce_sums<float>(*p, nparts, 2, static_cast<hipStream_t>(stream));
  return MAMBA_OK;
}

extern "C" int mamba1_scan_segments(const MambaScanParams *p, int backward) {
  if (!p || p->batch <= 0 || p->dim <= 0 || p->seqlen <= 0 || p->dstate <= 0 || p->ngroups <= 0 || p->dim % p->ngroups != 0)
    return MAMBA_E_BADARG;
  return p->seqlen < KI ? 1 : scan_segments(*p, backward != 0);
}
