// Pieces shared by the Mamba-1 scan kernels (mamba1_scan.hip, mamba1_scan_bwd_mx.hip): the tile constants,
// the staging of the B / C rows of a tile in LDS, row loads, and the channel geometry of a workgroup.
#pragma once
#include "common.hpp"

namespace {

constexpr int KI = 8;             // items per lane
constexpr int RL = 16;            // lanes per channel (one DPP row)
constexpr int ROWS = 4;           // channels per wave
constexpr int TILE = RL * KI;     // sequence positions per tile
constexpr int TILE_COMPLEX = 512; // tile of the complex kernels (mamba1_scan_complex.hip)
constexpr int NB16 = 16;          // states staged per LDS block
constexpr int NWAVES = 8;
constexpr int NTHREADS = NWAVES * 64;
constexpr int PASS_CH = NWAVES * ROWS;         // channels of a workgroup per pass
constexpr int BC_FLOATS = NB16 * TILE;         // one staged operand
constexpr int ACC_PITCH = TILE * ROWS;         // floats per state row of a dB / dC accumulator
constexpr int ACC_FLOATS = NB16 * ACC_PITCH;   // one accumulator: [n][half][lane][4]
constexpr int MAX_DSTATE = 256;
constexpr int MAX_PASSES = 8;

// How a kernel reaches the rows (positions contiguous): ROWS_SCALAR element by element (fewer than 8 positions),
// ROWS_ALIGNED 16-byte pieces (16-byte aligned rows, whole pieces), ROWS_ANY 16-byte pieces at any alignment with a
// ragged last piece, which is loaded from inside the row and moved into place.
constexpr int ROWS_SCALAR = 0, ROWS_ALIGNED = 1, ROWS_ANY = 2;

// B or C rows n0..n0+15 of the tile starting at t0 -> LDS as fp32, laid out [n][half][c][4] (c = the
// lane's place in its row) so that a lane reads its 8 items with two 16-byte LDS loads.
// BC: bit 0 set = B is not staged (input-independent), bit 1 = C likewise.
template <typename T, int MODE, int BC>
DEVI void stage_bc(float *Bs, float *Cs, const T *Bg, int64_t B_ns, const T *Cg, int64_t C_ns, int n0, int N, int t0,
                   int L, int tid) {
  constexpr int FIRST = (BC & 1) ? NB16 * RL : 0, LAST = (BC & 2) ? NB16 * RL : 2 * NB16 * RL;
  if constexpr (BC == 3) {
    return;  // nothing is staged
  } else {
    const int unit = FIRST + tid;  // one 8-item unit per thread: 2 operands x 16 states x 16 segments
    if (unit >= LAST) return;
    const int which = unit >> 8, n = (unit >> 4) & 15, j = unit & 15;
    float v[8];
    if constexpr (MODE != ROWS_SCALAR) {
      // from a clamped (valid) address, masked afterwards
      const int nc = min(n0 + n, N - 1), t = t0 + KI * j;
      const T *row = which ? Cg + (int64_t)nc * C_ns : Bg + (int64_t)nc * B_ns;
      if constexpr (MODE == ROWS_ALIGNED) {
        Pack8<T> raw;
        raw.load(row + min(t, L - KI));
        raw.unpack(v);
      } else {
        row8_raw<T>(row, t, L, v);
        if (t0 + TILE > L) row8_place(t, L, v);
      }
      const bool ok = n0 + n < N && t < L;
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = ok ? v[i] : 0.f;
    } else {
      const int t = t0 + KI * j;
      const T *src = (which ? Cg + (int64_t)(n0 + n) * C_ns : Bg + (int64_t)(n0 + n) * B_ns) + t;
      const int nvalid = (n0 + n < N) ? min(max(L - t, 0), KI) : 0;
      ld8_guard<T, false>(src, nvalid, 0.f, v);
    }
    float *dst = (which ? Cs : Bs) + n * TILE + j * 4;
    *reinterpret_cast<f32x4 *>(dst) = f32x4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4 *>(dst + 4 * RL) = f32x4{v[4], v[5], v[6], v[7]};
  }
}

// The 8 items of one (batch, channel) row owned by this lane, as stored: 16 bytes from a clamped position (the
// caller masks lanes past the end, and moves a ragged row's last piece into place: place_items), or element by element.
template <typename T, int MODE> DEVI void load_items(Pack8<T> &k, const T *row, int tl, int L, int nvalid) {
  if constexpr (MODE == ROWS_ALIGNED) {
    k.load_global(row + min(tl, L - KI));
  } else if constexpr (MODE == ROWS_ANY) {
    k.load_any(row + min(tl, L - KI));
  } else {
    float v[8];
    ld8_guard<T, false>(row + tl, nvalid, 0.f, v);
    k.pack(v);
  }
}

// After the unpacking of rows that load_items has read: only the last tile of a ragged row has anything to move.
template <int MODE> DEVI void place_items(float (&v)[8], int t0, int tl, int L) {
  if constexpr (MODE == ROWS_ANY) {
    if (t0 + TILE > L) row8_place(tl, L, v);
  }
}
// the values of a ragged row's last piece, element by element
template <typename T, int MODE> DEVI void st8_tail(T *dst, bool wanted, int t0, int L, int nvalid, const float (&v)[8]) {
  if constexpr (MODE == ROWS_ANY) {
    if (t0 + TILE > L && wanted && nvalid < KI) st8_guard<T, false>(dst, nvalid, v);
  }
}

// 8 floats of a [half][slot][4] LDS row: a slot's two 16-byte halves lie HALF_STRIDE floats apart
template <int HALF_STRIDE> DEVI void lds_st8(float *base, int slot, const float (&v)[8]) {
  *reinterpret_cast<f32x4 *>(base + slot * 4) = f32x4{v[0], v[1], v[2], v[3]};
  *reinterpret_cast<f32x4 *>(base + HALF_STRIDE + slot * 4) = f32x4{v[4], v[5], v[6], v[7]};
}
template <int HALF_STRIDE> DEVI void lds_ld8(const float *base, int slot, float (&o)[8]) {
  const f32x4 lo = *reinterpret_cast<const f32x4 *>(base + slot * 4);
  const f32x4 hi = *reinterpret_cast<const f32x4 *>(base + HALF_STRIDE + slot * 4);
  o[0] = lo.x; o[1] = lo.y; o[2] = lo.z; o[3] = lo.w;
  o[4] = hi.x; o[5] = hi.y; o[6] = hi.z; o[7] = hi.w;
}

// The 8 items of B (or C) for state n of channel d: from the staged tile, or, when the operand is an
// input-independent (dim, dstate) fp32 matrix, its one value for every position (0 for padded states).
template <int CONST>
DEVI void load_bc(float (&v)[8], const float *staged, const void *mat, int d, int N, int n_abs, int n_loc, int c) {
  if constexpr (CONST != 0) {
    const float x = n_abs < N ? static_cast<const float *>(mat)[(int64_t)d * N + n_abs] : 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = x;
  } else {
    lds_ld8<4 * RL>(staged + n_loc * TILE, c, v);
  }
}

// Where a workgroup's channels lie: workgroup cb of group g takes `passes` passes of CH channels, and the tiles
// [tile0, tile1) of segment blockIdx.z of the sequence.
struct Geo {
  int g, cb, b, Dg, dend, ntiles, cblocks, seg, nseg, tile0, tile1;
};
DEVI int tiles_per_segment(int ntiles, int nseg) { return (ntiles + nseg - 1) / nseg; }
template <int CH = PASS_CH> DEVI Geo geometry(const MambaScanParams &p, int passes) {
  Geo q;
  q.Dg = p.dim / p.ngroups;
  q.cblocks = (q.Dg + CH * passes - 1) / (CH * passes);
  q.g = blockIdx.x / q.cblocks;
  q.cb = blockIdx.x % q.cblocks;
  q.b = blockIdx.y;
  q.dend = (q.g + 1) * q.Dg;
  q.ntiles = (p.seqlen + TILE - 1) / TILE;
  q.seg = blockIdx.z;
  q.nseg = max(1, p.nseg);
  const int per = tiles_per_segment(q.ntiles, q.nseg);
  q.tile0 = q.seg * per;
  q.tile1 = min(q.ntiles, q.tile0 + per);
  return q;
}

// The workspace of a sequence cut into segments (mamba1_scan.hip).
DEVI int64_t seg_row(const MambaScanParams &p, int b, int seg, int d) { return ((int64_t)b * p.nseg + seg) * p.dim + d; }
DEVI float *seg_sums(const MambaScanParams &p) { return p.seg_ws + (int64_t)p.batch * p.nseg * p.dim * p.dstate; }
DEVI float *seg_firsts(const MambaScanParams &p) { return seg_sums(p) + (int64_t)p.batch * p.nseg * p.dim; }

// State entering this workgroup's segment (A2 = A log2 e)
DEVI float seg_state_in(const MambaScanParams &p, const Geo &q, int d, int n, float A2) {
  float h = 0.f;
  for (int s = 0; s < q.seg; ++s) {
    const int64_t row = seg_row(p, q.b, s, d);
    h = __builtin_fmaf(fast_exp2(A2 * seg_sums(p)[row]), h, p.seg_ws[row * p.dstate + n]);
  }
  return h;
}
// Row starts of one channel of the workgroup, kept in LDS: every (tile, pass) step needs nine
// addresses per lane, and as kernel arguments next to the loop state they did not fit the scalar
// registers (each step then re-read hundreds of spilled scalars through v_readlane).  Pointers read back
// from LDS carry no address space, so the rows are accessed through the helpers that name the global one.
template <typename T> struct BwdRow {
  const T *u, *delta, *dout, *z;
  T *du, *ddelta, *dz, *out_z;
  const float *ckpt;  // tile 0 of this channel
  float D, bias;
};

// 32 bytes per thread that nobody reads: a lane with nothing to store (past the end of the sequence, no z)
// stores there instead of branching around the store.  Shared by all workgroups.
static __device__ __align__(16) float bwd_spare[NTHREADS * 8];

}  // namespace
