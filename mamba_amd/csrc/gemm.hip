// bf16 matrix products: the projections inside a mixer (x_proj, dt_proj, out_proj and their gradients) where the problem is short
// or a library splits it badly.  A library product costs ~18 us of host time whatever its size, more than the product itself up
// to a few GFLOP; these cost a launch (~2 us), up to MAXG independent products share one, and operands are taken as
// they lie (either index contiguous, any alignment of the element's size), results in bf16 or fp32.
//
// Three tile sizes (form_of).  64 x 64 per workgroup of four waves, k in steps of 32 (the block core of the SSD kernels): what
// bounds a short product is the latency of its loads, not the matrix cores, so the operands of the next PF steps are in flight and
// the LDS tiles are double-buffered (one barrier a step).  128 x 128 and 256 x 256 for larger ones, which the 64 x 64 tiles'
// reading through the L2 would bound.  A product whose tiles do not fill the chip is split along k, the splits' fp32 tiles added
// up by a second kernel in a fixed order.
#include "ssd_common.hpp"

namespace {

constexpr int MAXG = 4, PF = 4;
struct Group {
  MambaGemm g[MAXG];
  int first[MAXG + 1];  // first workgroup of every product
  int helpers[MAXG];    // see Share
  float *ws[MAXG];
};

// The operand with rows r (m or n) and k: element (r, k) at base[r * s + k], or with TR at base[k * s + r].  A whole
// step of 32 k is read without guards: past the last row the rows before it are read again (their results are not
// stored), in the transposed layout up to 7 elements of the next k's row (`whole` says for which steps that stays
// inside the operand).
template <bool TR> struct Operand {
  const bf16_t *base;
  int64_t s;
  int rows, K;  // rows of this tile, whole extent of k
  int64_t rest;  // elements from base to the operand's end
  int t;
  DEVI Operand(const void *p, int64_t rs, int64_t ks, int row0, int all_rows, int K_, int t_)
      : base(static_cast<const bf16_t *>(p) + (int64_t)row0 * rs), s(TR ? ks : rs), rows(min(all_rows - row0, GB)), K(K_), t(t_) {
    rest = TR ? (int64_t)(K - 1) * ks + all_rows - row0 : 0;
  }
  DEVI bool whole(int k0) const {
    if (k0 + GK > K) return false;
    return !TR || rows == GB || (int64_t)(k0 + GK - 1) * s + (rows + 7) / 8 * 8 <= rest;
  }
  DEVI void fetch(Pack8<bf16_t> &q, int k0) const {
    if constexpr (TR) {
      const int r8 = (t & 7) * 8;
      q.load_any(base + (int64_t)(k0 + (t >> 3)) * s + (r8 < rows ? r8 : 0));
    } else {
      q.load_any(base + (int64_t)min(t >> 2, rows - 1) * s + k0 + (t & 3) * 8);
    }
  }
  DEVI void fetch_guarded(Pack8<bf16_t> &q, int k0) const {
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if constexpr (TR) {
      const int k = k0 + (t >> 3), r8 = (t & 7) * 8;
      if (k < K) {
        const bf16_t *src = base + (int64_t)k * s + r8;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (r8 + e < rows) v[e] = ld1<bf16_t>(src + e);
      }
    } else {
      const int k = k0 + (t & 3) * 8;
      const bf16_t *src = base + (int64_t)min(t >> 2, rows - 1) * s + k;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (k + e < K) v[e] = ld1<bf16_t>(src + e);
    }
    q.pack(v);
  }
  DEVI void commit(uint16_t *tile, const Pack8<bf16_t> &q) const {
    if constexpr (TR) put_raw<bf16_t>(tile, tr_off(t >> 3, (t & 7) * 8), q, true);
    else put_raw<bf16_t>(tile, tile_off(t >> 2, (t & 3) * 8), q, true);
  }
};

struct GemmTiles {
  uint16_t x[2][GTILE], y[2][GTILE];
};

template <bool XTR, bool YTR> DEVI void tile_mma(GemmAcc &acc, const uint16_t *x, const uint16_t *y, int wx, int wy, int lane) {
  const int i = lane & 15, g = lane >> 4;
  bf16x8_t a[2], b[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    a[u] = load_frag<XTR>(x, wx * 32 + u * 16, i, g);
    b[u] = load_frag<YTR>(y, wy * 32 + u * 16, i, g);
  }
#pragma unroll
  for (int tx = 0; tx < 2; ++tx)
#pragma unroll
    for (int ty = 0; ty < 2; ++ty) acc.v[tx][ty] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tx], b[ty], acc.v[tx][ty], 0, 0, 0);
}

// Steps [j0, j1) of the k axis.  X: the operand with the rows n, so that a lane's four accumulators are four
// neighbouring columns of a row of D; Y: the one with the rows m.
template <bool XTR, bool YTR>
DEVI void run_tile(GemmAcc &acc, GemmTiles &sh, const Operand<XTR> &X, const Operand<YTR> &Y, int j0, int j1, int tid) {
  const int lane = tid & 63, wave = tid >> 6, wx = wave & 1, wy = wave >> 1;
  int nf = j1;  // steps [j0, nf) are whole ones
  while (nf > j0 && !(X.whole((nf - 1) * GK) && Y.whole((nf - 1) * GK))) --nf;
  Pack8<bf16_t> qx[PF], qy[PF], rx, ry;
  if (nf > j0) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int k0 = min(j0 + u, nf - 1) * GK;
      X.fetch(qx[u], k0);
      Y.fetch(qy[u], k0);
    }
  }
  if (nf < j1) {
    X.fetch_guarded(rx, nf * GK);
    Y.fetch_guarded(ry, nf * GK);
  }
  auto step = [&](int j, const Pack8<bf16_t> &cx, const Pack8<bf16_t> &cy, auto &&next) {
    uint16_t *tx = sh.x[j & 1], *ty = sh.y[j & 1];
    X.commit(tx, cx);
    Y.commit(ty, cy);
    lds_barrier();  // (the tiles of step j - 2 were read before the barrier of step j - 1)
    next();
    tile_mma<XTR, YTR>(acc, tx, ty, wx, wy, lane);
  };
  int j = j0;
  auto piped = [&](int u) {
    step(j + u, qx[u], qy[u], [&] {
      const int k0 = min(j + u + PF, nf - 1) * GK;
      X.fetch(qx[u], k0);
      Y.fetch(qy[u], k0);
    });
  };
  for (; j + PF <= nf; j += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) piped(u);
  }
#pragma unroll
  for (int u = 0; u < PF - 1; ++u)
    if (j + u < nf) step(j + u, qx[u], qy[u], [] {});
  for (j = nf; j < j1; ++j) {  // what is left: the last, ragged step
    step(j, rx, ry, [] {});
    if (j + 1 < j1) {
      X.fetch_guarded(rx, (j + 1) * GK);
      Y.fetch_guarded(ry, (j + 1) * GK);
    }
  }
}

// four neighbouring columns n .. n + 3 of row m
DEVI void store4(const MambaGemm &g, int m, int n, f32x4 v) {
  if (m >= g.M || n >= g.N) return;
  const int64_t o = (int64_t)m * g.ldd + n;
  const int cols = min(4, g.N - n);
  float x[4] = {v.x, v.y, v.z, v.w};
  if (g.bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] += e < cols ? ld1<bf16_t>(static_cast<const bf16_t *>(g.bias) + n + e) : 0.f;
  }
  if (g.d_dtype == MAMBA_F32) {
    float *d = static_cast<float *>(g.D) + o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < cols) d[e] = g.accumulate ? d[e] + x[e] : x[e];
    return;
  }
  bf16_t *d = static_cast<bf16_t *>(g.D) + o;
  typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(2)));
  if (cols == 4) {
    if (g.accumulate) {
      const u32x2_any old = *reinterpret_cast<const u32x2_any *>(d);
      x[0] += bf16_lo(old.x), x[1] += bf16_hi(old.x), x[2] += bf16_lo(old.y), x[3] += bf16_hi(old.y);
    }
    *reinterpret_cast<u32x2_any *>(d) = u32x2_any{pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3])};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < cols) st1<bf16_t>(d + e, g.accumulate ? ld1<bf16_t>(d + e) + x[e] : x[e]);
  }
}
DEVI void place4(int q, int tid, int mt, int nt, int &m, int &n) {  // rows and columns of accumulator q = 2 tx + ty
  const int lane = tid & 63, wave = tid >> 6, wx = wave & 1, wy = wave >> 1;
  m = mt * GB + wy * 32 + (q & 1) * 16 + (lane & 15);
  n = nt * GB + wx * 32 + (q >> 1) * 16 + (lane >> 4) * 4;
}

DEVI int product_of(const Group &a, int block) {
  int i = 0;
#pragma unroll
  for (int j = 1; j < MAXG; ++j) i += block >= a.first[j];
  return i;
}

DEVI void store_tile(const Group &a, int i, const GemmAcc &acc, int tid, int tile, int split, int mt, int nt) {
  const MambaGemm &g = a.g[i];
  float *part = a.ws[i] + ((int64_t)tile * g.nsplit + split) * (GB * GB);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (g.nsplit > 1) {
      *reinterpret_cast<f32x4 *>(part + q * 1024 + tid * 4) = acc.v[q >> 1][q & 1];
    } else {
      int m, n;
      place4(q, tid, mt, nt, m, n);
      store4(g, m, n, acc.v[q >> 1][q & 1]);
    }
  }
}

__global__ __launch_bounds__(256) void gemm_kernel(const Group a) {
  __shared__ GemmTiles sh;
  const int tid = threadIdx.x, i = product_of(a, blockIdx.x);
  const MambaGemm &g = a.g[i];
  const int ntn = (g.N + GB - 1) / GB, tiles = ntn * ((g.M + GB - 1) / GB);
  const int block = blockIdx.x - a.first[i], split = block / tiles, tile = block % tiles;
  const int mt = tile / ntn, nt = tile % ntn;
  const int steps = (g.K + GK - 1) / GK, per = (steps + g.nsplit - 1) / g.nsplit;
  const int j0 = min(split * per, steps), j1 = min(j0 + per, steps);
  GemmAcc acc;
  acc.zero();
  auto run = [&](auto x_tr, auto y_tr) {
    constexpr bool XTR = decltype(x_tr)::value, YTR = decltype(y_tr)::value;
    const Operand<XTR> X(g.B, g.b_ns, g.b_ks, nt * GB, g.N, g.K, tid);
    const Operand<YTR> Y(g.A, g.a_ms, g.a_ks, mt * GB, g.M, g.K, tid);
    run_tile<XTR, YTR>(acc, sh, X, Y, j0, j1, tid);
  };
  const bool btr = g.b_ks != 1, atr = g.a_ks != 1;
  if (btr && atr) run(std::true_type{}, std::true_type{});
  else if (btr) run(std::true_type{}, std::false_type{});
  else if (atr) run(std::false_type{}, std::true_type{});
  else run(std::false_type{}, std::false_type{});
  store_tile(a, i, acc, tid, tile, split, mt, nt);
}

// ---- operands whose 16-byte pieces lie on 16 bytes: asynchronous loads into a ring of LDS stages of 64 k, one barrier per
// stage and two matrix instructions per accumulator between barriers (the form above: 32 k and one), no registers for what is in
// flight and no vector work to put it away.  2000 x 768 x 1536: 18.8 -> 14.2 us; its two gradients in one launch: 37 -> 31.
// What bounds it is the tiles' own reading, 150 MB through the L2 at 13 TB/s for the 6 + 2 MB of the former: 4 or 5 stages (14.6,
// 15.2 us), the k of a stage dealt to two sets of waves (15.6) and tiles dealt to the XCDs in runs (14.1, but 46 us for the two
// gradients, whose products have different lengths) are no faster.
constexpr int SK = 64, STAGES = 3, OPBYTES = GB * SK * 2;  // an operand's stage: 64 rows x 64 k, 8 KB
struct __align__(256) GemmRing {
  uint16_t x[STAGES][GB * SK], y[STAGES][GB * SK];
};
// One operand: 64 pieces of 16 bytes per wave and instruction, two instructions per wave and stage.  Rows past the last one,
// and k past the end, read others of the tile's own again; zero() puts zeros in the place of the latter.
template <bool TR> struct Ring {
  const bf16_t *base;
  int64_t s;
  int rows, K, wave, lane;
  DEVI Ring(const void *p, int64_t rs, int64_t ks, int row0, int all_rows, int K_, int wave_, int lane_)
      : base(static_cast<const bf16_t *>(p) + (int64_t)row0 * rs), s(TR ? ks : rs), rows(min(all_rows - row0, GB)), K(K_), wave(wave_), lane(lane_) {}
  // line of the stage (a row of 64 k, or with TR a k of 64 rows) and the piece of it that this lane moves
  DEVI int line(int q) const { return (q * 4 + wave) * 8 + (lane >> 3); }
  // pieces are permuted within a line: by bits of the row for the 16-byte reads of 16 rows, in pairs by bits of the k for the
  // transposing reads of 8 k
  DEVI static int swz(int l) { return TR ? ((l >> 1 & 1) | (l >> 3 & 1) << 1) << 1 : l >> 1 & 7; }
  DEVI void request(uint32_t lds, int k0) const {
    const bf16_t *src = base + (TR ? (int64_t)k0 * s : (int64_t)k0);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int l = line(q), c8 = ((lane & 7) ^ swz(l)) * 8;
      const uint32_t off = TR ? (uint32_t)min(l, K - 1 - k0) * (uint32_t)s + min(c8, rows - 8)
                              : (uint32_t)min(l, rows - 1) * (uint32_t)s + min(c8, K - 8 - k0);
      load_async16(src, off * 2u, lds + (q * 4 + wave) * 1024);
    }
  }
  DEVI void zero(uint32_t lds, int k0) const {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int l = line(q), k = k0 + (TR ? l : ((lane & 7) ^ swz(l)) * 8);
      if (k >= K) *(__attribute__((address_space(3))) u32x4 *)(uintptr_t)(lds + (q * 4 + wave) * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
    }
  }
};

// rows r0 + i, k = 32 kk + 8 g .. + 7 of 64 rows of a stage
template <bool TR> DEVI bf16x8_t ring_frag(uint32_t lds, int r0, int kk, int i, int g) {
  if constexpr (TR) {
    typedef __attribute__((address_space(3))) i16x4_t *lds_tr;
    typedef short i16x8_t __attribute__((ext_vector_type(8)));
    const int k = kk * 32 + 8 * g + (i >> 2);
    const uint32_t at = lds + k * 128 + (((r0 >> 3) ^ Ring<TR>::swz(k)) * 16) + (i & 3) * 8;
    const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)at);
    const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)(at + 4 * 128));
    return __builtin_bit_cast(bf16x8_t, (i16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  } else {
    const int r = r0 + i;
    return *(__attribute__((address_space(3))) bf16x8_t *)(uintptr_t)(lds + r * 128 + (((kk * 4 + g) ^ Ring<TR>::swz(r)) * 16));
  }
}

template <bool XTR, bool YTR>
DEVI void run_ring(GemmAcc &acc, const GemmRing &sh, const Ring<XTR> &X, const Ring<YTR> &Y, int k0, int k1, int wave, int lane) {
  const int i = lane & 15, g = lane >> 4, wx = wave & 1, wy = wave >> 1, n = (k1 - k0 + SK - 1) / SK;
  const uint32_t xs = lds_address(&sh.x[0][0]), ys = lds_address(&sh.y[0][0]);
  auto request = [&](int j) {
    X.request(xs + j % STAGES * OPBYTES, k0 + j * SK);
    Y.request(ys + j % STAGES * OPBYTES, k0 + j * SK);
  };
#pragma unroll
  for (int j = 0; j < STAGES - 1; ++j)
    if (j < n) request(j);
#pragma unroll 1
  for (int j = 0; j < n; ++j) {
    const uint32_t x = xs + j % STAGES * OPBYTES, y = ys + j % STAGES * OPBYTES;
    // four loads per wave and stage, in order
    if (j + STAGES - 2 < n) async_done<(STAGES - 2) * 4>();
    else async_done<0>();
    if (k0 + (j + 1) * SK > X.K) {
      X.zero(x, k0 + j * SK);
      Y.zero(y, k0 + j * SK);
    }
    lds_barrier();  // this stage is there, and the one before it has been read
    if (j + STAGES - 1 < n) request(j + STAGES - 1);
#pragma unroll
    for (int kk = 0; kk < SK / 32; ++kk) {
      bf16x8_t a[2], b[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        a[u] = ring_frag<XTR>(x, wx * 32 + u * 16, kk, i, g);
        b[u] = ring_frag<YTR>(y, wy * 32 + u * 16, kk, i, g);
      }
#pragma unroll
      for (int tx = 0; tx < 2; ++tx)
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) acc.v[tx][ty] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tx], b[ty], acc.v[tx][ty], 0, 0, 0);
    }
  }
}

__global__ __launch_bounds__(256) void gemm_ring_kernel(const Group a) {
  __shared__ GemmRing sh;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = product_of(a, blockIdx.x);
  const MambaGemm &g = a.g[i];
  const int ntn = (g.N + GB - 1) / GB, tiles = ntn * ((g.M + GB - 1) / GB);
  const int block = blockIdx.x - a.first[i], split = block / tiles, tile = block % tiles;
  const int mt = tile / ntn, nt = tile % ntn;
  const int steps = (g.K + GK - 1) / GK, per = (steps + g.nsplit - 1) / g.nsplit;
  const int k0 = min(split * per * GK, g.K), k1 = min(k0 + per * GK, g.K);
  GemmAcc acc;
  acc.zero();
  auto run = [&](auto x_tr, auto y_tr) {
    constexpr bool XTR = decltype(x_tr)::value, YTR = decltype(y_tr)::value;
    // (a split's k ends where the next one's begins)
    const Ring<XTR> X(g.B, g.b_ns, g.b_ks, nt * GB, g.N, k1, wave, lane);
    const Ring<YTR> Y(g.A, g.a_ms, g.a_ks, mt * GB, g.M, k1, wave, lane);
    run_ring<XTR, YTR>(acc, sh, X, Y, k0, k1, wave, lane);
  };
  const bool btr = g.b_ks != 1, atr = g.a_ks != 1;
  if (btr && atr) run(std::true_type{}, std::true_type{});
  else if (btr) run(std::true_type{}, std::false_type{});
  else if (atr) run(std::false_type{}, std::true_type{});
  else run(std::false_type{}, std::false_type{});
  store_tile(a, i, acc, tid, tile, split, mt, nt);
}

// ---- larger tiles for larger products: WX x WY waves of 16 FX x 16 FY each, operands in blocks of 64 rows, stages of WK k in a
// ring of LDS stages filled by asynchronous loads, one barrier a stage; a stage's fragments are read while the products of the one
// before it run.  What bounds them: up to 128 x 128 the reading through the L2 (2560 x 5120 x 32768: 13.4 GB, 11 TB/s), at 256 x 256
// the LDS (reading 96 KB and writing 32 KB per CU and stage is as long as its products), 1.0 - 1.2 PFLOP/s.
//   M x N x K                 us: library | 64 x 64 | 128 x 128 | 256 x 256 (with the splits that are chosen)
//   2560 x 5120 x 32768           965   |   -   | 1198 | 754        (200 tiles on 256 CUs: 832 without Share's helpers)
//   2560 x 5120 x 16384           513   |   -   |  605 | 384
//   192 x 5120 x 32768            234   |  156  |  121 - 138 | 124
//   768 x 1536 x 32768            183   |  218  |   89 |  90
//   1536 x 32768 x 48 (K short)    39   |   49  |   25 |  29
//   2560 x 32768 x 112, added      94   |  123  |   70 |  86
//   32768 x 2560 x 5120           650   |   -   | 1050 | 711        (left to the library)
// Tried: fragments read in front of their own products (256 x 256: 778 - 838 us where it is 712 - 773, 128 x 128 the same), four
// waves per SIMD of 64 x 64 (760 - 815), four stages (no change), two of 64 k at 128 x 128 (945, but 152 against 138 where K is
// short), 128 x 192 tiles (110 - 119 where 128 x 128 takes 121 - 135, for 192 rows alone), stages taken in another order by each
// workgroup against lines a power of two apart (no change).
constexpr int WK = 32, BLOCK = GB * WK * 2;  // a block's stage, 4 KB: four loads of a wave
template <int WX, int WY, int FX, int FY, int ST> struct WideTile {
  static constexpr int waves = WX * WY, stages = ST, rx = WX * FX * 16, ry = WY * FY * 16, bx = rx / GB, by = ry / GB;
  static constexpr int loads_x = 4 * bx / waves, loads_y = 4 * by / waves;  // of a wave and stage
  static constexpr int stage = (bx + by) * BLOCK;
  static_assert(rx % GB == 0 && ry % GB == 0 && loads_x * waves == 4 * bx && loads_y * waves == 4 * by, "whole loads per wave");
};
// An operand's blocks, one piece of 16 bytes per lane and load.  Lines: a row of WK k, or with TR a k of 64 rows.  Rows past the
// last one and k past the end are others of the operand's own again.
template <bool TR, int LOADS, int WAVES> struct WideRing {
  const bf16_t *base;
  int64_t s;
  int K, wave, lane;
  uint32_t off[LOADS];  // of its pieces in a whole stage, from base
  DEVI static int swz(int l) { return TR ? ((l >> 1 & 1) | (l >> 3 & 1) << 1) << 1 : l >> 2 & 3; }
  // load e of the stage: a quarter of block e / 4
  DEVI int line(int e) const { return TR ? (e & 3) * 8 + (lane >> 3) : (e & 3) * 16 + (lane >> 2); }
  DEVI int col(int e) const { return ((TR ? lane & 7 : lane & 3) ^ swz(line(e))) * 8; }
  DEVI WideRing(const void *p, int64_t rs, int64_t ks, int row0, int all_rows, int K_, int wave_, int lane_)
      : base(static_cast<const bf16_t *>(p) + (int64_t)row0 * rs), s(TR ? ks : rs), K(K_), wave(wave_), lane(lane_) {
    const int rows = all_rows - row0;
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
      const int e = q * WAVES + wave, r = (e >> 2) * GB;
      off[q] = 2u * (TR ? (uint32_t)line(e) * (uint32_t)s + min(r + col(e), rows - 8) : (uint32_t)min(r + line(e), rows - 1) * (uint32_t)s + col(e));
    }
  }
  DEVI void request(uint32_t lds, int k0) const {
    const bf16_t *src = base + (TR ? (int64_t)k0 * s : (int64_t)k0);
    const bool whole = k0 + WK <= K;
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
      const int e = q * WAVES + wave;
      const uint32_t back = whole ? 0u : TR ? (uint32_t)max(line(e) - (K - 1 - k0), 0) * (uint32_t)s * 2u : (uint32_t)max(col(e) - (K - 8 - k0), 0) * 2u;
      load_async16(src, off[q] - back, lds + e * 1024);
    }
  }
  DEVI void zero(uint32_t lds, int k0) const {
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
      const int e = q * WAVES + wave;
      if (k0 + (TR ? line(e) : col(e)) >= K) *(__attribute__((address_space(3))) u32x4 *)(uintptr_t)(lds + e * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
    }
  }
  // rows r0 + i, k = 8 g .. + 7
  DEVI static bf16x8_t frag(uint32_t lds, int r0, int i, int g) {
    if constexpr (TR) {
      typedef __attribute__((address_space(3))) i16x4_t *lds_tr;
      typedef short i16x8_t __attribute__((ext_vector_type(8)));
      const int k = 8 * g + (i >> 2);
      const uint32_t at = lds + (r0 >> 6) * BLOCK + k * 128 + (((r0 >> 3 & 7) ^ swz(k)) * 16) + (i & 3) * 8;
      const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)at);
      const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)(at + 4 * 128));
      return __builtin_bit_cast(bf16x8_t, (i16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      const int r = r0 + i;
      return *(__attribute__((address_space(3))) bf16x8_t *)(uintptr_t)(lds + r * (WK * 2) + ((g ^ swz(r)) * 16));
    }
  }
};

template <int FX, int FY> struct WideAcc {
  f32x4 v[FX][FY];
};
template <typename W, int FX, int FY, typename X_, typename Y_>
DEVI void run_wide(WideAcc<FX, FY> &acc, uint32_t sh, const X_ &X, const Y_ &Y, int k0, int k1, int wx, int wy, int lane) {
  const int i = lane & 15, g = lane >> 4, n = (k1 - k0 + WK - 1) / WK;
  constexpr int S = W::stages, LOADS = W::loads_x + W::loads_y;
  struct Frags {
    bf16x8_t a[FX], b[FY];
  } even, odd;
  auto request = [&](int slot, int j) {
    X.request(sh + slot * W::stage, k0 + j * WK);
    Y.request(sh + slot * W::stage + W::bx * BLOCK, k0 + j * WK);
  };
  auto zero = [&](int slot, int j) {
    if (k0 + (j + 1) * WK > X.K) {
      X.zero(sh + slot * W::stage, k0 + j * WK);
      Y.zero(sh + slot * W::stage + W::bx * BLOCK, k0 + j * WK);
    }
  };
  auto read = [&](Frags &f, int slot) {
    const uint32_t x = sh + slot * W::stage, y = x + W::bx * BLOCK;
#pragma unroll
    for (int u = 0; u < FX; ++u) f.a[u] = X.frag(x, wx * (FX * 16) + u * 16, i, g);
#pragma unroll
    for (int u = 0; u < FY; ++u) f.b[u] = Y.frag(y, wy * (FY * 16) + u * 16, i, g);
  };
#pragma unroll
  for (int j = 0; j < S; ++j)
    if (j < n) request(j, j);
  // the loads of a wave and stage, in order
  if (S <= n) async_done<(S - 1) * LOADS>();
  else async_done<0>();
  zero(0, 0);
  lds_barrier();
  read(even, 0);
  int slot = 0;
  // Stage j's fragments are in registers; those of stage j + 1 are read under its products
  auto step = [&](int j, const Frags &now, Frags &then) {
    const int next = slot + 1 == S ? 0 : slot + 1;
    if (j + S - 1 < n) async_done<(S - 2) * LOADS>();
    else async_done<0>();
    if (j + 1 < n) zero(next, j + 1);
    lds_barrier();  // stage j + 1 is there, and stage j has been read
    if (j + S < n) request(slot, j + S);
    read(then, next);  // (behind the last stage: what lies there, for nothing)
#pragma unroll
    for (int tx = 0; tx < FX; ++tx)
#pragma unroll
      for (int ty = 0; ty < FY; ++ty) acc.v[tx][ty] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now.a[tx], now.b[ty], acc.v[tx][ty], 0, 0, 0);
    // (a fragment's reads, then its share of the products)
#pragma unroll
    for (int q = 0; q < FX + FY; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x8, FX * FY / (FX + FY), 0);
    }
    slot = next;
  };
#pragma unroll 1
  for (int j = 0; j < n; j += 2) {
    step(j, even, odd);
    if (j + 1 < n) step(j + 1, odd, even);
  }
  lds_barrier();
}

// logical index of a workgroup of `count`, consecutive ones on one XCD
DEVI int xcd_run(int id, int count) {
  const int per = count / 8;
  return id < per * 8 ? id % 8 * per + id / 8 : id;
}
// row and first of four columns of accumulator q = FY tx + ty
template <int WX, int WY, int FX, int FY> DEVI void wide_place4(int q, int tid, int mt, int nt, int &m, int &n) {
  const int lane = tid & 63, wave = tid >> 6, wx = wave % WX, wy = wave / WX;
  m = (mt * WY + wy) * (FY * 16) + (q % FY) * 16 + (lane & 15);
  n = (nt * WX + wx) * (FX * 16) + (q / FY) * 16 + (lane >> 4) * 4;
}

// How the stages of a product's tiles are shared out where the tiles, their sums whole, leave `helpers` CUs idle: a tile's own
// workgroup takes its first `own` stages, so that all end together, and the helpers the rest of the tiles, `rest` stages each laid
// end to end, `span` stages per helper.  (Own workgroups walk k side by side, which keeps what neighbouring tiles share in the
// L2.)  2560 x 5120 x 32768, 200 tiles on 256 CUs: 832 -> 754 us (1.14 PFLOP/s).
struct Share {
  int tiles, own, rest, helpers, span;
  __host__ __device__ Share(int tiles_, int helpers_, int K) : tiles(tiles_), helpers(helpers_) {
    const int stages = (K + WK - 1) / WK;
    own = helpers ? (int)(((int64_t)stages * tiles + tiles + helpers - 1) / (tiles + helpers)) : stages;
    rest = stages - own;
    span = helpers ? (int)(((int64_t)tiles * rest + helpers - 1) / helpers) : 0;
  }
  // what helper h takes of tile u: stages [from, to), none where from >= to
  DEVI void part(int h, int u, int &from, int &to) const {
    from = own + max(h * span - u * rest, 0);
    to = own + min((h + 1) * span - u * rest, rest);
  }
  // places of the parts: the own ones', then the helpers', whose h and u both only grow from one part to the next
  DEVI int place(int h, int u) const { return tiles + h + u; }
  __host__ __device__ int64_t places() const { return 2 * (int64_t)tiles + helpers - 1; }
};

template <int WX, int WY, int FX, int FY, int ST, bool HELP>
__global__ __launch_bounds__(64 * WX * WY, WX * WY == 4 ? 3 : 2) void gemm_wide_kernel(const Group a) {
  typedef WideTile<WX, WY, FX, FY, ST> W;
  __shared__ __align__(256) char sh[ST * W::stage];
  int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = product_of(a, blockIdx.x), wx = wave % WX, wy = wave / WX;
  const MambaGemm &g = a.g[i];
  const int ntn = (g.N + W::rx - 1) / W::rx, ntm = (g.M + W::ry - 1) / W::ry, tiles = ntn * ntm;
  // consecutive tiles of the shorter side, which share the longer side's operand, on one XCD
  const int block = xcd_run(blockIdx.x - a.first[i], HELP ? tiles + a.helpers[i] : tiles * g.nsplit);
  WideAcc<FX, FY> acc;
  const uint32_t at = lds_address(sh);
  auto leave = [&](int64_t place) {  // for the kernel that adds the parts up
    float *part = a.ws[i] + place * (W::rx * W::ry);
#pragma unroll
    for (int q = 0; q < FX * FY; ++q) *reinterpret_cast<f32x4 *>(part + (q * W::waves * 64 + tid) * 4) = acc.v[q / FY][q % FY];
  };
  auto tile_at = [&](int tile, int &mt, int &nt) {
    mt = ntm < ntn ? tile % ntm : tile / ntn, nt = ntm < ntn ? tile / ntm : tile % ntn;
  };
  auto run = [&](auto x_tr, auto y_tr) {
    constexpr bool XTR = decltype(x_tr)::value, YTR = decltype(y_tr)::value;
    auto product = [&](int from, int to, int mt, int nt) {
      const int k0 = from * WK, k1 = min(to * WK, g.K);
#pragma unroll
      for (int q = 0; q < FX * FY; ++q) acc.v[q / FY][q % FY] = f32x4{0.f, 0.f, 0.f, 0.f};
      // (a part's k ends where the next one's begins)
      const WideRing<XTR, W::loads_x, W::waves> X(g.B, g.b_ns, g.b_ks, nt * W::rx, g.N, k1, wave, lane);
      const WideRing<YTR, W::loads_y, W::waves> Y(g.A, g.a_ms, g.a_ks, mt * W::ry, g.M, k1, wave, lane);
      run_wide<W>(acc, at, X, Y, k0, k1, wx, wy, lane);
    };
    int mt, nt;
    if constexpr (HELP) {
      const Share share(tiles, a.helpers[i], g.K);
      const bool helper = block >= tiles;
      const int h = block - tiles, u0 = helper ? h * share.span / share.rest : block, u1 = helper ? ((h + 1) * share.span - 1) / share.rest : block;
#pragma unroll 1
      for (int u = u0; u <= min(u1, tiles - 1); ++u) {
        int from = 0, to = share.own;
        if (helper) share.part(h, u, from, to);
        // (a new value to the compiler: what derives from it is formed where it is used instead of being carried along)
        asm volatile("" : "+v"(tid));
        lane = tid & 63;
        tile_at(u, mt, nt);
        product(from, to, mt, nt);
        leave(helper ? share.place(h, u) : u);
      }
    } else {
      const int stages = (g.K + WK - 1) / WK, per = (stages + g.nsplit - 1) / g.nsplit, from = block / tiles * per;
      tile_at(block % tiles, mt, nt);
      product(from, min(from + per, stages), mt, nt);
    }
  };
  const bool btr = g.b_ks != 1, atr = g.a_ks != 1;
  if (btr && atr) run(std::true_type{}, std::true_type{});
  else if (btr) run(std::true_type{}, std::false_type{});
  else if (atr) run(std::false_type{}, std::true_type{});
  else run(std::false_type{}, std::false_type{});
  if constexpr (HELP) return;
  if (g.nsplit > 1) {
    leave(block);
    return;
  }
  int mt, nt;
  tile_at(block, mt, nt);
  // whole rows of 16-byte pieces where D allows, 16 rows at a time through a patch of the wave's own
  const bool rows = g.d_dtype == MAMBA_BF16 && ((uintptr_t)g.D & 15) == 0 && g.ldd % 8 == 0 && g.N % 8 == 0;
  if (!rows) {
#pragma unroll
    for (int q = 0; q < FX * FY; ++q) {
      int m, n;
      wide_place4<WX, WY, FX, FY>(q, tid, mt, nt, m, n);
      store4(g, m, n, acc.v[q / FY][q % FY]);
    }
    return;
  }
  lds_barrier();
  constexpr int COLS = FX * 16, PITCH = COLS * 2 + 16, PIECES = COLS / 8, PER = (16 * PIECES + 63) / 64;
  static_assert(ST * W::stage >= W::waves * 16 * PITCH, "the patches lie where the stages lay");
  const uint32_t patch = at + wave * (16 * PITCH);
  const int n0 = (nt * WX + wx) * COLS, m0 = (mt * WY + wy) * (FY * 16);
  typedef __attribute__((address_space(3))) u32x4 *lds_u4;
  typedef __attribute__((address_space(3))) u32x2 *lds_u2;
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  f32x4 bias[FX];
#pragma unroll
  for (int tx = 0; tx < FX; ++tx) {
    bias[tx] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (g.bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) bias[tx][e] = ld1<bf16_t>(static_cast<const bf16_t *>(g.bias) + min(n0 + tx * 16 + (lane >> 4) * 4 + e, g.N - 1));
    }
  }
#pragma unroll
  for (int ty = 0; ty < FY; ++ty) {
    auto pieces = [&](auto f) {  // f(address in the patch, address in D)
#pragma unroll
      for (int q = 0; q < PER; ++q) {
        const int id = q * 64 + lane, r = id / PIECES, m = m0 + ty * 16 + r, n = n0 + id % PIECES * 8;
        if ((16 * PIECES % 64 == 0 || id < 16 * PIECES) && m < g.M && n < g.N)
          f((lds_u4)(uintptr_t)(patch + r * PITCH + id % PIECES * 16), reinterpret_cast<u32x4 *>(static_cast<bf16_t *>(g.D) + (int64_t)m * g.ldd + n));
      }
    };
    if (g.accumulate) {
      pieces([](lds_u4 at, const u32x4 *d) { *at = *d; });
      wave_sync();
    }
#pragma unroll
    for (int tx = 0; tx < FX; ++tx) {
      const lds_u2 at2 = (lds_u2)(uintptr_t)(patch + (lane & 15) * PITCH + (tx * 16 + (lane >> 4) * 4) * 2);
      f32x4 v = acc.v[tx][ty] + bias[tx];
      if (g.accumulate) {
        const u32x2 old = *at2;
        v += f32x4{bf16_lo(old.x), bf16_hi(old.x), bf16_lo(old.y), bf16_hi(old.y)};
      }
      *at2 = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    }
    wave_sync();
    pieces([](lds_u4 at, u32x4 *d) { *d = *at; });
    wave_sync();
  }
}

// the sum of the splits' tiles; an accumulator of every thread per workgroup
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const Group a) {
  const int tid = threadIdx.x, i = product_of(a, blockIdx.x);
  const MambaGemm &g = a.g[i];
  const int ntn = (g.N + GB - 1) / GB, block = blockIdx.x - a.first[i], tile = block >> 2, q = block & 3;
  int m, n;
  place4(q, tid, tile / ntn, tile % ntn, m, n);
  const float *part = a.ws[i] + (int64_t)tile * g.nsplit * (GB * GB) + q * 1024 + tid * 4;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < g.nsplit; ++s) v += *reinterpret_cast<const f32x4 *>(part + (int64_t)s * (GB * GB));
  store4(g, m, n, v);
}
template <int WX, int WY, int FX, int FY> __global__ __launch_bounds__(64 * WX * WY) void gemm_wide_reduce_kernel(const Group a) {
  typedef WideTile<WX, WY, FX, FY, 1> W;
  constexpr int QN = FX * FY;
  const int tid = threadIdx.x, i = product_of(a, blockIdx.x);
  const MambaGemm &g = a.g[i];
  const int ntn = (g.N + W::rx - 1) / W::rx, ntm = (g.M + W::ry - 1) / W::ry, tiles = ntn * ntm;
  const int block = blockIdx.x - a.first[i], tile = block / QN, q = block % QN;
  int m, n;
  wide_place4<WX, WY, FX, FY>(q, tid, ntm < ntn ? tile % ntm : tile / ntn, ntm < ntn ? tile / ntm : tile % ntn, m, n);
  const float *part = a.ws[i] + (q * W::waves * 64 + tid) * 4;
  auto at = [&](int64_t place) { return *reinterpret_cast<const f32x4 *>(part + place * (W::rx * W::ry)); };
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < g.nsplit; ++s) v += at(s * tiles + tile);
  if (a.helpers[i]) {
    const Share share(tiles, a.helpers[i], g.K);
    for (int h = tile * share.rest / share.span; h * share.span < (tile + 1) * share.rest; ++h) v += at(share.place(h, tile));
  }
  store4(g, m, n, v);
}

struct CastJobs {
  MambaCast c[MAXG];
  int64_t first[MAXG + 1];  // in groups of 8 elements
};
__global__ __launch_bounds__(256) void cast_bf16_kernel(const CastJobs a) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= a.first[MAXG]) return;
  int i = 0;
#pragma unroll
  for (int j = 1; j < MAXG; ++j) i += t >= a.first[j];
  const int64_t e0 = (t - a.first[i]) * 8;
  const float *src = a.c[i].src + e0;
  bf16_t *dst = static_cast<bf16_t *>(a.c[i].dst) + e0;
  const int n = (int)min((int64_t)8, a.c[i].n - e0);
  if (n == 8) {
    float v[8];
    ld8_any<float>(src, v);
    st8_any<bf16_t>(dst, v);
  } else {
    for (int e = 0; e < n; ++e) st1<bf16_t>(dst + e, src[e]);
  }
}

bool valid(const MambaGemm &g) {
  return g.A && g.B && g.D && g.M > 0 && g.N > 0 && g.K > 0 && (g.a_ks == 1 || g.a_ms == 1) && (g.b_ks == 1 || g.b_ns == 1) &&
         (g.d_dtype == MAMBA_BF16 || g.d_dtype == MAMBA_F32) && (g.nsplit >= 1 || g.nsplit == MAMBA_GEMM_SHARED) &&
         (int64_t)((g.M + GB - 1) / GB) * ((g.N + GB - 1) / GB) <= INT32_MAX / 1024;
}

// gemm_ring_kernel takes the operand with `rows` rows: 16-byte pieces on 16 bytes, offsets in a tile within 32 bits.  (At least 8
// of what is contiguous, and a multiple: no piece reaches past it.)
bool pieces(const void *p, int64_t row_stride, int64_t k_stride, int rows, int K) {
  const bool tr = k_stride != 1;
  return aligned(p, 16) && (tr ? k_stride : row_stride) % 8 == 0 && near_rows(tr ? k_stride : row_stride) && (tr ? rows : K) % 8 == 0;
}
bool ring(const MambaGemm &g) { return pieces(g.A, g.a_ms, g.a_ks, g.M, g.K) && pieces(g.B, g.b_ns, g.b_ks, g.N, g.K); }

enum { TILE64, TILE128, TILE256, FORMS };
constexpr int TILE[FORMS] = {GB, 128, 256};
int64_t tiles_of(const MambaGemm &g, int f) { return (int64_t)((g.M + TILE[f] - 1) / TILE[f]) * ((g.N + TILE[f] - 1) / TILE[f]); }
// 256 x 256 tiles where there are enough to be cut into few parts, 128 x 128 for what is left of 8 GFLOP and more and where they fill
// the chip uncut (2560 x 4096 x 80: 11 us against 17 at 64 x 64, 1536 x 2000 x 48 with 192 tiles 9.0 against 9.0).  Cut into parts, a
// smaller product is the faster one in 64 x 64 (768 x 1536 x 2000: 20 against 24 - 28).
int form_of(const MambaGemm &g) {
  if (!ring(g)) return TILE64;
  const double flop = 2.0 * g.M * g.N * g.K;
  if (flop > 16e9 && tiles_of(g, TILE256) >= 48) return TILE256;
  return flop > 8e9 || tiles_of(g, TILE128) >= cu_count() ? TILE128 : TILE64;
}
// The form of a product among those of one call: up to 8 GFLOP it stays in 64 x 64 tiles where another product of the call is in
// them, for launches of two forms run one after the other and each with an end of its own (the two gradients of a 768 x 1536
// projection over 3136 rows, the one 128 x 128 uncut and the other cut: 19 + 30 us, in one launch of 64 x 64 43).
int form_in(const MambaGemm *g, int i, int count) {
  const int f = form_of(g[i]);
  if (f != TILE128 || 2.0 * g[i].M * g[i].N * g[i].K > 8e9) return f;
  for (int k = 0; k < count; ++k)
    if (ring(g[k]) && form_of(g[k]) == TILE64) return TILE64;
  return f;
}
// Parts of the sum over k.  64 x 64: as many as give every CU two workgroups, of at least 8 steps (256 elements) each.  The others: the
// least of a stage's time by the workgroups on a CU, measured at 18 to 800 tiles in up to 32 parts, and what the parts' writing,
// reading and second launch take.  Helpers walk k apart from the tiles' own workgroups and from each other, which costs all of
// them a share of the L2: nothing at 56 helpers for 200 tiles, a fifth of a stage where they are as many as the tiles.  us, helped |
// two parts | three, cold operands: 1408 x 2816 x 16384 (66 tiles) 178 | 220 | 165; 1536 x 3072 x 16384 (72) 201 | 225 | 170, x 32768
// 363 | 427 | 322; 1664 x 3328 x 12288 (91) 161 | 177; 1792 x 3584 x 16384 (98) 253 | 232; 1920 x 3840 x 32768 (120) 535 | 486; 2304 x 4608
// x 32768 (162) 638, whole 823.  Cutting has to promise 1.5 % more than help.
double us_of(int64_t tiles, int splits, int helpers, int K, int f) {
  const int64_t units = tiles * splits, cus = cu_count(), stages = (K + WK - 1) / WK;
  const double crowd = std::min(1.0, (double)helpers / (double)tiles);
  const double stage = f == TILE256 ? 0.82 * (1 + 0.22 * crowd * crowd) : units <= cus ? 0.37 : units <= 2 * cus ? 0.41 : 0.62;
  const int64_t parts = (splits > 1 || helpers ? units : 0) + (helpers ? units + helpers : 0);
  return (helpers ? Share((int)tiles, helpers, K).own : (stages + splits - 1) / splits) * stage + (parts ? 6 + parts * TILE[f] * TILE[f] * 2e-6 : 0);
}
// CUs that 256 x 256 tiles with whole sums leave idle; 0 where there is nothing that they could take
int idle_of(int64_t tiles, int K, int f) {
  const int64_t idle = cu_count() - tiles;
  if (f != TILE256 || idle <= 0) return 0;
  const Share share((int)tiles, (int)idle, K);
  return share.rest && tiles * share.rest < 1 << 30 ? (int)idle : 0;
}
// ... and that are worth their parts.  (With the sums cut as well they never are, by these estimates at 48 to 255 tiles.)
int helpers_of(int64_t tiles, int K, int f) {
  const int idle = idle_of(tiles, K, f);
  return idle && us_of(tiles, 1, idle, K, f) < 0.97 * us_of(tiles, 1, 0, K, f) ? idle : 0;
}
int splits_of(const MambaGemm &g, int f) {
  const int64_t tiles = tiles_of(g, f), steps = (g.K + GK - 1) / GK, cus = cu_count();
  if (f == TILE64) return (int)std::max<int64_t>(1, std::min<int64_t>(2 * cus / tiles, steps / 8));
  int best = 1;
  double least = 1e30;
  const int64_t most = std::min<int64_t>((f == TILE256 ? 1 : 3) * cus / tiles, steps / 8);
  const int helped = helpers_of(tiles, g.K, f);
  for (int s = 1; s == 1 || s <= most; ++s) {
    const double us = us_of(tiles, s, s == 1 ? helped : 0, g.K, f);
    if (us < (best == 1 && helped ? 0.985 : 1.0) * least) least = us, best = s;
  }
  return best;
}
int planned_helpers(const MambaGemm &g, int f) { return g.nsplit == MAMBA_GEMM_SHARED ? idle_of(tiles_of(g, f), g.K, f) : 0; }
// fp32 elements of the parts' places
int64_t parts_of(const MambaGemm &g, int f) {
  const int64_t tiles = tiles_of(g, f);
  const int helpers = planned_helpers(g, f);
  if (g.nsplit == 1) return 0;
  return (helpers ? Share((int)tiles, helpers, g.K).places() : tiles * g.nsplit) * TILE[f] * TILE[f];
}

template <int WX, int WY, int FX, int FY, int ST, bool HELP> void launch_wide(const Group &a, int blocks, const Group &r, int rtiles, hipStream_t s) {
  hipLaunchKernelGGL((gemm_wide_kernel<WX, WY, FX, FY, ST, HELP>), dim3(blocks), dim3(64 * WX * WY), 0, s, a);
  if (rtiles) hipLaunchKernelGGL((gemm_wide_reduce_kernel<WX, WY, FX, FY>), dim3(rtiles * FX * FY), dim3(64 * WX * WY), 0, s, r);
}

}  // namespace

// Where the library takes over.  Up to 8 GFLOP its host time and choice of tiles cost more than any of these forms (whole mixer
// calls, forward + backward, library / own: products up to 0.5 GFLOP 350 / 180 us, up to 5 GFLOP 432 / 398).  Beyond:
// - sums over a long k into few tiles, which the library does not split, at three times the larger side and more: 1024 x 2048 x 16384 107 -
//   144 / 90 - 97, 2304 x 4608 x 16384 463 - 482 / 328 - 337, 2560 x 5120 x 32768 970 / 755; not always (2432 x 4864 x 16384 326 - 352 / 389 - 402).  Up to
//   16 GFLOP (270 products of 20 - 30 us) at twice the larger side: weight gradients take 0.4 - 0.8 of its time (calls of 4 x 1000 x
//   1792 409 / 394, 8 x 1000 x 1280 519 / 500), a projection to half the width 27 / 33, and where k is below the larger side the
//   two are within 10 % by themselves and a whole call is no faster with own products (1 x 1536 x 2560: 277 / 286).
// - where both operands lie along k the library is the better one at that: 1024 x 1024 x 4096 18 / 26, 1280 x 1280 x 4096 23 / 29, 2048 x 2048 x
//   6200 66 / 81, 3072 x 1536 x 16384 160 / 235.  It splits badly there from k 20000 or 48 times the shorter side on: 1024 x 4096 x
//   24576 280 / 210, 2048 x 2048 x 32768 377 / 319; 128 x 4096 x 12288 68 / 44, 126 x 3008 x 23808 117 / 51.
// - short k with up to 80 million results.  By whole mixer calls, forward + backward: 2304 channels x 32768 positions (75 million) 2950 /
//   2865, 4864 x 16384 3734 / 3582, 3584 x 12288 1976 / 1926, 2560 x 28672 2844 / 2812, though 4096 x 16384 2559 / 2578; with more of them 5120 x
//   16384 (84 million) 3620 / 3651, 3072 x 28672 3347 / 3376, 4480 x 20480 3903 / 3922, 2560 x 32768 3190 / 3186.
extern "C" int mamba_gemm_suits(const MambaGemm *g) {
  if (!g) return 0;
  const double flop = 2.0 * g->M * g->N * g->K;
  if (flop <= 8e9) return 1;
  if (!ring(*g)) return 0;
  const int64_t K = g->K, longer = std::max(g->M, g->N), shorter = std::min(g->M, g->N);
  if (g->a_ks != 1 || g->b_ks != 1 || K >= 20000 || K >= 48 * shorter) {
    if (flop <= 16e9 && K > 2 * longer) return 1;
    if (K >= 3 * longer && tiles_of(*g, TILE256) < cu_count()) return 1;
  }
  return K <= 256 && (int64_t)g->M * g->N <= 80000000;
}

extern "C" int64_t mamba_gemm_plan(MambaGemm *g, int count) {
  if (!g || count < 1 || count > MAXG) return MAMBA_E_BADARG;
  int64_t floats = 0;
  for (int i = 0; i < count; ++i) {
    g[i].nsplit = 1;
    if (!valid(g[i])) return MAMBA_E_BADARG;
    const int f = form_in(g, i, count);
    const int64_t steps = (g[i].K + GK - 1) / GK, want = splits_of(g[i], f);
    if (want > 1) {
      const int64_t per = (steps + want - 1) / want;
      g[i].nsplit = (int32_t)((steps + per - 1) / per);
    } else if (helpers_of(tiles_of(g[i], f), g[i].K, f)) {
      g[i].nsplit = MAMBA_GEMM_SHARED;
    }
    floats += parts_of(g[i], f);
  }
  return floats;
}

extern "C" int mamba_gemm(const MambaGemm *g, int count, float *ws, mamba_stream_t stream) {
  if (!g || count < 1 || count > MAXG) return MAMBA_E_BADARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  for (int i = 0; i < count; ++i) {
    if (!valid(g[i]) || (g[i].nsplit != 1 && !ws)) return MAMBA_E_BADARG;
    if (g[i].nsplit == MAMBA_GEMM_SHARED && !planned_helpers(g[i], form_in(g, i, count))) return MAMBA_E_BADARG;
  }
  // the products of one form in a launch, those with helpers (every workgroup leaves parts) apart from the others
  for (int form = FORMS; form >= 0; --form) {
    const int f = std::min(form, FORMS - 1);
    const bool helped = form == FORMS;
    Group a{}, r{};
    int blocks = 0, rtiles = 0, n = 0, nr = 0;
    bool all = true;
    const int per_tile = TILE[f] * TILE[f] / (f == TILE256 ? 2048 : 1024);  // workgroups that add up its splits
    for (int i = 0; i < count; ++i) {
      if (form_in(g, i, count) != f) continue;
      const int64_t tiles = tiles_of(g[i], f);
      const int helpers = planned_helpers(g[i], f);
      if ((helpers > 0) != helped) continue;
      MambaGemm p = g[i];
      p.nsplit = std::max(1, p.nsplit);
      a.g[n] = p, a.first[n] = blocks, a.helpers[n] = helpers, a.ws[n] = ws;
      blocks += (int)(tiles * p.nsplit) + helpers;
      all = all && ring(g[i]);
      if (const int64_t parts = parts_of(g[i], f)) {
        r.g[nr] = p, r.first[nr] = rtiles * per_tile, r.helpers[nr] = helpers, r.ws[nr] = ws;
        rtiles += (int)tiles;
        ws += parts;
        ++nr;
      }
      ++n;
    }
    if (!n) continue;
    for (int i = n; i <= MAXG; ++i) a.first[i] = INT32_MAX;
    for (int i = nr; i <= MAXG; ++i) r.first[i] = INT32_MAX;
    switch (f) {
      case TILE128: launch_wide<2, 2, 4, 4, 3, false>(a, blocks, r, rtiles, s); break;
      case TILE256:
        if (helped) launch_wide<2, 4, 8, 4, 3, true>(a, blocks, r, rtiles, s);
        else launch_wide<2, 4, 8, 4, 3, false>(a, blocks, r, rtiles, s);
        break;
      default:
        if (all) hipLaunchKernelGGL(gemm_ring_kernel, dim3(blocks), dim3(256), 0, s, a);
        else hipLaunchKernelGGL(gemm_kernel, dim3(blocks), dim3(256), 0, s, a);
        if (nr) hipLaunchKernelGGL(gemm_reduce_kernel, dim3(rtiles * 4), dim3(256), 0, s, r);
    }
    if (hipGetLastError() != hipSuccess) return MAMBA_E_LAUNCH;
  }
  return MAMBA_OK;
}

extern "C" int mamba_cast_bf16(const MambaCast *c, int count, mamba_stream_t stream) {
  if (!c || count < 1 || count > MAXG) return MAMBA_E_BADARG;
  CastJobs a{};
  int64_t groups = 0;
  for (int i = 0; i < count; ++i) {
    if (!c[i].src || !c[i].dst || c[i].n <= 0) return MAMBA_E_BADARG;
    a.c[i] = c[i], a.first[i] = groups;
    groups += (c[i].n + 7) / 8;
  }
  for (int i = count; i <= MAXG; ++i) a.first[i] = groups;
  if ((groups + 255) / 256 > INT32_MAX) return MAMBA_E_UNSUPPORTED;
  hipLaunchKernelGGL(cast_bf16_kernel, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), a);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}
