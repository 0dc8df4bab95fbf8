// Small bf16 matrix products: the projections inside a mixer (x_proj, dt_proj, out_proj and their gradients) where the
// problem is short.  A library product costs ~18 us of host time whatever its size, more than the product itself up
// to a few GFLOP; these cost a launch (~2 us), up to MAXG independent products share one, and operands are taken as
// they lie (either index contiguous, any alignment of the element's size), results in bf16 or fp32.
//
// Tile 64 x 64 per workgroup of four waves, k in steps of 32 (the block core of the SSD kernels).  What bounds a short
// product is the latency of its loads, not the matrix cores: the operands of the next PF steps are in flight, the LDS
// tiles are double-buffered (one barrier a step), and a product whose tiles do not fill the chip is split along k, the
// splits' fp32 tiles added up by a second kernel in a fixed order.
#include "ssd_common.hpp"

namespace {

constexpr int MAXG = 4, PF = 4;
struct Group {
  MambaGemm g[MAXG];
  int first[MAXG + 1];  // first workgroup of every product
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
  // rows r0 + i, k = 32 kk + 8 g .. + 7
  DEVI bf16x8_t frag(uint32_t lds, int r0, int kk, int i, int g) const {
    if constexpr (TR) {
      typedef __attribute__((address_space(3))) i16x4_t *lds_tr;
      typedef short i16x8_t __attribute__((ext_vector_type(8)));
      const int k = kk * 32 + 8 * g + (i >> 2);
      const uint32_t at = lds + k * 128 + (((r0 >> 3) ^ swz(k)) * 16) + (i & 3) * 8;
      const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)at);
      const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr)(uintptr_t)(at + 4 * 128));
      return __builtin_bit_cast(bf16x8_t, (i16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      const int r = r0 + i;
      return *(__attribute__((address_space(3))) bf16x8_t *)(uintptr_t)(lds + r * 128 + (((kk * 4 + g) ^ swz(r)) * 16));
    }
  }
};

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
        a[u] = X.frag(x, wx * 32 + u * 16, kk, i, g);
        b[u] = Y.frag(y, wy * 32 + u * 16, kk, i, g);
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

// the sum of the splits' tiles; a quarter of a tile per workgroup
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

int64_t tiles_of(const MambaGemm &g) { return (int64_t)((g.M + GB - 1) / GB) * ((g.N + GB - 1) / GB); }
bool valid(const MambaGemm &g) {
  return g.A && g.B && g.D && g.M > 0 && g.N > 0 && g.K > 0 && (g.a_ks == 1 || g.a_ms == 1) && (g.b_ks == 1 || g.b_ns == 1) &&
         (g.d_dtype == MAMBA_BF16 || g.d_dtype == MAMBA_F32) && g.nsplit >= 1 && tiles_of(g) <= INT32_MAX / 1024;
}

// gemm_ring_kernel takes the operand with `rows` rows: 16-byte pieces on 16 bytes, offsets in a tile within 32 bits.  (At least 8
// of what is contiguous, and a multiple: no piece reaches past it.)
bool pieces(const void *p, int64_t row_stride, int64_t k_stride, int rows, int K) {
  const bool tr = k_stride != 1;
  return aligned(p, 16) && (tr ? k_stride : row_stride) % 8 == 0 && near_rows(tr ? k_stride : row_stride) && (tr ? rows : K) % 8 == 0;
}
bool ring(const MambaGemm &g) { return pieces(g.A, g.a_ms, g.a_ks, g.M, g.K) && pieces(g.B, g.b_ns, g.b_ks, g.N, g.K); }

}  // namespace

// Splits along k: as many as give every CU two workgroups, of at least 8 steps (256 elements) each.
extern "C" int64_t mamba_gemm_plan(MambaGemm *g, int count) {
  if (!g || count < 1 || count > MAXG) return MAMBA_E_BADARG;
  int64_t floats = 0;
  for (int i = 0; i < count; ++i) {
    g[i].nsplit = 1;
    if (!valid(g[i])) return MAMBA_E_BADARG;
    const int64_t tiles = tiles_of(g[i]), steps = (g[i].K + GK - 1) / GK;
    const int64_t want = std::min<int64_t>(2 * (int64_t)cu_count() / tiles, steps / 8);
    if (want > 1) {
      const int64_t per = (steps + want - 1) / want;
      g[i].nsplit = (int32_t)((steps + per - 1) / per);
    }
    if (g[i].nsplit > 1) floats += tiles * g[i].nsplit * GB * GB;
  }
  return floats;
}

extern "C" int mamba_gemm(const MambaGemm *g, int count, float *ws, mamba_stream_t stream) {
  if (!g || count < 1 || count > MAXG) return MAMBA_E_BADARG;
  Group a{}, r{};
  int blocks = 0, rblocks = 0, nr = 0;
  int64_t used = 0;
  for (int i = 0; i < count; ++i) {
    if (!valid(g[i])) return MAMBA_E_BADARG;
    if (g[i].nsplit > 1 && !ws) return MAMBA_E_BADARG;
    const int64_t tiles = tiles_of(g[i]);
    a.g[i] = g[i], a.first[i] = blocks, a.ws[i] = ws + used;
    blocks += (int)(tiles * g[i].nsplit);
    if (g[i].nsplit > 1) {
      r.g[nr] = g[i], r.first[nr] = rblocks, r.ws[nr] = ws + used;
      rblocks += (int)(4 * tiles);
      used += tiles * g[i].nsplit * GB * GB;
      ++nr;
    }
  }
  for (int i = count; i <= MAXG; ++i) a.first[i] = INT32_MAX;
  for (int i = nr; i <= MAXG; ++i) r.first[i] = INT32_MAX;
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool all = true;
  for (int i = 0; i < count; ++i) all = all && ring(g[i]);
  if (all) hipLaunchKernelGGL(gemm_ring_kernel, dim3(blocks), dim3(256), 0, s, a);
  else hipLaunchKernelGGL(gemm_kernel, dim3(blocks), dim3(256), 0, s, a);
  if (nr) hipLaunchKernelGGL(gemm_reduce_kernel, dim3(rblocks), dim3(256), 0, s, r);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
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
