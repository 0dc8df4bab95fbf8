// Pieces shared by the norm kernels (gated group norm, residual-add norm): sums over a team of
// threads, one row of channels held in registers in its packed form, the reduction of the per-part
// partial sums of dweight / dbias.
#pragma once
#include "common.hpp"

#include <type_traits>

namespace {

// Sums over the TEAM threads that share a (row, group): lanes of one wave by xor shuffles, waves of
// a workgroup through LDS.
template <int TEAM> struct TeamSum {
  static constexpr int NW = TEAM / 64;
  float *red;  // LDS: 2 slots x NW x 2 floats
  int slot = 0;
  DEVI explicit TeamSum(float *lds) : red(lds) {}
  DEVI void sum2(float &a, float &b) {
#pragma unroll
    for (int off = (TEAM < 64 ? TEAM : 64) / 2; off >= 1; off >>= 1) {
      a += __shfl_xor(a, off, 64);
      b += __shfl_xor(b, off, 64);
    }
    if constexpr (NW > 1) {
      const int wave = threadIdx.x >> 6;
      float *s = red + slot * NW * 2;
      if ((threadIdx.x & 63) == 0) {
        s[wave * 2] = a;
        s[wave * 2 + 1] = b;
      }
      __syncthreads();
      a = 0.f;
      b = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        a += s[w * 2];
        b += s[w * 2 + 1];
      }
      slot ^= 1;  // the next sum uses the other slot, so one barrier per sum is enough
    }
  }
};

// K steps of 8 channels of one row, as loaded (16 bytes per step when VEC): the next row is fetched
// into this form while the current one is worked on, at half the registers of its fp32 values.
struct F8 {
  float f[8];
};
template <typename T, bool VEC, int K, int TEAM> struct RowBuf {
  using Slot = std::conditional_t<VEC, Pack8<T>, F8>;
  Slot s[K];
  DEVI void fetch(const T *row, int col, int gs) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = col + k * TEAM * 8;
      const int nv = min(max(gs - c, 0), 8);
      if constexpr (VEC) {
        if (nv == 8) s[k].load(row + c);
        else s[k].zero();
      } else {
        ld8_guard<T, false>(row + c, nv, 0.f, s[k].f);
      }
    }
  }
  DEVI void get(float (&v)[K][8]) const {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if constexpr (VEC) s[k].unpack(v[k]);
      else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[k][e] = s[k].f[e];
      }
    }
  }
};

template <typename T, bool VEC, int K, int TEAM>
DEVI void load_row(const T *row, int col, int gs, float (&v)[K][8]) {
  RowBuf<T, VEC, K, TEAM> b;
  b.fetch(row, col, gs);
  b.get(v);
}
template <typename T, bool VEC, int K, int TEAM>
DEVI void store_row(T *row, int col, int gs, const float (&v)[K][8]) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = col + k * TEAM * 8;
    const int nv = min(max(gs - c, 0), 8);
    if (nv > 0) st8_guard<T, VEC>(row + c, nv, v[k]);
  }
}

// The norm's parameters of this thread's channels, zero past the end.  The kernels call it after they have requested
// their first row: the conversion waits for the loads, and that wait is then the row's as well.
template <int K, int TEAM>
DEVI void load_params(const void *base, int dtype, int64_t off, int col, int gs, float (&v)[K][8]) {
  auto run = [&](auto *src) {
    typedef std::remove_const_t<std::remove_pointer_t<decltype(src)>> W;
    Pack8<W> q[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = col + k * TEAM * 8;
      if (c + 8 <= gs) {
        q[k].load_any(src + off + c);
      } else {
        float t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = c + e < gs ? ld1<W>(src + off + c + e) : 0.f;
        q[k].pack(t);
      }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) q[k].unpack(v[k]);
  };
  switch (dtype) {
    case MAMBA_BF16: run(static_cast<const bf16_t *>(base)); break;
    case MAMBA_F16: run(static_cast<const f16_t *>(base)); break;
    default: run(static_cast<const float *>(base)); break;
  }
}

// Sums over a workgroup of blockDim.x threads (whole waves, at most 16), whatever their number: DPP adds inside a wave,
// the waves' totals through LDS in alternating slots (one barrier per sum), of which every row of 16 lanes reads one per
// lane and adds them up by rotations.  (A loop over the waves' totals made a row of 5120 channels wait for ten LDS reads
// one after the other.)
struct WideSum {
  float *red;  // LDS: 2 slots x 16 waves x 2 floats
  int slot = 0, nw;
  DEVI explicit WideSum(float *lds) : red(lds), nw(blockDim.x >> 6) {
    if (threadIdx.x < 64 && (int)(threadIdx.x & 31) >= 2 * nw) red[threadIdx.x] = 0.f;  // waves that are not there
  }
  DEVI void sum2(float &a, float &b) {
    a = wave_sum_to_last(a);
    b = wave_sum_to_last(b);
    if (nw == 1) {
      a = readlane_f(a, 63);
      b = readlane_f(b, 63);
      return;
    }
    float *s = red + slot * 32;
    if ((threadIdx.x & 63) == 63) *reinterpret_cast<f32x2 *>(s + (threadIdx.x >> 6) * 2) = f32x2{a, b};
    lds_barrier();
    const f32x2 v = *reinterpret_cast<const f32x2 *>(s + (threadIdx.x & 15) * 2);
    a = row_sum_all(v.x);
    b = row_sum_all(v.y);
    slot ^= 1;
  }
};

// threads of a workgroup that holds `channels` channels (a multiple of 8, at most 8192), 8 per thread
inline int wide_threads(int channels) { return (channels / 8 + 63) / 64 * 64; }
// workgroups of that many threads which a CU holds at once at `waves_per_simd` waves per SIMD
inline int wide_resident(int threads, int waves_per_simd) { return max(1, waves_per_simd * 4 / (threads / 64)); }

// Column sums of up to four (nparts, dim) workspaces, in the order of the parts, written in the parameters' dtype:
// blockIdx.y is the workspace, a workgroup takes 16 channels (64 bytes of every row) on 128 slices of the parts, four
// of a thread's rows in flight.  (64 channels x 16 slices of 1024 threads took 25 us for 1024 parts of 2560 channels:
// 40 workgroups, one row at a time per thread.)
struct ReduceJobs {
  const float *part[4];
  void *out[4];
};
template <bool VEC> __global__ __launch_bounds__(512) void norm_reduce_kernel(const ReduceJobs jobs, int dtype, int nparts, int dim) {
  constexpr int SLICES = 128;
  __shared__ f32x4 s[SLICES][4];
  const float *src = jobs.part[blockIdx.y];
  const int q = threadIdx.x & 3, sl = threadIdx.x >> 2;
  const int c = blockIdx.x * 16 + q * 4;
  auto row4 = [&](int part) -> f32x4 {
    const float *r = src + (int64_t)part * dim + c;
    if constexpr (VEC) {
      return c < dim ? *(const GLOBAL_AS f32x4 *)r : f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (c < dim) v.x = r[0];
      if (c + 1 < dim) v.y = r[1];
      if (c + 2 < dim) v.z = r[2];
      if (c + 3 < dim) v.w = r[3];
      return v;
    }
  };
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int part = sl;
  for (; part + 3 * SLICES < nparts; part += 4 * SLICES) {
    const f32x4 v0 = row4(part), v1 = row4(part + SLICES), v2 = row4(part + 2 * SLICES), v3 = row4(part + 3 * SLICES);
    acc += (v0 + v1) + (v2 + v3);
  }
  for (; part < nparts; part += SLICES) acc += row4(part);
  s[sl][q] = acc;
  __syncthreads();
#pragma unroll
  for (int half = SLICES / 2; half >= 1; half >>= 1) {
    if (sl < half) s[sl][q] += s[sl + half][q];
    __syncthreads();
  }
  if (threadIdx.x < 16 && blockIdx.x * 16 + threadIdx.x < dim)
    st_param(jobs.out[blockIdx.y], dtype, blockIdx.x * 16 + threadIdx.x, reinterpret_cast<const float *>(&s[0][0])[threadIdx.x]);
}

inline int launch_reduce(const ReduceJobs &jobs, int njobs, int dtype, int nparts, int dim, hipStream_t st) {
  bool vec = dim % 4 == 0;
  for (int i = 0; i < njobs; ++i) vec = vec && (reinterpret_cast<uintptr_t>(jobs.part[i]) & 15) == 0;
  const dim3 grid((dim + 15) / 16, njobs), block(512);
  if (vec) norm_reduce_kernel<true><<<grid, block, 0, st>>>(jobs, dtype, nparts, dim);
  else norm_reduce_kernel<false><<<grid, block, 0, st>>>(jobs, dtype, nparts, dim);
  return hipGetLastError() == hipSuccess ? MAMBA_OK : MAMBA_E_LAUNCH;
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
