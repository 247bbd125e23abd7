// Alpha statistics of a K / V block (gfx950, wave64).
//
// The alpha of a cache layer is chosen from two statistics of the block it
// quantizes first (muzero/quantizer.py:46-83): percentiles of a strided
// subsample of |x|, and the mean distance of the groups' zero anchors from
// one half.  As torch operations that is about 20 launches per kind (position
// arithmetic, a gather, the group min / max, five elementwise passes over the
// group arrays, a sort of the subsample).  Here:
//
//   block_stats_kernel   reads the block once and writes each group's
//       |clamp((0 - min) / max(max - min, 1e-8), 0, 1) - 0.5| in the flattened
//       rows' group order (fp32, each operation rounded as torch rounds it;
//       min / max propagate NaN), and gathers the subsample's |x|.  The mean
//       over the groups stays torch's, whose summation order fixes its value.
//       A lane holds one 16-byte vector: for keys of all 64 tokens of a group
//       (consecutive lanes take consecutive vectors of a token's row, the loads
//       of 8 or 16 tokens in flight), for values of one token, reduced over the
//       group's 8 or 16 lanes by DPP.  Bound: HBM, one read of the block.
//   select16_kernel / select_kernel   take the three order statistics from the
//       subsample, one workgroup per kind (both kinds in one launch).
//
// Measured at [16, 8, 1856, 128] fp16 (65536 values in the subsample), profiled
// one at a time: 15 us for the keys, 18 us for the values (61 MB each), 9 us for
// both selections; with the fp16 quantize chain the whole 8-bit prefill went from
// 686 to 191 us.  A selection by three 11-bit passes, as fp32 runs it, took 30 us
// for 16-bit values: 8 compares and branches per value and pass, on one compute
// unit.
#include "common.hpp"

#include <algorithm>

namespace mz {
namespace stats {

constexpr int WG = 256;

__device__ __forceinline__ float vmin(float a, float b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ float vmax(float a, float b) { return __builtin_elementwise_maximum(a, b); }

template <int DT>
struct Vec {
  static constexpr int N = DT == MZ_F32 ? 4 : 8;                // values per 16 bytes
  static constexpr int KEY_LOADS = DT == MZ_F16 ? 8 : 16;  // tokens in flight per lane (registers for 4 waves per SIMD)
};

template <int DT>
__device__ __forceinline__ void unpack(float (&x)[Vec<DT>::N], const uint4 u) {
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (DT == MZ_F32) {
      x[k] = __uint_as_float(w[k]);
    } else if constexpr (DT == MZ_BF16) {
      x[2 * k] = __uint_as_float(w[k] << 16);
      x[2 * k + 1] = __uint_as_float(w[k] & 0xFFFF0000u);
    } else {
      x[2 * k] = h2f((uint16_t)w[k]);
      x[2 * k + 1] = h2f((uint16_t)(w[k] >> 16));
    }
  }
}

// |clamp((0 - lo) / max(hi - lo, 1e-8), 0, 1) - 0.5| of a group (quantizer.py:53-55)
__device__ __forceinline__ float anchor_offset(float lo, float hi) {
  const float span = clamp_min(hi - lo, 1e-8f);
  const float za = clamp01((0.f - lo) / span);
  return __builtin_fabsf(za - 0.5f);
}

struct Args {
  const void* x;
  int B, H, T, D;
  int64_t sb, sh, st;
  float* offsets;   // [groups]
  void* sample;     // [n_sample], the block's type
  int64_t n_sample, step;
  int64_t items;    // vectors of the min / max walk
  unsigned stat_blocks;  // blocks of that walk; the others gather the subsample
};

// Element `pos` of the flattened rows: keys in order (b, h, group, channel,
// token), values in order (b, h, token, channel).
template <int DT, bool KEYS>
__device__ __forceinline__ void gather(const Args& a, int64_t i) {
  const int64_t pos = i * a.step;
  int64_t bh, t, c;
  if constexpr (KEYS) {
    const int64_t tt = pos & 63, r = pos >> 6, r2 = r / a.D;
    c = r - r2 * a.D;
    const int64_t nsg = a.T / 64;
    bh = r2 / nsg;
    t = (r2 - bh * nsg) * 64 + tt;
  } else {
    const int64_t r = pos / a.D;
    c = pos - r * a.D;
    bh = r / a.T;
    t = r - bh * a.T;
  }
  const int64_t b = bh / a.H, h = bh - b * a.H;
  const int64_t at = b * a.sb + h * a.sh + t * a.st + c;
  if constexpr (DT == MZ_F32) ((uint32_t*)a.sample)[i] = ((const uint32_t*)a.x)[at] & 0x7FFFFFFFu;
  else ((uint16_t*)a.sample)[i] = ((const uint16_t*)a.x)[at] & 0x7FFFu;
}

template <int DT, bool KEYS>
__global__ __launch_bounds__(WG, 4) void block_stats_kernel(const Args a) {
  constexpr int NE = Vec<DT>::N, KEY_LOADS = Vec<DT>::KEY_LOADS;
  if (blockIdx.x >= a.stat_blocks) {
    const int64_t stride = (int64_t)(gridDim.x - a.stat_blocks) * WG;
    for (int64_t i = (int64_t)(blockIdx.x - a.stat_blocks) * WG + threadIdx.x; i < a.n_sample; i += stride)
      gather<DT, KEYS>(a, i);
    return;
  }
  const int vpr = a.D / NE;  // vectors per token
  const int es = DT == MZ_F32 ? 4 : 2;
  const int64_t stride = (int64_t)a.stat_blocks * WG;
  // (values: a group's lanes share an item range of 64 / NE, so they leave the loop together)
  for (int64_t it = (int64_t)blockIdx.x * WG + threadIdx.x; it < a.items; it += stride) {
    if constexpr (KEYS) {
      const int64_t tile = it / vpr;
      const int v = (int)(it - tile * vpr);
      const int nsg = a.T / 64;
      const int64_t bh = tile / nsg, b = bh / a.H, h = bh - b * a.H;
      const char* p = (const char*)a.x + (b * a.sb + h * a.sh + (tile - bh * nsg) * 64 * a.st + (int64_t)v * NE) * es;
      float lo[NE], hi[NE];
#pragma unroll
      for (int t0 = 0; t0 < 64; t0 += KEY_LOADS) {
        uint4 u[KEY_LOADS];
#pragma unroll
        for (int k = 0; k < KEY_LOADS; ++k) u[k] = *(const uint4*)(p + (int64_t)(t0 + k) * a.st * es);
#pragma unroll
        for (int k = 0; k < KEY_LOADS; k += 2) {
          float x[NE], y[NE];
          unpack<DT>(x, u[k]);
          unpack<DT>(y, u[k + 1]);
#pragma unroll
          for (int e = 0; e < NE; ++e) {
            const float m = vmin(x[e], y[e]), M = vmax(x[e], y[e]);
            lo[e] = t0 + k == 0 ? m : vmin(lo[e], m);
            hi[e] = t0 + k == 0 ? M : vmax(hi[e], M);
          }
        }
      }
      float* o = a.offsets + tile * a.D + (int64_t)v * NE;
#pragma unroll
      for (int e = 0; e < NE; e += 4)
        *(float4*)(o + e) = make_float4(anchor_offset(lo[e], hi[e]), anchor_offset(lo[e + 1], hi[e + 1]),
                                        anchor_offset(lo[e + 2], hi[e + 2]), anchor_offset(lo[e + 3], hi[e + 3]));
    } else {
      const int64_t tok = it / vpr;
      const int v = (int)(it - tok * vpr);
      const int64_t bh = tok / a.T, b = bh / a.H, h = bh - b * a.H;
      const uint4 u = *(const uint4*)((const char*)a.x +
                                      (b * a.sb + h * a.sh + (tok - bh * a.T) * a.st + (int64_t)v * NE) * es);
      float x[NE];
      unpack<DT>(x, u);
      float lo = x[0], hi = x[0];
#pragma unroll
      for (int e = 1; e < NE; ++e) lo = vmin(lo, x[e]), hi = vmax(hi, x[e]);
      constexpr int L = 64 / NE;  // lanes of a group
      lo = group_reduce<L>(lo, vmin);
      hi = group_reduce<L>(hi, vmax);
      if ((threadIdx.x & (L - 1)) == 0) a.offsets[it / L] = anchor_offset(lo, hi);
    }
  }
}

// ---------------------------------------------------------------- selection
constexpr int SEL = 1024;      // threads of a workgroup

// 16-bit values: one histogram over all 2^15 patterns (132 KB of LDS, a word
// of padding per thread's 32 bins), then a scan of it.  The patterns order as
// the values do (non-negative; NaN last, as torch's sort puts it).
constexpr int BINS16 = 32768, PER16 = BINS16 / SEL;
constexpr int LDS16 = (BINS16 + SEL + SEL / 64) * 4;

template <int DT>
__global__ __launch_bounds__(SEL) void select16_kernel(const uint16_t* __restrict__ v, int64_t v_stride, int64_t n,
                                                       uint32_t k0, uint32_t k1, uint32_t k2, float* __restrict__ out,
                                                       int64_t out_stride) {
  extern __shared__ uint32_t lds16[];
  uint32_t* scan = lds16 + BINS16 + SEL;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint16_t* u = v + blockIdx.x * v_stride;
  for (int i = t; i < BINS16 + SEL; i += SEL) lds16[i] = 0;
  __syncthreads();
  auto count = [&](uint32_t p) __attribute__((always_inline)) {
    p &= 0x7FFFu;
    atomicAdd(&lds16[p + p / PER16], 1u);
  };
  constexpr int LOADS = 8;  // 8 x 8 values in flight
  for (int64_t base = 0; base < n; base += (int64_t)SEL * 8 * LOADS) {
    uint4 r[LOADS];
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int64_t i = base + 8 * ((int64_t)k * SEL + t);
      if (i + 8 <= n) r[k] = *(const uint4*)(u + i);
    }
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int64_t i = base + 8 * ((int64_t)k * SEL + t);
      if (i + 8 <= n) {
        const uint32_t w[4] = {r[k].x, r[k].y, r[k].z, r[k].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) count(w[q]), count(w[q] >> 16);
      } else {
        for (int64_t j = i; j < n; ++j) count(u[j]);
      }
    }
  }
  __syncthreads();
  uint32_t c[PER16], own = 0;
#pragma unroll
  for (int i = 0; i < PER16; ++i) own += c[i] = lds16[t * (PER16 + 1) + i];
  uint32_t upto = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t x = __shfl_up(upto, o, 64);
    if (lane >= o) upto += x;
  }
  if (lane == 63) scan[wave] = upto;
  __syncthreads();
  uint32_t before = upto - own;
  for (int w = 0; w < wave; ++w) before += scan[w];
  const uint32_t rank[3] = {k0, k1, k2};
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    if (rank[j] < before || rank[j] >= before + own) continue;  // one thread's bins hold the rank
    uint32_t bin = t * PER16, below = before;
#pragma unroll
    for (int i = 0; i < PER16 - 1; ++i) {
      below += c[i];
      if (rank[j] >= below) bin = t * PER16 + i + 1;
    }
    out[blockIdx.x * out_stride + j] = DT == MZ_BF16 ? bf2f((uint16_t)bin) : h2f((uint16_t)bin);
  }
}

// fp32 values: radix selection by 11 + 10 + 10 bits of the patterns; the first
// histogram, where N(0, 1) data meets in few bins, in 4 copies by lane, and a
// wave per order statistic walks the bins.
constexpr int COPIES = 4;
constexpr int BINS = 2048, PER1 = BINS / 64, PITCH1 = BINS + 64 + 8;  // (a copy's bin in another bank than the next copy's)
constexpr int BINS2 = 1024, PER2 = BINS2 / 64, PITCH2 = BINS2 + 64;

// Bins are kept PER to a lane of the wave that walks them, a word of padding
// after each lane's, so that its 64 lanes read different banks.
template <int PER>
__device__ __forceinline__ uint32_t bin_at(uint32_t bin) {
  return bin + bin / PER;
}

// One wave: the bin (of 64 * PER) that holds the element of rank `rank`
// (0-based), and its rank within the bin.
template <int PER>
__device__ __forceinline__ uint32_t find_bin(const uint32_t* hist, uint32_t& rank) {
  const int lane = threadIdx.x & 63;
  uint32_t c[PER], own = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) own += c[i] = hist[lane * (PER + 1) + i];
  uint32_t upto = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t v = __shfl_up(upto, o, 64);
    if (lane >= o) upto += v;
  }
  // the lane whose bins hold the rank finds its bin; the others take the answer
  const bool mine = rank >= upto - own && rank < upto;
  uint32_t left = rank - (upto - own), bin = lane * PER, below = 0;
#pragma unroll
  for (int i = 0; i < PER - 1; ++i) {
    below += c[i];
    if (left >= below) bin = lane * PER + i + 1;
  }
  below = 0;
#pragma unroll
  for (int i = 0; i < PER - 1; ++i)
    if (lane * PER + i < bin) below += c[i];
  left -= below;
  const int src = __ffsll((unsigned long long)__ballot(mine)) - 1;
  rank = __shfl(left, src, 64);
  return __shfl(bin, src, 64);
}

// f(pattern of v[i] without its sign) for every i this thread takes, 8 loads of
// 4 values in flight.
template <typename F>
__device__ __forceinline__ void for_each(const uint32_t* __restrict__ u, int64_t n, F f) {
  constexpr int LOADS = 8;
  for (int64_t base = 0; base < n; base += (int64_t)SEL * 4 * LOADS) {
    uint4 r[LOADS];
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int64_t i = base + 4 * ((int64_t)k * SEL + threadIdx.x);
      if (i + 4 <= n) r[k] = *(const uint4*)(u + i);
    }
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int64_t i = base + 4 * ((int64_t)k * SEL + threadIdx.x);
      if (i + 4 <= n) {
        f(r[k].x & 0x7FFFFFFFu), f(r[k].y & 0x7FFFFFFFu), f(r[k].z & 0x7FFFFFFFu), f(r[k].w & 0x7FFFFFFFu);
      } else {
        for (int64_t j = i; j < n; ++j) f(u[j] & 0x7FFFFFFFu);
      }
    }
  }
}

// Workgroup s: out[s * out_stride + j] = the element of rank k[j] (0-based, < n)
// of the n values at v + s * v_stride, in ascending order.
__global__ __launch_bounds__(SEL) void select_kernel(const uint32_t* __restrict__ v, int64_t v_stride, int64_t n,
                                                     uint32_t k0, uint32_t k1, uint32_t k2, float* __restrict__ out,
                                                     int64_t out_stride) {
  __shared__ uint32_t hist[COPIES * PITCH1];
  __shared__ uint32_t found[3];
  const int t = threadIdx.x, wave = t >> 6;
  const uint32_t* u = v + blockIdx.x * v_stride;
  uint32_t rank = wave == 0 ? k0 : wave == 1 ? k1 : k2;  // waves 0..2 follow one order statistic each
  uint32_t prefix[3] = {0, 0, 0};
  for (int i = t; i < COPIES * PITCH1; i += SEL) hist[i] = 0;
  __syncthreads();
  for_each(u, n, [&](uint32_t x) { atomicAdd(&hist[(t & (COPIES - 1)) * PITCH1 + bin_at<PER1>(x >> 20)], 1u); });
  __syncthreads();
  for (int i = t; i < BINS + 64; i += SEL) {
    uint32_t c = hist[i];
    for (int k = 1; k < COPIES; ++k) c += hist[k * PITCH1 + i];
    hist[i] = c;
  }
  __syncthreads();
  if (wave < 3) {
    const uint32_t bin = find_bin<PER1>(hist, rank);
    if ((t & 63) == 0) found[wave] = bin;
  }
  __syncthreads();
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int sh = pass == 0 ? 10 : 0;  // the pass's 10 bits; those above must equal the prefix
#pragma unroll
    for (int j = 0; j < 3; ++j) prefix[j] = pass == 0 ? found[j] : (prefix[j] << 10) | found[j];
    for (int i = t; i < 3 * PITCH2; i += SEL) hist[i] = 0;
    __syncthreads();
    for_each(u, n, [&](uint32_t x) {
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if ((x >> (sh + 10)) == prefix[j]) atomicAdd(&hist[j * PITCH2 + bin_at<PER2>((x >> sh) & (BINS2 - 1))], 1u);
    });
    __syncthreads();
    if (wave < 3) {
      const uint32_t bin = find_bin<PER2>(hist + PITCH2 * wave, rank);
      if ((t & 63) == 0) found[wave] = bin;
    }
    __syncthreads();
  }
  if (t < 3)
    out[blockIdx.x * out_stride + t] = __uint_as_float(((t == 0 ? prefix[0] : t == 1 ? prefix[1] : prefix[2]) << 10) | found[t]);
}

}  // namespace stats
}  // namespace mz

using namespace mz;

extern "C" int muzero_block_stats(const void* x, int x_dtype, int keys, int B, int H, int T, int D, int64_t x_sb,
                                  int64_t x_sh, int64_t x_st, float* offsets, void* sample, int64_t n_sample,
                                  int64_t sample_step, mz_stream_t stream) {
  if (x_dtype != MZ_F32 && x_dtype != MZ_BF16 && x_dtype != MZ_F16) return MZ_EINVAL;
  if (B < 1 || H < 1 || T < 1 || D < 1 || !x || !offsets || !sample || n_sample < 0 || sample_step < 1) return MZ_EINVAL;
  const int64_t es = x_dtype == MZ_F32 ? 4 : 2, total = (int64_t)B * H * T * D;
  if (keys ? T % 64 : D % 64) return MZ_EINVAL;
  if (n_sample > 0 && (n_sample - 1) * sample_step >= total) return MZ_EINVAL;
  // 16-byte vectors; a key tile's vectors write 16-byte runs of offsets
  if (((uintptr_t)x | (uintptr_t)(x_sb * es) | (uintptr_t)(x_sh * es) | (uintptr_t)(x_st * es) | (uintptr_t)(D * es) |
       (uintptr_t)offsets) & 15)
    return MZ_EUNSUPPORTED;
  stats::Args a{x, B, H, T, D, x_sb, x_sh, x_st, offsets, sample, n_sample, sample_step, 0, 0};
  a.items = total / (16 / es) / (keys ? 64 : 1);
  const int64_t most = (int64_t)device_cu_count() * 8;
  a.stat_blocks = (unsigned)std::min<int64_t>((a.items + stats::WG - 1) / stats::WG, most);
  const int64_t gather = std::min<int64_t>((n_sample + stats::WG - 1) / stats::WG, most);
  const dim3 grid((unsigned)(a.stat_blocks + gather));
  hipStream_t s = (hipStream_t)stream;
#define MZ_STATS(DT) \
  if (keys) stats::block_stats_kernel<DT, true><<<grid, dim3(stats::WG), 0, s>>>(a); \
  else stats::block_stats_kernel<DT, false><<<grid, dim3(stats::WG), 0, s>>>(a)
  if (x_dtype == MZ_F32) { MZ_STATS(MZ_F32); }
  else if (x_dtype == MZ_BF16) { MZ_STATS(MZ_BF16); }
  else { MZ_STATS(MZ_F16); }
#undef MZ_STATS
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? MZ_OK : (int)e;
}

extern "C" int muzero_select3(const void* values, int dtype, int sets, int64_t set_stride, int64_t n, int64_t k0,
                              int64_t k1, int64_t k2, float* out, int64_t out_stride, mz_stream_t stream) {
  if (dtype != MZ_F32 && dtype != MZ_BF16 && dtype != MZ_F16) return MZ_EINVAL;
  if (!values || ((uintptr_t)values & 15) || !out || n < 1 || n >= (int64_t)1 << 31) return MZ_EINVAL;
  const int64_t es = dtype == MZ_F32 ? 4 : 2;
  if (sets < 1 || sets > 65535 || (sets > 1 && (set_stride < n || set_stride * es % 16 || out_stride < 3))) return MZ_EINVAL;
  for (const int64_t k : {k0, k1, k2})
    if (k < 0 || k >= n) return MZ_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == MZ_F32) {
    stats::select_kernel<<<dim3(sets), dim3(stats::SEL), 0, s>>>((const uint32_t*)values, set_stride, n, (uint32_t)k0,
                                                                 (uint32_t)k1, (uint32_t)k2, out, out_stride);
  } else {
    static std::atomic<uint64_t> raised[2];
    const auto kernel = dtype == MZ_BF16 ? stats::select16_kernel<MZ_BF16> : stats::select16_kernel<MZ_F16>;
    const hipError_t e = set_dynamic_lds((const void*)kernel, stats::LDS16, raised[dtype == MZ_BF16]);
    if (e != hipSuccess) return (int)e;
    kernel<<<dim3(sets), dim3(stats::SEL), stats::LDS16, s>>>((const uint16_t*)values, set_stride, n, (uint32_t)k0,
                                                             (uint32_t)k1, (uint32_t)k2, out, out_stride);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? MZ_OK : (int)e;
}
