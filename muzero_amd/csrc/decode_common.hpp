// Shared pieces of the decode-attention kernels (gfx950, wave64, MFMA 16x16x32).
#pragma once
#include "common.hpp"

namespace mz {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int IO> struct Mfma;
template <> struct Mfma<MZ_BF16> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                    0, 0, 0);
  }
  static __device__ __forceinline__ uint16_t cvt(float x) { return f2bf(x); }
  static __device__ __forceinline__ float load(uint16_t h) { return bf2f(h); }
};
template <> struct Mfma<MZ_F16> {
  static __device__ __forceinline__ f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                   0, 0);
  }
  static __device__ __forceinline__ uint16_t cvt(float x) { return f2h(x); }
  static __device__ __forceinline__ float load(uint16_t h) { return h2f(h); }
};

// Orders LDS writes and reads of one wave (the compiler must not move the
// reads of other lanes' data above the writes).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float meta_load(const void* p, int64_t i, int dt) { return load_any(p, i, dt); }

struct OpMax {
  __device__ __forceinline__ float operator()(float x, float y) const { return fmaxf(x, y); }
};
struct OpAdd {
  __device__ __forceinline__ float operator()(float x, float y) const { return x + y; }
};

// Wave-uniform maximum (NaN operands are ignored, as by fmaxf).
__device__ __forceinline__ float wave_max_fast(float v) {
  v = group_reduce<16>(v, OpMax());
  const int b = __builtin_bit_cast(int, v);
  const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0));
  const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16));
  const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32));
  const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48));
  return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

// Upper bounds of the wave-wide maxima of two non-negative floats, reduced
// together: each is cut to its top 16 bits rounded up (at most 2^-8 above the
// value, same or next binade), so both ride one DPP chain as u16 pairs.  NaN
// and overflowing inputs come back as the largest finite bound.
__device__ __forceinline__ void wave_max2_bound(float& x, float& y) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  const uint32_t hx = min(__float_as_uint(x) >> 16, 0x7F7Eu) + 1u;
  const uint32_t hy = min(__float_as_uint(y) >> 16, 0x7F7Eu) + 1u;
  u16x2 p = __builtin_bit_cast(u16x2, hx | (hy << 16));
  p = __builtin_elementwise_max(p, __builtin_bit_cast(u16x2, dpp_sel_u<DPP_QUAD_XOR1>(__builtin_bit_cast(uint32_t, p))));
  p = __builtin_elementwise_max(p, __builtin_bit_cast(u16x2, dpp_sel_u<DPP_QUAD_XOR2>(__builtin_bit_cast(uint32_t, p))));
  p = __builtin_elementwise_max(p, __builtin_bit_cast(u16x2, dpp_sel_u<DPP_ROW_HALF_MIRROR>(__builtin_bit_cast(uint32_t, p))));
  p = __builtin_elementwise_max(p, __builtin_bit_cast(u16x2, dpp_sel_u<DPP_ROW_MIRROR>(__builtin_bit_cast(uint32_t, p))));
  const uint32_t b = __builtin_bit_cast(uint32_t, p);
  u16x2 r = __builtin_bit_cast(u16x2, (uint32_t)__builtin_amdgcn_readlane((int)b, 0));
  r = __builtin_elementwise_max(r, __builtin_bit_cast(u16x2, (uint32_t)__builtin_amdgcn_readlane((int)b, 16)));
  r = __builtin_elementwise_max(r, __builtin_bit_cast(u16x2, (uint32_t)__builtin_amdgcn_readlane((int)b, 32)));
  r = __builtin_elementwise_max(r, __builtin_bit_cast(u16x2, (uint32_t)__builtin_amdgcn_readlane((int)b, 48)));
  const uint32_t rb = __builtin_bit_cast(uint32_t, r);
  x = __uint_as_float(rb << 16);
  y = __uint_as_float(rb & 0xFFFF0000u);
}

// The split count of a call the caller leaves to the library (host).  A
// workgroup of `waves` waves takes one split of a unit's (batch, kv-head)
// tiles, a tile per wave and round; `per_cu` workgroups are resident per CU.
// The cost of a count, in rounds of one wave per SIMD (3.2 us for the 4-bit
// codebook kernel): rounds of the workgroups that run one after another on a
// slot, a round slowed by `slope` per further wave on the SIMD; 0.05 per wave
// on the CU; 1.7 per repeated filling of the slots (tables, first loads, a last
// one that is nearly empty); 0.3 where workgroups share a CU; 0.5 for the merge
// of the splits.  The counts tried fill the CUs or the slots once, with the
// fewest splits of the same number of rounds, besides 1 and 2.  Measured
// (us per prebuilt call; a count that fills the slots rounded up, two tiles per wave / this rule):
// 4-bit, 1 sequence of 1000 tokens 16.3 / 12.3, of 4096 16.9 / 12.7; 48 of 2000
// 57.2 / 48.0; 70 of 2000 90.1 / 76.1; 7-bit, 1 of 4096 18.2 / 14.5; head_dim 64,
// 24 of 3001 32.4 / 25.9.
inline int choose_splits(int64_t units, int n_tiles, int waves, int per_cu, float slope) {
  units = units < 1 ? 1 : units;  // an empty batch splits nothing
  const int64_t cus = device_cu_count(), slots = cus * per_cu;
  auto cost = [&](int ns) {
    const int tps = (n_tiles + ns - 1) / ns;
    ns = (n_tiles + tps - 1) / tps;
    const int64_t wgs = units * ns, fills = (wgs + slots - 1) / slots;
    const int act = tps < waves ? tps : waves, shared = wgs > cus ? per_cu : 1;
    const float load = 0.25f * (float)(act * shared);
    const float round = load > 1.f ? 1.f + slope * (load - 1.f) : 1.f;
    return (float)fills * ((float)((tps + waves - 1) / waves) * round + 0.05f * (float)(act * shared)) +
           1.7f * (float)(fills - 1) + (shared > 1 ? 0.3f : 0.f) + (ns > 1 ? 0.5f : 0.f);
  };
  int best = 1;
  float least = cost(1);
  auto consider = [&](int64_t ns) {
    if (ns < 2 || ns > n_tiles) return;
    const float c = cost((int)ns);
    if (c < least) least = c, best = (int)ns;
  };
  consider(2);
  for (const int64_t cap : {cus, slots}) {
    const int64_t most = cap / units < n_tiles ? cap / units : n_tiles;
    if (most < 2) continue;
    const int64_t tps = (n_tiles + most - 1) / most, rounds = (tps + waves - 1) / waves;
    consider((n_tiles + rounds * waves - 1) / (rounds * waves));
    consider(most);
  }
  return best;
}

// Workspace record of one (batch, q-head, split): acc[D], m, l (fp32).
template <int D>
__device__ __forceinline__ float* ws_record(const mz_decode_args& a, int b, int qh, int split, int n_split) {
  const int Hq = a.kv_heads * a.n_rep;
  return (float*)a.workspace + (((int64_t)b * Hq + qh) * n_split + split) * (D + 2);
}

}  // namespace mz
