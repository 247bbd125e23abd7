// Quantize + dequantize of K or V without storing the codes (gfx950, wave64).
//
// The offline quality check (muzero/quantizer.py:273-323) quantizes a tensor's
// groups from fp32 and dequantizes them again.  As separate steps that is a
// cast, a permute, a quantize, a dequantize and a permute back per kind (11
// launches for K and V); here one kernel reads the tensor once and writes the
// result once, the codes staying in registers.  4 lanes share a 64-value group,
// 16 values each, so that a small tensor still fills the CUs: the fp32 chain
// (two IEEE divisions and a threshold search per value, about 100 VALU) is what
// bounds it, not the memory.
//   keys:   a workgroup takes 64 channels of one 64-token group, wave w tokens
//           16w .. 16w + 15, so each token's 64 lanes access consecutive
//           channels; the group's min / max cross the waves through LDS.
//   values: 4 consecutive lanes take the 64 channels of a group (min / max by
//           DPP), 16-byte accesses where rows are aligned.
// Minimum and scale are rounded to the metadata dtype between the two halves, as
// storing them rounds them.  K and V of [1, 8, 896, 128] bf16, 4-bit: 92 us as
// separate steps, 20 us here (two launches; profiled one at a time 11.1 and
// 10.3 us).
#include "quantize_core.hpp"

#include <algorithm>

namespace mz {
namespace rt {

constexpr int N = 16;  // values per lane

struct Args {
  const void* x;
  void* out;
  int B, H, T, D;
  int64_t sb, sh, st, osb, osh, ost;
  int mdt;
  float eps;
  const void* table;  // fp32 thresholds of the alpha
  const float* e;     // its expm1 rows
  int vec;            // 16-byte accesses fit the rows (values)
  int blocks_c;       // keys: channel blocks of 64; values: groups per token
  int64_t items;      // keys: (slice, group, channel block); values: (slice, token, group)
};

__device__ __forceinline__ float meta_round(float v, int dt) {
  return dt == MZ_F32 ? v : dt == MZ_BF16 ? bf2f(f2bf(v)) : h2f(f2h(v));
}

// expm1 rows of up to 6 bits in LDS after the thresholds, wider ones read from global memory
template <int BITS>
struct Tab {
  static constexpr int QMAX = (1 << BITS) - 1;
  static constexpr int TH = QTable<MZ_F32, BITS>::LDS_BYTES;
  static constexpr int EF = BITS <= 6 ? QMAX * (QMAX + 3) / 2 : 0;
  static constexpr int BYTES = TH + (EF * 4 + 15) / 16 * 16;
};

// x[i] -> its dequantized value, given the group's min and max.
template <int BITS>
__device__ __forceinline__ void roundtrip_lane(float (&x)[N], float mn, float mx, const Args& a, const uint8_t* lds) {
  QParams g = qparams<MZ_F32, BITS>(mn, mx, a.eps);
  if constexpr (BITS >= 5) set_estimate<BITS>(g, lds, a.table);
  const bool finite = QTable<MZ_F32, BITS>::IN_LDS && __builtin_isfinite(g.mn) && __builtin_isfinite(g.sc) &&
                      g.sc > 0.f && g.pe > 0.f && g.ne > 0.f;
  const DeqGroup d = make_group<Tab<BITS>::QMAX>(meta_round(g.mn, a.mdt), meta_round(g.sc, a.mdt));
  const float* E = Tab<BITS>::EF ? (const float*)(lds + Tab<BITS>::TH) : a.e;
  if (finite) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      x[i] = group_value(d, (int)value_code<MZ_F32, BITS, true, true>(x[i], g, lds, a.table), E);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i)
      x[i] = group_value(d, (int)value_code<MZ_F32, BITS, true, false>(x[i], g, lds, a.table), E);
  }
}

template <int IO, int BITS, bool KEYS>
__global__ __launch_bounds__(QWG) void roundtrip_kernel(const Args a) {
  __shared__ __align__(16) uint8_t lds[Tab<BITS>::BYTES];
  __shared__ float2 ends[KEYS ? 4 : 1][64];
  if constexpr (Tab<BITS>::EF > 0) {
    for (int i = threadIdx.x; i < Tab<BITS>::EF; i += QWG) ((float*)(lds + Tab<BITS>::TH))[i] = a.e[i];
  }
  stage_table<MZ_F32, BITS>(lds, a.table);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int ES = IO == MZ_F32 ? 4 : 2;
  if constexpr (KEYS) {
    for (int64_t it = blockIdx.x; it < a.items; it += gridDim.x) {
      const int64_t r = it / a.blocks_c;
      const int c = (int)(it - r * a.blocks_c) * 64 + lane;
      const int nsg = a.T / 64;
      const int64_t slice = r / nsg, b = slice / a.H, h = slice - b * a.H;
      const int64_t t0 = (r - slice * nsg) * 64 + N * wave;
      const bool in = c < a.D;
      float x[N], lo = 0.f, hi = 0.f;
      if (in) {
        const int64_t base = b * a.sb + h * a.sh + t0 * a.st + c;
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = load_val<IO>(a.x, base + i * a.st);
        lo = tree_min<N>(x), hi = tree_max<N>(x);
      }
      ends[wave][lane] = make_float2(lo, hi);
      __syncthreads();
      const float2 e0 = ends[0][lane], e1 = ends[1][lane], e2 = ends[2][lane], e3 = ends[3][lane];
      __syncthreads();  // (the next item overwrites them)
      if (in) {
        lo = fmin_nan(fmin_nan(e0.x, e1.x), fmin_nan(e2.x, e3.x));
        hi = fmax_nan(fmax_nan(e0.y, e1.y), fmax_nan(e2.y, e3.y));
        roundtrip_lane<BITS>(x, lo, hi, a, lds);
        const int64_t base = b * a.osb + h * a.osh + t0 * a.ost + c;
#pragma unroll
        for (int i = 0; i < N; ++i) store_val(a.out, base + i * a.ost, x[i], IO);
      }
    }
  } else {
    const int part = lane & 3;
    const int64_t stride = (int64_t)gridDim.x * (QWG / 4);
    for (int64_t it = (int64_t)blockIdx.x * (QWG / 4) + (threadIdx.x >> 2); it < a.items; it += stride) {
      const int64_t tok = it / a.blocks_c;  // (a group's 4 lanes share `it`)
      const int c = (int)(it - tok * a.blocks_c) * 64 + N * part;
      const int64_t slice = tok / a.T, b = slice / a.H, h = slice - b * a.H;
      const int64_t t = tok - slice * a.T;
      const int64_t src = b * a.sb + h * a.sh + t * a.st + c, dst = b * a.osb + h * a.osh + t * a.ost + c;
      float x[N];
#pragma unroll
      for (int k = 0; k < N; k += 8) {
        float (&x8)[8] = *(float(*)[8])(x + k);
        if (a.vec && c + k + 8 <= a.D) {
          load8<IO, true>(x8, a.x, src + k);
        } else {  // the last group's missing channels are zeros
#pragma unroll
          for (int e = 0; e < 8; ++e) x8[e] = c + k + e < a.D ? load_val<IO>(a.x, src + k + e) : 0.f;
        }
      }
      const float lo = group_min<4>(tree_min<N>(x)), hi = group_max<4>(tree_max<N>(x));
      roundtrip_lane<BITS>(x, lo, hi, a, lds);
#pragma unroll
      for (int k = 0; k < N; k += 8) {
        if (a.vec && c + k + 8 <= a.D) {
          if constexpr (IO == MZ_F32) {
            *(float4*)((float*)a.out + dst + k) = make_float4(x[k], x[k + 1], x[k + 2], x[k + 3]);
            *(float4*)((float*)a.out + dst + k + 4) = make_float4(x[k + 4], x[k + 5], x[k + 6], x[k + 7]);
          } else {
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
              w[e] = IO == MZ_BF16 ? (uint32_t)f2bf(x[k + 2 * e]) | (uint32_t)f2bf(x[k + 2 * e + 1]) << 16
                                   : (uint32_t)f2h(x[k + 2 * e]) | (uint32_t)f2h(x[k + 2 * e + 1]) << 16;
            *(uint4*)((uint16_t*)a.out + dst + k) = make_uint4(w[0], w[1], w[2], w[3]);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (c + k + e < a.D) store_val(a.out, dst + k + e, x[k + e], IO);
        }
      }
    }
  }
}

template <int IO, int BITS>
void launch(const Args& a, bool keys, hipStream_t s) {
  // the tables are staged per workgroup: at most 8 of them per CU, looping
  const int64_t per = keys ? 1 : QWG / 4;
  const int64_t grid = std::min<int64_t>((a.items + per - 1) / per, 8 * (int64_t)device_cu_count());
  if (keys) roundtrip_kernel<IO, BITS, true><<<dim3((unsigned)grid), dim3(QWG), 0, s>>>(a);
  else roundtrip_kernel<IO, BITS, false><<<dim3((unsigned)grid), dim3(QWG), 0, s>>>(a);
}

template <int IO>
void launch_bits(const Args& a, int bits, bool keys, hipStream_t s) {
  switch (bits) {
    case 1: return launch<IO, 1>(a, keys, s);
    case 2: return launch<IO, 2>(a, keys, s);
    case 3: return launch<IO, 3>(a, keys, s);
    case 4: return launch<IO, 4>(a, keys, s);
    case 5: return launch<IO, 5>(a, keys, s);
    case 6: return launch<IO, 6>(a, keys, s);
    case 7: return launch<IO, 7>(a, keys, s);
    default: return launch<IO, 8>(a, keys, s);
  }
}

}  // namespace rt
}  // namespace mz

using namespace mz;

extern "C" int muzero_roundtrip(const void* x, int dtype, int keys, int B, int H, int T, int D, int64_t x_sb,
                                int64_t x_sh, int64_t x_st, void* out, int64_t o_sb, int64_t o_sh, int64_t o_st,
                                int meta_dtype, int bits, float eps, const void* table, const float* e_table,
                                mz_stream_t stream) {
  const auto ok = [](int dt) { return dt == MZ_F32 || dt == MZ_BF16 || dt == MZ_F16; };
  if (!ok(dtype) || !ok(meta_dtype) || bits < 1 || bits > 8) return MZ_EINVAL;
  if (B < 0 || H < 0 || T < 0 || D < 1 || (keys && T % 64)) return MZ_EINVAL;
  if ((int64_t)B * H * T == 0) return MZ_OK;
  if (!x || !out || !table || !e_table) return MZ_EINVAL;
  rt::Args a{x, out, B, H, T, D, x_sb, x_sh, x_st, o_sb, o_sh, o_st, meta_dtype, eps, table, e_table, 0, 0, 0};
  const int64_t es = dtype == MZ_F32 ? 4 : 2;
  a.vec = (((uintptr_t)x | (uintptr_t)out | (uintptr_t)(x_sb * es) | (uintptr_t)(x_sh * es) | (uintptr_t)(x_st * es) |
            (uintptr_t)(o_sb * es) | (uintptr_t)(o_sh * es) | (uintptr_t)(o_st * es)) & 15) == 0;
  a.blocks_c = (D + 63) / 64;
  a.items = (int64_t)B * H * (keys ? T / 64 : T) * a.blocks_c;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == MZ_F32) rt::launch_bits<MZ_F32>(a, bits, keys, s);
  else if (dtype == MZ_BF16) rt::launch_bits<MZ_BF16>(a, bits, keys, s);
  else rt::launch_bits<MZ_F16>(a, bits, keys, s);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? MZ_OK : (int)e;
}
