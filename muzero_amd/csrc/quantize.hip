// Quantize + bit-pack kernels (gfx950, wave64).
//
// Quantize: 2 lanes per 64-value group, 32 consecutive values per lane, so a
// wave quantizes 32 groups.  The group min/max is an in-lane reduction plus
// one DPP step; the group's compander parameters are computed once per lane; every
// per-element op of the reference quantizer (muzero/quantizer.py:161-186) is
// evaluated in its own dtype with IEEE rounding and no contraction, and the
// one transcendental step (round(log1p(alpha*p)/lb*bins)) comes from a
// host-built constant table staged in LDS, so codes and metadata are
// bit-identical to the reference torch path.  8 codes of BITS bits are exactly
// BITS bytes of the LSB-first bitstream (quantizer.py:189-202), so each lane
// packs and stores its own bytes and a wave's stores are contiguous.  The grid
// is persistent (a few workgroups per CU loop over the groups), so each
// workgroup stages the table once.
#include "quantize_core.hpp"

#include <algorithm>
#include <type_traits>

namespace mz {

// Values per lane: each lane quantizes 32 values of a 64-value group (two
// lanes per group), so a wave quantizes 32 groups and a group's parameters
// are formed once per 32 values.  Key groups read their column from an LDS
// tile.
constexpr int QN_ROWS = 32;
constexpr int QN_KEYS = 32;

// 8 codes' BITS packed bytes.
template <int BITS>
__device__ __forceinline__ void store_codes8(uint8_t* dst, uint64_t w) {
  if constexpr (BITS == 8) *(uint64_t*)dst = w;
  else if constexpr (BITS == 4) *(uint32_t*)dst = (uint32_t)w;
  else if constexpr (BITS == 2) *(uint16_t*)dst = (uint16_t)w;
  else if constexpr (BITS == 1) *dst = (uint8_t)w;
  else {
#pragma unroll
    for (int k = 0; k < BITS; ++k) dst[k] = (uint8_t)(w >> (8 * k));
  }
}

// Quantize the 8 values x[0..7] of a chunk with the group's parameters and
// store their BITS packed bytes at dst.
template <int DT, int BITS>
__device__ __forceinline__ void quantize_chunk8(const float* x, const QParams& g, bool finite, uint8_t* dst,
                                                const uint8_t* lds, const void* table) {
  uint64_t w = 0;
  if (finite) {
#pragma unroll
    for (int i = 0; i < 8; ++i) w |= (uint64_t)value_code<DT, BITS, false, true>(x[i], g, lds, table) << (i * BITS);
  } else if (qfast<DT>(g)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) w |= (uint64_t)value_code<DT, BITS, true, false>(x[i], g, lds, table) << (i * BITS);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) w |= (uint64_t)value_code<DT, BITS, false, false>(x[i], g, lds, table) << (i * BITS);
  }
  store_codes8<BITS>(dst, w);
}

// Quantize this lane's N values x[0..N) (positions N*part .. N*part+N-1 of
// its group, which 64 / N lanes share) and store its N*BITS/8 packed bytes
// at prow + part*N*BITS/8; lane part 0 stores the group's metadata at index
// midx.  The group's parameters are formed once per lane, so a larger N
// spreads them over more values.  fp32 inputs, and the 16-bit groups that
// quantize_lane16 finds outside its finite chain.
template <int DT, int BITS, int N>
__device__ __forceinline__ void quantize_lane(const float (&x)[N], int part, uint8_t* prow, void* mn_out,
                                              void* sc_out, int64_t midx, int meta_dtype, float eps,
                                              const uint8_t* lds, const void* table) {
  constexpr int L = 64 / N;
  const float mn = group_min<L>(tree_min<N>(x));
  const float mx = group_max<L>(tree_max<N>(x));
  QParams g = qparams<DT, BITS>(mn, mx, eps);
  if constexpr (DT == MZ_F32 && BITS >= 5) set_estimate<BITS>(g, lds, table);
  // The fp32 8-bit thresholds stay in global memory, where the plain form's
  // binary search measured faster.
  const bool finite = DT == MZ_F32 && QTable<DT, BITS>::IN_LDS && __builtin_isfinite(g.mn) && __builtin_isfinite(g.sc) &&
                      g.sc > 0.f && g.pe > 0.f && g.ne > 0.f;
  uint8_t* dst = prow + part * (N / 8) * BITS;
#pragma unroll
  for (int c = 0; c < N / 8; ++c) quantize_chunk8<DT, BITS>(x + 8 * c, g, finite, dst + c * BITS, lds, table);
  if (part == 0) {
    store_val(mn_out, midx, mn, meta_dtype);
    store_val(sc_out, midx, g.sc, meta_dtype);
  }
}

// ------------------------------------------------------------- 16-bit pairs
// quantize_lane of 16-bit values held as they were loaded, 16 dwords of two
// (rows that cannot be read as vectors are read value by value and paired: K and
// V of 16 x 8 heads x 4096 tokens x 100, bf16, 4 bits, 200 us by the general chain,
// 166 paired).
// Min and max are taken two values at a time as fp16 patterns.  bf16 values
// order as their patterns read as fp16 do (sign and magnitude); a pattern fp16
// reads as infinite or NaN (bf16 magnitudes from 2^121, infinities, NaN) shows
// in the result, and such groups, like every group the finite chain does not
// take, run quantize_lane on the unpacked values.  The kernels are bound by
// VALU ops, so the raw dwords, unpacked by the ops that read them, are the
// gain: bf16 about 17 ops a value instead of 22, fp16 19 instead of 28, and 4
// instead of 64 for 32 values' min and max.  Prefill of K and V, 64 x 8 heads x
// 4096 tokens x 128, 4 bits: bf16 457 -> 400 us, fp16 563 -> 425 us.  (fp16 rounds
// eps to 0: a constant group, or za at 0 or 1, then divides by 0 and is not
// finite.)
template <int DT, int BITS>
__device__ __forceinline__ void quantize_lane16(const uint32_t (&w)[16], int part, uint8_t* prow, void* mn_out,
                                                void* sc_out, int64_t midx, int meta_dtype, float eps,
                                                const uint8_t* lds, const void* table) {
  auto h2 = [&](uint32_t u) { return __builtin_bit_cast(f16x2v, u); };
  auto value = [](uint32_t u) { return DT == MZ_BF16 ? bf2f((uint16_t)u) : h2f((uint16_t)u); };
  f16x2v lo = h2(w[0]), hi = lo;
#pragma unroll
  for (int i = 1; i < 15; i += 2) {
    lo = __builtin_elementwise_minimum(__builtin_elementwise_minimum(lo, h2(w[i])), h2(w[i + 1]));
    hi = __builtin_elementwise_maximum(__builtin_elementwise_maximum(hi, h2(w[i])), h2(w[i + 1]));
  }
  lo = __builtin_elementwise_minimum(lo, h2(w[15]));
  hi = __builtin_elementwise_maximum(hi, h2(w[15]));
  // the two halves, then the group's other lane
  const uint32_t lb = __builtin_bit_cast(uint32_t, lo), hb = __builtin_bit_cast(uint32_t, hi);
  lo = __builtin_elementwise_minimum(lo, h2(__builtin_amdgcn_alignbit(lb, lb, 16)));
  hi = __builtin_elementwise_maximum(hi, h2(__builtin_amdgcn_alignbit(hb, hb, 16)));
  lo = __builtin_elementwise_minimum(lo, h2(dpp_sel_u<DPP_QUAD_XOR1>(__builtin_bit_cast(uint32_t, lo))));
  hi = __builtin_elementwise_maximum(hi, h2(dpp_sel_u<DPP_QUAD_XOR1>(__builtin_bit_cast(uint32_t, hi))));
  const uint32_t mnb = __builtin_bit_cast(uint32_t, lo), mxb = __builtin_bit_cast(uint32_t, hi);
  const bool ordered = (mnb & 0x7C00u) != 0x7C00u && (mxb & 0x7C00u) != 0x7C00u;
  const float mn = value(mnb), mx = value(mxb);
  const QParams g = qparams<DT, BITS>(mn, mx, eps);
  if (ordered && qfast<DT>(g) && __builtin_isfinite(g.sc) && g.sc > 0.f && g.pe > 0.f && g.ne > 0.f) {
    const typename std::conditional<DT == MZ_BF16, BfGroup, HfGroup>::type cg(g, (float)((1 << BITS) - 1));
    uint8_t* dst = prow + part * 4 * BITS;
#pragma unroll
    for (int c = 0; c < 4; ++c) store_codes8<BITS>(dst + c * BITS, value_codes8<BITS>(w + 4 * c, cg, lds));
    if (part == 0) {
      store_val(mn_out, midx, mn, meta_dtype);
      store_val(sc_out, midx, g.sc, meta_dtype);
    }
  } else {
    float x[32];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[2 * i] = value(w[i]), x[2 * i + 1] = value(w[i] >> 16);
    quantize_lane<DT, BITS, 32>(x, part, prow, mn_out, sc_out, midx, meta_dtype, eps, lds, table);
  }
}

// ------------------------------------------------------------- rows
template <int DT, int BITS, bool VEC>
__global__ __launch_bounds__(QWG) void quantize_rows_kernel(const void* __restrict__ x, int64_t nrows,
                                                            int64_t xs, uint8_t* __restrict__ packed, int64_t ps,
                                                            void* mn, void* sc, int meta_dtype, int64_t ms,
                                                            float eps, const void* __restrict__ table) {
  __shared__ __align__(16) uint8_t lds[QTable<DT, BITS>::LDS_BYTES];
  stage_table<DT, BITS>(lds, table);
  constexpr int N = QN_ROWS, L = 64 / N;
  const int lane = threadIdx.x & 63;
  const int part = lane % L;
  const int64_t stride = (int64_t)gridDim.x * (QWG / 64) * N;
  for (int64_t row = ((int64_t)blockIdx.x * (QWG / 64) + (threadIdx.x >> 6)) * N + lane / L;
       row - lane / L < nrows; row += stride) {
    if (row < nrows) {  // lanes of a group share `row`: the whole group takes this branch
      if constexpr (DT != MZ_F32) {
        uint32_t w[N / 2];
        const uint16_t* xr = (const uint16_t*)x + row * xs + N * part;
        if constexpr (VEC) {
#pragma unroll
          for (int c = 0; c < N / 8; ++c) {
            const uint4 u = *(const uint4*)(xr + 8 * c);
            w[4 * c] = u.x, w[4 * c + 1] = u.y, w[4 * c + 2] = u.z, w[4 * c + 3] = u.w;
          }
        } else {
#pragma unroll
          for (int k = 0; k < N / 2; ++k) w[k] = (uint32_t)xr[2 * k] | (uint32_t)xr[2 * k + 1] << 16;
        }
        quantize_lane16<DT, BITS>(w, part, packed + row * ps, mn, sc, row * ms, meta_dtype, eps, lds, table);
      } else {
        float v[N];
#pragma unroll
        for (int c = 0; c < N / 8; ++c) load8<DT, VEC>(*(float(*)[8])(v + 8 * c), x, row * xs + N * part + 8 * c);
        quantize_lane<DT, BITS, N>(v, part, packed + row * ps, mn, sc, row * ms, meta_dtype, eps, lds, table);
      }
    }
  }
}

// ------------------------------------------------------------- index math
// n / d for 0 <= n < 2^31 by multiply-high (Granlund-Montgomery): l =
// ceil(log2 d), m = floor(2^32 (2^l - d) / d) + 1, n / d = (mulhi(n, m) + n) >> l.
struct FastDiv {
  uint32_t d, m, l;
  __device__ __forceinline__ uint32_t div(uint32_t n) const { return (__umulhi(n, m) + n) >> l; }
};

static FastDiv make_fastdiv(uint32_t d) {
  uint32_t l = 0;
  while ((1ull << l) < d) ++l;
  const uint64_t m = (((1ull << 32) * ((1ull << l) - d)) / d) + 1;
  return FastDiv{d, (uint32_t)m, l};
}

// ------------------------------------------------------------- values
// Row (b, h, t, j): channels 64j..64j+63 of token t, zero beyond D.  Rows
// are numbered b-major with j fastest; nrows < 2^31 per launch (the host
// splits the batch).
template <int DT, int BITS, bool VEC, bool NARROW>
__global__ __launch_bounds__(QWG) void quantize_values_kernel(const void* __restrict__ x, int nrows, FastDiv fng,
                                                              FastDiv fT, FastDiv fH, int D, int64_t sb, int64_t sh,
                                                              int64_t st, uint8_t* __restrict__ packed, int64_t psb,
                                                              int64_t psh, void* mn, void* sc, int meta_dtype,
                                                              int64_t msb, int64_t msh, float eps,
                                                              const void* __restrict__ table) {
  __shared__ __align__(16) uint8_t lds[QTable<DT, BITS>::LDS_BYTES];
  stage_table<DT, BITS>(lds, table);
  constexpr int QB = 8 * BITS;
  constexpr int N = QN_ROWS, L = 64 / N;  // values per lane, lanes per group
  const int ng = (int)fng.d, T = (int)fT.d, H = (int)fH.d;
  const int TN = T * ng;  // rows per (b, h)
  const int lane = threadIdx.x & 63;
  const int part = lane % L;
  const int k = lane / L;  // the lane's row within its wave's N
  // wave-uniform (the compiler cannot see that threadIdx.x >> 6 is): the
  // (b, h) decomposition of a wave's first row then runs on the scalar unit
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int stride = gridDim.x * (QWG / 64) * N;
  for (int w0 = (blockIdx.x * (QWG / 64) + wave) * N; w0 < nrows; w0 += stride) {
    const int row = w0 + k;
    if (row >= nrows) continue;  // lanes of a group share `row`: the whole group takes this branch
    int64_t xo, po, mo;
    int i;
    if (TN >= N) {
      // the wave's N rows lie in (b, h) slices o0 and o0 + 1 at most (rows
      // are b-major, (t, j) fastest): their offsets are scalar
      const int o0 = (int)fT.div((uint32_t)fng.div((uint32_t)w0));  // w0 / (T*ng)
      const int b0 = (int)fH.div((uint32_t)o0), h0 = o0 - b0 * H;
      const int b1 = h0 + 1 == H ? b0 + 1 : b0, h1 = h0 + 1 == H ? 0 : h0 + 1;
      i = w0 - o0 * TN + k;
      const bool next = i >= TN;
      if (next) i -= TN;
      xo = next ? b1 * sb + h1 * sh : b0 * sb + h0 * sh;
      po = next ? b1 * psb + h1 * psh : b0 * psb + h0 * psh;
      mo = next ? b1 * msb + h1 * msh : b0 * msb + h0 * msh;
    } else {
      // short slices (few tokens): each row decomposed on its own
      const int o = (int)fT.div((uint32_t)fng.div((uint32_t)row));
      const int b = (int)fH.div((uint32_t)o), h = o - b * H;
      i = row - o * TN;
      xo = b * sb + h * sh;
      po = b * psb + h * psh;
      mo = b * msb + h * msh;
    }
    const int t = (int)fng.div((uint32_t)i);
    const int j = i - t * ng;
    const int c = 64 * j + N * part;
    // NARROW: every offset within a slice fits 31 bits (checked on the host)
    const int64_t src = xo + (NARROW ? (int64_t)(t * (int)st + c) : (int64_t)t * st + c);
    uint8_t* prow = packed + po + (NARROW ? (int64_t)(i * QB) : (int64_t)i * QB);
    if constexpr (DT != MZ_F32) {
      uint32_t w[N / 2];
      const uint16_t* xr = (const uint16_t*)x + src;
#pragma unroll
      for (int e8 = 0; e8 < N / 8; ++e8) {
        const int c8 = c + 8 * e8;
        if constexpr (VEC) {
          // D % 8 == 0: a vector lies within D or past it (lanes past D read nothing)
          const uint4 u = c8 < D ? *(const uint4*)(xr + 8 * e8) : make_uint4(0, 0, 0, 0);
          w[4 * e8] = u.x, w[4 * e8 + 1] = u.y, w[4 * e8 + 2] = u.z, w[4 * e8 + 3] = u.w;
        } else if (c8 + 8 <= D) {
#pragma unroll
          for (int k = 4 * e8; k < 4 * e8 + 4; ++k) w[k] = (uint32_t)xr[2 * k] | (uint32_t)xr[2 * k + 1] << 16;
        } else {
          auto at = [&](int e) { return c + e < D ? (uint32_t)xr[e] : 0u; };
#pragma unroll
          for (int k = 4 * e8; k < 4 * e8 + 4; ++k) w[k] = at(2 * k) | at(2 * k + 1) << 16;
        }
      }
      quantize_lane16<DT, BITS>(w, part, prow, mn, sc, mo + i, meta_dtype, eps, lds, table);
    } else {
      float v[N];
#pragma unroll
      for (int e8 = 0; e8 < N / 8; ++e8) {
        float (&v8)[8] = *(float(*)[8])(v + 8 * e8);
        const int c8 = c + 8 * e8;
        if (c8 + 8 <= D) {  // VEC only picks the load width; lanes past D (D % 64 != 0) read nothing
          load8<DT, VEC>(v8, x, src + 8 * e8);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) v8[e] = c8 + e < D ? load_val<DT>(x, src + 8 * e8 + e) : 0.f;
        }
      }
      quantize_lane<DT, BITS, N>(v, part, prow, mn, sc, mo + i, meta_dtype, eps, lds, table);
    }
  }
}

// ------------------------------------------------------------- keys
// A workgroup loops over (b, h, token group) tiles: the [64 x D] tile is
// staged in LDS in the input dtype (16-bit inputs as they arrive, fp32 as
// fp32) and each wave quantizes 8 channels at a time reading the tile's
// columns, so the reference's permute + contiguous copy (layer.py:276-278)
// never touches HBM.  VEC: the tile arrives as 16-byte vectors (D % 8 == 0,
// D <= 256, aligned rows), and the next tile's vectors are loaded into
// registers before the current tile is quantized.  The grid holds as many
// workgroups per CU as the table and the tile leave room for in LDS (at most
// 4).
// 16-byte vectors per thread per tile on the vector path: 64 tokens x D
// channels / (16 / element bytes) / QWG, so at most D = 256 for 16-bit
// inputs and D = 128 for fp32 (the host sends wider fp32 tiles to the scalar
// path)
constexpr int KEY_MAX_VEC = 8;

template <int DT>
struct Vec16 {
  static constexpr int N = DT == MZ_F32 ? 4 : 8;  // elements per 16 bytes
};

template <int DT>
__device__ __forceinline__ void vec16_store_lds(float* dst, const uint4 u) {
  if constexpr (DT == MZ_F32) {
    dst[0] = __uint_as_float(u.x), dst[1] = __uint_as_float(u.y), dst[2] = __uint_as_float(u.z),
    dst[3] = __uint_as_float(u.w);
  } else {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      dst[2 * k] = DT == MZ_BF16 ? bf2f((uint16_t)w[k]) : h2f((uint16_t)w[k]);
      dst[2 * k + 1] = DT == MZ_BF16 ? bf2f((uint16_t)(w[k] >> 16)) : h2f((uint16_t)(w[k] >> 16));
    }
  }
}

// Staging element of the key tile: 16-bit inputs stay 16-bit in LDS (row
// pitch D + 2 halves), fp32 inputs stay fp32 (pitch D + 1).  Either pitch is
// an odd number of dwords, so a column read of a wave's 8 lane groups meets
// at most two distinct dwords per bank.
template <int DT>
struct KeyStage {
  using T = typename std::conditional<DT == MZ_F32, float, uint16_t>::type;
  static constexpr int PAD = DT == MZ_F32 ? 1 : 2;
};

// 16-bit inputs arriving as vectors are staged transposed instead: one row
// of KT_PITCH dwords per channel, dword m = tokens 2m (low half) and 2m + 1
// (high half), so a lane reads its 32 tokens of a column as four 16-byte
// LDS reads.  A staging thread loads the same 8 channels of two adjacent
// tokens and pairs them with v_perm; threads of a wave take consecutive
// token pairs, so their stores fill consecutive dwords of a row.  The pitch
// (36 dwords, a multiple of 4) keeps the 16-byte reads aligned, and the 8
// lanes served in one cycle (4 columns x 2 halves) cover distinct banks.
constexpr int KT_PITCH = 36;
template <int DT, bool VEC>
struct KeyTrans {
  static constexpr bool ON = VEC && DT != MZ_F32;
  static constexpr size_t bytes(int D) { return (size_t)D * KT_PITCH * 4; }
};

template <int DT, int BITS, bool VEC>
__global__ __launch_bounds__(QWG) void quantize_keys_kernel(const void* __restrict__ x, int B, int H, int T, int D,
                                                            int64_t sb, int64_t sh, int64_t st,
                                                            uint8_t* __restrict__ packed, int64_t psb, int64_t psh,
                                                            void* mn, void* sc, int meta_dtype, int64_t msb,
                                                            int64_t msh, float eps, const void* __restrict__ table) {
  using KS = KeyStage<DT>;
  using ET = typename KS::T;
  extern __shared__ __align__(16) uint8_t dyn[];
  uint8_t* lds = dyn;                                                 // compander table
  ET* tile = (ET*)(dyn + QTable<DT, BITS>::LDS_BYTES);                // [64][D + PAD]
  stage_table<DT, BITS>(lds, table);
  const int nsg = T / 64;
  const int ntiles = B * H * nsg;  // < 2^31 (host check)
  const int ld = D + KS::PAD;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int part = lane % (64 / QN_KEYS);
  constexpr int QB = 8 * BITS;
  constexpr int NE = Vec16<DT>::N;
  const int vpr = D / NE;             // vectors per token row (VEC)
  const int nvec = 64 * vpr;          // vectors per tile (VEC)
  auto tile_base = [&](int ti) -> int64_t {
    const int s = ti % nsg, h = (ti / nsg) % H, b = ti / (nsg * H);
    return b * sb + h * sh + (int64_t)(64 * s) * st;
  };
  constexpr bool TRANS = KeyTrans<DT, VEC>::ON;
  uint32_t* tileT = (uint32_t*)tile;  // TRANS: [D][KT_PITCH] token-pair dwords
  const int npair = 32 * vpr;         // TRANS: (token pair, 8-channel block) items per tile
  uint4 nxt[KEY_MAX_VEC];
  auto fetch = [&](int ti) {
    if constexpr (TRANS) {
      const int64_t base = tile_base(ti);
      const uint16_t* xb = (const uint16_t*)x;
#pragma unroll
      for (int k = 0; k < KEY_MAX_VEC / 2; ++k) {
        const int e = threadIdx.x + k * QWG;
        if (e < npair) {
          const int tp = e & 31, cb = e >> 5;
          const int64_t a = base + (int64_t)(2 * tp) * st + NE * cb;
          nxt[2 * k] = *(const uint4*)(xb + a);
          nxt[2 * k + 1] = *(const uint4*)(xb + a + st);
        }
      }
    } else if constexpr (VEC) {
      const int64_t base = tile_base(ti);
      const char* xb = (const char*)x;
#pragma unroll
      for (int k = 0; k < KEY_MAX_VEC; ++k) {
        const int e = threadIdx.x + k * QWG;
        if (e < nvec) {
          const int t = e / vpr, c = (e - t * vpr) * NE;
          nxt[k] = *(const uint4*)(xb + (base + (int64_t)t * st + c) * (DT == MZ_F32 ? 4 : 2));
        }
      }
    }
  };
  if (blockIdx.x < ntiles) fetch(blockIdx.x);
  for (int ti = blockIdx.x; ti < ntiles; ti += gridDim.x) {
    const int s = ti % nsg, h = (ti / nsg) % H, b = ti / (nsg * H);
    __syncthreads();  // the previous tile's columns are consumed
    if constexpr (TRANS) {
#pragma unroll
      for (int k = 0; k < KEY_MAX_VEC / 2; ++k) {
        const int e = threadIdx.x + k * QWG;
        if (e < npair) {
          const int tp = e & 31, cb = e >> 5;
          const uint32_t a4[4] = {nxt[2 * k].x, nxt[2 * k].y, nxt[2 * k].z, nxt[2 * k].w};
          const uint32_t b4[4] = {nxt[2 * k + 1].x, nxt[2 * k + 1].y, nxt[2 * k + 1].z, nxt[2 * k + 1].w};
          uint32_t* col = tileT + (NE * cb) * KT_PITCH + tp;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            col[(2 * q) * KT_PITCH] = __builtin_amdgcn_perm(b4[q], a4[q], 0x05040100u);      // channel 2q
            col[(2 * q + 1) * KT_PITCH] = __builtin_amdgcn_perm(b4[q], a4[q], 0x07060302u);  // channel 2q+1
          }
        }
      }
      if (ti + (int)gridDim.x < ntiles) fetch(ti + gridDim.x);  // lands while this tile is quantized
    } else if constexpr (VEC) {
#pragma unroll
      for (int k = 0; k < KEY_MAX_VEC; ++k) {
        const int e = threadIdx.x + k * QWG;
        if (e < nvec) {
          const int t = e / vpr, c = (e - t * vpr) * NE;
          if constexpr (DT == MZ_F32) {
            vec16_store_lds<DT>(tile + t * ld + c, nxt[k]);
          } else {
            uint32_t* d32 = (uint32_t*)(tile + t * ld + c);  // 4-byte aligned: ld and c are even
            d32[0] = nxt[k].x, d32[1] = nxt[k].y, d32[2] = nxt[k].z, d32[3] = nxt[k].w;
          }
        }
      }
      if (ti + (int)gridDim.x < ntiles) fetch(ti + gridDim.x);  // lands while this tile is quantized
    } else {
      const int64_t base = tile_base(ti);
      for (int e = threadIdx.x; e < 64 * D; e += QWG) {
        const int t = e / D, c = e - t * D;
        if constexpr (DT == MZ_F32) tile[t * ld + c] = load_val<DT>(x, base + t * st + c);
        else tile[t * ld + c] = ((const uint16_t*)x)[base + t * st + c];
      }
    }
    __syncthreads();
    uint8_t* gbase = packed + b * psb + h * psh + (int64_t)s * D * QB;
    const int64_t mbase = b * msb + h * msh + (int64_t)s * D;
    constexpr int N = QN_KEYS, L = 64 / N;  // values per lane, lanes per group (one column)
    for (int c0 = (64 / L) * wave; c0 < D; c0 += (64 / L) * (QWG / 64)) {
      const int c = c0 + lane / L;
      if (c < D) {  // a group's lanes share c
        uint8_t* prow = gbase + (int64_t)c * QB;
        if constexpr (DT != MZ_F32) {
          static_assert(N == 32, "a lane takes 16 token-pair dwords");
          uint32_t w[16];
          if constexpr (TRANS) {
            const uint4* src = (const uint4*)(tileT + c * KT_PITCH + 16 * part);
#pragma unroll
            for (int m4 = 0; m4 < 4; ++m4) {
              const uint4 u = src[m4];
              w[4 * m4] = u.x, w[4 * m4 + 1] = u.y, w[4 * m4 + 2] = u.z, w[4 * m4 + 3] = u.w;
            }
          } else {
            const ET* col = tile + (N * part) * ld + c;
#pragma unroll
            for (int k = 0; k < 16; ++k) w[k] = (uint32_t)col[(2 * k) * ld] | (uint32_t)col[(2 * k + 1) * ld] << 16;
          }
          quantize_lane16<DT, BITS>(w, part, prow, mn, sc, mbase + c, meta_dtype, eps, lds, table);
        } else {
          float v[N];
#pragma unroll
          for (int k = 0; k < N; ++k) v[k] = tile[(N * part + k) * ld + c];
          quantize_lane<DT, BITS, N>(v, part, prow, mn, sc, mbase + c, meta_dtype, eps, lds, table);
        }
      }
    }
  }
}

// ------------------------------------------------------------- dispatch
#define MZ_BITS_SWITCH(BITS, ...)                      \
  switch (BITS) {                                      \
    case 1: { constexpr int B_ = 1; __VA_ARGS__; } break; \
    case 2: { constexpr int B_ = 2; __VA_ARGS__; } break; \
    case 3: { constexpr int B_ = 3; __VA_ARGS__; } break; \
    case 4: { constexpr int B_ = 4; __VA_ARGS__; } break; \
    case 5: { constexpr int B_ = 5; __VA_ARGS__; } break; \
    case 6: { constexpr int B_ = 6; __VA_ARGS__; } break; \
    case 7: { constexpr int B_ = 7; __VA_ARGS__; } break; \
    case 8: { constexpr int B_ = 8; __VA_ARGS__; } break; \
    default: return MZ_EINVAL;                         \
  }

#define MZ_DT_SWITCH(DTV, ...)                                   \
  switch (DTV) {                                                 \
    case MZ_F32: { constexpr int D_ = MZ_F32; __VA_ARGS__; } break;   \
    case MZ_BF16: { constexpr int D_ = MZ_BF16; __VA_ARGS__; } break; \
    case MZ_F16: { constexpr int D_ = MZ_F16; __VA_ARGS__; } break;   \
    default: return MZ_EINVAL;                                   \
  }

static inline bool dtype_ok(int dt) { return dt == MZ_F32 || dt == MZ_BF16 || dt == MZ_F16; }

static inline int launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? MZ_OK : (int)e;
}

}  // namespace mz

using namespace mz;


// Persistent grid: enough workgroups to fill the GPU a few times over, each
// looping over its share of the 64-value groups (table staged once).
static int quantize_grid(int64_t work_groups, int groups_per_wave) {
  const int64_t per_wg = (int64_t)(QWG / 64) * groups_per_wave;
  const int64_t need = (work_groups + per_wg - 1) / per_wg;
  return (int)std::max<int64_t>(1, std::min<int64_t>(need, (int64_t)device_cu_count() * 8));
}

// Alignment the packed rows need: a lane stores its `bits` bytes as one
// 2/4/8-byte word when bits is 2/4/8, byte by byte otherwise.
static int packed_align(int bits) { return (bits == 2 || bits == 4 || bits == 8) ? bits : 1; }

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
static int64_t dtype_size(int dt) { return dt == MZ_F32 ? 4 : 2; }

extern "C" int muzero_quantize_rows(const void* x, int x_dtype, int64_t nrows, int64_t x_row_stride,
                                    uint8_t* packed, int64_t packed_row_stride, void* mn, void* scale,
                                    int meta_dtype, int64_t meta_stride, int bits, float eps, const void* table,
                                    mz_stream_t stream) {
  if (nrows < 0 || !dtype_ok(x_dtype) || !dtype_ok(meta_dtype) || bits < 1 || bits > 8) return MZ_EINVAL;
  if (nrows == 0) return MZ_OK;
  if (!x || !packed || !mn || !scale || !table) return MZ_EINVAL;
  if (x_row_stride < 64 || packed_row_stride < 8 * bits || meta_stride < 1) return MZ_EINVAL;
  // packed bytes are stored 1/2/4/8 at a time at offsets part*bits: rows must keep that alignment
  if (((uintptr_t)packed | (uintptr_t)packed_row_stride) % packed_align(bits) != 0) return MZ_EINVAL;
  const bool vec = aligned16(x) && x_row_stride % 8 == 0;
  const dim3 grid((unsigned)quantize_grid(nrows, QN_ROWS));
  hipStream_t s = (hipStream_t)stream;
  MZ_DT_SWITCH(x_dtype, MZ_BITS_SWITCH(bits,
      if (vec) hipLaunchKernelGGL((quantize_rows_kernel<D_, B_, true>), grid, dim3(QWG), 0, s, x, nrows,
                                  x_row_stride, packed, packed_row_stride, mn, scale, meta_dtype, meta_stride, eps,
                                  table);
      else hipLaunchKernelGGL((quantize_rows_kernel<D_, B_, false>), grid, dim3(QWG), 0, s, x, nrows,
                              x_row_stride, packed, packed_row_stride, mn, scale, meta_dtype, meta_stride, eps,
                              table)));
  return launch_status();
}

static int check_block(const void* x, int x_dtype, int B, int H, int T, int D, const uint8_t* packed,
                       const void* mn, const void* scale, int meta_dtype, int bits, const void* table) {
  if (!dtype_ok(x_dtype) || !dtype_ok(meta_dtype) || bits < 1 || bits > 8) return MZ_EINVAL;
  if (B < 0 || H < 0 || T < 0 || D <= 0) return MZ_EINVAL;
  if ((int64_t)B * H * T == 0) return 1;  // nothing to do
  if (!x || !packed || !mn || !scale || !table) return MZ_EINVAL;
  return MZ_OK;
}

extern "C" int muzero_quantize_keys(const void* keys, int x_dtype, int B, int H, int T, int D, int64_t x_sb,
                                    int64_t x_sh, int64_t x_st, uint8_t* packed, int64_t p_sb, int64_t p_sh,
                                    void* mn, void* scale, int meta_dtype, int64_t m_sb, int64_t m_sh, int bits,
                                    float eps, const void* table, mz_stream_t stream) {
  int st = check_block(keys, x_dtype, B, H, T, D, packed, mn, scale, meta_dtype, bits, table);
  if (st == 1) return MZ_OK;
  if (st) return st;
  if (T % 64) return MZ_EINVAL;
  if (((uintptr_t)packed | (uintptr_t)p_sb | (uintptr_t)p_sh) % packed_align(bits) != 0) return MZ_EINVAL;
  const int64_t ntiles = (int64_t)B * H * (T / 64);
  if (ntiles >= (int64_t)1 << 31) return MZ_EINVAL;
  const size_t es = x_dtype == MZ_F32 ? 4 : 2;
  // the vector path stages a whole tile in KEY_MAX_VEC 16-byte loads per thread
  const bool vec = aligned16(keys) && D % 8 == 0 && (int64_t)64 * D * (int64_t)es <= (int64_t)KEY_MAX_VEC * QWG * 16 &&
                   (x_sb * es) % 16 == 0 && (x_sh * es) % 16 == 0 && (x_st * es) % 16 == 0;
  hipStream_t s = (hipStream_t)stream;
  MZ_DT_SWITCH(x_dtype, MZ_BITS_SWITCH(bits,
      const size_t lds = (size_t)QTable<D_, B_>::LDS_BYTES +
                         (vec && D_ != MZ_F32 ? KeyTrans<D_, true>::bytes(D)
                                              : (size_t)64 * (D + KeyStage<D_>::PAD) * sizeof(typename KeyStage<D_>::T));
      if (lds > 160 * 1024) return MZ_EUNSUPPORTED;
      const void* fn = vec ? (const void*)quantize_keys_kernel<D_, B_, true> : (const void*)quantize_keys_kernel<D_, B_, false>;
      if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
      }
      const int per_cu = std::max<int>(1, std::min<int>(4, (int)((160 * 1024) / lds)));
      const dim3 grid((unsigned)std::max<int64_t>(1, std::min<int64_t>(ntiles, per_cu * (int64_t)device_cu_count())));
      if (vec) hipLaunchKernelGGL((quantize_keys_kernel<D_, B_, true>), grid, dim3(QWG), lds, s, keys, B, H, T, D,
                                  x_sb, x_sh, x_st, packed, p_sb, p_sh, mn, scale, meta_dtype, m_sb, m_sh, eps, table);
      else hipLaunchKernelGGL((quantize_keys_kernel<D_, B_, false>), grid, dim3(QWG), lds, s, keys, B, H, T, D,
                              x_sb, x_sh, x_st, packed, p_sb, p_sh, mn, scale, meta_dtype, m_sb, m_sh, eps, table)));
  return launch_status();
}

extern "C" int muzero_quantize_values(const void* values, int x_dtype, int B, int H, int T, int D, int64_t x_sb,
                                      int64_t x_sh, int64_t x_st, uint8_t* packed, int64_t p_sb, int64_t p_sh,
                                      void* mn, void* scale, int meta_dtype, int64_t m_sb, int64_t m_sh, int bits,
                                      float eps, const void* table, mz_stream_t stream) {
  int st = check_block(values, x_dtype, B, H, T, D, packed, mn, scale, meta_dtype, bits, table);
  if (st == 1) return MZ_OK;
  if (st) return st;
  if (((uintptr_t)packed | (uintptr_t)p_sb | (uintptr_t)p_sh) % packed_align(bits) != 0) return MZ_EINVAL;
  const int ng = (D + 63) / 64;
  const int64_t rows_per_b = (int64_t)H * T * ng;
  if (rows_per_b >= (int64_t)1 << 31) return MZ_EINVAL;
  const size_t es = x_dtype == MZ_F32 ? 4 : 2;
  const bool vec = aligned16(values) && D % 8 == 0 && (x_sb * es) % 16 == 0 && (x_sh * es) % 16 == 0 &&
                   (x_st * es) % 16 == 0;
  const FastDiv fng = make_fastdiv((uint32_t)ng), fT = make_fastdiv((uint32_t)T), fH = make_fastdiv((uint32_t)H);
  // offsets within one (b, h) slice in 32-bit arithmetic when they all fit
  const bool narrow = x_st >= 0 && (int64_t)(T - 1) * x_st + D < ((int64_t)1 << 31) &&
                      (int64_t)T * ng * 8 * bits < ((int64_t)1 << 31);
  hipStream_t s = (hipStream_t)stream;
  // row numbers stay below 2^31 per launch: batches go in slices of bstep
  const int bstep = (int)std::min<int64_t>(B, (((int64_t)1 << 31) - 1) / rows_per_b);
  for (int b0 = 0; b0 < B; b0 += bstep) {
    const int nb = std::min(bstep, B - b0);
    const int nrows = (int)(nb * rows_per_b);
    const void* xs = (const char*)values + b0 * x_sb * (int64_t)es;
    uint8_t* ps = packed + b0 * p_sb;
    void* mns = (char*)mn + b0 * m_sb * (int64_t)dtype_size(meta_dtype);
    void* scs = (char*)scale + b0 * m_sb * (int64_t)dtype_size(meta_dtype);
    const dim3 grid((unsigned)quantize_grid(nrows, QN_ROWS));
#define MZ_QV(VECV, NARV)                                                                                     \
  hipLaunchKernelGGL((quantize_values_kernel<D_, B_, VECV, NARV>), grid, dim3(QWG), 0, s, xs, nrows, fng, fT, fH, D, \
                     x_sb, x_sh, x_st, ps, p_sb, p_sh, mns, scs, meta_dtype, m_sb, m_sh, eps, table)
    MZ_DT_SWITCH(x_dtype, MZ_BITS_SWITCH(bits,
        if (vec && narrow) MZ_QV(true, true);
        else if (vec) MZ_QV(true, false);
        else if (narrow) MZ_QV(false, true);
        else MZ_QV(false, false)));
#undef MZ_QV
    const int st2 = launch_status();
    if (st2 != MZ_OK) return st2;
  }
  return MZ_OK;
}

extern "C" const char* muzero_version(void) { return "muzero_hip 0.1.0 gfx950"; }

extern "C" const char* muzero_strerror(int status) {
  switch (status) {
    case MZ_OK: return "ok";
    case MZ_EINVAL: return "invalid argument (pointer, size, stride, dtype or bit width)";
    case MZ_EUNSUPPORTED: return "shape not supported by the HIP path";
    case MZ_EWORKSPACE: return "workspace too small";
    case MZ_ESCRATCH: return "the call needs more than the static decode scratch (MZ_DECODE_SCRATCH_BYTES = 8 MiB)";
    default: return status > 0 ? hipGetErrorString((hipError_t)status) : "unknown error";
  }
}
