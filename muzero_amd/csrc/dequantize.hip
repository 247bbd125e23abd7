// Dequantize kernels (gfx950, wave64): packed groups back to dense K / V.
//
// Two walks over the same codec, both writing [B, H, T, D] rows directly:
//   keys:   a group is one channel's 64 tokens.  A lane owns a pair of adjacent
//           channels (one channel for fp32 outputs), so each token's 64 lanes
//           store one dword each, consecutive in the token's row: no transpose
//           through LDS, no permute copy (the reference dequantizes rows and
//           permutes them, muzero/cache/layer.py:303-345).
//   values: a group is 64 channels of one token (and the flat rows of
//           muzero_dequantize_rows are the same walk with one slice).  A lane
//           owns a group; its values cross the wave through a swizzled LDS
//           block so that 4 lanes store 64 consecutive bytes.
// A lane forms its groups' parameters (one IEEE division each) once per 64
// codes.  Up to 4 bits it then forms the 2^bits values of each group, rounded
// to the output type, into its own LDS column (entry q at q*256 + 4*lane: every
// read of a wave meets 64 distinct banks' dwords whatever the codes) and a code costs one
// address, one LDS read and half a merge; wider codes are formed one by one
// from the expm1 rows in LDS (128 KB at 8 bits: one workgroup of 16 waves per
// CU, the others' 4).  Every value is the reference's fp32 value
// (muzero/quantizer.py:229-255 op for op) rounded once to the output type.
//
// Bound: HBM (4-bit, bf16: 0.56 bytes read and 2 written per value); VALU close
// behind it (10 instructions per value at 4 bits).  A layer's whole dense read
// at B = 16, 4096 tokens, 8 heads of 128, 4-bit: 1004 us as row dequantization
// (one code per lane), permute and concatenation, 105 us here (3.3 TB/s of the
// 350 MB it must move; a large copy reaches 5.1 TB/s).
#include "decode_common.hpp"

#include <algorithm>
#include <atomic>

namespace mz {
namespace deq {

template <int BITS>
struct Cfg {
  static constexpr int QMAX = (1 << BITS) - 1;
  static constexpr int QB = 8 * BITS;                      // bytes per packed group
  static constexpr bool CB = BITS <= 4;                    // codebooks
  static constexpr int WAVES = BITS == 8 ? 16 : 4;         // per workgroup
  static constexpr bool STAGE = BITS < 8;                  // values: coalesced stores through LDS (no room at 8 bits)
  static constexpr int EF = QMAX * (QMAX + 3) / 2;         // expm1 rows of bins 1..QMAX
  static constexpr int EBYTES = (EF * 4 + 15) / 16 * 16;
  static constexpr int CB_BYTES = CB ? (1 << BITS) * 256 : 0;  // one wave's codebooks
  static constexpr int STAGE_BYTES = 64 * 64;                  // one wave's staging: 64 rows x 64 bytes
  static constexpr int key_lds() { return EBYTES + WAVES * CB_BYTES; }
  static constexpr int value_lds() { return EBYTES + WAVES * (CB_BYTES + (STAGE ? STAGE_BYTES : 0)); }
};

// (a call with only tail tokens has no table)
template <int BITS>
__device__ __forceinline__ void stage_e(float* lds, const float* __restrict__ e, int64_t waves) {
  if (waves == 0) return;
  for (int i = threadIdx.x; i < Cfg<BITS>::EF; i += Cfg<BITS>::WAVES * 64) lds[i] = e[i];
  __syncthreads();
}

template <int OT>
__device__ __forceinline__ uint32_t out_bits(float x) {
  if constexpr (OT == MZ_F32) return __float_as_uint(x);
  else if constexpr (OT == MZ_BF16) return f2bf(x);
  else return f2h(x);
}

// N bytes at p (any alignment) as dwords, zero beyond.
template <int N>
__device__ __forceinline__ void load_bytes(uint32_t (&w)[(N + 3) / 4], const uint8_t* p) {
  w[(N + 3) / 4 - 1] = 0;
  __builtin_memcpy(w, p, N);
}

// Code i of a group (i a constant after unrolling).
template <int BITS, int NW>
__device__ __forceinline__ uint32_t code_at(const uint32_t (&w)[NW], int i) {
  const int bit = i * BITS, k = bit >> 5, sh = bit & 31;
  if (sh + BITS <= 32) return (w[k] >> sh) & Cfg<BITS>::QMAX;
  return __builtin_amdgcn_alignbit(w[k + 1 < NW ? k + 1 : k], w[k], sh) & Cfg<BITS>::QMAX;
}

struct Args {
  const uint8_t* packed;
  const void* mn;
  const void* sc;
  void* out;
  const float* e;
  const void* tail;  // dense rows that follow the dequantized ones, copied (or null)
  int64_t psb, psh, pst, msb, msh, mst, osb, osh, ost, tsb, tsh, tst;
  int mdt, H, D, ng;
  int units;      // keys: 64-token groups; values: rows (T * ng), per (b, h)
  int per_slice;  // waves per (b, h) slice
  int ntail, tail_at;          // tail tokens, and the output token the first goes to
  int tail_vec;                // the tail is copied 16 bytes at a time
  int64_t waves, tail_waves;   // dequantizing waves, then copying waves
};

// ----------------------------------------------------------------- the tail
// Copy 16 tail tokens of one (b, h).
constexpr int TAIL_TOKENS = 16;
template <int OT>
__device__ __forceinline__ void copy_tail(const Args& a, int64_t w) {
  const int lane = threadIdx.x & 63;
  const int per = (a.ntail + TAIL_TOKENS - 1) / TAIL_TOKENS;
  const int64_t slice = w / per;
  const int t0 = (int)(w - slice * per) * TAIL_TOKENS, n = min(TAIL_TOKENS, a.ntail - t0);
  const int64_t b = slice / a.H, h = slice - b * a.H;
  constexpr int ES = OT == MZ_F32 ? 4 : 2;
  const char* src = (const char*)a.tail + (b * a.tsb + h * a.tsh + (int64_t)t0 * a.tst) * ES;
  char* dst = (char*)a.out + (b * a.osb + h * a.osh + (int64_t)(a.tail_at + t0) * a.ost) * ES;
  const int per_row = a.tail_vec ? a.D * ES / 16 : a.D;
  for (int i = lane; i < n * per_row; i += 64) {
    const int t = i / per_row, c = i - t * per_row;
    const char* s = src + (int64_t)t * a.tst * ES;
    char* d = dst + (int64_t)t * a.ost * ES;
    if (a.tail_vec) ((uint4*)d)[c] = ((const uint4*)s)[c];
    else if constexpr (OT == MZ_F32) ((uint32_t*)d)[c] = ((const uint32_t*)s)[c];
    else ((uint16_t*)d)[c] = ((const uint16_t*)s)[c];
  }
}

// ----------------------------------------------------------------- keys
// Wave = (slice, group, token part, column block): up to 64 column units of
// one group, TOK tokens each; `ls` = 2 gives lanes 32..63 the next TOK tokens
// of units 0..31 (at most 32 units: head_dim 64 in 16 bits).  TOK 16 splits a
// group over more waves where whole groups leave the chip idle.
// VEC: pairs are stored as dwords (even D, 4-byte aligned rows).
template <int BITS, int OT, int TOK, bool VEC>
__global__ __launch_bounds__(Cfg<BITS>::WAVES * 64) void keys_kernel(const Args a, int ls, int ncb) {
  using C = Cfg<BITS>;
  extern __shared__ __align__(16) uint8_t lds[];
  float* E = (float*)lds;
  stage_e<BITS>(E, a.e, a.waves);
  constexpr int W = OT == MZ_F32 ? 1 : 2;   // channels per lane
  constexpr int RB = TOK * BITS / 8;        // bytes of a row's TOK codes
  constexpr int NW = (RB + 3) / 4;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t* cb = (uint32_t*)(lds + C::EBYTES + wv * C::CB_BYTES) + lane;
  const int parts = 64 / TOK / ls;
  for (int64_t w = (int64_t)blockIdx.x * C::WAVES + wv; w < a.waves + a.tail_waves; w += (int64_t)gridDim.x * C::WAVES) {
    if (w >= a.waves) {
      copy_tail<OT>(a, w - a.waves);
      continue;
    }
    const int64_t slice = w / a.per_slice;
    int r = (int)(w - slice * a.per_slice);
    const int cblk = r % ncb;
    r /= ncb;
    const int part = r % parts, g = r / parts;
    const int64_t b = slice / a.H, h = slice - b * a.H;
    const int unit = ls == 2 ? (lane & 31) : 64 * cblk + lane;
    const int t0 = TOK * (ls == 2 ? 2 * part + (lane >> 5) : part);
    const int c0 = W * unit;
    if (c0 < a.D) {
      const bool two = W == 2 && c0 + 1 < a.D;
      const uint8_t* rows = a.packed + b * a.psb + h * a.psh + (int64_t)g * a.D * C::QB + t0 * BITS / 8;
      const int64_t m0 = b * a.msb + h * a.msh + (int64_t)g * a.D + c0;
      uint32_t q[W][NW];
      DeqGroup gr[W];
#pragma unroll
      for (int k = 0; k < W; ++k) {
        const int step = k == 0 || two ? k : 0;  // (odd D: the last lane's second channel repeats the first)
        load_bytes<RB>(q[k], rows + (int64_t)(c0 + step) * C::QB);
        gr[k] = make_group<C::QMAX>(load_any(a.mn, m0 + step, a.mdt), load_any(a.sc, m0 + step, a.mdt));
      }
      if constexpr (C::CB) {
#pragma unroll
        for (int v = 0; v <= C::QMAX; ++v) {
          uint32_t x = out_bits<OT>(group_value(gr[0], v, E));
          if constexpr (W == 2) x |= out_bits<OT>(group_value(gr[W - 1], v, E)) << 16;
          cb[64 * v] = x;
        }
      }
      constexpr int ES = OT == MZ_F32 ? 4 : 2;
      // a scalar base that steps through the tokens and a 32-bit lane offset (host check)
      char* obase = (char*)a.out + (b * a.osb + h * a.osh + (int64_t)(64 * g) * a.ost) * ES;
      const uint32_t ooff = (uint32_t)(t0 * (int)a.ost + c0) * ES;
#pragma unroll
      for (int i = 0; i < TOK; ++i) {
        uint32_t x;
        if constexpr (C::CB) {
          x = cb[64 * code_at<BITS>(q[0], i)];
          if constexpr (W == 2) x = (x & 0xFFFFu) | (cb[64 * code_at<BITS>(q[W - 1], i)] & 0xFFFF0000u);
        } else {
          x = out_bits<OT>(group_value(gr[0], (int)code_at<BITS>(q[0], i), E));
          if constexpr (W == 2) x |= out_bits<OT>(group_value(gr[W - 1], (int)code_at<BITS>(q[W - 1], i), E)) << 16;
        }
        char* o = obase + ooff;
        if constexpr (W == 1 || VEC) {
          *(uint32_t*)o = x;
        } else {
          ((uint16_t*)o)[0] = (uint16_t)x;
          if (two) ((uint16_t*)o)[1] = (uint16_t)(x >> 16);
        }
        obase += a.ost * ES;
      }
    }
  }
}

// ----------------------------------------------------------------- values
// Wave = 64 consecutive rows of one (b, h) slice, one per lane.  `half`s of 64
// output bytes are staged in turn: lane r writes its 16-byte chunk k at slot
// k ^ (r/2 & 3) of row r, and lane l then stores chunk l % 4 of rows
// l/4 + 16i, so 8 lanes served together meet 8 different 16-byte bank slots
// both ways.  VEC: 16-byte stores (D % 8 == 0 in 16 bits, % 4 in fp32, aligned rows).
template <int BITS, int OT, bool VEC>
__global__ __launch_bounds__(Cfg<BITS>::WAVES * 64) void values_kernel(const Args a) {
  using C = Cfg<BITS>;
  extern __shared__ __align__(16) uint8_t lds[];
  float* E = (float*)lds;
  stage_e<BITS>(E, a.e, a.waves);
  constexpr int ES = OT == MZ_F32 ? 4 : 2;
  constexpr int VPC = 16 / ES;            // values per 16-byte chunk
  constexpr int HALF = 64 / ES;           // values per staged half
  constexpr int NW = C::QB / 4;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint8_t* area = lds + C::EBYTES + wv * (C::CB_BYTES + (C::STAGE ? C::STAGE_BYTES : 0));
  uint32_t* cb = (uint32_t*)area + lane;
  uint4* stage = (uint4*)(area + C::CB_BYTES);
  for (int64_t w = (int64_t)blockIdx.x * C::WAVES + wv; w < a.waves + a.tail_waves; w += (int64_t)gridDim.x * C::WAVES) {
    if (w >= a.waves) {
      copy_tail<OT>(a, w - a.waves);
      continue;
    }
    const int64_t slice = w / a.per_slice;
    const int i0 = (int)(w - slice * a.per_slice) * 64;
    const int64_t b = slice / a.H, h = slice - b * a.H;
    const int last = a.units - 1;
    const int row = min(i0 + lane, last);  // (lanes past the slice repeat its last row and store nothing)
    uint32_t q[NW];
    load_bytes<C::QB>(q, a.packed + b * a.psb + h * a.psh + (int64_t)row * a.pst);
    const int64_t m = b * a.msb + h * a.msh + (int64_t)row * a.mst;
    const DeqGroup gr = make_group<C::QMAX>(load_any(a.mn, m, a.mdt), load_any(a.sc, m, a.mdt));
    if constexpr (C::CB) {
#pragma unroll
      for (int v = 0; v <= C::QMAX; ++v) {
        uint32_t x = out_bits<OT>(group_value(gr, v, E));
        if constexpr (OT != MZ_F32) x |= x << 16;
        cb[64 * v] = x;
      }
    }
    auto value = [&](int i) __attribute__((always_inline)) -> uint32_t {
      if constexpr (C::CB) return cb[64 * code_at<BITS>(q, i)];
      else return out_bits<OT>(group_value(gr, (int)code_at<BITS>(q, i), E));
    };
    auto chunk = [&](int c) __attribute__((always_inline)) -> uint4 {  // 16 output bytes: values VPC*c ..
      uint32_t x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if constexpr (OT == MZ_F32) x[k] = value(VPC * c + k);
        else if constexpr (C::CB) x[k] = (value(VPC * c + 2 * k) & 0xFFFFu) | (value(VPC * c + 2 * k + 1) & 0xFFFF0000u);
        else x[k] = value(VPC * c + 2 * k) | (value(VPC * c + 2 * k + 1) << 16);
      }
      return make_uint4(x[0], x[1], x[2], x[3]);
    };
    char* obase = (char*)a.out + (b * a.osb + h * a.osh) * ES;
    // store the 16 bytes of row rr whose first value is v0
    auto put = [&](int rr, int v0, const uint4 x) __attribute__((always_inline)) {
      if (rr > last) return;
      const int t = rr / a.ng, j = rr - t * a.ng;
      const int left = a.D - 64 * j - v0;
      char* o = obase + ((int64_t)t * a.ost + 64 * j + v0) * ES;
      if constexpr (VEC) {
        if (left > 0) *(uint4*)o = x;
      } else {
        const uint32_t u[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int k = 0; k < VPC; ++k)
          if (k < left) {
            if constexpr (OT == MZ_F32) ((uint32_t*)o)[k] = u[k];
            else ((uint16_t*)o)[k] = (uint16_t)(u[k / 2] >> (16 * (k & 1)));
          }
      }
    };
#pragma unroll
    for (int hf = 0; hf < 64 / HALF; ++hf) {
      if constexpr (C::STAGE) {
#pragma unroll
        for (int k = 0; k < 4; ++k) stage[4 * lane + (k ^ ((lane >> 1) & 3))] = chunk(4 * hf + k);
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * i + (lane >> 2), k = lane & 3;
          put(i0 + r, HALF * hf + VPC * k, stage[4 * r + (k ^ ((r >> 1) & 3))]);
        }
        wave_lds_sync();
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) put(i0 + lane, HALF * hf + VPC * k, chunk(4 * hf + k));
      }
    }
  }
}

// ----------------------------------------------------------------- host
inline bool dt_ok(int dt) { return dt == MZ_F32 || dt == MZ_BF16 || dt == MZ_F16; }
inline int64_t dt_size(int dt) { return dt == MZ_F32 ? 4 : 2; }
// whether `n`-byte accesses fit a [B, H, T, D] tensor's rows
inline bool rows_aligned(const void* p, int64_t sb, int64_t sh, int64_t st, int64_t es, int n) {
  return (((uintptr_t)p | (uintptr_t)(sb * es) | (uintptr_t)(sh * es) | (uintptr_t)(st * es)) & (uintptr_t)(n - 1)) == 0;
}

inline bool tail_vec(const Args& a, int64_t es) {
  return a.D * es % 16 == 0 && rows_aligned(a.out, a.osb, a.osh, a.ost, es, 16) &&
         rows_aligned(a.tail, a.tsb, a.tsh, a.tst, es, 16);
}

template <int BITS>
int64_t grid_for(int64_t waves, int lds_bytes) {
  const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(32 / Cfg<BITS>::WAVES, (160 * 1024) / std::max(lds_bytes, 1)));
  return std::max<int64_t>(1, std::min<int64_t>((waves + Cfg<BITS>::WAVES - 1) / Cfg<BITS>::WAVES, per_cu * device_cu_count()));
}

template <int BITS, int OT, int TOK, bool VEC>
int run_keys(const Args& a, int ls, int ncb, hipStream_t s) {
  static std::atomic<uint64_t> raised{0};
  using C = Cfg<BITS>;
  constexpr int lds = C::key_lds();
  if constexpr (lds > 64 * 1024) {
    const hipError_t e = set_dynamic_lds((const void*)keys_kernel<BITS, OT, TOK, VEC>, lds, raised);
    if (e != hipSuccess) return (int)e;
  }
  const int64_t grid = grid_for<BITS>(a.waves + a.tail_waves, lds);
  keys_kernel<BITS, OT, TOK, VEC><<<dim3((unsigned)grid), dim3(C::WAVES * 64), lds, s>>>(a, ls, ncb);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? MZ_OK : (int)e;
}

template <int BITS, int OT>
int keys_of(Args& a, int64_t slices, hipStream_t s) {
  constexpr int W = OT == MZ_F32 ? 1 : 2;
  const int64_t es = dt_size(OT);
  const int nc = (a.D + W - 1) / W;
  const int ls = nc <= 32 ? 2 : 1, ncb = ls == 2 ? 1 : (nc + 63) / 64;
  const bool vec = OT == MZ_F32 || (a.D % 2 == 0 && rows_aligned(a.out, a.osb, a.osh, a.ost, es, 4));
  // whole groups per lane (or half groups with two halves of the wave) unless
  // that leaves the chip's SIMDs without two waves each
  const bool small = slices * a.units * ncb < (int64_t)device_cu_count() * 8;
  const int tok = small ? 16 : ls == 2 ? 32 : 64;
  const int64_t per = (int64_t)a.units * ncb * (64 / tok / ls);
  if (per >= (int64_t)1 << 31) return MZ_EINVAL;
  a.per_slice = (int)per;
  a.waves = slices * per;
  a.tail_vec = tail_vec(a, es);
  a.tail_waves = slices * ((a.ntail + TAIL_TOKENS - 1) / TAIL_TOKENS);
  if (a.waves + a.tail_waves == 0) return MZ_OK;
#define MZ_DK(TOKV) \
  return vec ? run_keys<BITS, OT, TOKV, true>(a, ls, ncb, s) : run_keys<BITS, OT, TOKV, false>(a, ls, ncb, s)
  if (tok == 16) MZ_DK(16);
  if (tok == 32) MZ_DK(32);
  MZ_DK(64);
#undef MZ_DK
}

template <int BITS, int OT, bool VEC>
int run_values(const Args& a, hipStream_t s) {
  static std::atomic<uint64_t> raised{0};
  using C = Cfg<BITS>;
  constexpr int lds = C::value_lds();
  if constexpr (lds > 64 * 1024) {
    const hipError_t e = set_dynamic_lds((const void*)values_kernel<BITS, OT, VEC>, lds, raised);
    if (e != hipSuccess) return (int)e;
  }
  const int64_t grid = grid_for<BITS>(a.waves + a.tail_waves, lds);
  values_kernel<BITS, OT, VEC><<<dim3((unsigned)grid), dim3(C::WAVES * 64), lds, s>>>(a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? MZ_OK : (int)e;
}

template <int BITS, int OT>
int values_of(Args& a, int64_t slices, hipStream_t s) {
  const int64_t es = dt_size(OT);
  const bool vec = a.D * es % 16 == 0 && rows_aligned(a.out, a.osb, a.osh, a.ost, es, 16);
  a.per_slice = (int)(((int64_t)a.units + 63) / 64);
  a.waves = slices * a.per_slice;
  a.tail_vec = tail_vec(a, es);
  a.tail_waves = slices * ((a.ntail + TAIL_TOKENS - 1) / TAIL_TOKENS);
  if (a.waves + a.tail_waves == 0) return MZ_OK;
  return vec ? run_values<BITS, OT, true>(a, s) : run_values<BITS, OT, false>(a, s);
}

template <bool KEYS>
int dispatch(Args& a, int64_t slices, int bits, int ot, hipStream_t s) {
#define MZ_DQ(BV, OV) return KEYS ? keys_of<BV, OV>(a, slices, s) : values_of<BV, OV>(a, slices, s)
#define MZ_DQ_BITS(BV)                            \
  case BV:                                        \
    if (ot == MZ_F32) MZ_DQ(BV, MZ_F32);          \
    if (ot == MZ_BF16) MZ_DQ(BV, MZ_BF16);        \
    MZ_DQ(BV, MZ_F16);
  switch (bits) {
    MZ_DQ_BITS(1)
    MZ_DQ_BITS(2)
    MZ_DQ_BITS(3)
    MZ_DQ_BITS(4)
    MZ_DQ_BITS(5)
    MZ_DQ_BITS(6)
    MZ_DQ_BITS(7)
    MZ_DQ_BITS(8)
    default: return MZ_EINVAL;
  }
#undef MZ_DQ_BITS
#undef MZ_DQ
}

template <bool KEYS>
int block(const mz_dequant_args* p, mz_stream_t stream) {
  if (!p || !dt_ok(p->meta_dtype) || !dt_ok(p->out_dtype) || p->bits < 1 || p->bits > 8) return MZ_EINVAL;
  if (p->batch < 0 || p->heads < 0 || p->tokens < 0 || p->n_tail < 0 || p->head_dim <= 0) return MZ_EINVAL;
  if (KEYS && p->tokens % 64) return MZ_EINVAL;
  const int64_t slices = (int64_t)p->batch * p->heads;
  if (slices == 0 || (p->tokens == 0 && p->n_tail == 0)) return MZ_OK;
  if (!p->out || (p->tokens > 0 && (!p->packed || !p->mn || !p->scale || !p->e_table)) || (p->n_tail > 0 && !p->tail))
    return MZ_EINVAL;
  if ((int64_t)p->tokens + p->n_tail >= (int64_t)1 << 31) return MZ_EINVAL;
  const int ng = (p->head_dim + 63) / 64;
  // a key group's output offsets are 32-bit
  if (KEYS && (p->o_st < 0 || (64 * p->o_st + p->head_dim) * 4 >= (int64_t)1 << 31)) return MZ_EUNSUPPORTED;
  if (!KEYS && (int64_t)p->tokens * ng >= (int64_t)1 << 31) return MZ_EINVAL;
  Args a{};
  a.packed = p->packed, a.mn = p->mn, a.sc = p->scale, a.out = p->out, a.e = p->e_table, a.tail = p->tail;
  a.psb = p->p_sb, a.psh = p->p_sh, a.pst = 8 * p->bits;
  a.msb = p->m_sb, a.msh = p->m_sh, a.mst = 1;
  a.osb = p->o_sb, a.osh = p->o_sh, a.ost = p->o_st;
  a.tsb = p->t_sb, a.tsh = p->t_sh, a.tst = p->t_st;
  a.mdt = p->meta_dtype, a.H = p->heads, a.D = p->head_dim, a.ng = ng;
  a.units = KEYS ? p->tokens / 64 : p->tokens * ng;
  a.ntail = p->n_tail, a.tail_at = p->tokens;
  return dispatch<KEYS>(a, slices, p->bits, p->out_dtype, (hipStream_t)stream);
}

}  // namespace deq
}  // namespace mz

using namespace mz;

extern "C" int muzero_dequantize_keys(const mz_dequant_args* args, mz_stream_t stream) {
  return deq::block<true>(args, stream);
}

extern "C" int muzero_dequantize_values(const mz_dequant_args* args, mz_stream_t stream) {
  return deq::block<false>(args, stream);
}

extern "C" int muzero_dequantize_rows(const uint8_t* packed, int64_t nrows, int64_t packed_row_stride,
                                      const void* mn, const void* scale, int meta_dtype, int64_t meta_stride,
                                      void* out, int out_dtype, int64_t out_row_stride, int bits,
                                      const float* e_table, mz_stream_t stream) {
  if (nrows < 0 || !deq::dt_ok(meta_dtype) || !deq::dt_ok(out_dtype) || bits < 1 || bits > 8) return MZ_EINVAL;
  if (nrows == 0) return MZ_OK;
  if (!packed || !mn || !scale || !out || !e_table) return MZ_EINVAL;
  if (packed_row_stride < 8 * bits || out_row_stride < 64 || meta_stride < 1) return MZ_EINVAL;
  // rows as one slice of one-group tokens, in pieces whose row numbers fit 32 bits
  const int64_t ms = deq::dt_size(meta_dtype), os = deq::dt_size(out_dtype), most = (int64_t)1 << 30;
  for (int64_t r0 = 0; r0 < nrows; r0 += most) {
    deq::Args a{};
    a.packed = packed + r0 * packed_row_stride;
    a.mn = (const char*)mn + r0 * meta_stride * ms, a.sc = (const char*)scale + r0 * meta_stride * ms;
    a.out = (char*)out + r0 * out_row_stride * os, a.e = e_table;
    a.pst = packed_row_stride, a.mst = meta_stride, a.ost = out_row_stride;
    a.mdt = meta_dtype, a.H = 1, a.D = 64, a.ng = 1;
    a.units = (int)std::min(most, nrows - r0);
    const int st = deq::dispatch<false>(a, 1, bits, out_dtype, (hipStream_t)stream);
    if (st != MZ_OK) return st;
  }
  return MZ_OK;
}
