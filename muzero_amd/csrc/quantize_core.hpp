// The quantizer's arithmetic (gfx950, wave64): group parameters and codes, every
// operation rounded to the input dtype as the reference's torch operations are
// (muzero/quantizer.py:161-186), shared by the quantize kernels (quantize.hip)
// and the round trip (roundtrip.hip).
#pragma once
#include "common.hpp"

namespace mz {

constexpr int QWG = 256;  // threads per quantize workgroup

// Compander parameters of one group (quantizer.py:169-181), every op rounded
// to the input dtype DT.
struct QParams {
  float mn, sc, za, zl, pb, nb, pe, ne, eps;
  float rsc, rpe, rne;  // v_rcp_f32 of sc, pe, ne (16-bit inputs only)
  float ea, ec;         // fp32 inputs: the table's alpha estimate and 1 / log2(1 + ea) (see code_offset_f32)
};

// rnd<DT>(a / b) for a, b values of the 16-bit input dtype, given r = rcp(b).
// bf16: a and b have 8-bit significands, so a / b is never a bf16 rounding
// midpoint and lies at least 2^7 fp32 ulps from one (a = b * odd 9-bit
// significand is impossible; the distance is >= 1/B bf16 half-ulps with the
// odd part B < 2^8); a * rcp(b) is within 3 ulps, so rounding it to bf16 gives
// the reference's round(fp32 division).  fp16 (11-bit significands, distance
// >= 2 ulps) takes one residual correction (< 1 ulp) except where b is 0 or
// inf, where a * rcp(b) is already the IEEE quotient (inf, NaN or 0).  rcp of
// a b above 2^126 would be denormal: such groups use the IEEE division.
template <int DT, bool FAST>
__device__ __forceinline__ float qdiv(float a, float b, float r) {
  if constexpr (DT == MZ_F32 || !FAST) {
    return rnd<DT>(a / b);
  } else if constexpr (DT == MZ_BF16) {
    return rnd<DT>(a * r);
  } else {
    const float q0 = a * r;
    const float q1 = fmaf(fmaf(-b, q0, a), r, q0);
    return rnd<DT>((b != 0.f && b != __builtin_inff()) ? q1 : q0);
  }
}

// Whether the reciprocal form applies to every division of the group.
template <int DT>
__device__ __forceinline__ bool qfast(const struct QParams& g) {
  if constexpr (DT == MZ_F16) return true;  // an fp16 scale is <= 65504 or inf
  return DT != MZ_F32 && !(g.sc > 0x1p126f && g.sc < __builtin_inff());
}

template <int DT, int BITS>
__device__ __forceinline__ QParams qparams(float mn, float mx, float eps_in) {
  constexpr float qmax = (float)((1 << BITS) - 1);
  QParams g;
  g.eps = rnd<DT>(eps_in);
  g.mn = mn;
  g.sc = clamp_min(rnd<DT>(mx - mn), g.eps);
  if constexpr (DT == MZ_BF16) {
    // the reciprocal form of the division (exact for bf16 operands, see
    // qdiv) unless the scale's reciprocal would be denormal; the IEEE
    // division runs only in a wave that holds such a group
    g.rsc = __builtin_amdgcn_rcpf(g.sc);
    const float a = rnd<DT>(0.f - mn);
    float zq = rnd<DT>(a * g.rsc);
    const bool slow = g.sc > 0x1p126f && g.sc < __builtin_inff();
    if (__ballot(slow) != 0) {
      if (slow) zq = rnd<DT>(a / g.sc);
    }
    g.za = clamp01(zq);
  } else {
    g.za = clamp01(rnd<DT>(rnd<DT>(0.f - mn) / g.sc));
  }
  g.zl = rintf(rnd<DT>(g.za * qmax));
  g.pb = clamp_min(rnd<DT>(qmax - g.zl), 1.f);
  g.nb = clamp_min(g.zl, 1.f);
  g.pe = clamp_min(rnd<DT>(1.f - g.za), g.eps);
  g.ne = clamp_min(g.za, g.eps);
  if constexpr (DT != MZ_F32) {
    if constexpr (DT != MZ_BF16) g.rsc = __builtin_amdgcn_rcpf(g.sc);
    g.rpe = __builtin_amdgcn_rcpf(g.pe);
    g.rne = __builtin_amdgcn_rcpf(g.ne);
  }
  return g;
}

// Compander table in LDS: fp32 inputs use the threshold rows of bins 1..qmax
// (#{k : p >= T[bins][k]}, binary search); bf16/fp16 inputs the 16-bit ratio
// table indexed by the pattern of p.  Table bytes staged per workgroup:
template <int DT, int BITS>
struct QTable {
  static constexpr int QMAX = (1 << BITS) - 1;
  static constexpr int BYTES = DT == MZ_F32 ? QMAX * (QMAX + 1) / 2 * 4
                                            : ((DT == MZ_BF16 ? 0x3F80 : 0x3C00) + 1) * 2;
  static constexpr bool IN_LDS = BYTES <= 40 * 1024;  // 8-bit fp32 thresholds (128 KB) stay in global memory
  static constexpr int LDS_BYTES = IN_LDS ? (BYTES + 15) / 16 * 16 : 16;
};

template <int DT, int BITS>
__device__ __forceinline__ void stage_table(uint8_t* lds, const void* table) {
  using TB = QTable<DT, BITS>;
  if constexpr (TB::IN_LDS) {
    const uint16_t* src = (const uint16_t*)table;
    for (int i = threadIdx.x; i < TB::BYTES / 2; i += QWG) ((uint16_t*)lds)[i] = src[i];
    __syncthreads();
  }
}

// fp32 inputs: the code offset #{k in 1..bins : row[k-1] <= p} of a
// normalised distance p over the threshold row of `bins` (monotone: the
// offset is the reference's round(log1p(alpha*p) / lb * bins), tables.py).
// An estimate from the hardware log2 (bins * log2(1 + ea*p) * ec, ea the
// alpha the row of bins 1 implies) is within one of it; four independent
// reads of the thresholds around it give the count, and two of them check
// that the estimate's window [k0, k0 + 2] holds it (every threshold up to
// k0 at or below p, the one after k0 + 2 above).  Where the check fails the
// binary search runs, so the result is exact whatever the estimate.  Used
// from 5 bits (rows of up to 31 .. 255 thresholds: 5 to 8 dependent reads
// of the binary search); 8-bit keys / values 1.65x / 2.3x faster.
__device__ __forceinline__ int code_offset_f32(const float* row, int bins, float p, const QParams& g) {
  const float e = (float)bins * __builtin_amdgcn_logf(fmaf(g.ea, p, 1.f)) * g.ec;
  const float r = rintf(e) - 1.f;
  const int k0 = (int)__builtin_amdgcn_fmed3f(r == r ? r : 0.f, 0.f, (float)max(bins - 2, 0));
  // row[k0 - 1 .. k0 + 2], each index kept inside the row (an entry outside
  // it is not used: its test is decided by the bounds instead)
  const float t0 = row[max(k0 - 1, 0)], t1 = row[min(k0, bins - 1)], t2 = row[min(k0 + 1, bins - 1)],
              t3 = row[min(k0 + 2, bins - 1)];
  const bool below = k0 == 0 || t0 <= p;         // thresholds 1..k0 at or below p
  const bool above = k0 + 3 > bins || t3 > p;    // thresholds k0 + 3.. above p
  const int cnt = k0 + (k0 + 1 <= bins && t1 <= p ? 1 : 0) + (k0 + 2 <= bins && t2 <= p ? 1 : 0);
  if (below && above) return cnt;
  int lo = 0, hi = bins;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (row[mid] <= p) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// Code of one value given its group's parameters (quantizer.py:172-184).
// FINITE: the group's mn and scale are finite and every divisor (scale, pe,
// ne) is positive, so no intermediate is NaN or infinite and every clamped
// quantity is >= 0 (v >= mn; the side's offset from za is >= 0): the NaN
// cases and the lower clamps drop out and give the same results.
template <int DT, int BITS, bool FAST, bool FINITE>
__device__ __forceinline__ uint32_t value_code(float v, const QParams& g, const uint8_t* lds, const void* table) {
  constexpr float qmax = (float)((1 << BITS) - 1);
  const float n0 = qdiv<DT, FAST>(rnd<DT>(v - g.mn), g.sc, g.rsc);
  const float norm = FINITE ? fminf(n0, 1.f) : clamp01(n0);
  const bool up = norm >= g.za;  // torch.where(norm >= za, q_pos, q_neg); false on NaN
  // Only the selected side is evaluated: operands are chosen before the one
  // division, which computes exactly what the unselected-branch form would.
  const float p0 = qdiv<DT, FAST>(rnd<DT>(up ? norm - g.za : g.za - norm), up ? g.pe : g.ne, up ? g.rpe : g.rne);
  const float p = FINITE ? fminf(p0, 1.f) : clamp01(p0);
  const float bins = up ? g.pb : g.nb;
  float off;
  if constexpr (DT == MZ_F32) {
    const float* T = QTable<DT, BITS>::IN_LDS ? (const float*)lds : (const float*)table;
    const int ib = (FINITE || bins == bins) ? (int)bins : 1;
    const float* row = T + ib * (ib - 1) / 2;
    int lo;
    if constexpr (BITS >= 5) {
      lo = code_offset_f32(row, ib, p, g);
    } else {
      // up to 15 thresholds a row: the binary search's 4 steps measured as fast as the estimate
      lo = 0;
      int hi = ib;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (row[mid] <= p) lo = mid + 1; else hi = mid;
      }
    }
    off = (FINITE || p == p) ? (float)lo : __builtin_nanf("");
  } else {
    const uint16_t* Y = (const uint16_t*)lds;
    float y;
    if (FINITE || p == p) {
      const uint32_t pat = (DT == MZ_BF16 ? (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)p)  // p is not NaN
                                          : (uint32_t)f2h(p)) & 0x7FFFu;                          // -0 -> 0
      y = DT == MZ_BF16 ? bf2f(Y[pat]) : h2f(Y[pat]);
    } else {
      y = p;
    }
    off = rintf(rnd<DT>(y * bins));
  }
  // zl +- off is an integer in [-1, qmax + 1] <= 256 there: exact in every
  // input dtype, so its rounding is the identity
  const float q = FINITE ? (up ? g.zl + off : g.zl - off) : rnd<DT>(up ? g.zl + off : g.zl - off);
  // clamp(0, qmax).to(uint8); a NaN code converts to 0 (as on the reference CPU)
  if (!FINITE && !(q == q)) return 0u;
  return (uint32_t)fminf(fmaxf(q, 0.f), qmax);
}

// value_code<MZ_BF16, BITS, true, true> of 8 values (4 dwords) and their packed
// codes.
//
// The same values as the op-by-op chain, in fewer ops (every rewrite below is
// exact for a finite group: mn and the scale finite, the divisors positive):
//  - v - mn is one v_dot2_f32_bf16 on the dword as it was loaded: v * 1 + the
//    other half * 0 - mn (every value of the group is finite).  Its fp32 result
//    may differ from the subtraction's in the last bit, never in the bf16 it
//    rounds to: up to 15 binades apart, two 8-bit significands' difference has at
//    most 24 bits, exact in both; further apart it lies within 2^-15 of the larger
//    operand's binade, that operand is a bf16 value and half of the spacing of
//    bf16 values around it is at least 2^-9 of the binade.  Subnormal operands
//    are not flushed (the tests enumerate significand pairs and binades, and
//    sample the subnormals);
//  - each rounding to bf16 is one v_cvt_pk_bf16_f32 (rnd);
//  - min(rnd(x), 1) = rnd(min(x, 1)) (1 is a bf16 value and rounding is
//    monotone), and x >= 0, so the clamp rides on the multiply (med3 = the
//    VOP3 clamp bit);
//  - the selected side's difference, za - n below za and n - za above, is
//    |n - za| (fp32 negation is exact, and bf16 rounding is symmetric);
//  - the down side's offset is subtracted: zl - rint(rnd(y * nb)) =
//    zl + rint(rnd(y * -nb)) (both roundings are symmetric);
//  - p is a bf16 value >= +0 with a zero low half, so its ratio-table byte
//    address, pattern * 2, is its bit pattern >> 15;
//  - y * bins is a v_dot2_f32_bf16 on the table's 16-bit entry (8 bits by 8
//    bits: exact);
//  - rint is the addition of M = 1.5 * 2^23, whose sum's low bits are the
//    integer; the clamp to [0, qmax] is taken on the sum, from M - zl to
//    M - zl + qmax (exact), and M's and zl's bits leave once per packed word.
struct BfGroup {
  float nmn, rsc, za, rpe, rne, lo, hi;
  uint32_t pb, nb;  // bf16 bits of pb and -nb
  uint32_t base;    // bits of M - zl, the sum's where the code is 0
  __device__ __forceinline__ BfGroup(const QParams& g, float qmax)
      : nmn(-g.mn), rsc(g.rsc), za(g.za), rpe(g.rpe), rne(g.rne), lo(12582912.f - g.zl), hi(12582912.f - g.zl + qmax),
        pb(__float_as_uint(g.pb) >> 16), nb(__float_as_uint(-g.nb) >> 16), base(__float_as_uint(lo)) {}
};

// Dot products whose results other instructions read: they wait inside the
// block (three wait states after a dot, once for eight).
__device__ __forceinline__ void bf16_sub8(const uint32_t* w, float nmn, float (&a)[8]) {
  asm("v_dot2_f32_bf16 %0, %8, %12, %14\n\tv_dot2_f32_bf16 %1, %8, %13, %14\n\t"
      "v_dot2_f32_bf16 %2, %9, %12, %14\n\tv_dot2_f32_bf16 %3, %9, %13, %14\n\t"
      "v_dot2_f32_bf16 %4, %10, %12, %14\n\tv_dot2_f32_bf16 %5, %10, %13, %14\n\t"
      "v_dot2_f32_bf16 %6, %11, %12, %14\n\tv_dot2_f32_bf16 %7, %11, %13, %14\n\ts_nop 2"
      : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(a[4]), "=&v"(a[5]), "=&v"(a[6]), "=&v"(a[7])
      : "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "s"(0x00003F80u), "s"(0x3F800000u), "v"(nmn));
}
__device__ __forceinline__ void bf16_mul8(const uint32_t (&y)[8], const uint32_t (&b)[8], float (&o)[8]) {
  asm("v_dot2_f32_bf16 %0, %8, %16, 0\n\tv_dot2_f32_bf16 %1, %9, %17, 0\n\t"
      "v_dot2_f32_bf16 %2, %10, %18, 0\n\tv_dot2_f32_bf16 %3, %11, %19, 0\n\t"
      "v_dot2_f32_bf16 %4, %12, %20, 0\n\tv_dot2_f32_bf16 %5, %13, %21, 0\n\t"
      "v_dot2_f32_bf16 %6, %14, %22, 0\n\tv_dot2_f32_bf16 %7, %15, %23, 0\n\ts_nop 2"
      : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2]), "=&v"(o[3]), "=&v"(o[4]), "=&v"(o[5]), "=&v"(o[6]), "=&v"(o[7])
      : "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(y[4]), "v"(y[5]), "v"(y[6]), "v"(y[7]), "v"(b[0]), "v"(b[1]),
        "v"(b[2]), "v"(b[3]), "v"(b[4]), "v"(b[5]), "v"(b[6]), "v"(b[7]));
}

// 8 codes from their biased sums t (code + M - zl, clamped): 32-bit words of as
// many whole codes as fit, each the sum of (bits - base) << shift, the bases
// subtracted together (modulo 2^32).
template <int BITS>
__device__ __forceinline__ uint64_t pack_biased8(const float (&t)[8], uint32_t base) {
  constexpr int PER = BITS <= 4 ? 8 : 4;
  uint32_t word[8 / PER];
#pragma unroll
  for (int k = 0; k < 8 / PER; ++k) {
    constexpr uint32_t ones = (uint32_t)((((uint64_t)1 << (PER * BITS)) - 1) / ((1u << BITS) - 1));
    uint32_t acc = 0u - base * ones;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      acc = (__float_as_uint(t[PER * k + i]) << (i * BITS)) + acc;
      asm("" : "+v"(acc));  // one v_lshl_add_u32 each: the sum is not regrouped
    }
    word[k] = acc;
  }
  if constexpr (PER == 8) return word[0];
  else return (uint64_t)word[0] | ((uint64_t)word[1] << (4 * BITS));
}

template <int BITS>
__device__ __forceinline__ uint64_t value_codes8(const uint32_t* w, const BfGroup& g, const uint8_t* lds) {
  float a[8], o[8], t[8];
  uint32_t y[8], b[8];
  bf16_sub8(w, g.nmn, a);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float n = rnd<MZ_BF16>(__builtin_amdgcn_fmed3f(rnd<MZ_BF16>(a[i]) * g.rsc, 0.f, 1.f));
    const bool up = n >= g.za;
    const float d = rnd<MZ_BF16>(n - g.za);  // |rnd(x)| = rnd(|x|): the absolute value rides on the multiply's operand
    const float p = rnd<MZ_BF16>(__builtin_amdgcn_fmed3f(__builtin_fabsf(d) * (up ? g.rpe : g.rne), 0.f, 1.f));
    y[i] = *(const uint16_t*)(lds + (__float_as_uint(p) >> 15));
    b[i] = up ? g.pb : g.nb;
  }
  bf16_mul8(y, b, o);
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = __builtin_amdgcn_fmed3f(rnd<MZ_BF16>(o[i]) + 12582912.f, g.lo, g.hi);
  return pack_biased8<BITS>(t, g.base);
}

// value_code<MZ_F16, BITS, true, true> of 8 values (4 dwords) and their packed
// codes, with the rewrites of the bf16 form, which hold for fp16 as well (they
// use only that 1 is an fp16 value, that rounding is monotone and symmetric,
// and that in a finite group every quotient is >= +0).  The differences v - mn
// (two an op) and n - za are fp16 subtractions: fp32 carries 24 >= 2 * 11 + 2
// bits, so rounding its difference to fp16 gives the same value.  Each division
// is a * rcp(b) plus one residual correction (qdiv; b is positive and finite
// here), the clamp riding on the correction's FMA, the fp16 operands read as
// they are by v_fma_mix; its fp32 result is rounded before it is converted (an
// exact tie in fp16's subnormal range needs both).  p's fp16 pattern addresses
// the ratio table directly.
typedef _Float16 f16x2v __attribute__((ext_vector_type(2)));
struct HfGroup {
  float sc, rsc, pe, ne, rpe, rne, pb, nb, lo, hi;
  _Float16 mn, za;
  uint32_t base;
  __device__ __forceinline__ HfGroup(const QParams& g, float qmax)
      : sc(g.sc), rsc(g.rsc), pe(g.pe), ne(g.ne), rpe(g.rpe), rne(g.rne), pb(g.pb), nb(-g.nb), lo(12582912.f - g.zl),
        hi(12582912.f - g.zl + qmax), mn((_Float16)g.mn), za((_Float16)g.za), base(__float_as_uint(lo)) {}
};

template <int BITS>
__device__ __forceinline__ uint64_t value_codes8(const uint32_t* w, const HfGroup& g, const uint8_t* lds) {
  const f16x2v mn2 = {g.mn, g.mn};
  _Float16 y[8];
  float b[8], t[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const f16x2v a2 = __builtin_bit_cast(f16x2v, w[i / 2]) - mn2;
    const float a = (float)a2[i & 1];
    const float n0 = __builtin_fmaf(a, g.rsc, 0.f);  // a * rsc (a >= +0): one v_fma_mix
    const _Float16 n =
        (_Float16)__builtin_amdgcn_fmed3f(__builtin_fmaf(__builtin_fmaf(-g.sc, n0, a), g.rsc, n0), 0.f, 1.f);
    const bool up = n >= g.za;
    const float d = __builtin_fabsf((float)(_Float16)(n - g.za));
    const float q = up ? g.pe : g.ne, r = up ? g.rpe : g.rne;
    const float p0 = __builtin_fmaf(d, r, 0.f);
    const _Float16 p =
        (_Float16)__builtin_amdgcn_fmed3f(__builtin_fmaf(__builtin_fmaf(-q, p0, d), r, p0), 0.f, 1.f);
    y[i] = *(const _Float16*)(lds + (uint16_t)(__builtin_bit_cast(uint16_t, p) << 1));
    b[i] = up ? g.pb : g.nb;
  }
  float one = 1.f;
  asm("" : "+s"(one));  // opaque: o * 1 + M stays one v_fma_mix
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const _Float16 o = (_Float16)((float)y[i] * b[i]);
    t[i] = __builtin_amdgcn_fmed3f(__builtin_fmaf((float)o, one, 12582912.f), g.lo, g.hi);
  }
  return pack_biased8<BITS>(t, g.base);
}

// Min / max over the 8 lanes of a group (lanes 8k..8k+7), NaN-propagating:
// IEEE 754-2019 minimum / maximum (v_minimum3_f32 / v_maximum3_f32), which
// return NaN when either operand is NaN, as torch's amin / amax do.  (Between
// -0 and +0 they pick -0 / +0; torch's choice there depends on its
// vectorisation.  The codes are the same either way: only the sign of a zero
// minimum or maximum in the metadata can differ.)
__device__ __forceinline__ float fmin_nan(float a, float b) { return __builtin_elementwise_minimum(a, b); }
__device__ __forceinline__ float fmax_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }
// Over the L lanes of a group (aligned runs of L = 2, 4 or 8 lanes).
template <int L>
__device__ __forceinline__ float group_min(float v) {
  if constexpr (L >= 2) v = fmin_nan(v, dpp_sel<DPP_QUAD_XOR1>(v));
  if constexpr (L >= 4) v = fmin_nan(v, dpp_sel<DPP_QUAD_XOR2>(v));
  if constexpr (L >= 8) v = fmin_nan(v, dpp_sel<DPP_ROW_HALF_MIRROR>(v));
  return v;
}
template <int L>
__device__ __forceinline__ float group_max(float v) {
  if constexpr (L >= 2) v = fmax_nan(v, dpp_sel<DPP_QUAD_XOR1>(v));
  if constexpr (L >= 4) v = fmax_nan(v, dpp_sel<DPP_QUAD_XOR2>(v));
  if constexpr (L >= 8) v = fmax_nan(v, dpp_sel<DPP_ROW_HALF_MIRROR>(v));
  return v;
}

// NaN-propagating min / max of x[0..N) (a balanced tree).
template <int N, int S = 0>
__device__ __forceinline__ float tree_min(const float* x) {
  if constexpr (N == 1) return x[S];
  else return fmin_nan(tree_min<N / 2, S>(x), tree_min<N / 2, S + N / 2>(x));
}
template <int N, int S = 0>
__device__ __forceinline__ float tree_max(const float* x) {
  if constexpr (N == 1) return x[S];
  else return fmax_nan(tree_max<N / 2, S>(x), tree_max<N / 2, S + N / 2>(x));
}

// The offset estimate's constants (code_offset_f32) from the threshold t of
// bins 1 (index 0 of the table), where log1p(alpha*t) / lb crosses 1/2:
// (1 + alpha*t)^2 = 1 + alpha, so alpha = (1 - 2t) / t^2.
template <int BITS>
__device__ __forceinline__ void set_estimate(QParams& g, const uint8_t* lds, const void* table) {
  const float t = (QTable<MZ_F32, BITS>::IN_LDS ? (const float*)lds : (const float*)table)[0];
  g.ea = (1.f - 2.f * t) / (t * t);
  g.ec = 1.f / __builtin_amdgcn_logf(1.f + g.ea);
}

// 8 consecutive values at p[i..i+7] (VEC: one or two 16-byte loads).
template <int DT, bool VEC>
__device__ __forceinline__ void load8(float (&x)[8], const void* p, int64_t i) {
  if constexpr (VEC && DT == MZ_F32) {
    const float4 a = *(const float4*)((const float*)p + i);
    const float4 b = *(const float4*)((const float*)p + i + 4);
    x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
  } else if constexpr (VEC) {
    const uint4 a = *(const uint4*)((const uint16_t*)p + i);
    const uint32_t u[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[2 * k] = DT == MZ_BF16 ? bf2f((uint16_t)u[k]) : h2f((uint16_t)u[k]);
      x[2 * k + 1] = DT == MZ_BF16 ? bf2f((uint16_t)(u[k] >> 16)) : h2f((uint16_t)(u[k] >> 16));
    }
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = load_val<DT>(p, i + k);
  }
}

}  // namespace mz
