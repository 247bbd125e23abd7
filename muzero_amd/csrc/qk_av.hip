// Separate QK and AV launches over a packed prefix (gfx950, wave64).
//
// The reference's default decode path (muzero/cache/attention.py:179-295,
// MUZERO_FUSED_PREFIX_DECODE unset) runs three steps: qk writes the logits of
// the packed key prefix in the query dtype, torch takes the softmax, av writes
// the weighted sum of the packed value prefix.  This file implements qk and
// av with the reference's argument meaning (muzero/kernels/loader.py:46-53);
// the fused decode kernels (decode.hip, decode_fold.hip) do all three steps in
// one pass and are what the cache's decode hook runs.
//
// Both launches are one computation on 64-code rows: a wave takes a chunk of
// up to 64 rows, lane i dequantizes code i of every row and adds
// coefficient(row, head) * value to one accumulator per query head of the
// kv-head.
//   qk: rows = the D channels of one key group (64 tokens), lane = token,
//       coefficient = the query's channel; the accumulators are the group's
//       logits.  A wave owns one or two key groups.
//   av: rows = tokens of one value group (64 channels), lane = channel,
//       coefficient = the token's attention weight.  A workgroup owns a
//       (batch, kv-head, value group) or a split of its tokens; its 4 waves
//       take every 4th 64-token chunk and add their sums through LDS in a fixed
//       order (no atomics: results are deterministic).
// Per chunk, in the wave's LDS area: the rows' packed bytes (one row per lane,
// 8-byte global loads, written at an odd dword pitch so that neither the
// stores nor the per-row code reads meet on a bank), each row's
// dequantization parameters (from the stored metadata), and for codes of up
// to 5 bits a codebook of every code's value per row, lane r writing row r's
// 2^bits entries, so a row costs 2^bits / 64 dequantizations per lane instead
// of one.  Wider codes are dequantized one per lane and row from the row's
// parameters (an LDS broadcast).  Every value is the reference's fp32
// dequantized value exactly (group_value: muzero/quantizer.py:229-255 op for
// op, the expm1 rows read from the host-built table: copied to LDS once per
// workgroup for codes of up to 6 bits, read from global memory for 7 and 8);
// sums are fp32 multiply-adds, rounded once to the io dtype at the end.
//
// muzero_decode_unfused runs the whole of that default path for one decode
// token in four launches: qk over the prefix with the residual's logits in
// further workgroups of the same launch, the softmax with the residual's
// weighted sum, av over splits of the prefix's tokens, and the sum of the
// splits.  Logits, weights and sums are rounded to the io dtype where torch's
// steps round them.  As torch steps around the two launches it was 14 launches;
// at B = 8, 2100 tokens, 32/8 heads of 96, 4-bit: 182 us per call, now 33.2
// (profiled one at a time, when a kernel starts on an idle GPU: qk 12.8, softmax
// 9.0, av 11.8, sum 3.9; av 43 before, 128 workgroups walking 30 chunks each).
#include <algorithm>
#include <atomic>

#include "decode_common.hpp"

namespace mz {

namespace rowdot {

constexpr int kRows = 64;   // rows per chunk
constexpr int kWaves = 4;   // waves per workgroup
constexpr int kMaxHeadDim = 256;
constexpr int kMaxRep = 16;
constexpr int kGroupsPerWave = 2;  // qk: key groups per wave, once the waves fill the device

// The dense tail of an unfused decode call (none: `rows` null).
struct Tail {
  const void* rows = nullptr;  // residual keys (qk) or values (softmax) of the io dtype
  int64_t sb = 0, sh = 0, st = 0;
  int n = 0;       // residual tokens
  int first = 0;   // logits / weights column of the first one
  int vec = 0;     // rows are read 16 bytes at a time
  int blocks = 0;  // qk: workgroups before the tail's
};

// Byte layout of one wave's LDS area.
template <int BITS, int NR>
struct Area {
  static constexpr int QB = 8 * BITS;        // bytes per packed row
  static constexpr int PITCH = QB + 4;       // staged row pitch: an odd number of dwords
  static constexpr bool CB = BITS <= 5;      // codebook per row
  static constexpr int NCB = 1 << BITS;
  // codebook row pitch in floats: rows 8 apart share banks, so the 16-byte
  // stores of a row's entries (8 lanes at a time) do not conflict
  static constexpr int CBP = NCB == 2 ? 2 : NCB + 4;
  static constexpr int STAGE = kRows * PITCH + 16;  // + the dword read past the last row's end
  // wider codes: 32 bytes of parameters per row, read by every lane
  static constexpr int PAR_OFF = STAGE;
  static constexpr int CB_OFF = PAR_OFF + (CB ? 0 : kRows * 32);
  static constexpr int COEF_OFF = CB_OFF + (CB ? kRows * CBP * 4 : 0);
  // `coef`: the area also holds the chunk's coefficients [row][NR] (av)
  static constexpr int bytes(bool coef) { return COEF_OFF + (coef ? kRows * NR * 4 : 0); }
  static_assert(STAGE % 16 == 0 && (CB_OFF % 16) == 0, "16-byte aligned parts");
};

// expm1 rows in LDS (codes of up to 6 bits; 7- and 8-bit rows, up to 128 KB,
// stay in global memory): EF floats, rounded up to 16 bytes.
template <int BITS>
constexpr int etab_bytes() {
  return BITS <= 6 ? ((((1 << BITS) - 1) * ((1 << BITS) + 2) / 2) * 4 + 15) & ~15 : 0;
}

// Copy the expm1 rows to the start of LDS (all threads; the caller syncs).
template <int BITS>
__device__ __forceinline__ const float* stage_etab(uint8_t* lds, const float* e) {
  if constexpr (etab_bytes<BITS>() == 0) {
    return e;
  } else {
    constexpr int EF = ((1 << BITS) - 1) * ((1 << BITS) + 2) / 2;
    float* t = (float*)lds;
    for (int i = threadIdx.x; i < EF; i += 256) t[i] = e[i];
    return t;
  }
}

__device__ __forceinline__ void put_row(uint8_t* p, const DeqGroup& r) {
  float4* f = (float4*)p;
  f[0] = make_float4(r.mn, r.s, r.za, r.pe);
  f[1] = make_float4(r.nne, __int_as_float(r.zl), __int_as_float(r.offp), __int_as_float(r.offn));
}

__device__ __forceinline__ DeqGroup get_row(const uint8_t* p) {
  const float4* f = (const float4*)p;
  const float4 a = f[0], b = f[1];
  return DeqGroup{a.x, a.y, a.z, a.w, b.x, __float_as_int(b.y), __float_as_int(b.z), __float_as_int(b.w)};
}

// A chunk's global inputs, held in registers: a wave loads chunk c+1's while
// it computes chunk c.  Lane r holds row r's packed bytes and metadata (and,
// for av, the weights of token r).
template <int BITS, int NR>
struct Fetch {
  uint2 row[BITS];
  uint32_t mn, sc;  // raw metadata
  uint32_t w[NR];   // raw weights
};

// An entry's bits and their value: loads first, conversions when the value is
// used (a conversion behind its load's type branch would wait for it there).
__device__ __forceinline__ uint32_t load_raw(const void* p, int64_t i, int dt) {
  return dt == MZ_F32 ? ((const uint32_t*)p)[i] : (uint32_t)((const uint16_t*)p)[i];
}
__device__ __forceinline__ float raw_value(uint32_t u, int dt) {
  return dt == MZ_F32 ? __uint_as_float(u) : dt == MZ_BF16 ? bf2f((uint16_t)u) : h2f((uint16_t)u);
}

// Row r's packed bytes start at rows + r*row_stride, its metadata at index
// meta0 + r*meta_stride of mn / sc (r < nrows).
template <int BITS, int NR>
__device__ __forceinline__ void fetch_rows(Fetch<BITS, NR>& f, const uint8_t* rows, int64_t row_stride,
                                           const void* mn, const void* sc, int64_t meta0, int64_t meta_stride,
                                           int mdt, int nrows) {
  const int lane = threadIdx.x & 63;
  if (lane < nrows) {
    const uint2* src = (const uint2*)(rows + lane * row_stride);
#pragma unroll
    for (int k = 0; k < BITS; ++k) f.row[k] = src[k];
    const int64_t m = meta0 + lane * meta_stride;
    f.mn = load_raw(mn, m, mdt);
    f.sc = load_raw(sc, m, mdt);
  }
}

// One chunk of `nrows` (<= 64) fetched rows; row r's coefficients are
// coef[r*NR + h] (LDS).  acc[h] += coef[r][h] * value(r, lane) over the rows.
template <int BITS, int NR>
__device__ __forceinline__ void chunk(uint8_t* area, const Fetch<BITS, NR>& f, int mdt, const float* E,
                                      const float* coef, int nrows, float (&acc)[NR]) {
  using A = Area<BITS, NR>;
  const int lane = threadIdx.x & 63;
  if (lane < nrows) {
    uint32_t* dst = (uint32_t*)(area + lane * A::PITCH);
#pragma unroll
    for (int k = 0; k < BITS; ++k) {
      dst[2 * k] = f.row[k].x;
      dst[2 * k + 1] = f.row[k].y;
    }
    const DeqGroup r = make_group<(1 << BITS) - 1>(raw_value(f.mn, mdt), raw_value(f.sc, mdt));
    if constexpr (A::CB) {
      // lane r writes row r's codebook
      float* cbr = (float*)(area + A::CB_OFF) + lane * A::CBP;
      if constexpr (A::NCB == 2) {
        *(float2*)cbr = make_float2(group_value(r, 0, E), group_value(r, 1, E));
      } else {
#pragma unroll
        for (int q = 0; q < A::NCB; q += 4)
          *(float4*)(cbr + q) = make_float4(group_value(r, q, E), group_value(r, q + 1, E), group_value(r, q + 2, E),
                                            group_value(r, q + 3, E));
      }
    } else {
      put_row(area + A::PAR_OFF + 32 * lane, r);
    }
  }
  wave_lds_sync();
  const float* cb = (const float*)(area + A::CB_OFF);
  // lane's code: bits [lane*BITS, lane*BITS + BITS) of the row
  const int bit = lane * BITS;
  const uint8_t* lrow = area + (bit >> 5) * 4;
  const uint32_t sh = bit & 31;
  constexpr uint32_t mask = (1u << BITS) - 1u;
  constexpr bool straddle = (32 % BITS) != 0;
  auto row = [&](const int r) __attribute__((always_inline)) {
    const uint8_t* rp = lrow + r * A::PITCH;
    const uint32_t d0 = *(const uint32_t*)rp;
    uint32_t code;
    if constexpr (straddle) code = __builtin_amdgcn_alignbit(*(const uint32_t*)(rp + 4), d0, sh) & mask;
    else code = __builtin_amdgcn_ubfe(d0, sh, BITS);
    float x;
    if constexpr (A::CB) x = cb[r * A::CBP + code];
    else x = group_value(get_row(area + A::PAR_OFF + 32 * r), code, E);
#pragma unroll
    for (int h = 0; h < NR; ++h) acc[h] = __builtin_fmaf(coef[r * NR + h], x, acc[h]);
  };
  if (nrows == kRows) {
    // a full chunk: every row's offsets are compile-time constants (immediate
    // offsets of the LDS reads), so a row costs its extract and multiply-adds
#pragma unroll
    for (int r = 0; r < kRows; ++r) row(r);
  } else {
#pragma unroll 4
    for (int r = 0; r < nrows; ++r) row(r);
  }
}

__host__ __device__ constexpr int qc_bytes(int D, int NR) { return (D * NR * 4 + 15) & ~15; }

template <int BITS, int NR>
constexpr int qk_lds_bytes(int D) {
  return etab_bytes<BITS>() + qc_bytes(D, NR) + kWaves * Area<BITS, NR>::bytes(false);
}
template <int BITS, int NR>
constexpr int av_lds_bytes() {
  constexpr int areas = kWaves * Area<BITS, NR>::bytes(true);
  constexpr int red = kWaves * NR * kRows * 4;
  return etab_bytes<BITS>() + (areas > red ? areas : red);
}

// Residual logits: a thread takes one token's row, the query coefficients
// [D][NR] are LDS broadcasts; rounded to the io dtype after the product and
// after the scaling, as the product and the multiply by the scaling are.
template <int NR, int IO>
__device__ __forceinline__ void tail_logits(const mz_qk_args& a, const Tail& tl, const float* qc) {
  const int t = (blockIdx.x - tl.blocks) * 256 + threadIdx.x;
  if (t >= tl.n) return;
  const int kvh = blockIdx.y, b = blockIdx.z, D = a.head_dim;
  constexpr int ES = IO == MZ_F32 ? 4 : 2, NE = 16 / ES;
  const char* row = (const char*)tl.rows + (b * tl.sb + kvh * tl.sh + (int64_t)t * tl.st) * ES;
  float acc[NR];
#pragma unroll
  for (int h = 0; h < NR; ++h) acc[h] = 0.f;
  auto add = [&](float x, int d) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < NR; ++h) acc[h] = __builtin_fmaf(qc[d * NR + h], x, acc[h]);
  };
  if (tl.vec) {
#pragma unroll 4
    for (int d = 0; d < D; d += NE) {
      const uint4 u = *(const uint4*)(row + d * ES);
      const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if constexpr (IO == MZ_F32) {
          add(__uint_as_float(w[k]), d + k);
        } else {
          add(IO == MZ_BF16 ? bf2f((uint16_t)w[k]) : h2f((uint16_t)w[k]), d + 2 * k);
          add(IO == MZ_BF16 ? bf2f((uint16_t)(w[k] >> 16)) : h2f((uint16_t)(w[k] >> 16)), d + 2 * k + 1);
        }
      }
    }
  } else {
#pragma unroll 8
    for (int d = 0; d < D; ++d) add(load_val<IO>(row, d), d);
  }
  const int64_t o = b * a.o_sb + tl.first + t;
#pragma unroll
  for (int h = 0; h < NR; ++h)
    if (h < a.n_rep) store_val(a.logits, o + (int64_t)(kvh * a.n_rep + h) * a.o_sh, rnd<IO>(acc[h]) * a.scaling, IO);
}

// grid (ceil(n_groups / (4 gpw)) + the tail's workgroups of 256 tokens, kv_heads,
// batch); wave w of workgroup x takes key groups gpw (4x + w) .. + gpw - 1.
template <int BITS, int NR>
__global__ __launch_bounds__(256) void qk_kernel(const mz_qk_args a, const Tail tl, const int gpw) {
  using A = Area<BITS, NR>;
  extern __shared__ __align__(16) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kvh = blockIdx.y;
  const int b = blockIdx.z;
  const int D = a.head_dim;
  const bool tail = tl.rows && (int)blockIdx.x >= tl.blocks;
  const int g0 = (blockIdx.x * kWaves + wave) * gpw;
  const int groups = tail ? 0 : min(gpw, a.n_groups - g0);
  uint8_t* area = lds + etab_bytes<BITS>() + qc_bytes(D, NR) + wave * A::bytes(false);
  const uint8_t* gp = a.k_packed + b * a.kp_sb + kvh * a.kp_sh + (int64_t)g0 * D * A::QB;
  const int64_t m0 = b * a.km_sb + kvh * a.km_sh + (int64_t)g0 * D;
  // items = (group, chunk of up to 64 channels); the wave's groups are
  // contiguous rows, channel d of its group i being row i*D + d
  const int cpg = (D + kRows - 1) / kRows;
  const int items = groups * cpg;
  auto rows_of = [&](int it) { return min(kRows, D - (it % cpg) * kRows); };
  auto row0_of = [&](int it) { return (it / cpg) * D + (it % cpg) * kRows; };
  Fetch<BITS, NR> f;
  if (groups > 0) fetch_rows(f, gp, A::QB, a.k_mn, a.k_scale, m0, 1, a.meta_dtype, rows_of(0));
  const float* E = tail ? nullptr : stage_etab<BITS>(lds, a.e_key);
  // the kv-head's query rows as fp32 coefficients [D][NR] (heads past n_rep are 0)
  float* qc = (float*)(lds + etab_bytes<BITS>());
  for (int i = threadIdx.x; i < D * NR; i += 256) {
    const int d = i / NR, h = i % NR;
    qc[i] = h < a.n_rep ? load_any(a.query, b * a.q_sb + (int64_t)(kvh * a.n_rep + h) * a.q_sh + d, a.io_dtype) : 0.f;
  }
  __syncthreads();
  if (tail) {
    if (a.io_dtype == MZ_BF16) tail_logits<NR, MZ_BF16>(a, tl, qc);
    else if (a.io_dtype == MZ_F16) tail_logits<NR, MZ_F16>(a, tl, qc);
    else tail_logits<NR, MZ_F32>(a, tl, qc);
    return;
  }
  if (groups <= 0) return;
  float acc[NR];
  for (int it = 0; it < items; ++it) {
    const Fetch<BITS, NR> cur = f;
    if (it + 1 < items) {
      const int r1 = row0_of(it + 1);
      fetch_rows(f, gp + (int64_t)r1 * A::QB, A::QB, a.k_mn, a.k_scale, m0 + r1, 1, a.meta_dtype, rows_of(it + 1));
    }
    const int c = it % cpg;
    if (c == 0) {
#pragma unroll
      for (int h = 0; h < NR; ++h) acc[h] = 0.f;
    }
    wave_lds_sync();  // the previous item's reads of the area are done
    chunk<BITS, NR>(area, cur, a.meta_dtype, E, qc + c * kRows * NR, rows_of(it), acc);
    if (c == cpg - 1) {
      const int64_t o = b * a.o_sb + (int64_t)(g0 + it / cpg) * kRows + lane;
#pragma unroll
      for (int h = 0; h < NR; ++h)
        if (h < a.n_rep)
          store_val(a.logits, o + (int64_t)(kvh * a.n_rep + h) * a.o_sh, acc[h] * a.scaling, a.io_dtype);
    }
  }
}

// grid (value groups * splits, kv_heads, batch).  With `part` set, split s of
// the tokens (64 * `chunks` each) writes its fp32 sums to part[b, q-head, s, D]
// (`parts` records per q-head); else the one split writes the output.
template <int BITS, int NR>
__global__ __launch_bounds__(256) void av_kernel(const mz_av_args a, float* __restrict__ part, const int parts,
                                                 const int chunks) {
  using A = Area<BITS, NR>;
  extern __shared__ __align__(16) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ng = (a.head_dim + kRows - 1) / kRows;
  const int j = blockIdx.x % ng, split = blockIdx.x / ng;
  const int first = min(split * chunks * kRows, a.n_tokens);  // the split's tokens
  const int n_tokens = min(a.n_tokens - first, chunks * kRows);
  const int kvh = blockIdx.y;
  const int b = blockIdx.z;
  uint8_t* work = lds + etab_bytes<BITS>();
  uint8_t* area = work + wave * A::bytes(true);
  float* coef = (float*)(area + A::COEF_OFF);
  float acc[NR];
#pragma unroll
  for (int h = 0; h < NR; ++h) acc[h] = 0.f;
  const uint8_t* vp = a.v_packed + b * a.vp_sb + kvh * a.vp_sh + (int64_t)first * ng * A::QB + j * A::QB;
  const int64_t m0 = b * a.vm_sb + kvh * a.vm_sh + (int64_t)first * ng + j;
  const int64_t w0 = b * a.w_sb + (int64_t)kvh * a.n_rep * a.w_sh + first;
  auto weights_of = [&](uint32_t (&w)[NR], int t) {
#pragma unroll
    for (int h = 0; h < NR; ++h) w[h] = h < a.n_rep ? load_raw(a.weights, w0 + h * a.w_sh + t, a.io_dtype) : 0u;
  };
  // chunk t0 = 64*(wave + 4k): its rows (tokens) and its tokens' weights
  auto fetch = [&](Fetch<BITS, NR>& f, int t0) {
    const int nrows = min(kRows, n_tokens - t0);
    fetch_rows(f, vp + (int64_t)t0 * ng * A::QB, (int64_t)ng * A::QB, a.v_mn, a.v_scale, m0 + (int64_t)t0 * ng, ng,
               a.meta_dtype, nrows);
    if (lane < nrows) weights_of(f.w, t0 + lane);
  };
  Fetch<BITS, NR> f;
  int t0 = wave * kRows;
  if (t0 < n_tokens) fetch(f, t0);
  // (no table to read when there are no tokens: the call writes zeros)
  const float* E = n_tokens > 0 ? stage_etab<BITS>(lds, a.e_value) : nullptr;
  if constexpr (etab_bytes<BITS>() > 0) __syncthreads();
  for (; t0 < n_tokens; t0 += kWaves * kRows) {
    const Fetch<BITS, NR> cur = f;
    if (t0 + kWaves * kRows < n_tokens) fetch(f, t0 + kWaves * kRows);
    const int nrows = min(kRows, n_tokens - t0);
    wave_lds_sync();  // the previous chunk's reads of the area are done
    if (lane < nrows) {
#pragma unroll
      for (int h = 0; h < NR; ++h) coef[lane * NR + h] = raw_value(cur.w[h], a.io_dtype);
    }
    chunk<BITS, NR>(area, cur, a.meta_dtype, E, coef, nrows, acc);
  }
  // the 4 waves' sums, added in wave order
  __syncthreads();
  float* red = (float*)work;  // [wave][NR][64]
#pragma unroll
  for (int h = 0; h < NR; ++h) red[(wave * NR + h) * kRows + lane] = acc[h];
  __syncthreads();
  const int c = j * kRows + lane;
  for (int h = wave; h < a.n_rep; h += kWaves) {
    float s = red[h * kRows + lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) s += red[(w * NR + h) * kRows + lane];
    if (c >= a.head_dim) continue;
    if (part) part[(((int64_t)b * a.kv_heads * a.n_rep + kvh * a.n_rep + h) * parts + split) * a.head_dim + c] = s;
    else store_val(a.out, b * a.o_sb + (int64_t)(kvh * a.n_rep + h) * a.o_sh + c, s, a.io_dtype);
  }
}

// Softmax of one (batch, q-head)'s logits in place: fp32 over the io-dtype
// logits (plus the additive mask, rounded to the io dtype as its addition is),
// weights rounded to the io dtype.  The row is held in LDS between its passes
// (HELD: up to kHeldLogits), else read again.  The same workgroup then sums the
// dense tail's values with its weights into part[row, parts - 1, D]: a thread
// takes 16 bytes of a token's channels, the tokens are dealt over the threads.
// (As further splits of the av launch the tail cost it a second filling of the
// CUs, 26 us instead of 11.)
constexpr int kHeldLogits = 12 * 1024;
template <int IO, bool HELD>
__global__ __launch_bounds__(256) void softmax_kernel(void* __restrict__ logits, int64_t ld, int len, int kv_heads,
                                                      int n_rep, const float* __restrict__ mask, int64_t mask_sb,
                                                      const Tail tl, int D, float* __restrict__ part, int parts) {
  extern __shared__ __align__(16) float row[];
  __shared__ float red[2 * kWaves];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t bh = blockIdx.x, base = bh * ld;
  const int64_t b = bh / (kv_heads * n_rep), kvh = (bh - b * (kv_heads * n_rep)) / n_rep;
  const float* m = mask ? mask + b * mask_sb : nullptr;
  auto logit = [&](int i) __attribute__((always_inline)) {
    float x = load_val<IO>(logits, base + i);
    if (m) x = rnd<IO>(x + rnd<IO>(m[i]));
    return x;
  };
  float top = -INFINITY;
#pragma unroll 4
  for (int i = t; i < len; i += 256) {
    const float x = logit(i);
    if constexpr (HELD) row[i] = x;
    top = nmax(top, x);  // NaN propagates, as through torch's softmax
  }
  top = wave_max(top);
  if (lane == 0) red[wave] = top;
  __syncthreads();
  top = nmax(nmax(red[0], red[1]), nmax(red[2], red[3]));
  float sum = 0.f;
#pragma unroll 4
  for (int i = t; i < len; i += 256) {
    const float e = expf((HELD ? row[i] : logit(i)) - top);
    if constexpr (HELD) row[i] = e;
    sum += e;
  }
  sum = group_reduce<64>(sum, OpAdd());
  if (lane == 0) red[kWaves + wave] = sum;
  __syncthreads();
  sum = (red[kWaves] + red[kWaves + 1]) + (red[kWaves + 2] + red[kWaves + 3]);
#pragma unroll 4
  for (int i = t; i < len; i += 256) {
    const float w = (HELD ? row[i] : expf(logit(i) - top)) / sum;
    store_val(logits, base + i, w, IO);
    if constexpr (HELD) row[i] = rnd<IO>(w);
  }
  if (!tl.rows) return;
  __syncthreads();
  // thread (token group p, channels c .. c + N - 1)
  constexpr int ES = IO == MZ_F32 ? 4 : 2, NE = 16 / ES;
  const char* rows = (const char*)tl.rows + (b * tl.sb + kvh * tl.sh) * ES;
  auto weight = [&](int i) __attribute__((always_inline)) {
    return HELD ? row[tl.first + i] : load_val<IO>(logits, base + tl.first + i);
  };
  const int N = tl.vec ? NE : 1, lanes = D / N, groups = 256 / lanes;  // D <= 256, a multiple of N
  const int p = t / lanes, c = (t - p * lanes) * N;
  float acc[NE];
#pragma unroll
  for (int k = 0; k < NE; ++k) acc[k] = 0.f;
  if (p < groups) {
    if (tl.vec) {
#pragma unroll 4
      for (int i = p; i < tl.n; i += groups) {
        const uint4 u = *(const uint4*)(rows + ((int64_t)i * tl.st + c) * ES);
        const uint32_t x[4] = {u.x, u.y, u.z, u.w};
        const float w = weight(i);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if constexpr (IO == MZ_F32) {
            acc[k] = __builtin_fmaf(w, __uint_as_float(x[k]), acc[k]);
          } else {
            acc[2 * k] = __builtin_fmaf(w, IO == MZ_BF16 ? bf2f((uint16_t)x[k]) : h2f((uint16_t)x[k]), acc[2 * k]);
            acc[2 * k + 1] = __builtin_fmaf(w, IO == MZ_BF16 ? bf2f((uint16_t)(x[k] >> 16)) : h2f((uint16_t)(x[k] >> 16)),
                                            acc[2 * k + 1]);
          }
        }
      }
    } else {
#pragma unroll 4
      for (int i = p; i < tl.n; i += groups) acc[0] = __builtin_fmaf(weight(i), load_val<IO>(rows, (int64_t)i * tl.st + c), acc[0]);
    }
  }
  __syncthreads();  // the weights in LDS are read; their space takes the groups' sums [groups][D]
  if (p < groups) {
#pragma unroll
    for (int k = 0; k < NE; ++k)
      if (k < N) row[p * D + c + k] = acc[k];
  }
  __syncthreads();
  if (t < D) {
    float s = 0.f;
    for (int g = 0; g < groups; ++g) s += row[g * D + t];
    part[(bh * parts + parts - 1) * D + t] = s;
  }
}
// bytes of its LDS row: the logits held, or the tail's sums (at most 256 * 8 floats)
inline int softmax_lds(int len) { return std::max(len <= kHeldLogits ? len : 0, 256 * 8) * (int)sizeof(float); }

// out[b, q-head] = the prefix's sum (splits 0 .. prefix - 1, in order) plus the
// residual's, each rounded to the io dtype and the sum of the two again, as the
// separate av, product and addition are.
constexpr int kSumLoads = 8;
template <int IO>
__global__ __launch_bounds__(256) void sum_splits_kernel(const float* __restrict__ part, int splits, int prefix, int D,
                                                         int Hq, void* out, int64_t o_sb, int64_t o_sh) {
  const int64_t bh = blockIdx.x;
  const int b = (int)(bh / Hq), h = (int)(bh - (int64_t)b * Hq);
  const int c = threadIdx.x;
  if (c >= D) return;
  const float* p = part + bh * splits * D + c;
  float packed = 0.f, dense = 0.f;
  for (int s0 = 0; s0 < splits; s0 += kSumLoads) {
    float x[kSumLoads];
#pragma unroll
    for (int k = 0; k < kSumLoads; ++k) x[k] = p[(int64_t)min(s0 + k, splits - 1) * D];
#pragma unroll
    for (int k = 0; k < kSumLoads; ++k) {
      packed += s0 + k < prefix ? x[k] : 0.f;
      dense += s0 + k >= prefix && s0 + k < splits ? x[k] : 0.f;
    }
  }
  store_val(out, b * o_sb + (int64_t)h * o_sh + c, rnd<IO>(packed) + rnd<IO>(dense), IO);
}

// Query heads per kv-head rounded up to the accumulator count of a kernel.
inline int nr_for(int n_rep) { return n_rep <= 1 ? 1 : n_rep <= 2 ? 2 : n_rep <= 4 ? 4 : n_rep <= 8 ? 8 : 16; }

template <int BITS, int NR>
hipError_t launch_qk(const mz_qk_args& a, Tail tl, hipStream_t s) {
  static std::atomic<uint64_t> raised{0};
  const int bytes = qk_lds_bytes<BITS, NR>(a.head_dim);
  if (bytes > 65536) {
    const hipError_t e = set_dynamic_lds((const void*)qk_kernel<BITS, NR>, bytes, raised);
    if (e != hipSuccess) return e;
  }
  // one group per wave until the workgroups fill the CUs four times (their LDS holds about four per CU)
  const int64_t wide = (int64_t)((a.n_groups + kWaves - 1) / kWaves) * a.kv_heads * a.batch;
  const int gpw = wide <= 4 * (int64_t)device_cu_count() ? 1 : kGroupsPerWave;
  tl.blocks = (a.n_groups + kWaves * gpw - 1) / (kWaves * gpw);
  const dim3 grid(tl.blocks + (tl.rows ? (tl.n + 255) / 256 : 0), a.kv_heads, a.batch);
  qk_kernel<BITS, NR><<<grid, dim3(256), bytes, s>>>(a, tl, gpw);
  return hipGetLastError();
}

template <int BITS, int NR>
hipError_t launch_av(const mz_av_args& a, float* part, int parts, int splits, int chunks, hipStream_t s) {
  static std::atomic<uint64_t> raised{0};
  constexpr int bytes = av_lds_bytes<BITS, NR>();
  if constexpr (bytes > 65536) {
    const hipError_t e = set_dynamic_lds((const void*)av_kernel<BITS, NR>, bytes, raised);
    if (e != hipSuccess) return e;
  }
  const dim3 grid((a.head_dim + kRows - 1) / kRows * splits, a.kv_heads, a.batch);
  av_kernel<BITS, NR><<<grid, dim3(256), bytes, s>>>(a, part, parts, chunks);
  return hipGetLastError();
}

template <int BITS>
hipError_t qk_nr(const mz_qk_args& a, const Tail& tl, hipStream_t s) {
  switch (nr_for(a.n_rep)) {
    case 1: return launch_qk<BITS, 1>(a, tl, s);
    case 2: return launch_qk<BITS, 2>(a, tl, s);
    case 4: return launch_qk<BITS, 4>(a, tl, s);
    case 8: return launch_qk<BITS, 8>(a, tl, s);
    default: return launch_qk<BITS, 16>(a, tl, s);
  }
}

template <int BITS>
hipError_t av_nr(const mz_av_args& a, float* part, int parts, int splits, int chunks, hipStream_t s) {
  switch (nr_for(a.n_rep)) {
    case 1: return launch_av<BITS, 1>(a, part, parts, splits, chunks, s);
    case 2: return launch_av<BITS, 2>(a, part, parts, splits, chunks, s);
    case 4: return launch_av<BITS, 4>(a, part, parts, splits, chunks, s);
    case 8: return launch_av<BITS, 8>(a, part, parts, splits, chunks, s);
    default: return launch_av<BITS, 16>(a, part, parts, splits, chunks, s);
  }
}

hipError_t run_qk(const mz_qk_args& a, const Tail& tl, hipStream_t s) {
  switch (a.bits) {
    case 1: return qk_nr<1>(a, tl, s);
    case 2: return qk_nr<2>(a, tl, s);
    case 3: return qk_nr<3>(a, tl, s);
    case 4: return qk_nr<4>(a, tl, s);
    case 5: return qk_nr<5>(a, tl, s);
    case 6: return qk_nr<6>(a, tl, s);
    case 7: return qk_nr<7>(a, tl, s);
    default: return qk_nr<8>(a, tl, s);
  }
}

hipError_t run_av(const mz_av_args& a, float* part, int parts, int splits, int chunks, hipStream_t s) {
  switch (a.bits) {
    case 1: return av_nr<1>(a, part, parts, splits, chunks, s);
    case 2: return av_nr<2>(a, part, parts, splits, chunks, s);
    case 3: return av_nr<3>(a, part, parts, splits, chunks, s);
    case 4: return av_nr<4>(a, part, parts, splits, chunks, s);
    case 5: return av_nr<5>(a, part, parts, splits, chunks, s);
    case 6: return av_nr<6>(a, part, parts, splits, chunks, s);
    case 7: return av_nr<7>(a, part, parts, splits, chunks, s);
    default: return av_nr<8>(a, part, parts, splits, chunks, s);
  }
}

inline bool dtype_ok(int dt) { return dt == MZ_F32 || dt == MZ_BF16 || dt == MZ_F16; }
inline bool aligned8(const void* p) { return ((uintptr_t)p & 7u) == 0; }

int status(hipError_t e) { return e == hipSuccess ? MZ_OK : (int)e; }

}  // namespace rowdot
}  // namespace mz

using namespace mz;
using namespace mz::rowdot;

extern "C" int muzero_qk(const mz_qk_args* a, mz_stream_t stream) {
  if (a == nullptr) return MZ_EINVAL;
  if (a->batch < 0 || a->kv_heads < 1 || a->n_rep < 1 || a->head_dim < 1 || a->n_groups < 0) return MZ_EINVAL;
  if (a->bits < 1 || a->bits > 8 || !dtype_ok(a->io_dtype) || !dtype_ok(a->meta_dtype)) return MZ_EINVAL;
  if (a->n_rep > kMaxRep || a->head_dim > kMaxHeadDim) return MZ_EUNSUPPORTED;
  if (a->batch > 65535 || a->kv_heads > 65535) return MZ_EUNSUPPORTED;
  if (a->batch == 0 || a->n_groups == 0) return MZ_OK;
  if (!a->query || !a->k_packed || !a->k_mn || !a->k_scale || !a->e_key || !a->logits) return MZ_EINVAL;
  if (!aligned8(a->k_packed) || (a->kp_sb & 7) || (a->kp_sh & 7)) return MZ_EINVAL;
  return status(run_qk(*a, Tail{}, (hipStream_t)stream));
}

extern "C" int muzero_av(const mz_av_args* a, mz_stream_t stream) {
  if (a == nullptr) return MZ_EINVAL;
  if (a->batch < 0 || a->kv_heads < 1 || a->n_rep < 1 || a->head_dim < 1 || a->n_tokens < 0) return MZ_EINVAL;
  if (a->bits < 1 || a->bits > 8 || !dtype_ok(a->io_dtype) || !dtype_ok(a->meta_dtype)) return MZ_EINVAL;
  if (a->n_rep > kMaxRep || a->head_dim > kMaxHeadDim) return MZ_EUNSUPPORTED;
  if (a->batch > 65535 || a->kv_heads > 65535) return MZ_EUNSUPPORTED;
  if (a->batch == 0) return MZ_OK;
  if (!a->out || (a->n_tokens > 0 && (!a->weights || !a->v_packed || !a->v_mn || !a->v_scale || !a->e_value)))
    return MZ_EINVAL;
  if (a->n_tokens > 0 && (!aligned8(a->v_packed) || (a->vp_sb & 7) || (a->vp_sh & 7))) return MZ_EINVAL;
  return status(run_av(*a, nullptr, 1, 1, (a->n_tokens + kRows - 1) / kRows, (hipStream_t)stream));
}

// ---------------------------------------------------------------- the whole default path

namespace {

struct Unfused {
  int vp, n_v, len;          // quantized value tokens, dense value rows, all tokens
  int splits, parts, chunks;  // of the prefix's tokens; records per q-head (one more for the tail); 64-token chunks per split
  int64_t ld, rows, logits_bytes, bytes;
};

// whether 16-byte reads fit dense rows [B, H, T, D]
bool tail_vec(const void* p, int64_t sb, int64_t sh, int64_t st, int64_t D, int64_t es) {
  return (((uintptr_t)p | (uintptr_t)(sb * es) | (uintptr_t)(sh * es) | (uintptr_t)(st * es) | (uintptr_t)(D * es)) & 15) == 0;
}

int plan_unfused(const mz_decode_args* a, Unfused& u) {
  if (!a) return MZ_EINVAL;
  if (a->batch < 0 || a->kv_heads < 1 || a->n_rep < 1 || a->head_dim < 1 || a->n_groups < 0 || a->n_residual < 0)
    return MZ_EINVAL;
  if (a->bits < 1 || a->bits > 8 || !dtype_ok(a->io_dtype) || !dtype_ok(a->meta_dtype) || a->out_dtype != a->io_dtype)
    return MZ_EINVAL;
  if (a->n_rep > kMaxRep || a->head_dim > kMaxHeadDim || a->batch > 65535 || a->kv_heads > 65535) return MZ_EUNSUPPORTED;
  const int64_t lk = (int64_t)a->n_groups * kRows, len = lk + a->n_residual;
  const int64_t vp = a->v_prefix ? a->v_prefix : lk;
  if (len < 1 || len >= (int64_t)1 << 30 || vp < lk || vp > len) return MZ_EINVAL;
  u.vp = (int)vp, u.len = (int)len, u.n_v = (int)(len - vp);
  u.ld = (len + 7) / 8 * 8;
  u.rows = (int64_t)a->batch * a->kv_heads * a->n_rep;
  // av: splits of whole chunks, a chunk per wave at least, while the
  // workgroups fill the CUs up to four times (about what their LDS admits at once)
  const int64_t units = std::max<int64_t>(1, (int64_t)a->batch * a->kv_heads * ((a->head_dim + kRows - 1) / kRows));
  const int total = (u.vp + kRows - 1) / kRows;
  int64_t want = 4 * (int64_t)device_cu_count() / units;
  want = std::max<int64_t>(1, std::min<int64_t>(want, (total + kWaves - 1) / kWaves));
  u.chunks = (int)((total + want - 1) / want);
  u.splits = total > 0 ? (total + u.chunks - 1) / u.chunks : 0;
  u.parts = u.splits + (u.n_v > 0 ? 1 : 0);
  const int64_t es = a->io_dtype == MZ_F32 ? 4 : 2;
  u.logits_bytes = (u.rows * u.ld * es + 255) / 256 * 256;
  u.bytes = u.logits_bytes + u.rows * u.parts * a->head_dim * (int64_t)sizeof(float);
  return MZ_OK;
}

}  // namespace

extern "C" int64_t muzero_decode_unfused_workspace_bytes(const mz_decode_args* a) {
  Unfused u;
  return plan_unfused(a, u) == MZ_OK ? u.bytes : -1;
}

extern "C" int muzero_decode_unfused(const mz_decode_args* a, mz_stream_t stream) {
  Unfused u;
  const int st = plan_unfused(a, u);
  if (st != MZ_OK) return st;
  if (a->batch == 0) return MZ_OK;
  if (!a->query || !a->out) return MZ_EINVAL;
  if (a->n_groups > 0 && (!a->k_packed || !a->k_mn || !a->k_scale || !a->e_key)) return MZ_EINVAL;
  if (a->n_groups > 0 && (!aligned8(a->k_packed) || (a->kp_sb & 7) || (a->kp_sh & 7))) return MZ_EINVAL;
  if (u.vp > 0 && (!a->v_packed || !a->v_mn || !a->v_scale || !a->e_value)) return MZ_EINVAL;
  if (u.vp > 0 && (!aligned8(a->v_packed) || (a->vp_sb & 7) || (a->vp_sh & 7))) return MZ_EINVAL;
  if ((a->n_residual > 0 && !a->k_res) || (u.n_v > 0 && !a->v_res)) return MZ_EINVAL;
  if (!a->workspace || ((uintptr_t)a->workspace & 15) || a->workspace_bytes < u.bytes) return MZ_EWORKSPACE;
  const hipStream_t s = (hipStream_t)stream;
  const int64_t es = a->io_dtype == MZ_F32 ? 4 : 2;
  void* logits = a->workspace;
  float* part = (float*)((uint8_t*)a->workspace + u.logits_bytes);
  const int Hq = a->kv_heads * a->n_rep;

  mz_qk_args q{};
  q.batch = a->batch, q.kv_heads = a->kv_heads, q.n_rep = a->n_rep, q.head_dim = a->head_dim, q.bits = a->bits;
  q.n_groups = a->n_groups, q.meta_dtype = a->meta_dtype, q.io_dtype = a->io_dtype, q.scaling = a->scaling;
  q.query = a->query, q.q_sb = a->q_sb, q.q_sh = a->q_sh;
  q.k_packed = a->k_packed, q.kp_sb = a->kp_sb, q.kp_sh = a->kp_sh;
  q.k_mn = a->k_mn, q.k_scale = a->k_scale, q.km_sb = a->km_sb, q.km_sh = a->km_sh, q.e_key = a->e_key;
  q.logits = logits, q.o_sb = Hq * u.ld, q.o_sh = u.ld;
  Tail kt;
  if (a->n_residual > 0) {
    kt.rows = a->k_res, kt.sb = a->kr_sb, kt.sh = a->kr_sh, kt.st = a->kr_st;
    kt.n = a->n_residual, kt.first = a->n_groups * kRows;
    kt.vec = tail_vec(a->k_res, a->kr_sb, a->kr_sh, a->kr_st, a->head_dim, es);
  }
  hipError_t e = run_qk(q, kt, s);
  if (e != hipSuccess) return (int)e;

  const dim3 rows((unsigned)u.rows);
  Tail vt;
  if (u.n_v > 0) {
    vt.rows = a->v_res, vt.sb = a->vr_sb, vt.sh = a->vr_sh, vt.st = a->vr_st, vt.n = u.n_v, vt.first = u.vp;
    vt.vec = tail_vec(a->v_res, a->vr_sb, a->vr_sh, a->vr_st, a->head_dim, es);
  }
#define MZ_SOFTMAX(IOV, HELDV)                                                                                       \
  softmax_kernel<IOV, HELDV><<<rows, dim3(256), softmax_lds(u.len), s>>>(logits, u.ld, u.len, a->kv_heads, a->n_rep, \
                                                                        a->mask, a->mask_sb, vt, a->head_dim, part, u.parts)
#define MZ_SOFTMAX_IO(IOV)                                \
  if (u.len <= kHeldLogits) { MZ_SOFTMAX(IOV, true); } \
  else { MZ_SOFTMAX(IOV, false); }
  if (a->io_dtype == MZ_BF16) { MZ_SOFTMAX_IO(MZ_BF16) }
  else if (a->io_dtype == MZ_F16) { MZ_SOFTMAX_IO(MZ_F16) }
  else { MZ_SOFTMAX_IO(MZ_F32) }
#undef MZ_SOFTMAX_IO
#undef MZ_SOFTMAX
  e = hipGetLastError();
  if (e != hipSuccess) return (int)e;

  if (u.vp > 0) {
    mz_av_args v{};
    v.batch = a->batch, v.kv_heads = a->kv_heads, v.n_rep = a->n_rep, v.head_dim = a->head_dim, v.bits = a->bits;
    v.n_tokens = u.vp, v.meta_dtype = a->meta_dtype, v.io_dtype = a->io_dtype;
    v.weights = logits, v.w_sb = Hq * u.ld, v.w_sh = u.ld;
    v.v_packed = a->v_packed, v.vp_sb = a->vp_sb, v.vp_sh = a->vp_sh;
    v.v_mn = a->v_mn, v.v_scale = a->v_scale, v.vm_sb = a->vm_sb, v.vm_sh = a->vm_sh, v.e_value = a->e_value;
    e = run_av(v, part, u.parts, u.splits, u.chunks, s);
    if (e != hipSuccess) return (int)e;
  }

  const auto sum = a->io_dtype == MZ_BF16  ? sum_splits_kernel<MZ_BF16>
                   : a->io_dtype == MZ_F16 ? sum_splits_kernel<MZ_F16>
                                           : sum_splits_kernel<MZ_F32>;
  sum<<<rows, dim3(256), 0, s>>>(part, u.parts, u.splits, a->head_dim, Hq, a->out, a->out_sb, a->out_sh);
  return status(hipGetLastError());
}
