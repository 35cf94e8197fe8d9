// Logits step of tree construction for gfx950: per row of bf16 draft logits, the top-k (value descending,
// token id ascending) and their log-probabilities value - log Z.
//
// Reference semantics: inference/hf/tree_logits.py:34-46 (torch.topk on the bf16 logits, log Z from an
// fp32 online max/sum) and the fp32 variant inference/hf/ddtree.py:240-245. Here log Z is computed in one
// fixed order of IEEE operations, so that the CPU restatement produces the same bits:
//   the row is cut into pieces of MFD_LZ_PIECE = 2048 elements; piece c has max m_c, and its element
//   512 j + 8 l + e belongs to lane l (l < 64, j < 4, e < 8), which sums its 32 elements in (j, e) order
//   starting from 0:
//     s = fma(E(x), C, s),  C = E(-m_c)             if -60 <= m_c < 64 (E: e^x for every bf16 x with
//                                                    2^-25 <= |x| < 128, rounded to float: exp_bf16_table.h)
//     s = s + exp_det(max(x - m_c, -80))            otherwise (an all -inf piece sums to 0)
//   the 64 lane sums are added pairwise over lane distances 32, 16, 8, 4, 2, 1 (every lane ends with the
//   same value S_c);
//   Z = sum_c S_c exp_det(max(m_c - m, -80)) in piece order (fp64), log Z = float(m + log_det(Z)).
// exp_det and log_det use only IEEE +, *, fma, division and exact power-of-two scaling, with contraction
// disabled; log Z agrees with an fp64 logsumexp to about one fp32 ulp.
//
// Kernel 1 (topk_piece_kernel): one wave per piece: its maximum, its sum S_c, and the largest key of each of its 16
//           groups of 128 elements. No selection and no synchronisation between waves.
// Kernel 2 (topk_row_kernel): one workgroup per row: the k-th largest group maximum t; at least k elements reach t,
//           and all that do lie in the few groups whose maximum does, which are read again (from the caches): their
//           elements from t up are the candidates, whose exact top k it takes. Log Z and the outputs.
// A row of at most 16 pieces is done by one workgroup in one launch.
#include <algorithm>

#include "mfd_common.h"
#include "exp_bf16_table.h"

#define MFD_LZ_PIECE 2048

namespace {

constexpr int PIECE = MFD_LZ_PIECE;  // log Z piece: one wave, 32 elements per lane
constexpr int PW = 16;               // waves per workgroup of kernel 1
constexpr int NT1 = PW * 64;
constexpr int KMAX = 256;
constexpr int MERGE_MAX = 8192;      // accepted sizes (interface): pieces * k (k <= 32), ceil(V / 8192) * k above

__device__ __forceinline__ float pow2i(int k) { return __uint_as_float((uint32_t)(k + 127) << 23); }

__device__ float exp_det(float d) {
#pragma clang fp contract(off)
  const float k = __builtin_rintf(d * 1.44269504088896341f);
  float r = __builtin_fmaf(k, -0.693145751953125f, d);
  r = __builtin_fmaf(k, -1.42860676533018592e-06f, r);
  float p = 2.48015873015873016e-05f;
  p = __builtin_fmaf(p, r, 1.98412698412698413e-04f);
  p = __builtin_fmaf(p, r, 1.38888888888888889e-03f);
  p = __builtin_fmaf(p, r, 8.33333333333333333e-03f);
  p = __builtin_fmaf(p, r, 4.16666666666666667e-02f);
  p = __builtin_fmaf(p, r, 1.66666666666666667e-01f);
  p = __builtin_fmaf(p, r, 0.5f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  return p * pow2i((int)k);
}

__device__ double log_det(double z) {
#pragma clang fp contract(off)
  int e;
  double f = frexp(z, &e);
  if (f < 0.70710678118654752440) {
    f = f * 2.0;
    e -= 1;
  }
  const double s = (f - 1.0) / (f + 1.0);
  const double s2 = s * s;
  double p = 1.0 / 23.0;
  p = __builtin_fma(p, s2, 1.0 / 21.0);
  p = __builtin_fma(p, s2, 1.0 / 19.0);
  p = __builtin_fma(p, s2, 1.0 / 17.0);
  p = __builtin_fma(p, s2, 1.0 / 15.0);
  p = __builtin_fma(p, s2, 1.0 / 13.0);
  p = __builtin_fma(p, s2, 1.0 / 11.0);
  p = __builtin_fma(p, s2, 1.0 / 9.0);
  p = __builtin_fma(p, s2, 1.0 / 7.0);
  p = __builtin_fma(p, s2, 1.0 / 5.0);
  p = __builtin_fma(p, s2, 1.0 / 3.0);
  p = __builtin_fma(p, s2, 1.0);
  const double logf_ = 2.0 * s * p;
  const double de = (double)e;
  return __builtin_fma(de, 6.93147180369123816490e-01, __builtin_fma(de, 1.90821492927058770002e-10, logf_));
}
// ---- the e^x table ------------------------------------------------------------------------------------
// In LDS the 8192 entries are split by sign: e^x of the non-negative magnitudes i at byte 4 i, of the negative
// ones at byte 32768 + 4 i, so that the byte offset of a bf16 bit pattern b is
//   4 min(max((b & 0x7FFF) - 0x3300, 0), 4095) + (b & 0x8000),
// five packed 16-bit operations for two elements. Entry 4095 of the non-negative half (x = 127.5, and every
// larger magnitude and NaN) holds 0: no element of a piece with m_c < 64 is that large, and a NaN adds nothing.
constexpr int ETAB = MFD_EXP_BF16_TABLE_SIZE;
constexpr int ETAB_NEG = 32768;              // byte offset of the negative half; the 16 KB in between are free
constexpr int ETAB_BYTES = ETAB_NEG + ETAB * 2;
__device__ const uint32_t exp_tab_g[ETAB] = {MFD_EXP_BF16_TABLE_INIT};
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t etab_offsets(uint32_t pair) {
  const u16x2 b = __builtin_bit_cast(u16x2, pair);
  u16x2 i = __builtin_elementwise_sub_sat((u16x2)(b << (u16x2){1, 1}), (u16x2){0x6600, 0x6600});
  i = __builtin_elementwise_min(i, (u16x2){ETAB - 2, ETAB - 2});
  // (pair & 0x80008000) | 2 i in one operation (the compiler takes it apart into three)
  uint32_t off;
  asm("v_and_or_b32 %0, %1, %2, %3"
      : "=v"(off)
      : "v"(pair), "s"(0x80008000u), "v"(__builtin_bit_cast(uint32_t, (u16x2)(i << (u16x2){1, 1}))));
  return off;
}
__device__ __forceinline__ float etab_at(const unsigned char* etab, uint32_t byte_off) {
  return *reinterpret_cast<const float*>(etab + byte_off);
}
// The table into LDS by all NT1 threads: entries 8 t .. 8 t + 7 (magnitudes 4 t .. 4 t + 3, both signs).
__device__ __forceinline__ void etab_stage(unsigned char* etab) {
  static_assert(ETAB == 8 * NT1, "eight entries per thread");
  const int t = threadIdx.x;
  const u32x4 a = reinterpret_cast<const u32x4*>(exp_tab_g)[2 * t];
  const u32x4 b = reinterpret_cast<const u32x4*>(exp_tab_g)[2 * t + 1];
  *reinterpret_cast<u32x4*>(etab + 16 * t) = (u32x4){a[0], a[2], b[0], t == NT1 - 1 ? 0u : b[2]};
  *reinterpret_cast<u32x4*>(etab + ETAB_NEG + 16 * t) = (u32x4){a[1], a[3], b[1], b[3]};
}

// Lane sum of one piece: the lane's 32 elements raw[j][e] (piece element 512 j + 8 lane + e) in (j, e) order,
// against the piece maximum m. Elements at piece positions >= nvalid are past the row end: NaNs in raw,
// contributing nothing. The polynomial path (m outside the table's range, rare) reads the elements again
// from psrc, the piece's first element.
__device__ __forceinline__ float piece_lane_sum(const u32x4 (&raw)[4], float m, const uint16_t* psrc, int nvalid,
                                                const unsigned char* etab) {
#pragma clang fp contract(off)
  float s = 0.f;
  if (m >= -60.0f && m < 64.0f) {
    // -m is a bf16 value too: its bits are m's upper half with the sign flipped
    const uint32_t mneg = ((__float_as_uint(m) >> 16) ^ 0x8000u) * 0x10001u;
    const float C = etab_at(etab, etab_offsets(mneg) & 0xFFFFu);
    // the eight table reads of group j + 1 are in flight while those of group j are added (left to itself the compiler
    // waits for every read before the next)
    float x[2][8];
    auto fetch = [&](int j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t off = etab_offsets(raw[j][q]);
        x[j & 1][2 * q] = etab_at(etab, off & 0xFFFFu);
        x[j & 1][2 * q + 1] = etab_at(etab, off >> 16);
      }
    };
    fetch(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < 3) fetch(j + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 8; ++e) s = __builtin_fmaf(x[j & 1][e], C, s);
    }
  } else if (m != -INFINITY) {
    const int l8 = 8 * (int)(threadIdx.x & 63);
#pragma unroll 1
    for (int j = 0; j < 4; ++j)
#pragma unroll 1
      for (int e = 0; e < 8; ++e) {
        const int idx = 512 * j + l8 + e;
        float t = 0.0f;
        if (idx < nvalid) {
          float d = bf2f(psrc[idx]) - m;
          d = d > -80.0f ? d : -80.0f;
          t = exp_det(d);
        }
        s = s + t;
      }
  }
  return s;
}

// ---- wave reductions ------------------------------------------------------------------------------------
template <int N>
__device__ __forceinline__ uint32_t row_ror32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + N, 0xF, 0xF, false);
}
// Sum over the wave, pairwise over lane distances 32, 16, 8, 4, 2, 1: every lane ends with the same value. Once
// the distances above d are added, a lane's value depends only on its number modulo 2 d, so a rotation by d
// within the row of 16 reads the same value as lane ^ d.
__device__ __forceinline__ float wave_sum_tree(float v) {
#pragma clang fp contract(off)
  {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
  {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
  v = v + __uint_as_float(row_ror32<8>(__float_as_uint(v)));
  v = v + __uint_as_float(row_ror32<4>(__float_as_uint(v)));
  v = v + __uint_as_float(row_ror32<2>(__float_as_uint(v)));
  v = v + __uint_as_float(row_ror32<1>(__float_as_uint(v)));
  return v;
}
// wave maximum of a float (uniform result): DPP rotations within rows of 16, then the four row maxima
__device__ __forceinline__ float wave_max_dpp(float v) {
  v = fmaxf(v, __uint_as_float(row_ror32<1>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(row_ror32<2>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(row_ror32<4>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(row_ror32<8>(__float_as_uint(v))));
  const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__float_as_uint(v), 0));
  const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__float_as_uint(v), 16));
  const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__float_as_uint(v), 32));
  const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__float_as_uint(v), 48));
  return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}
// wave maximum of an int, the same way
__device__ __forceinline__ int wave_max_i32(int v) {
  v = std::max(v, (int)row_ror32<1>((uint32_t)v));
  v = std::max(v, (int)row_ror32<2>((uint32_t)v));
  v = std::max(v, (int)row_ror32<4>((uint32_t)v));
  v = std::max(v, (int)row_ror32<8>((uint32_t)v));
  const int r0 = __builtin_amdgcn_readlane(v, 0), r1 = __builtin_amdgcn_readlane(v, 16);
  const int r2 = __builtin_amdgcn_readlane(v, 32), r3 = __builtin_amdgcn_readlane(v, 48);
  return std::max(std::max(r0, r1), std::max(r2, r3));
}
// sum of an int over the wave (uniform result)
__device__ __forceinline__ int wave_sum_i32(int v) {
  v += (int)row_ror32<1>((uint32_t)v);
  v += (int)row_ror32<2>((uint32_t)v);
  v += (int)row_ror32<4>((uint32_t)v);
  v += (int)row_ror32<8>((uint32_t)v);
  return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) + __builtin_amdgcn_readlane(v, 32) +
         __builtin_amdgcn_readlane(v, 48);
}
// inclusive prefix sum over the lanes: within rows of 16, then the row totals handed on
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_add(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ int wave_scan_i32(int v) {
  v = dpp_add<0x111, 0xF>(v);  // row_shr:1, 2, 4, 8
  v = dpp_add<0x112, 0xF>(v);
  v = dpp_add<0x114, 0xF>(v);
  v = dpp_add<0x118, 0xF>(v);
  v = dpp_add<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

// ---- keys -----------------------------------------------------------------------------------------------
// Selection keys are the bf16 bit patterns as signed 16-bit numbers with the magnitude bits of negative values
// flipped (larger value = larger key; -0 has key -1, right below +0). For patterns without the sign bit the key is
// the pattern itself.
constexpr int KEY_MIN = -32768;
__device__ __forceinline__ uint32_t keys2(uint32_t pair) {  // two at once
  const i16x2 s = __builtin_bit_cast(i16x2, pair) >> (i16x2){15, 15};
  return pair ^ (__builtin_bit_cast(uint32_t, s) & 0x7FFF7FFFu);
}
__device__ __forceinline__ int key1(uint16_t b) { return (int)(int16_t)(b ^ (((int16_t)b >> 15) & 0x7FFF)); }
__device__ __forceinline__ uint32_t max2(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t,
                            __builtin_elementwise_max(__builtin_bit_cast(i16x2, a), __builtin_bit_cast(i16x2, b)));
}
// candidate key: larger = better (value descending, then token id ascending); never 0
__device__ __forceinline__ uint64_t cand_key(uint16_t raw, uint32_t idx) {
  return ((uint64_t)float_order_key(bf2f(raw) + 0.0f) << 32) | (uint64_t)(0xFFFFFFFFu - idx);
}
__device__ __forceinline__ float key_value(uint64_t key) {
  const uint32_t hi = (uint32_t)(key >> 32);
  return __uint_as_float((hi & 0x80000000u) ? (hi & 0x7FFFFFFFu) : ~hi);
}

struct TopkArgs {
  const uint16_t* logits;
  int64_t row_stride;
  int rows, V, k;
  int npieces;         // (m, S) pairs per row
  int ng;              // group keys per piece: 16 (128 elements each), 4 (512 each) for k < 4
  float* ws_m;         // [rows * npieces]
  double* ws_s;        // [rows * npieces]
  int16_t* ws_g;       // [rows * npieces * ng] the largest key1 of each group, in index order
  float* out_logp;     // [rows, k]
  void* out_ids;       // [rows, k] int32 or int64
  int ids_int64;
  float* out_logz;     // [rows] or null
  const int32_t* vocab_ids;  // [V] token id of each logit column, or null (column = token id)
};

// The (m, S) of the row's first 256 pieces, piece c in lane c % 64, entry c / 64 (loaded before they are needed).
struct PieceSums {
  float m[4];
  double s[4];
};
__device__ __forceinline__ PieceSums load_piece_sums(const TopkArgs& a, int row) {
  const int lane = threadIdx.x & 63;
  const int np = a.npieces;
  PieceSums p;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int c = lane + 64 * r;
    p.m[r] = c < np ? a.ws_m[(int64_t)row * np + c] : -INFINITY;
    p.s[r] = c < np ? a.ws_s[(int64_t)row * np + c] : 0.0;
  }
  return p;
}
// log Z of row `row` from its pieces' (m, S), formed by one wave: the terms S_c exp_det(m_c - m) in parallel,
// added in piece order by a chain of lane reads (pieces past 256 through LDS scratch `terms` of npieces
// doubles); wave-uniform result.
__device__ float row_logz(const TopkArgs& a, int row, const PieceSums& p, double* terms) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int np = a.npieces;
  const float* mc = a.ws_m + (int64_t)row * np;
  const double* sc = a.ws_s + (int64_t)row * np;
  float m = fmaxf(fmaxf(p.m[0], p.m[1]), fmaxf(p.m[2], p.m[3]));
  for (int c = lane + 256; c < np; c += 64) m = fmaxf(m, mc[c]);
  m = wave_max_dpp(m);
  if (m == -INFINITY) return -INFINITY;
  // a piece whose maximum is -inf adds +0, which leaves the non-negative sum unchanged
  auto term = [&](float mcc, double s) -> double {
    if (mcc == -INFINITY) return 0.0;
    float d = mcc - m;
    d = d > -80.0f ? d : -80.0f;
    return s * (double)exp_det(d);
  };
  // the terms go to LDS, then every lane adds them in piece order (two per 16-byte read, eight reads in flight)
  for (int r = 0; r < 4; ++r)
    if (lane + 64 * r < np) terms[lane + 64 * r] = term(p.m[r], p.s[r]);
  for (int c = lane + 256; c < np; c += 64) terms[c] = term(mc[c], sc[c]);
  const int np2 = (np + 1) & ~1;
  if (lane == 0 && np2 != np) terms[np] = 0.0;  // adding +0 leaves the non-negative sum unchanged
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_wave_barrier();
  typedef double f64x2 __attribute__((ext_vector_type(2)));
  const f64x2* t2 = reinterpret_cast<const f64x2*>(terms);
  double z = 0.0;
  int c = 0;
  for (; c + 16 <= np2; c += 16) {
    f64x2 x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = t2[c / 2 + i];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      z = z + x[i][0];
      z = z + x[i][1];
    }
  }
  for (; c < np2; c += 2) {
    const f64x2 x = t2[c / 2];
    z = z + x[0];
    z = z + x[1];
  }
  return (float)((double)m + log_det(z));
}

// ---- the top k of a row's candidates ----------------------------------------------------------------------
constexpr int NBIN = 1024;
constexpr int COUNT_MAX = 256;  // up to here a candidate's rank is counted against all others
constexpr int CAND_MAX = 1024;
constexpr int TIED_MAX = 512;   // k <= 32: beyond, the bisection
// Counters of the bisections: one for each of the 16 bits of a key, one for the elements above it, one for each bit of
// an element's index (k = 1 takes MERGE_MAX pieces: up to 2^24 elements, whose number has 25 bits)
constexpr int VBITS = 32 - __builtin_clz(MERGE_MAX * PIECE);
constexpr int NCOUNT = 16 + 1 + VBITS;
static_assert((int64_t)MERGE_MAX * PIECE < (int64_t)1 << 31 && NCOUNT <= 64, "cleared by one wave");
struct MergeLds {
  uint32_t hist[NBIN];
  __attribute__((aligned(16))) uint64_t cand[CAND_MAX + 2];
  __attribute__((aligned(16))) uint64_t sel[KMAX];
  uint16_t bnd[CAND_MAX];
  uint16_t glist[2 * KMAX];  // the groups whose elements are looked at
  int wmax[16], wsum[16];
  int count[NCOUNT];
  int n, nsel, nb, bin, need, ng, top;
  float logz;
};

__device__ __forceinline__ void put_one(const TopkArgs& a, int row, int pos, uint64_t key, float logz) {
  uint32_t idx = 0xFFFFFFFFu - (uint32_t)key;
  if (a.vocab_ids) idx = (uint32_t)a.vocab_ids[idx];
  a.out_logp[(int64_t)row * a.k + pos] = key_value(key) - logz;
  if (a.ids_int64)
    static_cast<int64_t*>(a.out_ids)[(int64_t)row * a.k + pos] = (int64_t)idx;
  else
    static_cast<int32_t*>(a.out_ids)[(int64_t)row * a.k + pos] = (int32_t)idx;
}

// The bin b that holds the k-th largest of the histogrammed values and how many of that bin are needed, by one wave:
// lane l holds bins 16 (63 - l) .. + 15, an inclusive scan over the lanes gives the suffix sums. False (every lane) if
// fewer than k values are histogrammed.
__device__ __forceinline__ bool kth_bin(const uint32_t* hist, int k, int* bin, int* need) {
  const int lane = threadIdx.x & 63;
  const int b0 = 16 * (63 - lane);
  int h[16];
#pragma unroll
  for (int i = 0; i < 16; i += 4) {
    const u32x4 x = *reinterpret_cast<const u32x4*>(hist + b0 + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) h[i + e] = (int)x[e];
  }
  int own = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) own += h[i];
  const int inc = wave_scan_i32(own);
  const bool here = inc >= k && inc - own < k;  // one lane, if any
  if (here) {
    int above = inc - own, b = -1;
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      if (b < 0) {
        if (above + h[i] >= k)
          b = b0 + i;
        else
          above += h[i];
      }
    }
    *bin = b;
    *need = k - above;
  }
  return __builtin_amdgcn_ballot_w64(here) != 0;
}

// Called by all NTH threads of a workgroup, after a barrier, with n >= k candidates in ml.cand and log Z in ml.logz;
// top: the largest candidate's 16-bit value key. Few candidates (what k <= 32 nearly always leaves) are ranked by
// counting, n broadcast reads each. More: the value keys' distance from the largest, clamped to 1024 bins, is
// histogrammed, the bin that holds the k-th largest is read off the suffix sums, the candidates above it are taken,
// those in it by their rank among themselves (one value unless clamped, so ties by token id), and the k taken are
// ranked by counting, four threads each. False, with nothing written, if that bin holds more than max_tied candidates.
template <int NTH>
__device__ bool merge_row(const TopkArgs& a, int row, int n, int top, int max_tied, MergeLds& ml) {
  const int tid = threadIdx.x;
  const int k = a.k;
  uint64_t* cand = ml.cand;
  const float logz = ml.logz;
  if (n <= COUNT_MAX) {
    if (tid < n) {
      const uint64_t v = cand[tid];
      int r = 0;
      for (int i = 0; i < n; i += 2) {
        const u64x2 x = *reinterpret_cast<const u64x2*>(cand + i);
        r += (x[0] > v ? 1 : 0) + (x[1] > v && i + 1 < n ? 1 : 0);
      }
      if (r < k) put_one(a, row, r, v, logz);
    }
    return true;
  }
  for (int i = tid; i < NBIN; i += NTH) ml.hist[i] = 0;
  if (tid < KMAX) ml.sel[tid] = 0;
  if (tid == 0) ml.nsel = ml.nb = 0;
  auto bin_of = [&](uint64_t v) -> int {
    const int d = NBIN - 1 - (top - (int)(v >> 48));
    return d < 0 ? 0 : (d > NBIN - 1 ? NBIN - 1 : d);
  };
  __syncthreads();
  for (int i = tid; i < n; i += NTH) atomicAdd(&ml.hist[bin_of(cand[i])], 1u);
  __syncthreads();
  if (tid < 64) kth_bin(ml.hist, k, &ml.bin, &ml.need);
  __syncthreads();
  const int bin = ml.bin, need = ml.need;
  if ((int)ml.hist[bin] > max_tied) return false;
  for (int i = tid; i < n; i += NTH) {
    const uint64_t v = cand[i];
    const int b = bin_of(v);
    if (b > bin)
      ml.sel[atomicAdd(&ml.nsel, 1)] = v;
    else if (b == bin)
      ml.bnd[atomicAdd(&ml.nb, 1)] = (uint16_t)i;
  }
  __syncthreads();
  const int nb = ml.nb;
  for (int i = tid; i < nb; i += NTH) {
    const uint64_t v = cand[ml.bnd[i]];
    int r = 0;
    if (nb > need)
      for (int j = 0; j < nb; ++j) r += cand[ml.bnd[j]] > v ? 1 : 0;
    if (r < need) ml.sel[atomicAdd(&ml.nsel, 1)] = v;
  }
  __syncthreads();
  // four threads per selected key: thread p of a key reads entries 8 i + 2 p, + 1
  static_assert(NTH / 4 >= KMAX || NTH / 4 >= 32, "one pass");
  const int s = tid >> 2;
  const uint64_t v = s < k ? ml.sel[s] : 0ull;
  int r = 0;
  for (int i = 2 * (tid & 3); i < k; i += 8) {
    const u64x2 x = *reinterpret_cast<const u64x2*>(ml.sel + i);
    r += (x[0] > v ? 1 : 0) + (x[1] > v ? 1 : 0);
  }
  r += __builtin_amdgcn_update_dpp(0, r, 0xB1, 0xF, 0xF, false);  // lane ^ 1
  r += __builtin_amdgcn_update_dpp(0, r, 0x4E, 0xF, 0xF, false);  // lane ^ 2
  if (s < k && (tid & 3) == 0) put_one(a, row, r, v, logz);
  return true;
}

// Kernel 2's work for one row, by all NTH threads of a workgroup, once the row's (m, S) and group keys are in memory.
// The groups' keys are histogrammed by their distance from the largest (1024 bins, 8 octaves of bf16) and the k-th
// largest, t, is read off the suffix sums (or found by bisection, where it lies further down). Listed are the groups
// above t (fewer than k) and the first k of those at t in index order, which hold the first k elements equal to t:
// nearly always k groups and a few, never more than 2 k. Their elements from t up are the candidates; should they not
// fit (rows of ties, masked rows), the k-th largest key among the listed groups and the index of the last equal
// element taken are found by bisection over counts. Wave 0 forms log Z while the others wait for the elements.
// What bounds it: a chain of two trips to memory and about ten barriers. 128 rows, k = 8: 5.7 us (5.4 for merging
// the pieces' top-8 lists); 120 rows, k = 256: 11.2 us (1.83 ms for 256 serial maxima over 7936 listed keys).
template <int NTH>
__device__ void row_topk(const TopkArgs& a, int row, MergeLds& ml, double* terms) {
  constexpr int NW = NTH / 64;
  constexpr int NQ = 4;  // loads of four keys held in registers per thread; further ones are read again in every pass
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int k = a.k;
  PieceSums ps;
  if (w == 0) ps = load_piece_sums(a, row);
  if (k == 0) {
    if (w == 0) {
      const float z = row_logz(a, row, ps, terms);
      if (lane == 0) a.out_logz[row] = z;
    }
    return;
  }
  // thread t holds the groups [t gp, (t + 1) gp)
  const int ngroups = a.npieces * a.ng;
  const int gp = ((ngroups + NTH - 1) / NTH + 3) & ~3;
  const uint64_t* gsrc = reinterpret_cast<const uint64_t*>(a.ws_g + (int64_t)row * ngroups);
  const int g0 = tid * gp, g1 = std::min(ngroups, g0 + gp);
  uint64_t kq[NQ];
#pragma unroll
  for (int c = 0; c < NQ; ++c) kq[c] = g0 + 4 * c < g1 ? gsrc[(g0 >> 2) + c] : 0ull;
  auto for_groups = [&](auto visit) {  // visit(key, group)
    auto four = [&](uint64_t q, int g) {
#pragma unroll
      for (int i = 0; i < 4; ++i) visit((int)(int16_t)(uint16_t)(q >> (16 * i)), g + i);
    };
#pragma unroll
    for (int c = 0; c < NQ; ++c)
      if (g0 + 4 * c < g1) four(kq[c], g0 + 4 * c);
    for (int g = g0 + 4 * NQ; g < g1; g += 4) four(gsrc[g >> 2], g);
  };
  for (int i = tid; i < NBIN; i += NTH) ml.hist[i] = 0;
  if (tid == 0) {
    ml.n = 0;
    ml.bin = -1;
  }
  if (tid < NCOUNT) ml.count[tid] = 0;
  int top = KEY_MIN;
  for_groups([&](int key, int) { top = std::max(top, key); });
  top = wave_max_i32(top);
  if (lane == 0) ml.wmax[w] = top;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NW; ++i) top = std::max(top, ml.wmax[i]);
  const int lsh = a.ng == 16 ? 4 : 6;  // a group is 8 << lsh elements
  int t = k == 1 ? top : KEY_MIN;      // KEY_MIN: fewer than k groups, every element is taken
  bool below = false;
  if (k > 1 && (a.V + (8 << lsh) - 1) >> (lsh + 3) >= k) {
    for_groups([&](int key, int) {
      const int d = NBIN - 1 - (top - key);
      if (d >= 0) atomicAdd(&ml.hist[d], 1u);
    });
    __syncthreads();
    if (w == 0) kth_bin(ml.hist, k, &ml.bin, &ml.need);
    __syncthreads();
    below = ml.bin < 0;
    t = top - (NBIN - 1 - ml.bin);
  }
  if (below) {
    // further down than the bins reach
    uint32_t T = 0;
#pragma unroll 1
    for (int bit = 15; bit >= 0; --bit) {
      const int cut = (int)(T | (1u << bit)) - 32768;
      int own = 0;
      for_groups([&](int key, int) { own += key >= cut ? 1 : 0; });
      own = wave_sum_i32(own);
      if (lane == 0 && own) atomicAdd(&ml.count[bit], own);
      __syncthreads();
      if (ml.count[bit] >= k) T |= 1u << bit;
    }
    t = (int)T - 32768;
    __syncthreads();
    if (tid < NCOUNT) ml.count[tid] = 0;
  }
  if (t == 0) t = -1;  // -0 counts as 0
  auto at_t = [&](int key) -> bool { return t == -1 ? key == 0 || key == -1 : key == t; };
  // the list; both counts in one prefix sum (fewer than k groups above t, at most 2^15 at it)
  int both = 0;
  for_groups([&](int key, int) { both += at_t(key) ? 1 : key > t ? 1 << 16 : 0; });
  const int inc = wave_scan_i32(both);
  if (lane == 63) ml.wsum[w] = inc;
  __syncthreads();
  int before = inc - both, all = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int x = ml.wsum[i];
    before += i < w ? x : 0;
    all += x;
  }
  const int nabove = all >> 16, nl = nabove + std::min(all & 0xFFFF, k);
  if (both) {
    int pa = before >> 16, pe = before & 0xFFFF;
    for_groups([&](int key, int g) {
      if (at_t(key)) {
        if (pe < k) ml.glist[nabove + pe] = (uint16_t)g;
        ++pe;
      } else if (key > t) {
        ml.glist[pa++] = (uint16_t)g;
      }
    });
  }
  __syncthreads();
  // The listed groups' elements, eight per lane and step: step u is 16 or 64 lanes' share of a group.
  const uint16_t* src = a.logits + (int64_t)row * a.row_stride;
  const int steps = nl << lsh;
  auto start_of = [&](int u) -> int { return 8 * (((int)ml.glist[u >> lsh] << lsh) + (u & ((1 << lsh) - 1))); };
  if (w == 0) {
    const float z = row_logz(a, row, ps, terms);
    if (lane == 0) ml.logz = z;
  } else {
    constexpr int ST = NTH - 64;
    const i16x2 under = {(int16_t)(t - 1), (int16_t)(t - 1)};  // t > KEY_MIN here or every element is taken
    for (int u0 = tid - 64 - lane; u0 < steps; u0 += 4 * ST) {
      u32x4 x[4];
      int i0[4];
#pragma unroll
      for (int h = 0; h < 4; ++h) {  // four loads in flight; past the list the row's first elements, not counted
        const int u = u0 + lane + h * ST;
        i0[h] = u < steps ? start_of(u) : a.V;
        x[h] = *reinterpret_cast<const u32x4*>(src + (i0[h] < a.V ? i0[h] : 0));
      }
      uint32_t hits = 0;  // bit 8 h + e
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        uint32_t m = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          // key > t - 1: the sign of the saturated difference, in both halves
          const uint32_t d = __builtin_bit_cast(
              uint32_t, __builtin_elementwise_sub_sat(under, __builtin_bit_cast(i16x2, keys2(x[h][q]))));
          m |= (((d >> 15) & 1u) | ((d >> 30) & 2u)) << (2 * q);
        }
        if (t == KEY_MIN) m = 0xFFu;
        const int rest = a.V - i0[h];
        if (rest < 8) m &= rest <= 0 ? 0u : (1u << rest) - 1u;
        hits |= m << (8 * h);
      }
      const int mine = __builtin_popcount(hits);
      const int inc = wave_scan_i32(mine);
      const int total = __builtin_amdgcn_readlane(inc, 63);
      if (total == 0) continue;
      int base = 0;
      if (lane == 0) base = atomicAdd(&ml.n, total);
      int pos = __builtin_amdgcn_readfirstlane(base) + inc - mine;
      for (; hits && pos < CAND_MAX; hits &= hits - 1, ++pos) {
        const int b = __builtin_ctz(hits);
        const int idx = start_of(u0 + lane + (b >> 3) * ST) + (b & 7);
        ml.cand[pos] = cand_key(src[idx], (uint32_t)idx);
      }
    }
  }
  __syncthreads();
  const int n = ml.n;
  if (tid == 0 && a.out_logz) a.out_logz[row] = ml.logz;
  // (For k <= 32 hundreds of candidates are a row of few groups, or one whose largest values lie close together, or
  // ties. 8 rows, k = 8, by the bisection and so: 512 values 35 -> 11 us, 20000 falling from the first column on
  // 35 -> 13, 151936 sorted 39 -> 16. Many equal ones are settled sooner by the bisection than by counting them against each
  // other: 151936 equal values 41 against 86.)
  if (n > CAND_MAX || !merge_row<NTH>(a, row, n, top + 32768, k <= 32 ? TIED_MAX : CAND_MAX, ml)) {
    auto norm = [](int key) -> int { return key == -1 ? 0 : key; };
    auto elem = [](const u32x4& x, int e) -> uint16_t { return (uint16_t)((e & 1) ? x[e >> 1] >> 16 : x[e >> 1] & 0xFFFFu); };
    auto for_elements = [&](auto visit) {  // visit(the eight elements, the index of the first)
      for (int u = tid; u < steps; u += NTH) {
        const int i0 = start_of(u);
        if (i0 < a.V) visit(*reinterpret_cast<const u32x4*>(src + i0), i0);
      }
    };
    auto count = [&](int slot, auto pred) -> int {  // elements with pred, over the workgroup
      int own = 0;
      for_elements([&](const u32x4& x, int i0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) own += i0 + e < a.V && pred(norm(key1(elem(x, e))), i0 + e) ? 1 : 0;
      });
      own = wave_sum_i32(own);
      if (lane == 0 && own) atomicAdd(&ml.count[slot], own);
      __syncthreads();
      return ml.count[slot];
    };
    __syncthreads();
    if (tid == 0) ml.n = 0;
    uint32_t T = 0;
#pragma unroll 1
    for (int bit = 15; bit >= 0; --bit) {
      const int cut = (int)(T | (1u << bit)) - 32768;
      if (count(bit, [&](int key, int) { return key >= cut; }) >= k) T |= 1u << bit;
    }
    const int cut = (int)T - 32768;
    const int need = k - count(16, [&](int key, int) { return key > cut; });
    uint32_t I = 0;  // the largest I with fewer than `need` equal elements below it: the last one taken
    const int top_bit = 31 - __builtin_clz(a.V);
#pragma unroll 1
    for (int bit = top_bit; bit >= 0; --bit) {
      const int c = (int)(I | (1u << bit));
      if (count(17 + top_bit - bit, [&](int key, int idx) { return key == cut && idx < c; }) < need) I |= 1u << bit;
    }
    const int last = (int)I;
    for_elements([&](const u32x4& x, int i0) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int key = norm(key1(elem(x, e)));
        if (i0 + e < a.V && (key > cut || (key == cut && i0 + e <= last))) {
          const int pos = atomicAdd(&ml.n, 1);
          if (pos < CAND_MAX) ml.cand[pos] = cand_key(elem(x, e), (uint32_t)(i0 + e));
        }
      }
    });
    __syncthreads();
    merge_row<NTH>(a, row, k, top + 32768, CAND_MAX, ml);
  }
}

// ---- kernel 1 -------------------------------------------------------------------------------------------
// What bounds it: the read of the logits, then per element 4.5 VALU and one LDS read of the sum (the table lookups),
// about half of the load's time at eight waves per SIMD. The selection's share is the group maxima, about one
// operation per element: the maximum of raw patterns (one packed operation per two elements) is the key of the largest
// value unless every value is negative; a wave with such a group, or a NaN, forms the keys. 128 x 151936: 10.8 us
// (3.6 TB/s; loads and maxima alone about 9), against 15.4 for a kernel that also took every piece's top 8;
// 120 x 248320: 13 us, against 3.9 ms for one that kept sorted lists of 32 keys per thread for k > 32. Selecting per
// workgroup of 16 pieces (thresholds exchanged over LDS between two barriers) instead of per row: 14.4 us.
// ROW: rows of at most PW pieces, one workgroup per row, which also takes its top k.
template <bool ROW>
__global__ __launch_bounds__(NT1) __attribute__((amdgpu_waves_per_eu(ROW ? 4 : 8))) void topk_piece_kernel(TopkArgs a) {
  __shared__ __attribute__((aligned(16))) unsigned char etab[ETAB_BYTES];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int step = ROW ? PW : (int)gridDim.x * PW;
  const int total = ROW ? a.npieces : a.rows * a.npieces;
  int pid = ROW ? w : (int)blockIdx.x * PW + w;
  int row = ROW ? (int)blockIdx.x : pid / a.npieces;
  int piece = ROW ? w : pid - row * a.npieces;
  const int drow = ROW ? 0 : step / a.npieces, dpiece = step - drow * a.npieces;
  // group j of a piece: elements 512 j + 8 lane + e; past the row end a NaN of the lowest key, which adds nothing
  auto load = [&](u32x4(&raw)[4]) {
    const uint16_t* psrc = a.logits + (int64_t)row * a.row_stride + (int64_t)piece * PIECE;
    const int nvalid = a.V - piece * PIECE;
    if (nvalid >= PIECE) {
#pragma unroll
      for (int j = 0; j < 4; ++j) raw[j] = *reinterpret_cast<const u32x4*>(psrc + 512 * j + 8 * lane);
    } else {
      // a group starting before the row end is read whole (the buffer holds rows * row_stride elements, row_stride a
      // multiple of 8)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i0 = 512 * j + 8 * lane;
        u32x4 x = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};
        if (i0 < nvalid) x = *reinterpret_cast<const u32x4*>(psrc + i0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (i0 + 2 * q >= nvalid) x[q] |= 0xFFFFu;
          if (i0 + 2 * q + 1 >= nvalid) x[q] |= 0xFFFF0000u;
        }
        raw[j] = x;
      }
    }
  };
  u32x4 raw[4];
  if (pid < total) load(raw);
  etab_stage(etab);
  __syncthreads();
  while (pid < total) {
    int gm[4];  // the largest key of the lane's row of 16 lanes, in group j
    auto group_max = [&](bool keyed) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t x = keyed ? keys2(raw[j][0]) : raw[j][0];
#pragma unroll
        for (int q = 1; q < 4; ++q) x = max2(x, keyed ? keys2(raw[j][q]) : raw[j][q]);
        gm[j] = std::max((int)(int16_t)(x & 0xFFFFu), (int)x >> 16);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) gm[j] = std::max(gm[j], (int)row_ror32<1>((uint32_t)gm[j]));
#pragma unroll
      for (int j = 0; j < 4; ++j) gm[j] = std::max(gm[j], (int)row_ror32<2>((uint32_t)gm[j]));
#pragma unroll
      for (int j = 0; j < 4; ++j) gm[j] = std::max(gm[j], (int)row_ror32<4>((uint32_t)gm[j]));
#pragma unroll
      for (int j = 0; j < 4; ++j) gm[j] = std::max(gm[j], (int)row_ror32<8>((uint32_t)gm[j]));
    };
    auto wave_of_rows = [&](int v) -> int {
      return std::max(std::max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
                      std::max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
    };
    group_max(false);
    const int wmax = wave_of_rows(std::max(std::max(gm[0], gm[1]), std::max(gm[2], gm[3])));
    float m = __uint_as_float((uint32_t)wmax << 16);
    const bool neg = std::min(std::min(gm[0], gm[1]), std::min(gm[2], gm[3])) < 0;
    if (__builtin_amdgcn_ballot_w64(neg) != 0 || wmax > 0x7F80) {
      // negative maxima or a NaN: from the keys, and the maximum (which leaves NaNs out) from the values
      group_max(true);
      float x = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          x = fmaxf(x, fmaxf(__uint_as_float(raw[j][q] << 16), __uint_as_float(raw[j][q] & 0xFFFF0000u)));
      m = wave_max_dpp(x);
    }
    const int64_t at = (int64_t)row * a.npieces + piece;
    if (a.k > 0) {
      if (a.ng == 16) {
        // lane row r has the maxima of groups 4 j + r: a 4 x 4 transpose over the rows, then it has those of 4 r + j
        auto swap16 = [](int& x, int& y) {
          const auto p = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)y, false, false);
          x = (int)p[0];
          y = (int)p[1];
        };
        auto swap32 = [](int& x, int& y) {
          const auto p = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)y, false, false);
          x = (int)p[0];
          y = (int)p[1];
        };
        swap16(gm[0], gm[1]);
        swap16(gm[2], gm[3]);
        swap32(gm[0], gm[2]);
        swap32(gm[1], gm[3]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) gm[j] = wave_of_rows(gm[j]);
      }
      const uint32_t lo = ((uint32_t)gm[0] & 0xFFFFu) | ((uint32_t)gm[1] << 16);
      const uint32_t hi = ((uint32_t)gm[2] & 0xFFFFu) | ((uint32_t)gm[3] << 16);
      if ((lane & 15) == 0 && lane < a.ng * 4)
        reinterpret_cast<uint64_t*>(a.ws_g)[at * (a.ng / 4) + (lane >> 4)] = ((uint64_t)hi << 32) | lo;
    }
    const uint16_t* psrc = a.logits + (int64_t)row * a.row_stride + (int64_t)piece * PIECE;
    const float ssum = wave_sum_tree(piece_lane_sum(raw, m, psrc, a.V - piece * PIECE, etab));
    if (lane == 0) {
      a.ws_m[at] = m;
      a.ws_s[at] = (double)ssum;
    }
    if constexpr (ROW) break;
    pid += step;
    row += drow;
    piece += dpiece;
    if (piece >= a.npieces) {
      piece -= a.npieces;
      ++row;
    }
    if (pid < total) load(raw);
  }
  if constexpr (ROW) {
    __shared__ MergeLds ml;
    __shared__ double terms[PW + 2];
    __syncthreads();  // the row's maxima, sums and group keys are written
    row_topk<NT1>(a, blockIdx.x, ml, terms);
  }
}

// ---- kernel 2 -------------------------------------------------------------------------------------------
template <int NTH>
__global__ __launch_bounds__(NTH) void topk_row_kernel(TopkArgs a) {
  extern __shared__ __align__(16) unsigned char dyn[];  // npieces + 1 doubles
  __shared__ MergeLds ml;
  row_topk<NTH>(a, blockIdx.x, ml, reinterpret_cast<double*>(dyn));
}

}  // namespace

extern "C" int64_t mfd_topk_logz_workspace_bytes(int rows, int V, int k) {
  const int64_t npieces = ((int64_t)V + PIECE - 1) / PIECE;
  // per piece: m (4 bytes), S (8) and 8 per rank, of which the group keys take at most 32 (the size is the interface's)
  return (int64_t)rows * npieces * (4 + 8 + 8 * (int64_t)(k > 0 ? k : 1)) + 64;
}

static int topk_logz_impl(const uint16_t* logits, int rows, int V, int64_t row_stride, int k, float* out_logp,
                          void* out_ids, int ids_int64, float* out_logz, const int32_t* vocab_ids, void* workspace,
                          int64_t workspace_bytes, void* stream) {
  if (rows < 0 || V < 1 || k < 0 || k > V)
    return mfd_set_error(MFD_ERR_INVALID_ARG, "mfd_topk_logz: bad sizes rows=%d V=%d k=%d", rows, V, k);
  if (k > KMAX) return mfd_set_error(MFD_ERR_UNSUPPORTED, "mfd_topk_logz: k=%d > %d", k, KMAX);
  const int npieces = (V + PIECE - 1) / PIECE;
  const int kk = k > 0 ? k : 1;
  const int nlists = kk <= 32 ? npieces : (V + 8191) / 8192;
  if ((int64_t)nlists * kk > MERGE_MAX)
    return mfd_set_error(MFD_ERR_UNSUPPORTED, "mfd_topk_logz: V=%d with k=%d exceeds the merge capacity", V, k);
  if (row_stride < V || (row_stride % 8) != 0 || (reinterpret_cast<uintptr_t>(logits) % 16) != 0)
    return mfd_set_error(MFD_ERR_UNSUPPORTED, "mfd_topk_logz: rows must be 16-byte aligned (stride %lld)",
                         (long long)row_stride);
  if (rows == 0) return MFD_OK;
  if (!logits || (k > 0 && (!out_logp || !out_ids)) || (k == 0 && !out_logz))
    return mfd_set_error(MFD_ERR_INVALID_ARG, "mfd_topk_logz: null pointer");
  const int64_t need = mfd_topk_logz_workspace_bytes(rows, V, k);
  if (!workspace || workspace_bytes < need)
    return mfd_set_error(MFD_ERR_INVALID_ARG, "mfd_topk_logz: workspace of %lld bytes needed", (long long)need);
  char* ws = static_cast<char*>(workspace);
  double* s = reinterpret_cast<double*>(ws + (int64_t)rows * npieces * kk * 8);
  float* m = reinterpret_cast<float*>(ws + (int64_t)rows * npieces * (kk * 8 + 8));
  // the group keys take up to 32 of the 8 max(k, 1) bytes per piece
  const int ng = kk >= 4 ? 16 : 4;
  TopkArgs a{logits, row_stride, rows, V, k, npieces, ng, m, s, reinterpret_cast<int16_t*>(ws), out_logp, out_ids, ids_int64,
             out_logz, vocab_ids};
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (npieces <= PW) {
    hipLaunchKernelGGL(topk_piece_kernel<true>, dim3((unsigned)rows), dim3(NT1), 0, st, a);
    MFD_CHECK_LAUNCH();
    return MFD_OK;
  }
  // one wave per piece while that fits two workgroups per CU; beyond, the waves take further pieces in turn
  const int64_t total = (int64_t)rows * npieces;
  const dim3 grid((unsigned)std::min<int64_t>((total + PW - 1) / PW, 2 * (int64_t)mfd_num_cus()));
  hipLaunchKernelGGL(topk_piece_kernel<false>, grid, dim3(NT1), 0, st, a);
  MFD_CHECK_LAUNCH();
  const size_t smem = (size_t)((npieces + 3) & ~1) * sizeof(double);
  if (kk <= 32) {
    const int rc = mfd_set_max_lds(reinterpret_cast<const void*>(&topk_row_kernel<256>), 128 * 1024);
    if (rc != MFD_OK) return rc;
    hipLaunchKernelGGL(topk_row_kernel<256>, dim3(rows), dim3(256), smem, st, a);
  } else {
    const int rc = mfd_set_max_lds(reinterpret_cast<const void*>(&topk_row_kernel<1024>), 128 * 1024);
    if (rc != MFD_OK) return rc;
    hipLaunchKernelGGL(topk_row_kernel<1024>, dim3(rows), dim3(1024), smem, st, a);
  }
  MFD_CHECK_LAUNCH();
  return MFD_OK;
}

extern "C" int mfd_topk_logz(const uint16_t* logits, int rows, int V, int64_t row_stride, int k, float* out_logp,
                             void* out_ids, int ids_int64, float* out_logz, void* workspace, int64_t workspace_bytes,
                             void* stream) {
  return topk_logz_impl(logits, rows, V, row_stride, k, out_logp, out_ids, ids_int64, out_logz, nullptr, workspace,
                        workspace_bytes, stream);
}

extern "C" int mfd_topk_logz_vocab(const uint16_t* logits, int rows, int V, int64_t row_stride, int k,
                                   float* out_logp, void* out_ids, int ids_int64, float* out_logz,
                                   const int32_t* vocab_ids, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!vocab_ids) return mfd_set_error(MFD_ERR_INVALID_ARG, "mfd_topk_logz_vocab: vocab_ids is required");
  return topk_logz_impl(logits, rows, V, row_stride, k, out_logp, out_ids, ids_int64, out_logz, vocab_ids, workspace,
                        workspace_bytes, stream);
}
