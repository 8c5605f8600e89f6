// Fused encode + bitpack + page build + V placement (gfx950).
//
// One 8-wave workgroup per four consecutive pages (eight at dh 64); a wave's
// lanes are the 64 tokens of four pages and the wave takes 16 of their
// dimensions: it places those dimensions of V (and of dense pages' K), and
// encodes the codebook group they form (32 dimensions, in half of the waves,
// at tier 3).  Then one wave per page packs it.  Per (token, group) the radius
// and code reproduce torch CPU's operation order of
// _encode_keys_with_codebooks (spherical_kv_pipeline.py:1136-1144) bit for
// bit:
//   r    = sqrtf(sum over 8 lanes of fmaf(x, x, .) chains, lanes summed in order)
//   dir  = x / (r + 1e-8f)                     (IEEE division)
//   code = first index of the maximum similarity, where the similarity is
//          scored in the order of the torch path the page's size selects
//          (code_sim / code_sim_m1 below).
// The codes are found on MFMA from the keys themselves and the codebook rows
// as two fp16 terms: wherever the best approximate similarity leads the second
// by more than the proven error of both, it is the exact maximum; the others
// (about one token-group in 2,000 for random keys) are scored exactly.  The
// page of pagebuilder.py:8-33 (header, fp32 scales, LSB-first theta codes,
// int8 radius codes) is built in LDS and stored.  This file is compiled with
// -ffp-contract=off so no multiply/add pair is fused except where fmaf is
// written.
#include "sphkv_common.h"
#include "sphkv_internal.h"

namespace sphkv {

struct EncodeArgs {
  const void* k;
  int32_t k_is_fp32;
  const __half* v;
  int64_t num_src_rows;
  const int64_t* src_rows;
  const int32_t* tier;
  const int32_t* count;
  const int32_t* ptable;
  const int32_t* vslot;
  const int32_t* seq_head;
  int32_t num_pages;
  int32_t num_kv;
  const float* cb[4];
  uint8_t* pages;
  int64_t pages_bytes;
  __half* v_pool;
  int64_t num_vpages;
  float* r_out;
  int32_t* code_out;
  const int32_t* order_n;   // per page: N of the torch call whose summation order applies (NULL: count)
  int32_t codes_only;       // 1: write r_out / code_out only (no pages, no V)
};

typedef const float __attribute__((address_space(4)))* cb_ptr;   // read through the scalar cache

constexpr int kEncWaves = 8;       // waves per workgroup
constexpr int kEncMaxG = 8;        // groups per token (dh / g)
constexpr int kSetPages = 4;       // pages of a wave: one lane per token

// Pages per workgroup: dh/16 waves cover the dimensions of four pages.
template <int DH>
__host__ __device__ constexpr int enc_pages() { return kSetPages * kEncWaves / (DH / 16); }

// LDS: the wave-private staging area holds, one after the other, V on its way
// to dim-major order and the MFMA's B operand: per page 16 rows of the keys'
// fp16 values (fp32 keys: a plane of their high halves, then one of the low
// ones).  Rows are packed, so the operand reads of a wave are contiguous.
template <int DH, bool K32>
struct EncodeLds {
  static constexpr int GW = DH / 16;                       // waves per set of pages
  static constexpr int wide = (K32 ? 2 : 1) * 1024;        // bytes of a page's keys, 32 dimensions a row
  // waves w < DH/32 of a set may hold 32-dimension rows, the others 16
  __host__ __device__ static constexpr int page_bytes(int w) { return w < DH / 32 ? wide : wide / 2; }
  __host__ __device__ static constexpr int base(int wave) {
    const int set = wave / GW, w = wave % GW;
    const int per_set = kSetPages * wide * (DH / 32) * 3 / 2;
    return set * per_set + kSetPages * (w < DH / 32 ? w * wide : (DH / 32) * wide + (w - DH / 32) * (wide / 2));
  }
  static constexpr int xs_bytes = kSetPages * wide * (DH / 32) * 3 / 2 * (kEncWaves / GW);
  uint8_t xs[xs_bytes];
  float r[enc_pages<DH>() * kTile][kEncMaxG + 1];          // radius of (token, group), rows padded
  int32_t code[enc_pages<DH>() * kTile][kEncMaxG + 1];     // code of (token, group)
  // (the rows' padding holds the page's tier, tokens and offset, at its first
  // three tokens; after the barrier a page image takes 512 bytes of xs)
  static_assert(xs_bytes >= enc_pages<DH>() * 512, "page images");
  __device__ int32_t& meta(int page, int i) { return code[page * kTile + i][kEncMaxG]; }
};

// Gap between the two largest approximate similarities S = <x, c> (in units of
// r = |x|) past which the largest is the exact first maximum.  |S - s r| <=
// eps r for the exactly scored s, from: the codebook row's two fp16 terms
// (2^-20, and 2^-24 sqrt(g) where the second is denormal: the unit keeps fp16
// denormals), fp32 keys' two terms (2^-19), the fp32 sums of up to 96 products
// (5.7e-6), the six low bits of S that carry the code (63 ulp: 7.5e-6 at the
// bottom of a binade), the rounding of the exact chain and of its direction
// (2e-6).  With rows of |c|^2 <= 1.1 that is eps < 1.95e-5, and two values may
// err apart: 3.9e-5, which the slack passes by a quarter.  About 0.05 % of the
// token-groups of Gaussian keys are scored exactly; fp16 terms of the direction
// alone need 5e-3, which left more than one candidate to one lane of nearly
// every wave.
constexpr float kGapSlack = 5e-5f;
// The bound above scales with |c|: it holds for rows with |c|^2 within
// kUnitTol of 1.  Against a codebook with any other row (scaled or
// unnormalised rows: _encode_keys_with_codebooks accepts any codebook, only
// codebook_loader.py:43-44 normalises) every code is scored exactly.
constexpr float kUnitTol = 0.1f;
// fp32 keys are ranked at length 256, through their norm.  Below 1e-18 the
// squares lose bits to underflow and the norm with them (at 4e-23 it is 3 times
// too short), so such groups are scored exactly.
constexpr float kMinNorm = 1e-18f;
// A code left to the exact scoring is the bits of its best approximate
// similarity, at least this (values that small rank as zeros).
constexpr uint32_t kOpenCode = 0x100;
// Most codes of a wave that are scored one at a time.  Gaussian keys leave one
// to a wave in 30, and such a wave ends its workgroup: the pass over pages and
// candidates takes 5,000 cycles for one code as for 64, score_alone a fifth of
// that.  8,192 x 8 tokens at three tiers 25.3 -> 22.4 us (fp32 keys 36.3 ->
// 32.6), 4 x 500 of dh 64 6.7 -> 5.6 (fp32 7.9 -> 6.6; 7.2 with candidates
// scored by every wave).  2 to 8 are the same there; with one row of each group
// twice 2 and 4 33 us, 6 35, 8 38.
constexpr int kFewOpen = 4;
constexpr float kNoSim = -1e30f;       // no similarity yet (finite: its low bits carry a code too)

// Nearest centroid of one (token, group) against the codebook rows cbg[c * GG ..]
// (wave-uniform, so every centroid coordinate is a scalar operand): the fmaf
// chain over i of torch's batched path, or its separate multiply and add when
// the page is small (N*g*C < 400); first index of the maximum, codes scored in
// ascending order.
template <int GG, bool NAIVE>
__device__ __forceinline__ float code_sim(const float* dir, const float* w) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < GG; ++i) {
    if (NAIVE) s = __fadd_rn(s, __fmul_rn(dir[i], w[i]));
    else s = __builtin_fmaf(dir[i], w[i], s);
  }
  return s;
}

// torch's N = 1 path for a contraction of 16 with C = 64 (tier 1, one token:
// N*g*C >= 400 with M = 1) runs MKL's M = 1 sgemm kernel, whose order is
//   s01 = fmaf(d1, c1, d0*c0); L_l = d_{l+2}c_{l+2} + d_{l+10}c_{l+10} (l < 6);
//   L_6 = d8 c8; L_7 = d9 c9 + s01; M_l = L_l + L_{l+4}; (M_0 + M_2) + (M_1 + M_3)
// (identified with exact power-of-two probes against torch 2.10 / oneMKL
// 2024.2 and pinned by near-tie single-token fixtures).
__device__ __forceinline__ float code_sim_m1(const float* d, const float* c) {
  float L[8];
  const float s01 = __builtin_fmaf(d[1], c[1], __fmul_rn(d[0], c[0]));
#pragma unroll
  for (int l = 0; l < 6; ++l) L[l] = __fadd_rn(__fmul_rn(d[l + 2], c[l + 2]), __fmul_rn(d[l + 10], c[l + 10]));
  L[6] = __fmul_rn(d[8], c[8]);
  L[7] = __fadd_rn(__fmul_rn(d[9], c[9]), s01);
  float M[4];
#pragma unroll
  for (int l = 0; l < 4; ++l) M[l] = __fadd_rn(L[l], L[l + 4]);
  return __fadd_rn(__fadd_rn(M[0], M[2]), __fadd_rn(M[1], M[3]));
}

constexpr int kOrderFma = 0, kOrderNaive = 1, kOrderM1 = 2;

// Codes are scored in batches of NB rows (NB * GG = 64 floats, the scalar
// registers one batch holds): scalar loads return in any order, so a batch's
// rows are waited for together and their NB chains run side by side.
template <int GG, int ORDER>
__device__ __forceinline__ int argmax_codes(const float* dir, cb_ptr cbg, int C) {
  constexpr int NB = 64 / GG;
  float best_sim = 0.f;
  int best = 0;
  for (int c = 0; c < C; c += NB) {
    float w[NB][GG];
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int i = 0; i < GG; ++i) w[q][i] = cbg[(c + q) * GG + i];
    float sim[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      if constexpr (ORDER == kOrderM1) sim[q] = code_sim_m1(dir, w[q]);
      else sim[q] = code_sim<GG, ORDER == kOrderNaive>(dir, w[q]);
    }
#pragma unroll
    for (int q = 0; q < NB; ++q)
      if (c + q == 0 || sim[q] > best_sim) { best_sim = sim[q]; best = c + q; }
  }
  return best;
}

// Code of the group of GG values (of norm r) at element kofs of K, every code
// scored exactly in the order of torch's call over `ord` tokens.
template <int GG, bool K32>
__device__ __forceinline__ int encode_group(const EncodeArgs& a, int64_t kofs, int ord, cb_ptr cbg, int C, float r) {
  float x[GG];
  if constexpr (K32) {
    const float4* src = reinterpret_cast<const float4*>(static_cast<const float*>(a.k) + kofs);
#pragma unroll
    for (int i = 0; i < GG / 4; ++i) {
      const float4 v4 = src[i];
      x[4 * i] = v4.x; x[4 * i + 1] = v4.y; x[4 * i + 2] = v4.z; x[4 * i + 3] = v4.w;
    }
  } else {
    const half8* src = reinterpret_cast<const half8*>(static_cast<const __half*>(a.k) + kofs);
#pragma unroll
    for (int i = 0; i < GG / 8; ++i) {
      const half8 hv = src[i];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[8 * i + e] = (float)hv[e];
    }
  }
  float dir[GG];
  group_directions<GG>(x, __fadd_rn(r, 1e-8f), !K32, dir);
  if (ord * GG * C < 400) return argmax_codes<GG, kOrderNaive>(dir, cbg, C);   // torch's own small-bmm loop
  if (GG == 16 && ord == 1) return argmax_codes<GG, GG == 16 ? kOrderM1 : kOrderFma>(dir, cbg, C);
  return argmax_codes<GG, kOrderFma>(dir, cbg, C);
}

// The code of one token's 16-value group among the candidate codes of mask mk
// (not empty; their rows at cb + 16 c): the first maximum in ascending order
// (calls over one token at C = 64, whose order is code_sim_m1's, are left to
// encode_group).  Codes whose row repeats the first one's score the same and
// lose to it, so directions(dir) and the scores are formed only where a row
// differs.
template <typename D>
__device__ __forceinline__ int best_candidate(D directions, bool naive, const float* cb, uint64_t mk) {
  auto load = [&](int c, float (&w)[16]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(cb + 16 * c + 4 * q);
      w[4 * q] = v.x; w[4 * q + 1] = v.y; w[4 * q + 2] = v.z; w[4 * q + 3] = v.w;
    }
  };
  int best = (int)__builtin_ctzll(mk);
  float f[16], dir[16];
  load(best, f);
  uint64_t rest = mk & (mk - 1);
  mk = 0;
  while (rest) {
    const int c = (int)__builtin_ctzll(rest);
    rest &= rest - 1;
    float w[16];
    load(c, w);
    uint32_t differ = 0u;
#pragma unroll
    for (int i = 0; i < 16; ++i) differ |= __builtin_bit_cast(uint32_t, w[i]) ^ __builtin_bit_cast(uint32_t, f[i]);
    if (differ != 0u) mk |= 1ull << c;
  }
  if (mk == 0) return best;
  directions(dir);
  float best_sim = naive ? code_sim<16, true>(dir, f) : code_sim<16, false>(dir, f);
  for (; mk; mk &= mk - 1) {
    const int c = (int)__builtin_ctzll(mk);
    load(c, f);
    const float sc = naive ? code_sim<16, true>(dir, f) : code_sim<16, false>(dir, f);
    if (sc > best_sim) { best_sim = sc; best = c; }
  }
  return best;
}

// hi + lo = x to 2^-20 |x|, as fp16 (both terms rounded towards zero).
__device__ __forceinline__ void split_half4(const float (&x)[4], half4& hi, half4& lo) {
  const auto h0 = __builtin_amdgcn_cvt_pkrtz(x[0], x[1]), h1 = __builtin_amdgcn_cvt_pkrtz(x[2], x[3]);
  const auto l0 = __builtin_amdgcn_cvt_pkrtz(x[0] - (float)h0[0], x[1] - (float)h0[1]);
  const auto l1 = __builtin_amdgcn_cvt_pkrtz(x[2] - (float)h1[0], x[3] - (float)h1[1]);
  hi = half4{(_Float16)h0[0], (_Float16)h0[1], (_Float16)h1[0], (_Float16)h1[1]};
  lo = half4{(_Float16)l0[0], (_Float16)l0[1], (_Float16)l1[0], (_Float16)l1[1]};
}

// The codebook rows of one (tier, kv head, group) as the MFMA's A operand, two
// fp16 terms.  g = 16: block b of 16 codes, lane (tl, kg) holds dimensions 4 kg
// .. 4 kg + 3 of code 16 b + tl.  g = 32: dimensions 8 kg .. 8 kg + 7 of code
// tl < 8 (blocks 0 and 1; rows 8..15 are zero).  bad: a row's length leaves
// kUnitTol.
struct Codebook {
  half4 hi[4], lo[4];
  int tid, h;
  bool bad;
};

template <int DH, bool G32>
__device__ __forceinline__ void load_codebook(const EncodeArgs& a, int tid, int h, int w, int lane, Codebook& cb) {
  const int tl = lane & 15, kg = lane >> 4;
  const int C = G32 ? 8 : tier_C(tid);
  constexpr int NB = G32 ? 2 : 4;
  const float* c = G32 ? a.cb[3] + ((int64_t)h * (DH / 32) + w) * (8 * 32) + (tl & 7) * 32 + 8 * kg
                       : a.cb[tid] + ((int64_t)h * (DH / 16) + w) * C * 16 + tl * 16 + 4 * kg;
  float4 v[NB];
  v[0] = *reinterpret_cast<const float4*>(c);
  if constexpr (G32) {
    v[1] = *reinterpret_cast<const float4*>(c + 4);
  } else if (C == 64) {
#pragma unroll
    for (int b = 1; b < 4; ++b) v[b] = *reinterpret_cast<const float4*>(c + 256 * b);
  }
  float n2[NB];                                          // squared length of the lane's part of each row
  auto convert = [&](int b) __attribute__((always_inline)) {
    float x[4] = {v[b].x, v[b].y, v[b].z, v[b].w};
    n2[b] = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      n2[b] = __builtin_fmaf(x[e], x[e], n2[b]);
      if (G32) x[e] = tl < 8 ? x[e] : 0.f;
    }
    split_half4(x, cb.hi[b], cb.lo[b]);
  };
  convert(0);
  float row2;
  if constexpr (G32) {
    convert(1);
    row2 = rows_sum(n2[0] + n2[1]);
  } else if (C == 64) {
    convert(1);
    convert(2);
    convert(3);
    // the four lane rows' parts added: each lane ends with one block's row
    float a0 = n2[0], a1 = n2[1], b0 = n2[2], b1 = n2[3];
    swap32(a0, a1);
    swap32(b0, b1);
    float c0 = a0 + a1, c1 = b0 + b1;
    swap16(c0, c1);
    row2 = c0 + c1;
  } else {
    row2 = rows_sum(n2[0]);
  }
  const bool bad = !(fabsf(row2 - 1.f) <= kUnitTol);
  cb.tid = tid;
  cb.h = h;
  cb.bad = __builtin_amdgcn_ballot_w64(bad) != 0;
}

// fmaxf without the instruction that quiets its operands first
__device__ __forceinline__ float max_raw(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float min_raw(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// Largest and second largest of a running pair (m1 >= m2) and s, whose six low
// bits are replaced by (code bits of the caller); NaNs are passed over.
__device__ __forceinline__ void top2(float s, int bits, float& m1, float& m2) {
  const float k = __builtin_bit_cast(float, (__builtin_bit_cast(uint32_t, s) & ~63u) | (uint32_t)bits);
  m2 = __builtin_amdgcn_fmed3f(m1, m2, k);
  m1 = max_raw(m1, k);
}
__device__ __forceinline__ void top2_merge(float& a1, float& a2, float b1, float b2) {
  const float lo = min_raw(a1, b1);
  a1 = max_raw(a1, b1);
  a2 = max_raw(lo, max_raw(a2, b2));
}

// K values of one token's GG dimensions of a wave: fp16 as loaded, or fp32.
template <int GG, bool K32> struct KeyRegs { half8 h[GG / 8]; };
template <int GG> struct KeyRegs<GG, true> { float f[GG]; };

// The loads are unconditional, so nothing waits between them: lanes without a
// token read 128 bytes of the caller's row table instead.
template <int GG, bool K32>
__device__ __forceinline__ void load_keys(const EncodeArgs& a, int64_t kofs, bool ok, const void* none,
                                          KeyRegs<GG, K32>& k) {
  if constexpr (K32) {
    const float4* src = ok ? reinterpret_cast<const float4*>(static_cast<const float*>(a.k) + kofs)
                           : static_cast<const float4*>(none);
#pragma unroll
    for (int i = 0; i < GG / 4; ++i) {
      const float4 v4 = src[i];
      k.f[4 * i] = v4.x; k.f[4 * i + 1] = v4.y; k.f[4 * i + 2] = v4.z; k.f[4 * i + 3] = v4.w;
    }
  } else {
    const half8* src = ok ? reinterpret_cast<const half8*>(static_cast<const __half*>(a.k) + kofs)
                          : static_cast<const half8*>(none);
#pragma unroll
    for (int i = 0; i < GG / 8; ++i) k.h[i] = src[i];
  }
}

// Similarities of 16 tokens (B, Bl: their keys' high and low halves) x the 16
// codes of block b.
template <bool K32>
__device__ __forceinline__ floatx4 sims16(const Codebook& cb, int b, half4 B, half4 Bl) {
  floatx4 D = __builtin_amdgcn_mfma_f32_16x16x16f16(cb.hi[b], B, (floatx4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  D = __builtin_amdgcn_mfma_f32_16x16x16f16(cb.lo[b], B, D, 0, 0, 0);
  if constexpr (K32) D = __builtin_amdgcn_mfma_f32_16x16x16f16(cb.hi[b], Bl, D, 0, 0, 0);
  return D;
}

// What the second group size and the exact scoring need of a token, loaded
// again where they run (so that the usual path does not hold it in registers).
struct TokenMeta {
  int64_t row;
  int ord;
};
template <bool CODES>
__device__ __forceinline__ TokenMeta reload_token(const EncodeArgs& a, int pc, int t) {
  asm volatile("" : "+v"(pc));
  TokenMeta m;
  m.row = a.src_rows[(int64_t)pc * kTile + t];
  // the summation order follows torch's call over ord tokens: the page's own
  // count, or the caller's N (a whole head's tokens in one call)
  m.ord = CODES && a.order_n ? max(a.order_n[pc], 1) : min(max(a.count[pc], 0), kTile);
  return m;
}

// The wave's tokens of the pages in `comp` (a ballot: whole 16-lane rows) at
// group size GG: radius and code of each live lane.  The keys go to LDS as the
// MFMA's B operand; per page 16 tokens x 16 codes per MFMA, lane (tl, kg)
// keeping the two largest similarities of token tl over codes 16 b + 4 kg + i;
// the rows' pairs are then merged into the lanes that hold the tokens.
template <int DH, int GG, bool K32>
__device__ __forceinline__ void encode_tokens(const EncodeArgs& a, const KeyRegs<GG, K32>& k, uint8_t* xs,
                                              int PB, uint64_t comp, bool mine_l, bool live, int tid_l, int head_l,
                                              int w, int lane, Codebook& cb, float& r, int& code) {
  constexpr bool G32 = GG == 32;
  constexpr int RB = 2 * GG;                             // bytes per staged row
  const int j = lane >> 4, t = lane & 15;
  r = 0.f;
  bool zero = false;                                     // every value of a live group is zero
  uint8_t* dst = xs + PB * j + RB * t;
  if constexpr (K32) {
    if (live) r = torch_norm(k.f, GG);
    const bool none = live && r == 0.f;                  // (also where every square underflows)
    if (__builtin_amdgcn_ballot_w64(none)) {
      uint32_t any = 0u;
#pragma unroll
      for (int i = 0; i < GG; ++i) any |= __builtin_bit_cast(uint32_t, k.f[i]) << 1;
      zero = none && any == 0u;
    }
    // scaled to length 256 (a factor common to a token's similarities leaves
    // their order): high and low fp16 halves
    const float sc = 256.f * __builtin_amdgcn_rcpf(r);
    if (mine_l) {
#pragma unroll
      for (int q = 0; q < GG / 4; ++q) {
        const float x4[4] = {k.f[4 * q] * sc, k.f[4 * q + 1] * sc, k.f[4 * q + 2] * sc, k.f[4 * q + 3] * sc};
        half4 hi, lo;
        split_half4(x4, hi, lo);
        *reinterpret_cast<half4*>(dst + 8 * q) = hi;
        *reinterpret_cast<half4*>(dst + 16 * RB + 8 * q) = lo;
      }
    }
  } else {
    if (mine_l) {
#pragma unroll
      for (int q = 0; q < GG / 8; ++q) *reinterpret_cast<half8*>(dst + 16 * q) = k.h[q];
    }
    float x[GG];
#pragma unroll
    for (int i = 0; i < GG; ++i) x[i] = (float)k.h[i / 8][i % 8];
    if (live) r = torch_norm(x, GG);
    zero = live && r == 0.f;
  }
  wave_lds_sync();
  float m1[kSetPages], m2[kSetPages];
  uint32_t bad_pages = 0u;
#pragma unroll
  for (int jj = 0; jj < kSetPages; ++jj) {
    m1[jj] = kNoSim;
    m2[jj] = kNoSim;
    if (((comp >> (16 * jj)) & 0xFFFFull) == 0) continue;
    const int tid = G32 ? 3 : uniform(__builtin_amdgcn_readlane(tid_l, 16 * jj));
    const int h = uniform(__builtin_amdgcn_readlane(head_l, 16 * jj));
    if (tid != cb.tid || h != cb.h) load_codebook<DH, G32>(a, tid, h, w, lane, cb);
    bad_pages |= (uint32_t)cb.bad << jj;
    const uint8_t* xp = xs + PB * jj + RB * t;
    if constexpr (G32) {
      const half8 A0 = __builtin_shufflevector(cb.hi[0], cb.hi[1], 0, 1, 2, 3, 4, 5, 6, 7);
      const half8 A1 = __builtin_shufflevector(cb.lo[0], cb.lo[1], 0, 1, 2, 3, 4, 5, 6, 7);
      const half8 B = *reinterpret_cast<const half8*>(xp + 16 * j);
      floatx4 D = __builtin_amdgcn_mfma_f32_16x16x32_f16(A0, B, (floatx4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      D = __builtin_amdgcn_mfma_f32_16x16x32_f16(A1, B, D, 0, 0, 0);
      if constexpr (K32) {
        const half8 Bl = *reinterpret_cast<const half8*>(xp + 16 * RB + 16 * j);
        D = __builtin_amdgcn_mfma_f32_16x16x32_f16(A0, Bl, D, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) top2(j < 2 ? D[i] : kNoSim, i, m1[jj], m2[jj]);   // rows 8..15 hold no code
    } else {
      const half4 B = *reinterpret_cast<const half4*>(xp + 8 * j);
      half4 Bl{};
      if constexpr (K32) Bl = *reinterpret_cast<const half4*>(xp + 16 * RB + 8 * j);
      auto block = [&](int b) __attribute__((always_inline)) { return sims16<K32>(cb, b, B, Bl); };
      if (tier_C(tid) == 64) {
        const floatx4 D[4] = {block(0), block(1), block(2), block(3)};
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) top2(D[b][i], 16 * b + i, m1[jj], m2[jj]);
      } else {
        const floatx4 D = block(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) top2(D[i], i, m1[jj], m2[jj]);
      }
    }
    m1[jj] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, m1[jj]) | (uint32_t)(4 * j));
  }
  // two rounds of row swaps: row r ends with page r
  float a0 = m1[0], a1 = m1[2], b0 = m1[1], b1 = m1[3];
  float c0 = m2[0], c1 = m2[2], d0 = m2[1], d1 = m2[3];
  swap32(a0, a1);
  swap32(c0, c1);
  swap32(b0, b1);
  swap32(d0, d1);
  top2_merge(a0, c0, a1, c1);
  top2_merge(b0, d0, b1, d1);
  swap16(a0, b0);
  swap16(c0, d0);
  top2_merge(a0, c0, b0, d0);
  code = (int)(__builtin_bit_cast(uint32_t, a0) & 63u);
  const float unit = K32 ? 256.f : r;
  // a zero key scores 0 on every finite row: the first code wins (8,192 x 8
  // tokens at three tiers, every fp16 key zero: 66 -> 21 us; every eighth: 66
  // -> 23; fp32: 75 -> 29 and 74 -> 31; none: 22 and 33)
  const bool open = live && (((bad_pages >> j) & 1u) || (!zero && (!(a0 - c0 > kGapSlack * unit + 1e-30f) ||
                                                                   !(a0 > 0.1f * kNoSim) || (K32 && r < kMinNorm))));
  const uint32_t best = __builtin_bit_cast(uint32_t, a0);
  code = live ? (open ? (int)(best < kOpenCode ? kOpenCode : best) : zero ? 0 : code) : 0;
}

__device__ __forceinline__ float lane_value(float x, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}

// Value of the lane N places along in each row of 16 (DPP row_ror).
template <int N>
__device__ __forceinline__ float row_ror(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x120 + N, 0xF, 0xF, true));
}

// Code of one (token, group) by the whole wave, a lane per code (lanes past C
// repeat the last): its value `lane mod GG` is x, its norm r, its codebook's
// rows at cb.  Same operations and the same winner as encode_group.
template <int GG>
__device__ __forceinline__ int score_alone(const float* cb, int C, float x, float r, bool fp16_in, int ord, int lane) {
  float w[GG];
#pragma unroll
  for (int q = 0; q < GG / 4; ++q) {
    const float4 v = *reinterpret_cast<const float4*>(cb + GG * min(lane, C - 1) + 4 * q);
    w[4 * q] = v.x; w[4 * q + 1] = v.y; w[4 * q + 2] = v.z; w[4 * q + 3] = v.w;
  }
  float d, dir[GG];
  group_directions<1>(&x, __fadd_rn(r, 1e-8f), fp16_in, &d);
#pragma unroll
  for (int i = 0; i < GG; ++i) dir[i] = lane_value(d, i);
  float sim;
  if (ord * GG * C < 400) {
    sim = code_sim<GG, true>(dir, w);
  } else if (GG == 16 && ord == 1) {
    if constexpr (GG == 16) sim = code_sim_m1(dir, w);
  } else {
    sim = code_sim<GG, false>(dir, w);
  }
  // the first maximum: NaNs are passed over, but nothing exceeds a first NaN
  const float first = lane_value(sim, 0);
  if (!(first == first)) return 0;
  float mx = rows_max(sim);
  mx = fmaxf(mx, row_ror<8>(mx));
  mx = fmaxf(mx, row_ror<4>(mx));
  mx = fmaxf(mx, row_ror<2>(mx));
  mx = fmaxf(mx, row_ror<1>(mx));
  return (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(sim == mx));
}

// The wave's (token, group)s that encode_tokens left open, scored exactly.
// Their metadata and fp32 keys are loaded again, so that the usual path holds
// nothing for it.
template <int DH, bool K32, bool CODES>
__device__ __forceinline__ void score_open(const EncodeArgs& a, const uint8_t* xs, int PB, int pc, int tid_l, int head_l, int w, int lane,
                                           bool open, Codebook& cb, float r, int& code) {
  asm volatile("" : "+v"(lane));
  const int j = lane >> 4, t = lane & 15;
  const TokenMeta mt = reload_token<CODES>(a, pc, t);
  // a few: one after the other, their metadata and keys as scalars
  uint64_t few = __builtin_amdgcn_ballot_w64(open);
  if (__builtin_popcountll(few) <= kFewOpen) {
    for (; few; few &= few - 1) {
      const int lead = (int)__builtin_ctzll(few);
      const int tid = uniform(__builtin_amdgcn_readlane(tid_l, lead)), h = uniform(__builtin_amdgcn_readlane(head_l, lead));
      const int ord = uniform(__builtin_amdgcn_readlane(mt.ord, lead));
      const float r1 = lane_value(r, lead);
      const int64_t row = (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(mt.row >> 32), lead) << 32 |
                                    (uint32_t)__builtin_amdgcn_readlane((int)mt.row, lead));
      const uint8_t* key = xs + PB * (lead >> 4);
      int c;
      if (tid != 3) {
        const float* rows = a.cb[tid] + ((int64_t)h * (DH / 16) + w) * tier_C(tid) * 16;
        const float x = K32 ? static_cast<const float*>(a.k)[row * DH + 16 * w + t]
                            : (float)reinterpret_cast<const _Float16*>(key + 32 * (lead & 15))[t];
        c = score_alone<16>(rows, tier_C(tid), x, r1, !K32, ord, lane);
      } else {
        const float* rows = a.cb[3] + ((int64_t)h * (DH / 32) + w) * 8 * 32;
        const float x = K32 ? static_cast<const float*>(a.k)[row * DH + 32 * w + (lane & 31)]
                            : (float)reinterpret_cast<const _Float16*>(key + 64 * (lead & 15))[lane & 31];
        c = score_alone<32>(rows, 8, x, r1, !K32, ord, lane);
      }
      if (lane == lead) code = c;
    }
    return;
  }
  // a gap within the slack: the page's similarities again, for the codes
  // within it of the best (whose bits `code` holds); then all pages' tokens
  // together, codes of repeated rows without scoring.  A wave in 30 comes here
  // for Gaussian keys and random rows, nearly every one against repeated rows,
  // and then VALU issue and the lanes' gathers of rows are what it costs: the
  // sign of a difference is a code's candidate bit (2 instructions per code;
  // compares against a maximum formed here took 5), and the rows are gathered
  // once (fp32 keys against rows with a twin one ulp away: 73 -> 60 us).  8,192
  // x 8 fp16 tokens at three tiers, with one row of each group twice / every
  // row / every row four times: 33 / 39 / 43 us (every lane scoring its
  // candidates: 41 / 42 / 45), fp32 keys 45 / 49 / 53 (52 / 52 / 54); without
  // ties 22 and 33.  (Tier 3 by candidates too was slower: 40 and 48 for 36
  // and 41.)
  uint64_t mk = 0;                                       // this lane's token: codes within the slack
  const float thr = __builtin_bit_cast(float, code) - (kGapSlack * (K32 ? 256.f : r) + 1e-30f);
#pragma unroll 1
  for (int jj = 0; jj < kSetPages; ++jj) {
    const int tid = uniform(__builtin_amdgcn_readlane(tid_l, 16 * jj));
    if (((__builtin_amdgcn_ballot_w64(open) >> (16 * jj)) & 0xFFFFull) == 0 || tid == 3) continue;
    const int h = uniform(__builtin_amdgcn_readlane(head_l, 16 * jj));
    const int C = tier_C(tid);
    if (tid != cb.tid || h != cb.h) load_codebook<DH, false>(a, tid, h, w, lane, cb);
    if (cb.bad) continue;
    const uint8_t* xp = xs + PB * jj + 32 * t;
    const half4 B = *reinterpret_cast<const half4*>(xp + 8 * j);
    half4 Bl{};
    if constexpr (K32) Bl = *reinterpret_cast<const half4*>(xp + 512 + 8 * j);
    const float thr_t = __shfl(thr, 16 * jj + t, 64);
    uint32_t below = 0u;                                 // bit 4 b + i: code 16 b + 4 j + i is below the threshold
#pragma unroll
    for (int b = 3; b >= 0; --b)
      if (16 * b < C) {
        const floatx4 D = sims16<K32>(cb, b, B, Bl);
#pragma unroll
        for (int i = 3; i >= 0; --i)
          below = __builtin_amdgcn_alignbit(below, __builtin_bit_cast(uint32_t, D[i] - thr_t), 31);
      }
    const uint32_t m = ~below & (C == 64 ? 0xFFFFu : 0xFu);
    const uint32_t lo = rows_or(((m & 0xFu) | ((m & 0xF0u) << 12)) << (4 * j));
    const uint32_t hi = rows_or((((m >> 8) & 0xFu) | ((m & 0xF000u) << 4)) << (4 * j));
    if (j == jj) mk = (uint64_t)lo | ((uint64_t)hi << 32);
  }
  {
    const int C = tid_l == 1 ? 64 : 16;
    const bool naive = mt.ord * 16 * C < 400;
    const float* rows = (tid_l == 1 ? a.cb[1] : a.cb[2]) + ((int64_t)head_l * (DH / 16) + w) * C * 16;
    // (keys with an infinity or NaN rank nothing: every code scored)
    if (open && mk != 0 && __builtin_popcountll(mk) <= 8 && (naive || mt.ord > 1) && r < INFINITY && (!K32 || r >= kMinNorm)) {
      auto directions = [&](float (&dir)[16]) __attribute__((always_inline)) {
        float x[16];
        if constexpr (K32) {
          KeyRegs<16, K32> k;
          load_keys<16, K32>(a, mt.row * DH + 16 * w, true, nullptr, k);
#pragma unroll
          for (int i = 0; i < 16; ++i) x[i] = k.f[i];
        } else {
          const half8* src = reinterpret_cast<const half8*>(xs + PB * j + 32 * t);
#pragma unroll
          for (int i = 0; i < 16; ++i) x[i] = (float)src[i / 8][i % 8];
        }
        group_directions<16>(x, __fadd_rn(r, 1e-8f), !K32, dir);
      };
      code = best_candidate(directions, naive, rows, mk);
      open = false;
    }
  }
  // many ties, NaNs, fp32 keys too small to rank, non-unit rows and tier 3: every code
  // scored, with the codebook rows as scalar operands, lanes of one (tier,
  // head) at a time
  uint64_t todo = __builtin_amdgcn_ballot_w64(open);
  while (todo) {
    const int lead = (int)__builtin_ctzll(todo);                 // first lane not yet encoded
    const int tid = uniform(__builtin_amdgcn_readlane(tid_l, lead));
    const int h = uniform(__builtin_amdgcn_readlane(head_l, lead));
    const bool mine = open && tid_l == tid && head_l == h;
    todo &= ~__builtin_amdgcn_ballot_w64(mine);
    const int g = uniform(tier_g(tid)), C = uniform(tier_C(tid));
    const uint64_t cba = (uint64_t)(a.cb[tid] + ((int64_t)h * (DH / g) + w) * C * g);
    const cb_ptr cbg = (cb_ptr)(((uint64_t)(uint32_t)uniform((int)(cba >> 32)) << 32) |
                                (uint32_t)uniform((int)(uint32_t)cba));
    if (mine) {
      if (g == 16) code = encode_group<16, K32>(a, mt.row * DH + 16 * w, mt.ord, cbg, C, r);
      else code = encode_group<32, K32>(a, mt.row * DH + 32 * w, mt.ord, cbg, C, r);
    }
  }
}

// What bounds it: a workgroup is two round trips (page metadata; then keys, V
// and codebook) and about 650 VALU instructions per wave, some 10 us under
// load, so the rate is the workgroups resident: three per CU at 80 VGPRs and
// 29 KB of LDS (fp32 keys 52.5 KB; at dh 64 57 KB and two.  With an area of
// their own for the page images it was two at dh 128 too, a fifth slower).
// Eight waves per SIMD (64 VGPRs) spill: 462 us against 315 for the
// 98,000-token batch below.  Measured (per launch): 16 prompts of 500..12,000
// tokens 254 -> 180 us (3.9 TB/s of traffic), 8,192 tokens 26.7 -> 19.7, the
// same tokens' codes at three tiers 43.4 -> 23.0, of fp32 keys 52 -> 33.
template <int DH, bool K32, bool CODES>
__global__ __launch_bounds__(kEncWaves * 64) __attribute__((amdgpu_waves_per_eu(6, 6))) void encode_pages_kernel(EncodeArgs a) {
  using L = EncodeLds<DH, K32>;
  constexpr int GW = L::GW, PG = enc_pages<DH>();
  __shared__ __attribute__((aligned(16))) L sm;
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int set = wave / GW, w = wave % GW;
  const int p0 = blockIdx.x * PG;                                  // the workgroup's first page
  const int ps = p0 + kSetPages * set;                             // the wave's first page

  // ---- this lane's token: page j, slot t; its page's metadata -------------
  const int j = lane >> 4, t = lane & 15;
  const int p = ps + j;
  const bool p_ok = p < a.num_pages;
  const int pc = p_ok ? p : a.num_pages - 1;
  // the token's source row is loaded together with the page's metadata (its
  // address does not depend on them) and masked by the count afterwards; no
  // load is conditional, so they share one round trip
  const int64_t* rows = a.src_rows + (int64_t)pc * kTile;
  int64_t row_raw = rows[t];
  int tid_raw = a.tier[pc], n_raw = a.count[pc], sh_raw = a.seq_head[pc];
  int vs_l = -1, off_l = -1, th_l = -1;
  if constexpr (!CODES) {
    vs_l = a.vslot[pc];
    off_l = a.ptable[3 * (int64_t)pc];
    th_l = a.ptable[3 * (int64_t)pc + 1];
  }
  // (left alone, the compiler sinks loads into the branches that use them)
  asm volatile("" : "+v"(row_raw), "+v"(tid_raw), "+v"(n_raw), "+v"(sh_raw), "+v"(vs_l), "+v"(off_l), "+v"(th_l));
  vs_l = p_ok ? vs_l : -1;
  const int tid_l = p_ok ? tid_raw : 0;
  const int n_l = p_ok ? min(max(n_raw, 0), kTile) : 0;
  const int sh_l = p_ok ? sh_raw : -1;
  const int head_l = sh_l >= 0 ? sh_l % a.num_kv : 0;
  const bool row_ok = t < n_l && row_raw >= 0 && row_raw < a.num_src_rows;
  const int64_t row = row_ok ? row_raw : 0;
  // a page is encoded only with its tier's codebook and a valid (seq, head)
  const int have = (a.cb[1] ? 2 : 0) | (a.cb[2] ? 4 : 0) | (a.cb[3] ? 8 : 0);
  const bool comp_l = tid_l >= 1 && tid_l <= 3 && w < DH / tier_g(tid_l) && sh_l >= 0 && ((have >> (tid_l & 3)) & 1);
  const bool comp16_l = comp_l && tid_l != 3, comp32_l = comp_l && tid_l == 3;
  const bool dense_l = !CODES && tid_l == kDenseTier;
  const uint64_t comp16 = __builtin_amdgcn_ballot_w64(comp16_l), comp32 = __builtin_amdgcn_ballot_w64(comp32_l);
  uint8_t* xs = sm.xs + L::base(wave);
  const int PB = L::page_bytes(w);                       // bytes of a page's staged keys

  // ---- K and V of the wave's dimensions, the first codebook ----------------
  KeyRegs<16, K32> k16;
  load_keys<16, K32>(a, row * DH + 16 * w, row_ok && (comp16_l || dense_l), rows, k16);
  half8 vh[2];
  if constexpr (!CODES) {
    const half8* src = row_ok ? reinterpret_cast<const half8*>(a.v + row * DH + 16 * w) : reinterpret_cast<const half8*>(rows);
    vh[0] = src[0];
    vh[1] = src[1];
  }
  Codebook cb;
  cb.tid = 0;
  if (comp16) {
    const int l0 = (int)__builtin_ctzll(comp16);
    load_codebook<DH, false>(a, uniform(__builtin_amdgcn_readlane(tid_l, l0)), uniform(__builtin_amdgcn_readlane(head_l, l0)),
                             w, lane, cb);
  }

  // ---- V: 64 rows of the wave's 16 dimensions through LDS; the transposing
  //      read gives lane (i, q) tokens 4 q .. 4 q + 3 of dimension i, 8 bytes
  //      of its dim-major row (element (token k, dim d) at d * 16 + k) --------
  if constexpr (!CODES) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      uint4 d = __builtin_bit_cast(uint4, vh[k]);
      d.x = row_ok ? d.x : 0u; d.y = row_ok ? d.y : 0u; d.z = row_ok ? d.z : 0u; d.w = row_ok ? d.w : 0u;
      *reinterpret_cast<uint4*>(xs + 32 * lane + 16 * k) = d;
    }
    wave_lds_sync();
#pragma unroll
    for (int jj = 0; jj < kSetPages; ++jj) {
      const int64_t vs = __builtin_amdgcn_readlane(vs_l, 16 * jj);
      if (vs < 0 || vs >= a.num_vpages) continue;
      typedef short short4v __attribute__((ext_vector_type(4)));
      const uint8_t* src = xs + (16 * jj + 4 * j + (t >> 2)) * 32 + 8 * (t & 3);
      const short4v tr = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v*)src);
      *reinterpret_cast<short4v*>(a.v_pool + (vs * DH + 16 * w + t) * kTile + 4 * j) = tr;
    }
    wave_lds_sync();
  }

  // ---- dense pages: header (tier id, count, six zero bytes) and fp16 K rows
  //      at a 16-byte aligned theta offset.  A pointer-table row that does not
  //      place the whole page inside the byte pool (negative or misaligned
  //      offsets included) writes nothing, as a compressed page's does -------
  if (dense_l && off_l >= 0 && (int64_t)off_l + 8 <= a.pages_bytes && (int64_t)th_l >= (int64_t)off_l + 8 &&
      (th_l & 15) == 0 && (int64_t)th_l + (int64_t)n_l * DH * 2 <= a.pages_bytes) {
    if (w == 0 && t < 8) a.pages[off_l + t] = t == 0 ? (uint8_t)kDenseTier : (t == 1 ? (uint8_t)n_l : 0);
    if (t < n_l) {
      half8* dst = reinterpret_cast<half8*>(a.pages + (int64_t)th_l + ((int64_t)t * DH + 16 * w) * 2);
      if constexpr (K32) {
        half8 h0, h1;
#pragma unroll
        for (int e = 0; e < 8; ++e) { h0[e] = (_Float16)k16.f[e]; h1[e] = (_Float16)k16.f[8 + e]; }
        dst[0] = row_ok ? h0 : half8{};
        dst[1] = row_ok ? h1 : half8{};
      } else {
        dst[0] = row_ok ? k16.h[0] : half8{};
        dst[1] = row_ok ? k16.h[1] : half8{};
      }
    }
  }

  if (w == 0 && t == 0) {
    sm.meta(kSetPages * set + j, 0) = tid_l;
    sm.meta(kSetPages * set + j, 1) = n_l;
    sm.meta(kSetPages * set + j, 2) = off_l;
  }

  // ---- radii and codes ------------------------------------------------------
  if (comp16) {
    float r;
    int code;
    const bool live = comp16_l && row_ok;
    encode_tokens<DH, 16, K32>(a, k16, xs, PB, comp16, comp16_l, live, tid_l, head_l, w, lane, cb, r, code);
    if (comp16_l) {
      sm.r[64 * set + lane][w] = r;
      sm.code[64 * set + lane][w] = code;
    }
  }
  if (comp32) {
    float r;
    int code;
    const bool live = comp32_l && row_ok;
    KeyRegs<32, K32> k32;
    const int64_t row32 = reload_token<CODES>(a, pc, t).row;
    load_keys<32, K32>(a, row32 * DH + 32 * w, live, a.src_rows + (int64_t)pc * kTile, k32);
    const int l0 = (int)__builtin_ctzll(comp32);
    load_codebook<DH, true>(a, 3, uniform(__builtin_amdgcn_readlane(head_l, l0)), w, lane, cb);
    wave_lds_sync();
    encode_tokens<DH, 32, K32>(a, k32, xs, PB, comp32, comp32_l, live, tid_l, head_l, w, lane, cb, r, code);
    if (comp32_l) {
      sm.r[64 * set + lane][w] = r;
      sm.code[64 * set + lane][w] = code;
    }
  }
  if (comp16 | comp32) {
    int code = sm.code[64 * set + lane][w];
    const bool open = (((comp16 | comp32) >> lane) & 1ull) && (uint32_t)code >= kOpenCode;
    if (__builtin_amdgcn_ballot_w64(open)) {
      score_open<DH, K32, CODES>(a, xs, PB, pc, tid_l, head_l, w, lane, open, cb, sm.r[64 * set + lane][w], code);
      if (open) sm.code[64 * set + lane][w] = code;
    }
  }
  __syncthreads();

  if constexpr (CODES) {
    // radii and codes of every (token, group) of the workgroup's compressed
    // pages, [page][slot][DH / 16]
    for (int e = threadIdx.x; e < PG * kTile * (DH / 16); e += kEncWaves * 64) {
      const int tk = e / (DH / 16), gi = e % (DH / 16);
      const int tid = sm.meta(tk / kTile, 0);
      if (tid < 1 || tid > 3 || tk % kTile >= sm.meta(tk / kTile, 1) || gi >= DH / tier_g(tid)) continue;
      const int64_t o = (int64_t)p0 * kTile * (DH / 16) + e;
      if (a.r_out) a.r_out[o] = sm.r[tk][gi];
      if (a.code_out) a.code_out[o] = sm.code[tk][gi];
    }
    return;
  }
  if (wave >= PG || p0 + wave >= a.num_pages) return;

  // ---- page build: wave = page; lane = (token t, quarter gs) -----------------
  const int tid = uniform(sm.meta(wave, 0)), n = uniform(sm.meta(wave, 1));
  const int64_t page_off = uniform(sm.meta(wave, 2));
  const int64_t pg = p0 + wave;
  if (tid < 1 || tid > 3) return;
  int tx = threadIdx.x;
  asm volatile("" : "+v"(tx));                           // (formed again rather than held, and spilled, until here)
  const int lane_b = tx & 63, tk = tx & 15, gs = lane_b >> 4;
  const bool tok_ok = tk < n;
  const int g = tier_g(tid), b = tier_b(tid);
  const int G = DH / g;
  const int nk = (G + 3) / 4;                   // groups per lane_b (2 for g=16, 1 for g=32 at DH=128)
  float rr_[2] = {0.f, 0.f};
  int best_[2] = {0, 0};
  for (int k = 0; k < nk; ++k) {
    const int gi = gs + 4 * k;
    if (gi < G) { rr_[k] = sm.r[16 * wave + tk][gi]; best_[k] = sm.code[16 * wave + tk][gi]; }
  }
  // radius scale per group: max over the page's tokens (lanes of one 16-row)
  float scale_[2];
  for (int k = 0; k < 2; ++k) {
    float m = tok_ok ? rr_[k] : 0.f;
    for (int o = 1; o < 16; o <<= 1) m = fmaxf(m, shfl_xor(m, o));
    scale_[k] = m;
  }
  uint8_t* st = sm.xs + 512 * wave;
  const int nG = n * G;
  const int tb = (nG * b + 7) / 8;
  const int hdr = kHeaderBytes + 4 * G;
  const int size = hdr + tb + nG;
  if (lane_b < kHeaderBytes) st[lane_b] = lane_b == 0 ? (uint8_t)tid : (lane_b == 1 ? (uint8_t)n : 0);
  for (int k = 0; k < nk; ++k) {
    const int gi = gs + 4 * k;
    if (tk == 0 && gi < G) *reinterpret_cast<float*>(st + kHeaderBytes + 4 * gi) = scale_[k];
  }
  // LSB-first bit stream (bitpacking.py:14-27): bit j of item i = (token t,
  // group gi), i = t*G + gi, at bit i*b + j.  The theta section's dwords (hdr
  // = 8 + 4G is a multiple of 4) are cleared, then every item ORs its b bits
  // into the one or two dwords they fall in.
  uint32_t* thw = reinterpret_cast<uint32_t*>(st + hdr);
  for (int w = lane_b; w < (tb + 3) / 4; w += kWave) thw[w] = 0u;
  wave_lds_sync();
  for (int k = 0; k < nk; ++k) {
    const int gi = gs + 4 * k;
    if (!tok_ok || gi >= G) continue;
    const uint32_t c = (uint32_t)best_[k];
    const int o = (tk * G + gi) * b, w = o >> 5, sh = o & 31;
    __hip_atomic_fetch_or(thw + w, c << sh, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (sh + b > 32) __hip_atomic_fetch_or(thw + w + 1, c >> (32 - sh), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  // the radius codes, after the ORs (the first radius bytes can share the
  // last theta dword)
  wave_lds_sync();
  for (int k = 0; k < nk; ++k) {
    const int gi = gs + 4 * k;
    if (!tok_ok || gi >= G) continue;
    const int item = tk * G + gi;
    const float safe = scale_[k] < 1e-8f ? 1e-8f : scale_[k];
    float qv = __fmul_rn(__fdiv_rn(rr_[k], safe), 127.0f);
    qv = __builtin_rintf(qv);
    qv = fminf(fmaxf(qv, -127.f), 127.f);
    st[hdr + tb + item] = (uint8_t)(int8_t)(int)qv;
    if (a.r_out) a.r_out[(pg * kTile + tk) * (DH / 16) + gi] = rr_[k];
    if (a.code_out) a.code_out[(pg * kTile + tk) * (DH / 16) + gi] = best_[k];
  }
  wave_lds_sync();
  if (page_off >= 0 && page_off + size <= a.pages_bytes) {
    // whole dwords where the page is 4-byte aligned, then its last bytes
    // (the next page may start right after it)
    const int nw = (page_off & 3) == 0 ? size >> 2 : 0;
    uint32_t* dw = reinterpret_cast<uint32_t*>(a.pages + page_off);
    for (int i = lane_b; i < nw; i += kWave) dw[i] = reinterpret_cast<const uint32_t*>(st)[i];
    for (int i = 4 * nw + lane_b; i < size; i += kWave) a.pages[page_off + i] = st[i];
  }
}

int launch_encode(const EncodeLaunch& L, hipStream_t stream) {
  EncodeArgs a;
  a.k = L.k; a.k_is_fp32 = L.k_is_fp32; a.v = reinterpret_cast<const __half*>(L.v);
  a.num_src_rows = L.num_src_rows; a.src_rows = L.src_rows; a.tier = L.tier; a.count = L.count;
  a.ptable = L.ptable; a.vslot = L.vslot; a.seq_head = L.seq_head; a.num_pages = L.num_pages;
  a.num_kv = L.num_kv; a.cb[0] = nullptr; a.cb[1] = L.cb1; a.cb[2] = L.cb2; a.cb[3] = L.cb3;
  a.pages = L.pages; a.pages_bytes = L.pages_bytes; a.v_pool = reinterpret_cast<__half*>(L.v_pool);
  a.num_vpages = L.num_vpages; a.r_out = L.r_out; a.code_out = L.code_out;
  a.order_n = L.order_n; a.codes_only = L.codes_only;
  const int per = L.dh == 128 ? enc_pages<128>() : enc_pages<64>();
  const dim3 grid((L.num_pages + per - 1) / per), block(kEncWaves * 64);
#define SPHKV_ENC(D, K, C) if (L.dh == D && (L.k_is_fp32 != 0) == K && (L.codes_only != 0) == C) \
    hipLaunchKernelGGL((encode_pages_kernel<D, K, C>), grid, block, 0, stream, a);
  SPHKV_ENC(128, false, false) SPHKV_ENC(128, true, false) SPHKV_ENC(128, false, true) SPHKV_ENC(128, true, true)
  SPHKV_ENC(64, false, false) SPHKV_ENC(64, true, false) SPHKV_ENC(64, false, true) SPHKV_ENC(64, true, true)
#undef SPHKV_ENC
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace sphkv
