// Several tokens against F32, F16, IQ4_NL or Q8_0 weights on the matrix cores, to the precision of the fp32 kernels:
//   out[m][o] = (residual ? residual[m][o] : 0) + sum_j x[m][j] * w(o, j)
// These types have no fp16-precision prefill form (the reference computes them in full precision at every token count,
// src/ml/gguf/quant_matmul.cr:216-368), so every operand is split into bfloat16 terms that lose nothing: an fp32 value is
// exactly three of them (8 + 8 + 8 significand bits, by truncation),
// a binary16 weight two, a Q8_0 or IQ4_NL code one (the block scale is applied to the 32-value sum in fp32). Truncated terms are
// below 2^-7 and 2^-15 of the value and have its sign, so what is left out of a product is a bias: all term products are taken
// but the last one of fp32 weights, x2 w2, below 2^-30. 3 instructions of v_mfma_f32_16x16x32_bf16 per 16 x 16 x 32 for the
// codes, 6 for binary16, 8 for fp32 weights. (Without x1 w2 and x2 w1: up to 7.8 x 2^-24 of a product, 0.7 on average.)
// The instruction reads a term below 2^-126 as zero, and the third term of a value is as small as its last place: fp32 operands are
// split times 2^24, which brings the last place of the smallest subnormal above that, and the sums are brought back at the end
// (unscaled, activations around 2^-112 / 2^-120 / 2^-128 were off by 2.6e-7 / 7e-5 / 0.018 of the result, the row kernels by 9e-8).
//
// Kernel ABI: (w_raw, x, residual | null, out, in_dim:u32, out_dim:u32, tokens:u32), names <type>_gemm_terms_f32_<TM>x<TN>:
// a workgroup of eight wavefronts takes 16 TM tokens x 16 TN rows, grid gemm_terms_plan (gemv_config.h). The
// wavefronts are eight k-slices (contiguous runs of 32-value steps), whose sums meet in LDS in a fixed order.
//
// A lane of the instruction's operand holds eight consecutive k values of one row (row = lane % 16, k-group = lane / 16).
// Loaded that way every load instruction touches 64 cache lines and the loads are what the kernel waits for (4096 x 4096
// IQ4_NL, 64 tokens: 34 us against 18.7; with four steps in flight instead of one 40), so a wavefront loads its steps with
// neighbouring lanes on neighbouring bytes of a row, up to two ahead, and turns them through a region of LDS that no other
// wavefront uses: no barrier in the loop.
// What bounds it: small calls the chain load - LDS - sums (4 us), large ones the issue slots of a SIMD: Q8_0 4096 -> 4096, 256 tokens, 13300
// instructions per SIMD, 82 % of its cycles, where a kernel without any load still takes 36 of the 42 us and one without the splitting of
// x 39. A matrix instruction takes 7 to 8 clocks of issue, but its sum is there only 16 clocks later. Interleaved, the products of a token tile go out row tile by
// row tile (TN independent sums), with the next tile's terms and the last one's sums in between, instead of one sum after the other: Q8_0 1024 ->
// 3584, 200 tokens 15.1 -> 14.6 us, 4096 -> 4096, 256 tokens 43.5 -> 42.3; F16 2048 -> 2048, 33 tokens 8.65 -> 8.45; F32 4096 -> 4096, 256 tokens 79 -> 72. Smaller
// tiles have less to put between the products and lose by it on short rows: which take it is measured (gemm_terms_interleaved, gemv_config.h).
// Splitting by v_cvt_pk_bf16_f32 and v_dot2_f32_bf16, half the instructions, gained nothing: the second takes twice as long.
// Measured, weights from memory, row kernels (Q8_0: one-pass launches of eight tokens) -> these: Q8_0 1024 -> 3584, 9 / 48 / 200
// tokens 9.6 / 35 / 143 -> 5.0 / 7.8 / 15.4 us; F16 2048 -> 2048, 33 tokens 41.8 -> 9.1; F32 4096 -> 4096, 33 tokens 174 -> 26; IQ4_NL
// 4096 -> 4096, 1 / 64 tokens 40 / 1926 -> 10.5 / 21.
#pragma once
#include "common.hpp"
#include "dequant.hpp"
#include "gemv_config.h"
#include <type_traits>


typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float terms_f4 __attribute__((ext_vector_type(4)));

// the upper halves of two dwords (b behind a): two truncated bfloat16 values
__device__ __forceinline__ u32 terms_pair(u32 a, u32 b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
__device__ __forceinline__ bf16x8_t terms_op(const u32 (&q)[4]) {
  uint4 o = make_uint4(q[0], q[1], q[2], q[3]);
  return __builtin_bit_cast(bf16x8_t, o);
}
// v -> N truncated terms
template <int N>
__device__ __forceinline__ void terms_split(const float (&v)[8], bf16x8_t (&t)[N]) {
  float r[8];
#pragma unroll
  for (int e = 0; e < 8; e++) r[e] = v[e];
#pragma unroll
  for (int k = 0; k < N; k++) {
    u32 q[4];
#pragma unroll
    for (int p = 0; p < 4; p++) q[p] = terms_pair(__float_as_uint(r[2 * p]), __float_as_uint(r[2 * p + 1]));
    t[k] = terms_op(q);
    if (k + 1 < N) {
#pragma unroll
      for (int e = 0; e < 8; e++) r[e] -= __uint_as_float(__float_as_uint(r[e]) & 0xFFFF0000u);
    }
  }
}

// Four consecutive values of an fp32 row of n; FULL: all of them exist, else zeros behind the end.
template <bool FULL>
__device__ __forceinline__ float4 terms_load4(const float* row, u32 k, u32 n) {
  if constexpr (FULL) {
    float4 a;
    __builtin_memcpy(&a, row + k, 16);
    return a;
  } else {
    return make_float4(k < n ? row[k] : 0.f, k + 1 < n ? row[k + 1] : 0.f, k + 2 < n ? row[k + 2] : 0.f, k + 3 < n ? row[k + 3] : 0.f);
  }
}

// Rows of 32 fp32 values in LDS, 36 dwords apart (the 16-byte reads of sixteen rows then fall on all 64 banks). get(): the
// lane's operand times TERMS_F32_SCALE (from 2^104 on an infinity, whose sums are taken again).
#define TERMS_F32_STRIDE 36u
#define TERMS_F32_SCALE 0x1p24f
struct TermsF32Tile {   // 16 rows: two loads of eight rows x 8 lanes x 16 bytes
  float4 v[2];
  template <bool FULL>
  __device__ __forceinline__ void load(const float* const (&rows)[2], u32 s, u32 lane, u32 n) {
#pragma unroll
    for (int i = 0; i < 2; i++) v[i] = terms_load4<FULL>(rows[i], 32 * s + 4 * (lane & 7), n);
  }
  __device__ __forceinline__ void put(u32* lds, u32 lane) const {
#pragma unroll
    for (int i = 0; i < 2; i++) *reinterpret_cast<float4*>(lds + (8 * i + (lane >> 3)) * TERMS_F32_STRIDE + 4 * (lane & 7)) = v[i];
  }
  static __device__ __forceinline__ void get(const u32* lds, u32 lane, float (&o)[8]) {
    const float4* q = reinterpret_cast<const float4*>(lds + (lane & 15) * TERMS_F32_STRIDE + 8 * (lane >> 4));
    const float4 a = q[0], b = q[1];
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
    o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] *= TERMS_F32_SCALE;
  }
};

// ---- weight formats: sixteen rows x 32 values. rows(): the addresses a lane loads from; load<FULL>() / put(): registers, LDS;
// terms(): the operand's terms; scale(): what the step's sum is multiplied by; UNSCALE: what brings the sums back from the scale
// of the terms (those of x are always scaled).
struct TermsF32 {
  static constexpr int TERMS = 3;
  static constexpr bool SCALED = false;
  static constexpr float UNSCALE = 1.0f / (TERMS_F32_SCALE * TERMS_F32_SCALE);
  static constexpr u32 LDS_DWORDS = 16 * TERMS_F32_STRIDE;
  static constexpr int ROWS = 2;   // row addresses per lane
  static __device__ __forceinline__ size_t row_bytes(u32 n) { return (size_t)n * 4; }
  static __device__ __forceinline__ u32 row_of(u32 lane, int i) { return 8 * i + (lane >> 3); }
  static __device__ __forceinline__ float at(const uint8_t* row, u32 k) { return reinterpret_cast<const float*>(row)[k]; }
  TermsF32Tile t;
  template <bool FULL>
  __device__ __forceinline__ void load(const uint8_t* const (&rows)[2], u32 s, u32 lane, u32 n) {
    const float* const r[2] = {reinterpret_cast<const float*>(rows[0]), reinterpret_cast<const float*>(rows[1])};
    t.load<FULL>(r, s, lane, n);
  }
  __device__ __forceinline__ void put(u32* lds, u32 lane) const { t.put(lds, lane); }
  static __device__ __forceinline__ float scale(const u32*, u32) { return 1.0f; }
  static __device__ __forceinline__ void terms(const u32* lds, u32 lane, bf16x8_t (&o)[3]) {
    float v[8];
    TermsF32Tile::get(lds, lane, v);
    terms_split<3>(v, o);
  }
};
struct TermsF16 {   // one load: four lanes x 16 bytes per row; rows 20 dwords apart
  static constexpr int TERMS = 2;
  static constexpr bool SCALED = false;
  static constexpr float UNSCALE = 1.0f / TERMS_F32_SCALE;
  static constexpr u32 STRIDE = 20, LDS_DWORDS = 16 * STRIDE;
  static constexpr int ROWS = 1;
  static __device__ __forceinline__ size_t row_bytes(u32 n) { return (size_t)n * 2; }
  static __device__ __forceinline__ u32 row_of(u32 lane, int) { return lane >> 2; }
  static __device__ __forceinline__ float at(const uint8_t* row, u32 k) { return h2f(ld2(row + (size_t)k * 2)); }
  uint4 q;
  template <bool FULL>
  __device__ __forceinline__ void load(const uint8_t* const (&rows)[1], u32 s, u32 lane, u32 n) {
    const u32 k = 32 * s + 8 * (lane & 3);
    if constexpr (FULL) {
      q = ld16(rows[0] + (size_t)k * 2);
    } else {
      u32 h[8];
#pragma unroll
      for (u32 e = 0; e < 8; e++) h[e] = k + e < n ? ld2(rows[0] + (size_t)(k + e) * 2) : 0u;
      q = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
    }
  }
  __device__ __forceinline__ void put(u32* lds, u32 lane) const { *reinterpret_cast<uint4*>(lds + (lane >> 2) * STRIDE + 4 * (lane & 3)) = q; }
  static __device__ __forceinline__ float scale(const u32*, u32) { return 1.0f; }
  static __device__ __forceinline__ void terms(const u32* lds, u32 lane, bf16x8_t (&o)[2]) {
    const uint4 r = *reinterpret_cast<const uint4*>(lds + (lane & 15) * STRIDE + 4 * (lane >> 4));
    const u32 d[4] = {r.x, r.y, r.z, r.w};
    float v[8];
#pragma unroll
    for (int p = 0; p < 4; p++) {
      v[2 * p] = h2f(d[p]);
      v[2 * p + 1] = h2f(d[p] >> 16);
    }
    terms_split<2>(v, o);
  }
};
// eight signed bytes -> one bfloat16 term (every value is exact)
__device__ __forceinline__ void terms_from_bytes(u32 a, u32 b, bf16x8_t& t) {
  u32 q[4];
#pragma unroll
  for (int p = 0; p < 4; p++) {
    const u32 w = p < 2 ? a : b;
    const int sh = 16 * (p & 1);
    const float lo = (float)(int)(int8_t)(w >> sh), hi = (float)(int)(int8_t)(w >> (sh + 8));
    q[p] = terms_pair(__float_as_uint(lo), __float_as_uint(hi));
  }
  t = terms_op(q);
}
// Q8_0 and IQ4_NL: a block (f16 scale, then 32 or 16 bytes of codes) is one step of a row; four lanes per row take a quarter
// of the codes each and the scale. A block is whole in memory also where the row ends inside it.
struct TermsQ80 {
  static constexpr int TERMS = 1;
  static constexpr bool SCALED = true;
  static constexpr float UNSCALE = 1.0f / TERMS_F32_SCALE;
  static constexpr u32 STRIDE = 10, LDS_DWORDS = 16 * STRIDE + 16;   // rows of 8 dwords 10 apart, then the scales
  static constexpr int ROWS = 1;
  static __device__ __forceinline__ size_t row_bytes(u32 n) { return (size_t)((n + 31) >> 5) * 34; }
  static __device__ __forceinline__ u32 row_of(u32 lane, int) { return lane >> 2; }
  static __device__ __forceinline__ float at(const uint8_t* row, u32 k) {
    const uint8_t* b = row + (size_t)(k >> 5) * 34;
    return h2f(ld2(b)) * (float)(int)(int8_t)b[2 + (k & 31)];
  }
  uint2 q;
  u32 d;
  template <bool FULL>
  __device__ __forceinline__ void load(const uint8_t* const (&rows)[1], u32 s, u32 lane, u32) {
    const uint8_t* b = rows[0] + (size_t)s * 34;
    d = ld2(b);
    q = ld8(b + 2 + 8 * (lane & 3));
  }
  __device__ __forceinline__ void put(u32* lds, u32 lane) const {
    *reinterpret_cast<uint2*>(lds + (lane >> 2) * STRIDE + 2 * (lane & 3)) = q;
    lds[16 * STRIDE + (lane >> 2)] = d;
  }
  static __device__ __forceinline__ float scale(const u32* lds, u32 lane) { return h2f(lds[16 * STRIDE + (lane & 15)]); }
  static __device__ __forceinline__ void terms(const u32* lds, u32 lane, bf16x8_t (&o)[1]) {
    const uint2 r = *reinterpret_cast<const uint2*>(lds + (lane & 15) * STRIDE + 2 * (lane >> 4));
    terms_from_bytes(r.x, r.y, o[0]);
  }
};
struct TermsIq4nl {   // values 0..15 of a block are the low nibbles of its 16 bytes, 16..31 the high ones
  static constexpr int TERMS = 1;
  static constexpr bool SCALED = true;
  static constexpr float UNSCALE = 1.0f / TERMS_F32_SCALE;
  static constexpr u32 STRIDE = 6, LDS_DWORDS = 16 * STRIDE + 16;
  static constexpr int ROWS = 1;
  static __device__ __forceinline__ size_t row_bytes(u32 n) { return (size_t)((n + 31) >> 5) * 18; }
  static __device__ __forceinline__ u32 row_of(u32 lane, int) { return lane >> 2; }
  static __device__ __forceinline__ float at(const uint8_t* row, u32 k) {
    const uint8_t* b = row + (size_t)(k >> 5) * 18;
    return h2f(ld2(b)) * (float)(int)(int8_t)look(((u32)b[2 + (k & 15)] >> (k & 16 ? 4 : 0)) & 15u);
  }
  u32 q, d;
  template <bool FULL>
  __device__ __forceinline__ void load(const uint8_t* const (&rows)[1], u32 s, u32 lane, u32) {
    const uint8_t* b = rows[0] + (size_t)s * 18;
    d = ld2(b);
    q = ld4(b + 2 + 4 * (lane & 3));
  }
  __device__ __forceinline__ void put(u32* lds, u32 lane) const {
    lds[(lane >> 2) * STRIDE + (lane & 3)] = q;
    lds[16 * STRIDE + (lane >> 2)] = d;
  }
  static __device__ __forceinline__ float scale(const u32* lds, u32 lane) { return h2f(lds[16 * STRIDE + (lane & 15)]); }
  // four nibbles (one per byte) through the 16-byte table: both halves of the table are indexed by the low three bits, the
  // fourth picks between them byte by byte
  static __device__ __forceinline__ u32 look(u32 n) {
    const u32 i7 = n & 0x07070707u;
    const u32 lo = __builtin_amdgcn_perm(0xF6EADDCFu, 0xBFAD9881u, i7);   // -49 -35 -22 -10 | -127 -104 -83 -65
    const u32 hi = __builtin_amdgcn_perm(0x71594535u, 0x26190D01u, i7);   // 53 69 89 113 | 1 13 25 38
    return __builtin_amdgcn_perm(hi, lo, 0x03020100u + ((n & 0x08080808u) >> 1));
  }
  static __device__ __forceinline__ void terms(const u32* lds, u32 lane, bf16x8_t (&o)[1]) {
    const u32 kg = lane >> 4, sh = kg >= 2 ? 4u : 0u;
    const uint2 r = *reinterpret_cast<const uint2*>(lds + (lane & 15) * STRIDE + 2 * (kg & 1));
    terms_from_bytes(look((r.x >> sh) & 0x0F0F0F0Fu), look((r.y >> sh) & 0x0F0F0F0Fu), o[0]);
  }
};

// What has no such terms: an infinity (inf - inf, and inf times a term that is zero), and sums that leave the range of fp32 times the
// scale of the terms, or before the block scale brings them back. A sum that is no finite number is therefore taken again from plain fp32 products, as
// the row kernels do: a wavefront takes four tokens against one row at a time, lanes over k, all wavefronts of the workgroup share
// the tile's. F16 2048 x 2048, 33 tokens, us (a lane per sum, walking the row alone | this | the row kernel): one infinity 178 | 24 | 42, one
// in every token 818 | 63 | 42, every value a NaN 10 | 16 | 41; F32 4096 x 4096, 33 tokens, one infinity 383 | 59 | 177; Q8_0 1024 -> 3584,
// 200 tokens, one infinity 140 | 43, one in every token 3650 | 310.
template <class W>
__device__ __forceinline__ void terms_plain_sums(const uint8_t* row, const float* const (&x)[4], u32 n, u32 lane, float (&s)[4]) {
#pragma unroll
  for (int v = 0; v < 4; v++) s[v] = 0.f;
#pragma unroll 4
  for (u32 k = lane; k < n; k += 64) {
    const float w = W::at(row, k);
#pragma unroll
    for (int v = 0; v < 4; v++) s[v] = fmaf(x[v][k], w, s[v]);
  }
#pragma unroll
  for (int v = 0; v < 4; v++) s[v] = wave_sum(s[v]);
}

// D: steps whose loads are in flight while one is computed (a ring of registers). INTERLEAVED: the order of a step's instructions
// (gemm_terms_interleaved in gemv_config.h).
template <class W, int TM, int TN, int D, bool INTERLEAVED>
__device__ __forceinline__ void gemm_terms_core(const uint8_t* __restrict__ w, const float* __restrict__ x, const float* residual,
                                                float* out, u32 in_dim, u32 out_dim, u32 tokens) {
  constexpr u32 XD = 16 * TERMS_F32_STRIDE;                      // dwords of 16 rows of x
  constexpr u32 WAVE_DWORDS = TM * XD + TN * W::LDS_DWORDS;      // a wavefront's region
  constexpr u32 PART_DWORDS = GEMM_TERMS_WAVES * TM * TN * 256;  // the k-slices' sums, behind the loop
  constexpr u32 END_DWORDS = PART_DWORDS + GEMM_TERMS_WAVES;     // and a flag of each wavefront
  constexpr u32 LDS_DWORDS = GEMM_TERMS_WAVES * WAVE_DWORDS > END_DWORDS ? GEMM_TERMS_WAVES * WAVE_DWORDS : END_DWORDS;
  __shared__ uint4 lds4[(LDS_DWORDS + 3) / 4];
  const u32 lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const u32 row = lane & 15, kg = lane >> 4;
  u32 mt, nt;
  gemm_terms_tile(blockIdx.x, (tokens + 16 * TM - 1) / (16 * TM), &mt, &nt);
  const u32 n0 = nt * (16 * TN), m0 = mt * (16 * TM);
  if (n0 >= out_dim) return;   // (the grid is rounded up to whole rows of tiles per XCD)
  u32* const mine = reinterpret_cast<u32*>(lds4) + wave * WAVE_DWORDS;
  // rows and tokens behind the last are the last one again; nothing of them is stored
  const uint8_t* wr[TN][W::ROWS];
  const float* xr[TM][2];
#pragma unroll
  for (int c = 0; c < TN; c++)
#pragma unroll
    for (int i = 0; i < W::ROWS; i++) wr[c][i] = w + (size_t)min(n0 + 16 * c + W::row_of(lane, i), out_dim - 1) * W::row_bytes(in_dim);
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int i = 0; i < 2; i++) xr[t][i] = x + (size_t)min(m0 + 16 * t + 8 * i + (lane >> 3), tokens - 1) * in_dim;
  terms_f4 acc[TM][TN];
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int c = 0; c < TN; c++) acc[t][c] = terms_f4{0.f, 0.f, 0.f, 0.f};

  struct Step {
    W w[TN];
    TermsF32Tile x[TM];
  };
  auto request = [&](Step& r, u32 s, auto full) {
#pragma unroll
    for (int c = 0; c < TN; c++) r.w[c].template load<decltype(full)::value>(wr[c], s, lane, in_dim);
#pragma unroll
    for (int t = 0; t < TM; t++) r.x[t].template load<decltype(full)::value>(xr[t], s, lane, in_dim);
  };
  auto put = [&](const Step& r) {
#pragma unroll
    for (int c = 0; c < TN; c++) r.w[c].put(mine + TM * XD + c * W::LDS_DWORDS, lane);
#pragma unroll
    for (int t = 0; t < TM; t++) r.x[t].put(mine + t * XD, lane);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the lanes read what other lanes of the wavefront wrote
  };
  // One step. INTERLEAVED: token tile t's matrix instructions go out term product by term product across the TN row tiles (TN independent
  // sums), with tile t + 1's terms and tile t - 1's sums made in between; else row tile by row tile, the three to eight products of a sum one after the
  // other. The same sums, bit for bit.
  auto compute = [&]() {
    if constexpr (INTERLEAVED) {
      constexpr bool AHEAD = W::TERMS == 1 || TM < 4;   // room for two sets of terms of x
      constexpr int XB = AHEAD ? 2 : 1;
      bf16x8_t B[TN][W::TERMS], X[XB][3];
      float d[TN];
      terms_f4 p[2][TN];
      float v[8];
      TermsF32Tile::get(mine, lane, v);
#pragma unroll
      for (int c = 0; c < TN; c++) {
        const u32* wl = mine + TM * XD + c * W::LDS_DWORDS;
        W::terms(wl, lane, B[c]);
        d[c] = W::scale(wl, lane);
      }
      terms_split<3>(v, X[0]);
      auto fold = [&](int t) {   // the sum over the step's 32 values joins the running sum in one rounding
#pragma unroll
        for (int c = 0; c < TN; c++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[t][c][e] = W::SCALED ? fmaf(d[c], p[t & 1][c][e], acc[t][c][e]) : acc[t][c][e] + p[t & 1][c][e];
      };
#pragma unroll
      for (int t = 0; t < TM; t++) {
        if (TM > 1) __builtin_amdgcn_sched_barrier(0);
        if (AHEAD && t + 1 < TM) TermsF32Tile::get(mine + (t + 1) * XD, lane, v);
        if (!AHEAD && t > 0) {
          TermsF32Tile::get(mine + t * XD, lane, v);
          terms_split<3>(v, X[0]);
        }
#pragma unroll
        for (int c = 0; c < TN; c++) p[t & 1][c] = terms_f4{0.f, 0.f, 0.f, 0.f};
        // term i of x against term j of w, i + j <= 3, smallest first
#pragma unroll
        for (int ij = 3; ij >= 0; ij--)
#pragma unroll
          for (int j = 0; j < W::TERMS; j++)
            if (ij - j >= 0 && ij - j < 3) {
#pragma unroll
              for (int c = 0; c < TN; c++) p[t & 1][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(X[t % XB][ij - j], B[c][j], p[t & 1][c], 0, 0, 0);
            }
        if (AHEAD && t + 1 < TM) terms_split<3>(v, X[(t + 1) % XB]);
        if (t > 0) fold(t - 1);
        if (AHEAD && TM > 1) {
          constexpr int MFMAS = TN * (W::TERMS == 1 ? 3 : (W::TERMS == 2 ? 6 : 8)), VALU = (72 + 4 * TN + MFMAS - 1) / MFMAS;
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
          for (int i = 0; i < MFMAS; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
          }
        }
      }
      if (TM > 1) __builtin_amdgcn_sched_barrier(0);
      fold(TM - 1);
    } else {
      bf16x8_t X[TM][3];
#pragma unroll
      for (int t = 0; t < TM; t++) {
        float v[8];
        TermsF32Tile::get(mine + t * XD, lane, v);
        terms_split<3>(v, X[t]);
      }
#pragma unroll
      for (int c = 0; c < TN; c++) {
        const u32* wl = mine + TM * XD + c * W::LDS_DWORDS;
        bf16x8_t B[W::TERMS];
        W::terms(wl, lane, B);
        const float d = W::scale(wl, lane);
#pragma unroll
        for (int t = 0; t < TM; t++) {
          // term i of x against term j of w, i + j <= 3, smallest first; the sum over the step's 32 values joins the running sum
          // in one rounding
          terms_f4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ij = 3; ij >= 0; ij--)
#pragma unroll
            for (int j = 0; j < W::TERMS; j++)
              if (ij - j >= 0 && ij - j < 3) p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(X[t][ij - j], B[j], p, 0, 0, 0);
#pragma unroll
          for (int v = 0; v < 4; v++) acc[t][c][v] = W::SCALED ? fmaf(d, p[v], acc[t][c][v]) : acc[t][c][v] + p[v];
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  // whole steps: contiguous runs of them per wavefront; a last step that the row ends inside is added by the last wavefront
  const u32 steps = in_dim >> 5;
  const u32 s0 = wave * steps / GEMM_TERMS_WAVES, s1 = (wave + 1) * steps / GEMM_TERMS_WAVES;
  if (s0 < s1) {
    Step ring[D];
#pragma unroll
    for (int d = 0; d < D; d++) request(ring[d], min(s0 + d, s1 - 1), std::true_type{});
    for (u32 s = s0; s < s1; s += D) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        put(ring[d]);
        request(ring[d], min(s + D + d, s1 - 1), std::true_type{});
        if (s + d < s1) compute();
      }
    }
  }
  if ((in_dim & 31u) != 0 && wave == GEMM_TERMS_WAVES - 1) {
    Step last;
    request(last, steps, std::false_type{});
    put(last);
    compute();
  }
  __syncthreads();   // the regions are free: the k-slices' sums take their place
  terms_f4* const part = reinterpret_cast<terms_f4*>(lds4);
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int c = 0; c < TN; c++) part[(wave * (TM * TN) + t * TN + c) * 64 + lane] = acc[t][c];
  __syncthreads();
  // a lane's four sums are tokens 4 (lane / 16) .. + 3 of its tile for weight row lane % 16
  u32 again = 0;   // four bits a tile: the lane's sums that are no finite numbers
#pragma unroll
  for (u32 i = wave, j = 0; i < TM * TN; i += GEMM_TERMS_WAVES, j++) {
    terms_f4 p[GEMM_TERMS_WAVES];
#pragma unroll
    for (u32 k = 0; k < GEMM_TERMS_WAVES; k++) p[k] = part[(k * (TM * TN) + i) * 64 + lane];
#pragma unroll
    for (u32 h = GEMM_TERMS_WAVES / 2; h; h >>= 1)   // in pairs: three roundings on the way, not seven
#pragma unroll
      for (u32 k = 0; k < h; k++) p[k] += p[k + h];
    const u32 n = n0 + 16 * (i % TN) + row;
    const u32 mb = m0 + 16 * (i / TN) + 4 * kg;
    if (n < out_dim) {
#pragma unroll
      for (u32 v = 0; v < 4; v++)
        if (mb + v < tokens) {
          const size_t at = (size_t)(mb + v) * out_dim + n;
          const float r = p[0][v] * W::UNSCALE;   // exact, but for one rounding of a subnormal result
          if (__builtin_isfinite(r)) out[at] = residual ? residual[at] + r : r;
          else again |= 1u << (4 * j + v);
        }
    }
  }
  u32* const flag = reinterpret_cast<u32*>(lds4) + PART_DWORDS;
  const bool any = __builtin_amdgcn_ballot_w64(again != 0) != 0;
  if (lane == 0) flag[wave] = any;
  __syncthreads();
  u32 sum = 0;
#pragma unroll
  for (u32 k = 0; k < GEMM_TERMS_WAVES; k++) sum |= flag[k];
  if (__builtin_amdgcn_readfirstlane(sum) == 0) return;
  // All wavefronts share the tile's sums that have to be taken again (the k-slices' sums in LDS have been read). A NaN among the first
  // values of a token, as in a row of NaNs, is the answer for all its sums.
  u32* const todo = reinterpret_cast<u32*>(lds4);
  u32* const nan = todo + TM * TN * 64;
  for (u32 i = wave, j = 0; i < TM * TN; i += GEMM_TERMS_WAVES, j++) todo[i * 64 + lane] = (again >> (4 * j)) & 15u;
  for (u32 t = wave; t < 16 * TM; t += GEMM_TERMS_WAVES) {
    const float v = lane < in_dim ? x[(size_t)min(m0 + t, tokens - 1) * in_dim + lane] : 0.f;
    const bool is = __builtin_amdgcn_ballot_w64(v != v) != 0;
    if (lane == 0) nan[t] = is;
  }
  __syncthreads();
  for (u32 q = wave; q < TM * TN * 64; q += GEMM_TERMS_WAVES) {
    const u32 which = __builtin_amdgcn_readfirstlane(todo[q]);
    if (which == 0) continue;
    const u32 i = q >> 6, n = n0 + 16 * (i % TN) + (q & 15), t0 = 16 * (i / TN) + 4 * ((q >> 4) & 3), mb = m0 + t0;
    u32 known = 0;
    const float* xs[4];
#pragma unroll
    for (u32 v = 0; v < 4; v++) {
      known |= nan[t0 + v] << v;
      xs[v] = x + (size_t)min(mb + v, tokens - 1) * in_dim;
    }
    known = __builtin_amdgcn_readfirstlane(known);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    if (which & ~known) terms_plain_sums<W>(w + (size_t)n * W::row_bytes(in_dim), xs, in_dim, lane, s);
    if (lane == 0) {
#pragma unroll
      for (u32 v = 0; v < 4; v++)
        if (which & (1u << v)) {
          const size_t at = (size_t)(mb + v) * out_dim + n;
          const float r = known & (1u << v) ? __builtin_nanf("") : s[v];
          out[at] = residual ? residual[at] + r : r;
        }
    }
  }
}

#define GEMM_TERMS_ENTRY(NAME, W, TM, TN, D, INTERLEAVED)                                                                       \
  extern "C" __global__ __launch_bounds__(64 * GEMM_TERMS_WAVES) void NAME(const uint8_t* w, const float* x, const float* residual, \
                                                                           float* out, u32 in_dim, u32 out_dim, u32 tokens) {  \
    gemm_terms_core<W, TM, TN, D, INTERLEAVED>(w, x, residual, out, in_dim, out_dim, tokens);                                  \
  }
// The tiles that are interleaved at every row length or at none have one kernel, the others a second one of the name with "_i".
#define GEMM_TERMS_TYPE(PREFIX, W, SHORT)                            \
  GEMM_TERMS_ENTRY(PREFIX##_gemm_terms_f32_1x1, W, 1, 1, 2, false)   \
  GEMM_TERMS_ENTRY(PREFIX##_gemm_terms_f32_1x2, W, 1, 2, 2, SHORT)   \
  GEMM_TERMS_ENTRY(PREFIX##_gemm_terms_f32_2x2, W, 2, 2, 2, false)   \
  GEMM_TERMS_ENTRY(PREFIX##_gemm_terms_f32_2x2_i, W, 2, 2, 2, true)  \
  GEMM_TERMS_ENTRY(PREFIX##_gemm_terms_f32_2x4, W, 2, 4, 1, false)   \
  GEMM_TERMS_ENTRY(PREFIX##_gemm_terms_f32_4x4, W, 4, 4, 1, true)
GEMM_TERMS_TYPE(f32, TermsF32, true)
GEMM_TERMS_TYPE(f16, TermsF16, true)
GEMM_TERMS_TYPE(iq4_nl, TermsIq4nl, false)
GEMM_TERMS_TYPE(q8_0, TermsQ80, false)
GEMM_TERMS_ENTRY(f16_gemm_terms_f32_2x4_i, TermsF16, 2, 4, 1, true)
GEMM_TERMS_ENTRY(iq4_nl_gemm_terms_f32_2x4_i, TermsIq4nl, 2, 4, 1, true)
GEMM_TERMS_ENTRY(q8_0_gemm_terms_f32_2x4_i, TermsQ80, 2, 4, 1, true)
