// Prefill GEMM over raw Q4_K weights, tiles of 256 tokens x 256 weight rows: launches of many tokens (gemm_tall_takes in gemv_config.h).
// Operands and element order of gemm_q4k.hpp; precision as there (x and the dequantized weights rounded to half, fp32 sums).
//
//   q4_k_gemm_tall_f16 (list: GemmManyArgs by value, tile_end in tiles of 256 rows, xp, in_dim:u32, m:u32)
//                      block 256, grid gemm_tiles_grid(ceil(m/256), tiles) from gemv_config.h, no dynamic LDS (160 KiB static)
//   q4_k_gemm_tall_pack_f16 (list, next: GemmNextArgs by value, xp, in_dim, m): next.xq[i] gets out[i] as the packed input of a following GEMM
//   q4_k_gemm_tall_swiglu_pack_q4k|q6k_f16 (w_gate, w_up, xp, out | null, xq, in_dim, out_dim, m): a tile is 128 rows of each matrix;
//                      grid gemm_tiles_grid(ceil(m/256), ceil(out_dim/128)); products and packed activations as the kernels of gemm_q4k.hpp
//   xp is the image pack_x_f16_q4k writes.
//
// Why this tile. On this chip a matrix instruction takes 7 to 8 clocks of the SIMD's issue beside the 4 of every vector one (32x32x16 with 8
// vector instructions each: 19.1 ns where they take 14.4 and 15.9 alone), and the 128-token kernels, which decode a weight once per 128 tokens, spend
// 5.6 vector instructions per matrix instruction: issue is what they run out of (46 % vector, 56 % matrix cycles). Here a wavefront
// has 256 tokens x 64 rows (8 x 2 tiles of v_mfma_f32_32x32x16_f16, all 256 accumulator registers), so a decoded operand is used eight
// times, and an operand of x twice; one wavefront per SIMD, the four of a workgroup share the 256 tokens' activations in LDS.
// The k range is walked by one wavefront in order (the 128-token kernels add two halves at the end), so the sums are not theirs bit for bit: with operands that are
// exact in half, 2-norm of the error against 64 bits, 128-token kernels | these, 4096 columns 2.89e-7 | 4.05e-7, 512 1.06e-7 | 1.45e-7, 12288 4.98e-7 | 7.09e-7. Of the outputs, whose
// operands are rounded to half, it is the same: 3.57372e-4 both, 3.57230e-4 both, 3.62460e-4 | 3.62461e-4 (300 tokens of 2304 columns 3.70261e-4 | 3.70260e-4).
// 512 x 30720 x 4096 in one launch: 116 us = 1.11 PFLOP/s, 139 to 149 on the eight-wavefront kernel (two rounds of tiles there, one here); 2048 tokens
// 438 | 522, and 6.1 us a super-block = 1.34 PFLOP/s between start and end, which are 18 us of a round (12 without the stores). What bounds
// the loop is the chip's power: with half the compute units a super-block takes 4.1 us. torch's fp16 product of the shape 1.32 PFLOP/s.
//
// Staging. x: the super-block in quarters of four k-steps (256 tokens: 32 KiB), each in a buffer of its own. A quarter's buffer is free behind the
// barrier in front of its last k-step, is filled again at once (the next super-block's quarter, global_load_lds_dwordx4) and needed eleven
// k-steps later, about 5600 clocks. Weights: a wavefront copies the 128 bytes of codes of its 64 rows into a region of its own when it has
// taken the super-block before into registers; headers go straight to registers. Loads are waited for by count: a super-block issues, in
// order, 8 copies of weights (k-step 0), 2 loads of headers (1), and 8 copies of x in k-steps 3, 7, 11 and 15.
#pragma once
#include "gemm_q4k_wide.hpp"

#define GEMM_TALL_BM 256
#define GEMM_TALL_BN 256

__shared__ uint4 gemm_tall_x0[2048];   // [128-token tile 2][k-step 4][k-group][128 tokens]: k-steps 0..3 of a super-block
__shared__ uint4 gemm_tall_x1[2048];
__shared__ uint4 gemm_tall_x2[2048];
__shared__ uint4 gemm_tall_x3[2048];
__shared__ uint4 gemm_tall_w[4 * 512];   // [wavefront][64 rows][8 pieces]: piece q of row r in slot 8 r + (q ^ (r & 7))

// 16 bytes per lane from base + voff (base uniform) to the LDS byte address lds + 16 lane (lds uniform). In asm, so that the compiler, which takes a
// read of LDS for one of any copy in flight once it has too many of them to tell apart, does not wait for all of them in front of the
// operand reads: the copies are waited for by the counted waits of the loop alone. (Volatile, so they stay between those; M0 is written nowhere else
// in these kernels, check_hazards.py.)
__device__ __forceinline__ void gemm_tall_copy(u32 lds, const void* base, u32 voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(voff), "s"(base));
}

// 16 bytes per lane from base + voff into registers, valid behind the counted wait that covers the load and a gemm_tall_pin (a plain load would be
// waited for with all the copies behind it; check_hazards.py looks that nothing touches the registers earlier)
typedef u32 gemm_tall_u4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void gemm_tall_load(gemm_tall_u4& dst, const void* base, u32 voff) {
  asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(dst) : "v"(voff), "s"(base));
}
__device__ __forceinline__ void gemm_tall_pin(gemm_tall_u4& v) { asm volatile("" : "+v"(v)); }

// A lane's sums: acc[r][c][4 g4 + v] is token 32 r + j, row 32 c + 8 g4 + 4 kg + v of the wavefront's 64: stored as they lie, an instruction
// would write 32 pieces of 32 bytes. They go through the wavefront's own quarter of x instead (no barrier), 128 tokens at a time, and out as
// four whole runs of 256 bytes an instruction.
__device__ __forceinline__ void gemm_tall_store(const float16_t (&acc)[8][2], float4* lds, float* out, u32 out_dim, u32 m, u32 token0, u32 col0, u32 j,
                                                u32 kg, u32 lane) {
  const bool vec = (out_dim & 3u) == 0;
  const u32 piece = lane & 15, n = col0 + 4 * piece;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    // piece q of token t of the 128 in slot 16 t + (q ^ (t & 15))
#pragma unroll
    for (int rr = 0; rr < 4; rr++)
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
          const float16_t& t = acc[4 * h + rr][c];
          lds[(32 * rr + j) * 16 + ((8 * c + 2 * g4 + kg) ^ (j & 15))] = make_float4(t[4 * g4], t[4 * g4 + 1], t[4 * g4 + 2], t[4 * g4 + 3]);
        }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const u32 first = token0 + 128 * h + (lane >> 4);
    auto put = [&](auto whole, auto vec16) {
#pragma unroll 8
      for (u32 i = 0; i < 32; i++) {
        const u32 t = 4 * i + (lane >> 4), token = first + 4 * i;
        const float4 v = lds[t * 16 + (piece ^ (t & 15))];
        if (!decltype(whole)::value && (token >= m || n >= out_dim)) continue;
        float* dst = out + (size_t)token * out_dim + n;
        if (decltype(vec16)::value && (decltype(whole)::value || n + 4 <= out_dim)) {
          *reinterpret_cast<float4*>(dst) = v;
        } else {
          const float ov[4] = {v.x, v.y, v.z, v.w};
          for (u32 e = 0; e < 4 && n + e < out_dim; e++) dst[e] = ov[e];
        }
      }
    };
    if (vec && token0 + GEMM_TALL_BM <= m && col0 + 64 <= out_dim) put(std::true_type{}, std::true_type{});
    else if (vec) put(std::false_type{}, std::true_type{});
    else put(std::false_type{}, std::false_type{});
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

// silu(g) * u as swiglu_one gives it, in 20 instructions instead of 30 (a tile's products are 128 a lane, with one wavefront per SIMD to make them). e^-g is
// 2^n 2^f with n whole and n + f = -g log2 e in two parts; g is held to 200, behind which e^-g is 0 or infinite and its parts would be no numbers. 1 / (1 + e^-g) is
// taken of a quarter of the sum, so that it is not flushed where e^-g nears the largest float; the quotient is corrected once and put right for infinities and
// NaN by the last step of a division. The bits of swiglu_one on all of ten times 2^24 gates tried (scales of 0.01 to 60, the ends of the range, -104 to -86). With
// swiglu_one the products of a tile are 11 of its 130 us; 16 instructions that round once more (2-norm of the error 4.72e-8 where swiglu_one has 4.67e-8) are 0.3 % faster over the
// whole FFN block of 2048 tokens.
__device__ __forceinline__ float gemm_tall_silu(float g, float u) {
  const float x = __builtin_amdgcn_fmed3f(g, -200.0f, 200.0f), h = x * -0x1.715476p+0f, n = __builtin_rintf(h);
  const float l = fmaf(x, -0x1.4ae0c0p-26f, fmaf(x, -0x1.715476p+0f, -h));   // log2 e = 0x1.715476p+0 + 0x1.4ae0c0p-26
  const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((h - n) + l), (int)n);
  const float d = 1.0f + e, r = 0.25f * __builtin_amdgcn_rcpf(fmaf(e, 0.25f, 0.25f)), q = g * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, g), r, q), d, g) * u;
}

// Gate (nh = 0, 1) and up (nh = 2, 3) wavefronts of the same 64 rows exchange half of their sums through LDS, each stores silu(gate) * up for
// half of the column quads: gemm_wide_epilogue_swiglu_half without the k halves.
template <int PACK>
__device__ __forceinline__ void gemm_tall_swiglu(const float16_t (&acc)[8][2], float* out, u32 out_dim, u32 m, u32 mt, u32 nt, u32 nh, u32 j, u32 kg,
                                                 u32 lane, uint2* xq) {
  const u32 col0 = nt * (GEMM_TALL_BN / 2) + (nh & 1) * 64, mtiles = (m + GEMM_BM - 1) / GEMM_BM;
  const bool vec = (out_dim & 3u) == 0;
  auto region = [&](u32 of) {
    return reinterpret_cast<float4*>(of == 0 ? gemm_tall_x0 : (of == 1 ? gemm_tall_x1 : (of == 2 ? gemm_tall_x2 : gemm_tall_x3))) + lane;
  };
  auto half = [&](auto upc) {
    constexpr int UP = decltype(upc)::value;
    float4* const mine = region(nh);
#pragma unroll
    for (int r = 0; r < 8; r++)
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int gg = 0; gg < 2; gg++) {
          const int g4 = UP == 0 ? 2 + gg : gg;   // the quad given away
          const float16_t& t = acc[r][c];
          mine[((r * 2 + c) * 2 + gg) * 64] = make_float4(t[4 * g4], t[4 * g4 + 1], t[4 * g4 + 2], t[4 * g4 + 3]);
        }
    __syncthreads();
    const float4* const theirs = region(nh ^ 2u);
#pragma unroll
    for (int r = 0; r < 8; r++) {
      const u32 token = mt * GEMM_TALL_BM + 32 * r + j, tile = 2 * mt + (r >> 2);
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int gg = 0; gg < 2; gg++) {
          const int g4 = UP == 0 ? gg : 2 + gg;   // the quad finished here
          const float16_t& t = acc[r][c];
          const float4 other = theirs[((r * 2 + c) * 2 + gg) * 64];
          const float4 own = make_float4(t[4 * g4], t[4 * g4 + 1], t[4 * g4 + 2], t[4 * g4 + 3]);
          const float4 g = UP == 0 ? own : other, u = UP == 0 ? other : own;
          const float4 o = make_float4(gemm_tall_silu(g.x, u.x), gemm_tall_silu(g.y, u.y), gemm_tall_silu(g.z, u.z), gemm_tall_silu(g.w, u.w));
          const u32 n8 = col0 + 32 * c + 8 * g4, n = n8 + 4 * kg;
          if (out && token < m && n < out_dim) {
            float* dst = out + (size_t)token * out_dim + n;
            if (vec && n + 4 <= out_dim) {
              *reinterpret_cast<float4*>(dst) = o;
            } else {
              const float ov[4] = {o.x, o.y, o.z, o.w};
              for (u32 e = 0; e < 4 && n + e < out_dim; e++) dst[e] = ov[e];
            }
          }
          if (n8 < out_dim && tile < mtiles) {
            // half kg of the cell that rows n8 .. n8 + 7 fill as k values of the next matrix; absent tokens are zeros
            const u32 kb = n8 >> 8, k = n8 & 255u;
            u32 ks, kgr;
            if (PACK == 14) {
              ks = 8 * (k >> 7) + 2 * ((k >> 5) & 3) + ((k >> 3) & 1);
              kgr = (k >> 4) & 1;
            } else {
              const u32 g6 = k >> 6;
              ks = 8 * (g6 >> 1) + 4 * ((k >> 4) & 1) + 2 * ((k >> 5) & 1) + ((k >> 3) & 1);
              kgr = g6 & 1;
            }
            const float4 z = token < m ? o : make_float4(0.f, 0.f, 0.f, 0.f);
            const __half2 p0 = __floats2half2_rn(z.x, z.z), p1 = __floats2half2_rn(z.y, z.w);   // slot order 0,2,1,3
            xq[(((size_t)tile * (out_dim >> 8) + kb) * 4096 + (ks * 2 + kgr) * 128 + 32 * (r & 3) + j) * 2 + kg] =
                make_uint2(__builtin_bit_cast(u32, p0), __builtin_bit_cast(u32, p1));
          }
        }
    }
  };
  if (nh < 2) half(std::integral_constant<int, 0>{});
  else half(std::integral_constant<int, 1>{});
}

// The sums as packed inputs of following GEMMs, straight from the registers: the lanes j and 32 + j hold the halves of a cell, two quads of them
// are exchanged so that each lane has a whole one. (out_dim is whole super-blocks, so all 64 rows exist or none.) 512 tokens x 30720 x 4096, 16384 of the
// rows packed: 123 us, 129 with a pack launch behind the list; with stores of half cells there was nothing to gain.
__device__ __forceinline__ void gemm_tall_next(const float16_t (&acc)[8][2], uint4* xq, bool q6, u32 out_dim, u32 m, u32 mt, u32 row0, u32 j, u32 kg) {
  const u32 mtiles = (m + GEMM_BM - 1) / GEMM_BM;
  if (row0 >= out_dim) return;
  uint4* const dst = xq + ((size_t)(2 * mt) * (out_dim >> 8) + (row0 >> 8)) * 4096 + j;
  const size_t tile = (size_t)(out_dim >> 8) * 4096;
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int g4 = 0; g4 < 4; g4 += 2) {
      const u32 cell = gemm_next_cell(q6, (row0 & 255u) + 32 * c + 8 * (g4 + kg));
#pragma unroll
      for (int r = 0; r < 8; r++) {
        if (2 * mt + (r >> 2) >= mtiles) break;
        const bool there = mt * GEMM_TALL_BM + 32 * r + j < m;
        const float16_t& t = acc[r][c];
        const uint2 e = gemm_next_half(make_float4(t[4 * g4], t[4 * g4 + 1], t[4 * g4 + 2], t[4 * g4 + 3]), there);
        const uint2 o = gemm_next_half(make_float4(t[4 * g4 + 4], t[4 * g4 + 5], t[4 * g4 + 6], t[4 * g4 + 7]), there);
        const auto x = __builtin_amdgcn_permlane32_swap(e.x, o.x, false, false), y = __builtin_amdgcn_permlane32_swap(e.y, o.y, false, false);
        dst[(r >> 2) * tile + cell * 128 + 32 * (r & 3)] = make_uint4(x[0], y[0], x[1], y[1]);
      }
    }
}

// PACK 0: a list of matrices, NEXT: their outputs as packed inputs too. 12 | 14: gate | up with SwiGLU, the products packed for a next matrix of that type.
template <int PACK, bool NEXT = false>
__device__ __forceinline__ void gemm_tall_core(const uint8_t* w, const uint8_t* w_b, const uint4* xp, float* out, uint2* xq, u32 in_dim, u32 out_dim,
                                               u32 m, const GemmManyArgs* many, const GemmNextArgs* next = nullptr) {
  constexpr u32 BS = 144, TILE_ROWS = PACK ? GEMM_TALL_BN / 2 : GEMM_TALL_BN;   // rows of a matrix a tile covers
  const u32 tid = threadIdx.x, lane = tid & 63;
  const u32 nh = __builtin_amdgcn_readfirstlane(tid >> 6);
  const u32 j = lane & 31, kg = lane >> 5;
  const u32 nkb = in_dim >> 8;
  const u32 mtiles = (m + GEMM_TALL_BM - 1) / GEMM_TALL_BM;
  const u32 ntiles = PACK ? (out_dim + TILE_ROWS - 1) / TILE_ROWS : many->tile_end[many->count - 1];
  u32 mt, nt;
  if (!gemm_tile_of(blockIdx.x, mtiles, ntiles, &mt, &nt)) return;
  [[maybe_unused]] u32 mi = 0;
  if constexpr (PACK == 0) {   // the tile's matrix, uniform over the workgroup
    u32 i = 0, first = 0;
    while (i + 1 < many->count && nt >= many->tile_end[i]) first = many->tile_end[i++];
    nt -= first;
    w = many->w[i];
    out = many->out[i];
    out_dim = many->out_dim[i];
    if constexpr (NEXT) mi = i;
  }
  const size_t row_bytes = (size_t)nkb * BS;
  const u32 sh = 16u * kg;
  u32 magic_lo = 0x64006400u, magic_hi = 0x54005400u;
  asm volatile("" : "+v"(magic_lo), "+v"(magic_hi));

  // the wavefront's 64 rows of its matrix (one past the last row: the last row again)
  const u32 row0 = nt * TILE_ROWS + (PACK ? nh & 1 : nh) * 64;
  const u32 base_row = min(row0, out_dim - 1);
  const uint8_t* wbase = (PACK && nh >= 2 ? w_b : w) + (size_t)base_row * row_bytes;   // uniform
  // copy i: rows 8 i .. 8 i + 7, eight lanes a row; lane l brings the piece that belongs in slot l % 8 of its row
  u32 woff[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const u32 r = 8u * i + (lane >> 3);
    woff[i] = (min(row0 + r, out_dim - 1) - base_row) * (u32)row_bytes + 16u + 16u * ((lane & 7u) ^ (lane >> 3));
  }
  u32 hoff[2];
#pragma unroll
  for (int c = 0; c < 2; c++) hoff[c] = (min(row0 + 32 * c + j, out_dim - 1) - base_row) * (u32)row_bytes;
  const uint4* const wrow = gemm_tall_w + nh * 512 + j * 8;   // the lane's row c = 0 (c = 1: 256 further; 32 c + j and j agree modulo 8)
  const u32 jx = j & 7u;
  // the two 128-token tiles (behind the last one: the last again; nothing of it is stored)
  const u32 tile1 = min(2 * mt + 1, (m + GEMM_BM - 1) / GEMM_BM - 1);
  const uint4* const xt0 = xp + (size_t)(2 * mt) * nkb * 4096;
  const uint4* const xt1 = xp + (size_t)tile1 * nkb * 4096;

  float16_t acc[8][2];
#pragma unroll
  for (int r = 0; r < 8; r++)
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[r][c][v] = 0.0f;

  auto stage = [&](auto qc) -> uint4* {
    constexpr int Q = decltype(qc)::value;
    if constexpr (Q == 0) return gemm_tall_x0;
    else if constexpr (Q == 1) return gemm_tall_x1;
    else if constexpr (Q == 2) return gemm_tall_x2;
    else return gemm_tall_x3;
  };
  auto lds_of = [&](const uint4* at) { return (u32)(uintptr_t)(lds_void*)at; };
  auto copy_x = [&](u32 kb, auto qc, int i) {
    constexpr int Q = decltype(qc)::value;
    const uint4* src = (i < 4 ? xt0 : xt1) + (size_t)kb * 4096 + Q * 1024 + (i & 3) * 256 + nh * 64;
    gemm_tall_copy(lds_of(stage(qc)) + (i * 256 + nh * 64) * 16, src, lane * 16);
  };
  auto copy_w = [&](u32 kb, int i) { gemm_tall_copy(lds_of(gemm_tall_w) + (nh * 512 + i * 64) * 16, wbase + (size_t)kb * BS, woff[i]); };
  gemm_tall_u4 nhdr[2], hdr[2];
  auto load_hdr = [&](u32 kb, int c) { gemm_tall_load(nhdr[c], wbase + (size_t)kb * BS, hoff[c]); };

  uint4 raw[2][4];   // the lane's pieces of its two rows: 2 kg, 2 kg + 1 (k-steps 0..7), 4 + 2 kg, 5 + 2 kg (8..15)
  u32 S[2][4];
  uint4 A[2][8];
  half8_t B[2][2];
  auto take_raw = [&]() {
#pragma unroll
    for (int c = 0; c < 2; c++) {
      gemm_tall_pin(nhdr[c]);
      hdr[c] = nhdr[c];
#pragma unroll
      for (int q = 0; q < 4; q++) raw[c][q] = wrow[256 * c + ((4u * (q >> 1) + 2u * kg + (q & 1)) ^ jx)];
    }
  };
  auto decode_scales = [&](auto hc) {
    constexpr int H = decltype(hc)::value;
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const float d = h2f(hdr[c].x), dm = h2f(hdr[c].x >> 16);
      const u32 a0 = hdr[c].y >> sh, a1 = hdr[c].z >> sh, a2 = hdr[c].w >> sh;
      const u32 scp = H == 0 ? a0 & 0x3F3Fu : (a2 & 0x0F0Fu) | ((a0 >> 2) & 0x3030u);
      const u32 mp = H == 0 ? a1 & 0x3F3Fu : ((a2 >> 4) & 0x0F0Fu) | ((a1 >> 2) & 0x3030u);
      S[c][0] = h2_dup(d * ubyte_f<0>(scp));
      S[c][1] = h2_dup(-(dm * ubyte_f<0>(mp)));
      S[c][2] = h2_dup(d * ubyte_f<1>(scp));
      S[c][3] = h2_dup(-(dm * ubyte_f<1>(mp)));
    }
  };
  auto build_b = [&](half8_t (&Bd)[2], int ks) {
    const int h = (ks >> 2) & 1, op = ks & 3, hi = op >> 1;
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const uint4 Q = raw[c][2 * (ks >> 3) + h];
      const u32 qa = (op & 1) ? Q.z : Q.x, qb = (op & 1) ? Q.w : Q.y;
      const u32 mask = hi ? 0x00F000F0u : 0x000F000Fu;
      const u32 magic = hi ? magic_hi : magic_lo;
      const u32 off = hi ? 0xD400D400u : 0xE400E400u;
      const u32 sc = S[c][2 * hi], nm = S[c][2 * hi + 1];
      uint4 bw;
      bw.x = h2_fma_off((qa & mask) | magic, off, sc, nm);
      bw.y = h2_fma_off(((qa >> 8) & mask) | magic, off, sc, nm);
      bw.z = h2_fma_off((qb & mask) | magic, off, sc, nm);
      bw.w = h2_fma_off(((qb >> 8) & mask) | magic, off, sc, nm);
      Bd[c] = *reinterpret_cast<const half8_t*>(&bw);
    }
  };
  const u32 xlane = kg * 128 + j;
  auto read_a = [&](uint4 (&Ad)[8], auto ksc) {
    constexpr int KS = decltype(ksc)::value;
    const uint4* arow = stage(std::integral_constant<int, KS / 4>{}) + xlane + (KS % 4) * 256;
#pragma unroll
    for (int r = 0; r < 8; r++) Ad[r] = arow[(r >> 2) * 1024 + (r & 3) * 32];
  };

  // super-block 0: weights, headers, then the quarters of x; the first quarter is waited for with 24 copies behind it in flight
#pragma unroll
  for (int i = 0; i < 8; i++) copy_w(0, i);
  load_hdr(0, 0);
  load_hdr(0, 1);
#pragma unroll
  for (int i = 0; i < 8; i++) copy_x(0, std::integral_constant<int, 0>{}, i);
#pragma unroll
  for (int i = 0; i < 8; i++) copy_x(0, std::integral_constant<int, 1>{}, i);
#pragma unroll
  for (int i = 0; i < 8; i++) copy_x(0, std::integral_constant<int, 2>{}, i);
#pragma unroll
  for (int i = 0; i < 8; i++) copy_x(0, std::integral_constant<int, 3>{}, i);
  asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  take_raw();
  read_a(A[0], std::integral_constant<int, 0>{});
  decode_scales(std::integral_constant<int, 0>{});
  build_b(B[0], 0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  for (u32 kb = 0; kb < nkb; kb++) {
    const u32 kn = min(kb + 1, nkb - 1);   // the last iteration copies its own super-block again; it is not used
    auto step = [&](auto tc) {
      constexpr int t = decltype(tc)::value, p = t & 1;
      if constexpr (t == 1) {
        load_hdr(kn, 0);
        load_hdr(kn, 1);
      }
      if constexpr (t < 15) {
        read_a(A[p ^ 1], std::integral_constant<int, t + 1>{});
        if constexpr (t == 7) decode_scales(std::integral_constant<int, 1>{});
        build_b(B[p ^ 1], t + 1);
      } else {
        // the next super-block's weights, headers and first quarter are there (wait and barrier behind k-step 14)
        take_raw();
        read_a(A[0], std::integral_constant<int, 0>{});
        decode_scales(std::integral_constant<int, 0>{});
        build_b(B[0], 0);
      }
#pragma unroll
      for (int r = 0; r < 8; r++) {
        const half8_t Ar = *reinterpret_cast<const half8_t*>(&A[p][r]);
#pragma unroll
        for (int c = 0; c < 2; c++) acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(B[p][c], Ar, acc[r][c], 0, 0, 0);
        if constexpr (t == 0) copy_w(kn, r);
        if constexpr (t % 4 == 3) copy_x(kn, std::integral_constant<int, t / 4>{}, r);
      }
#pragma unroll
      for (int c = 0; c < 2; c++) asm volatile("" : "+v"(B[p ^ 1][c]));
      if constexpr (t < 15) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, t == 7 ? 5 : 3, 0);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, t == 7 ? 6 : 3, 0);
        }
      } else {
        __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
        for (int i = 0; i < 8; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (t % 4 == 2) {
        // the quarter the next k-step reads from is there (26 younger loads may be in flight; behind k-step 14, where the next
        // super-block's weights and headers have to be there too, 16), and this wavefront's reads of the quarter it leaves are done; behind the barrier
        // that holds for every wavefront
        if constexpr (t == 14) asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(26) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
    step(std::integral_constant<int, 4>{});
    step(std::integral_constant<int, 5>{});
    step(std::integral_constant<int, 6>{});
    step(std::integral_constant<int, 7>{});
    step(std::integral_constant<int, 8>{});
    step(std::integral_constant<int, 9>{});
    step(std::integral_constant<int, 10>{});
    step(std::integral_constant<int, 11>{});
    step(std::integral_constant<int, 12>{});
    step(std::integral_constant<int, 13>{});
    step(std::integral_constant<int, 14>{});
    step(std::integral_constant<int, 15>{});
    // the raw bytes taken in the last k-step are in registers before the next iteration's copies overwrite the region
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last (unused) copies
  __syncthreads();
  if constexpr (NEXT) {
    if (next->xq[mi]) gemm_tall_next(acc, reinterpret_cast<uint4*>(next->xq[mi]), next->q6 >> mi & 1u, out_dim, m, mt, row0, j, kg);
  }
  if constexpr (PACK != 0) gemm_tall_swiglu<PACK>(acc, out, out_dim, m, mt, nt, nh, j, kg, lane, xq);
  else gemm_tall_store(acc, reinterpret_cast<float4*>(nh == 0 ? gemm_tall_x0 : (nh == 1 ? gemm_tall_x1 : (nh == 2 ? gemm_tall_x2 : gemm_tall_x3))), out, out_dim, m,
                       mt * GEMM_TALL_BM, row0, j, kg, lane);
}

#define GEMM_TALL_KERNEL extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void
GEMM_TALL_KERNEL q4_k_gemm_tall_f16(const GemmManyArgs list, const uint4* xp, u32 in_dim, u32 m) {
  gemm_tall_core<0>(nullptr, nullptr, xp, nullptr, nullptr, in_dim, 0, m, &list);
}
GEMM_TALL_KERNEL q4_k_gemm_tall_pack_f16(const GemmManyArgs list, const GemmNextArgs next, const uint4* xp, u32 in_dim, u32 m) {
  gemm_tall_core<0, true>(nullptr, nullptr, xp, nullptr, nullptr, in_dim, 0, m, &list, &next);
}
GEMM_TALL_KERNEL q4_k_gemm_tall_swiglu_pack_q4k_f16(const uint8_t* w_gate, const uint8_t* w_up, const uint4* xp, float* out, uint2* xq, u32 in_dim,
                                                    u32 out_dim, u32 m) {
  gemm_tall_core<12>(w_gate, w_up, xp, out, xq, in_dim, out_dim, m, nullptr);
}
GEMM_TALL_KERNEL q4_k_gemm_tall_swiglu_pack_q6k_f16(const uint8_t* w_gate, const uint8_t* w_up, const uint4* xp, float* out, uint2* xq, u32 in_dim,
                                                    u32 out_dim, u32 m) {
  gemm_tall_core<14>(w_gate, w_up, xp, out, xq, in_dim, out_dim, m, nullptr);
}
