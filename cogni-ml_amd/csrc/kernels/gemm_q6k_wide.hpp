// Prefill GEMM over raw Q6_K weights with eight wavefronts per workgroup: the wavefront roles of gemm_q4k_wide.hpp with the
// operands of gemm_q6k.hpp (block layout, element order and assembly of the codes there).
//
//   q6_k_gemm_wide_f16 (w_raw, xp, bias|null, out:f32 [m][out_dim], in_dim:u32, out_dim:u32, m:u32, bias_stride:u32)
//                      block 512, grid gemm_grid_x(ceil(m/128), ceil(out_dim/256)), no dynamic LDS (112 KiB static); no k split
//
// A workgroup owns 128 tokens x 256 rows; wavefront (row quarter nh, k half kh) accumulates 128 tokens x 64 rows over half
// kh of every super-block and copies the bytes that it decodes itself, so no two wavefronts share weights. Those are, of each
// row, ql[64 kh, +64) and qh[32 kh, +32): six pieces of 16 bytes, 6 KiB = six copies a super-block into a region of its own;
// the eight scale bytes of the half and d go from global memory to the lanes that need them.
// Two x tiles of a whole super-block (128 KiB) and these 48 KiB do not fit LDS. So x is staged by half super-blocks, the
// k-steps 0..3 and 4..7 of both k halves (32 KiB each, always in the same buffer): while one is consumed the other is filled,
// copies issued three k-steps ahead of the barrier that hands them over. Every load goes through a buffer descriptor: as 64-bit
// addresses the offsets of the copies cost 14 more registers, which spilled, and the compiler waited for all loads in flight in front
// of the operand reads. 12288 -> 4096 at 2048 tokens: 211 us = 0.98 PFLOP/s, 237 on 128 x 128 tiles.
#pragma once
#include "gemm_q4k_wide.hpp"
#include "gemm_q6k.hpp"

__shared__ uint4 gemm_q6w_x0[2048];        // [kh][k-step 0..3][k-group][128 tokens]
__shared__ uint4 gemm_q6w_x1[2048];        // the same of k-steps 4..7
__shared__ uint4 gemm_q6w_wbuf[8 * 384];   // [wavefront][64 rows][ql 4 pieces, qh 2 pieces]

// T4: raw Q4_K weights (codes 64 kh of a row's super-block, four copies into the same region; headers from global memory) in the same loop, T5: Q5_K
// (the 32 bytes of fifth bits behind the codes, six copies as here). Tile (mt, nt) of the matrix, super-blocks [kb0, kb1) of its rows.
enum GemmWideType { T6, T4, T5 };
template <GemmWideType W>
__device__ __forceinline__ void gemm_q6k_wide_core(const uint8_t* w, const uint4* xp, const float* bias, float* out, u32 in_dim, u32 out_dim, u32 m,
                                                   u32 bias_stride, u32 mt, u32 nt, u32 kb0, u32 kb1) {
  constexpr bool Q4 = W != T6, Q5 = W == T5;
  constexpr u32 BS = Q5 ? 176 : (Q4 ? 144 : 210);
  constexpr int NW = W == T4 ? 4 : 6;   // copies of a wavefront's weights per super-block
  const u32 tid = threadIdx.x, lane = tid & 63;
  const u32 wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const u32 nh = wave & 3, kh = wave >> 2;
  const u32 j = lane & 31, kg = lane >> 5;
  const u32 nkb = in_dim >> 8;
  const size_t row_bytes = (size_t)nkb * BS;
  // constants of the code assembly, kept in registers (as literals each (a & mask) | b would be two instructions): the masks
  // in scalar ones, of which an instruction takes one
  u32 mask_lo = 0x000F000Fu, mask_hi = 0x00F000F0u, magic_lo = 0x64006400u, magic_hi = 0x54005400u, m3_lo = 0x00300030u, m3_hi = 0x03000300u;
  asm volatile("" : "+s"(mask_lo), "+s"(mask_hi), "+s"(m3_lo), "+s"(m3_hi));
  asm volatile("" : "+v"(magic_lo), "+v"(magic_hi));

  const u32 row0 = nt * GEMM_WIDE_BN + nh * 64;        // first weight row of this wavefront
  const u32 base_row = min(row0, out_dim - 1);
  // loads through a buffer descriptor: scalar base, scalar offset of the super-block, a 32-bit offset per lane
  const __amdgpu_buffer_rsrc_t wrsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(w + (size_t)base_row * row_bytes), 0, 0xFFFFFFFFu, 0x00027000);
  // copy i of this wavefront: piece p = 64 i + lane is piece p % 6 of wave-local row p / 6 (Q4_K: of row p / 4 the piece that belongs in slot p % 4,
  // as in gemm_q4k_wide.hpp)
  u32 woff[NW];
#pragma unroll
  for (int i = 0; i < NW; i++) {
    const u32 p = 64u * i + lane, r = p / (u32)NW, part = p - NW * r;
    const u32 at = Q5 ? (part < 4u ? 48u + 64u * kh + 16u * part : 16u * (part - 3u)) : Q4 ? 16u + 64u * kh + 16u * (part ^ ((r >> 2) & 3u)) : part < 4u ? 64u * kh + 16u * part : 128u + 32u * kh + 16u * (part - 4u);
    woff[i] = (min(row0 + r, out_dim - 1) - base_row) * (u32)row_bytes + at;
  }
  u32 soff[2];   // scales of the half, row c of this lane (d is 16 - 8 kh bytes further); Q4_K: the header
#pragma unroll
  for (int c = 0; c < 2; c++) soff[c] = (min(row0 + 32 * c + j, out_dim - 1) - base_row) * (u32)row_bytes + (Q4 ? 0u : 192u + 8u * kh);
  const u32 wrow = wave * 384 + j * 6 + kg;   // the lane's first ql piece of its row c = 0 (c = 1: 192 further)
  const u32 wrow4 = wave * 384 + j * 4, slot4 = (2u * kg) ^ ((j >> 2) & 3u);   // its two pieces 2 kg, 2 kg + 1: slots slot4, slot4 ^ 1 (c = 1: 128 further)
  const __amdgpu_buffer_rsrc_t xrsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(xp + (size_t)mt * nkb * 4096), 0, 0xFFFFFFFFu, 0x00027000);

  float16_t acc[4][2];
#pragma unroll
  for (int r = 0; r < 4; r++)
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[r][c][v] = 0.0f;

  auto copy_w = [&](u32 kb, int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wrsrc, (lds_void*)(gemm_q6w_wbuf + wave * 384 + i * 64), 16, woff[i], kb * BS, 0, 0);
  };
  uint2 nsc[2];
  u32 nd[2];
  uint4 nh4[2];
  auto load_sc = [&](u32 kb, int c) {
    if constexpr (Q4) {
      nh4[c] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, soff[c], kb * BS, 0));
      return;
    }
    nsc[c] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(wrsrc, soff[c], kb * BS, 0));
    nd[c] = (u32)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(wrsrc, soff[c], kb * BS + (16u - 8u * kh), 0);
  };
  // copy i of half `hs` of a super-block's x: KiB 8 i + wave of the buffer, 16 of each kh
  const u32 xw = (wave & 7u) * 64;
  auto copy_x = [&](u32 kb, int hs, int i) {
    const u32 src = kb * 65536u + ((i >> 1) * 2048 + hs * 1024 + (i & 1) * 512 + xw) * 16u;   // uniform; 32 bits: GEMM_Q6W_MAX_KB
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xrsrc, (lds_void*)((hs ? gemm_q6w_x1 : gemm_q6w_x0) + i * 512 + xw), 16, lane * 16, src, 0, 0);
  };

  GemmRaw6 cur[2];
  uint4 cur5[2];   // Q5_K: the fifth bits of values 16 .. 31 of a run of 32 (cur.qh: 0 .. 15)
  u32 S[2][4];
  uint4 A[2][4];
  half8_t B[2][2];
  auto take_raw = [&]() {
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if constexpr (Q5) {
        cur[c].qa = gemm_q6w_wbuf[wrow + kg + 192 * c];
        cur[c].qb = gemm_q6w_wbuf[wrow + kg + 192 * c + 1];
        cur[c].qh = gemm_q6w_wbuf[wrow - kg + 192 * c + 4];
        cur5[c] = gemm_q6w_wbuf[wrow - kg + 192 * c + 5];
        continue;
      }
      if constexpr (Q4) {
        cur[c].qa = gemm_q6w_wbuf[wrow4 + 128 * c + slot4];
        cur[c].qb = gemm_q6w_wbuf[wrow4 + 128 * c + (slot4 ^ 1u)];
        continue;
      }
      cur[c].qa = gemm_q6w_wbuf[wrow + 192 * c];
      cur[c].qb = gemm_q6w_wbuf[wrow + 192 * c + 2];
      cur[c].qh = gemm_q6w_wbuf[wrow + 192 * c + 4];
    }
  };
  // d * sc of the four 16-value sub-blocks of the lane's group (scale bytes kg, kg + 2, kg + 4, kg + 6 of the half's eight)
  auto decode_scales = [&]() {
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if constexpr (Q4) {
        const float d4 = h2f(nh4[c].x), dm = h2f(nh4[c].x >> 16);
        const u32 a0 = nh4[c].y >> (16 * kg), a1 = nh4[c].z >> (16 * kg), a2 = nh4[c].w >> (16 * kg);
        const u32 scp = kh ? (a2 & 0x0F0Fu) | ((a0 >> 2) & 0x3030u) : a0 & 0x3F3Fu;
        const u32 mp = kh ? ((a2 >> 4) & 0x0F0Fu) | ((a1 >> 2) & 0x3030u) : a1 & 0x3F3Fu;
        S[c][0] = h2_dup(d4 * ubyte_f<0>(scp));
        S[c][1] = h2_dup(-(dm * ubyte_f<0>(mp)));
        S[c][2] = h2_dup(d4 * ubyte_f<1>(scp));
        S[c][3] = h2_dup(-(dm * ubyte_f<1>(mp)));
        continue;
      }
      const float d = h2f(nd[c]);
      const u32 lo = nsc[c].x >> (8 * kg), hi = nsc[c].y >> (8 * kg);
      S[c][0] = h2_dup(d * (float)(int)(signed char)(lo & 0xFFu));
      S[c][1] = h2_dup(d * (float)(int)(signed char)((lo >> 16) & 0xFFu));
      S[c][2] = h2_dup(d * (float)(int)(signed char)(hi & 0xFFu));
      S[c][3] = h2_dup(d * (float)(int)(signed char)((hi >> 16) & 0xFFu));
    }
  };
  auto build_b = [&](half8_t (&Bd)[2], int t) {   // as in gemm_q6k_core
    const int qd = t >> 1, h8 = t & 1, hi = qd >> 1;
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if constexpr (Q4) {   // as in gemm_wide_core
        const int op = t & 3, up = op >> 1;
        const uint4 P = (t >> 2) ? cur[c].qb : cur[c].qa;
        const u32 q0 = (op & 1) ? P.z : P.x, q1 = (op & 1) ? P.w : P.y;
        const u32 msk = up ? mask_hi : mask_lo, mag = up ? magic_hi : magic_lo, of = up ? 0xD400D400u : 0xE400E400u;
        if constexpr (Q5) {   // the fifth bit beside the nibble, as in gemm_k45_core
          const uint4 H = (t >> 2) ? cur5[c] : cur[c].qh;
          const u32 s5 = 2 * (2 * kh + kg) + up;
          const u32 h0 = ((op & 1) ? H.z : H.x) >> s5, h1 = ((op & 1) ? H.w : H.y) >> s5;
          constexpr u32 one = 0x00010001u;
          const int at = up ? 8 : 4;
          uint4 b5;
          b5.x = h2_fma_off((q0 & msk) | mag | ((h0 & one) << at), of, S[c][2 * up], S[c][2 * up + 1]);
          b5.y = h2_fma_off(((q0 >> 8) & msk) | mag | (((h0 >> 8) & one) << at), of, S[c][2 * up], S[c][2 * up + 1]);
          b5.z = h2_fma_off((q1 & msk) | mag | ((h1 & one) << at), of, S[c][2 * up], S[c][2 * up + 1]);
          b5.w = h2_fma_off(((q1 >> 8) & msk) | mag | (((h1 >> 8) & one) << at), of, S[c][2 * up], S[c][2 * up + 1]);
          Bd[c] = *reinterpret_cast<const half8_t*>(&b5);
          continue;
        }
        uint4 b4;
        b4.x = h2_fma_off((q0 & msk) | mag, of, S[c][2 * up], S[c][2 * up + 1]);
        b4.y = h2_fma_off(((q0 >> 8) & msk) | mag, of, S[c][2 * up], S[c][2 * up + 1]);
        b4.z = h2_fma_off((q1 & msk) | mag, of, S[c][2 * up], S[c][2 * up + 1]);
        b4.w = h2_fma_off(((q1 >> 8) & msk) | mag, of, S[c][2 * up], S[c][2 * up + 1]);
        Bd[c] = *reinterpret_cast<const half8_t*>(&b4);
        continue;
      }
      const uint4 Q = (qd & 1) ? cur[c].qb : cur[c].qa;
      const u32 qa = h8 ? Q.z : Q.x, qb = h8 ? Q.w : Q.y;
      const u32 ha = h8 ? cur[c].qh.z : cur[c].qh.x, hb = h8 ? cur[c].qh.w : cur[c].qh.y;
      const u32 mask = hi ? mask_hi : mask_lo, magic = hi ? magic_hi : magic_lo, m3 = hi ? m3_hi : m3_lo;
      const u32 off = hi ? 0xD600D600u : 0xE420E420u;   // half2(-96) : half2(-1056)
      const int sl = (qd & 1) ? 2 : 4, sr = (qd & 1) ? 6 : 4;
      const u32 sc = S[c][qd];
      u32 n0 = (qa & mask) | magic, n1 = ((qa >> 8) & mask) | magic, n2 = (qb & mask) | magic, n3 = ((qb >> 8) & mask) | magic;
      asm("" : "+v"(n0), "+v"(n1), "+v"(n2), "+v"(n3));
      uint4 bw;
      bw.x = h2_sub_mul(((ha << sl) & m3) | n0, off, sc);
      bw.y = h2_sub_mul(((ha >> sr) & m3) | n1, off, sc);
      bw.z = h2_sub_mul(((hb << sl) & m3) | n2, off, sc);
      bw.w = h2_sub_mul(((hb >> sr) & m3) | n3, off, sc);
      Bd[c] = *reinterpret_cast<const half8_t*>(&bw);
    }
  };
  const u32 xrow = kh * 1024 + kg * 128 + j;
  auto read_a = [&](uint4 (&Ad)[4], int t) {   // 32 lanes read 512 contiguous bytes
    const uint4* arow = ((t & 4) ? gemm_q6w_x1 : gemm_q6w_x0) + xrow + (t & 3) * 256;
#pragma unroll
    for (int r = 0; r < 4; r++) Ad[r] = arow[r * 32];
  };

#pragma unroll
  for (int i = 0; i < NW; i++) copy_w(kb0, i);
#pragma unroll
  for (int c = 0; c < 2; c++) load_sc(kb0, c);
#pragma unroll
  for (int i = 0; i < 4; i++) copy_x(kb0, 0, i);
#pragma unroll
  for (int i = 0; i < 4; i++) copy_x(kb0, 1, i);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  take_raw();
  read_a(A[0], 0);
  decode_scales();
  build_b(B[0], 0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  for (u32 kb = kb0; kb < kb1; kb++) {
    const u32 kn = min(kb + 1, kb1 - 1);   // the last iteration copies its own tile again; it is not used
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const int p = t & 1;
      // The raw bytes were taken into registers in the last k-step of the iteration before, so the region is free. x: half 0
      // is free behind the barrier of k-step 2, half 1 behind that of k-step 6; the copies into one follow the first reads of the
      // other, in front of which the compiler waits for every load in flight.
      if (t == 0) {
#pragma unroll
        for (int i = 0; i < NW; i++) copy_w(kn, i);
      }
      if (t == 3) {
        read_a(A[p ^ 1], t + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; i++) copy_x(kn, 0, i);
      }
      if (t == 5) {
        load_sc(kn, 0);
        load_sc(kn, 1);
      }
      if (t < 7) {
        if (t != 3) read_a(A[p ^ 1], t + 1);
        build_b(B[p ^ 1], t + 1);
      } else {
        take_raw();
        read_a(A[0], 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; i++) copy_x(kn, 1, i);
        decode_scales();
        build_b(B[0], 0);
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const half8_t Ar = *reinterpret_cast<const half8_t*>(&A[p][r]);
#pragma unroll
        for (int c = 0; c < 2; c++) acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(B[p][c], Ar, acc[r][c], 0, 0, 0);
      }
#pragma unroll
      for (int c = 0; c < 2; c++) asm volatile("" : "+v"(B[p ^ 1][c]));
      if (t < 7) {
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 7, 0);
#pragma unroll
        for (int i = 0; i < 8; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
        }
      } else {
        __builtin_amdgcn_sched_group_barrier(0x020, 4, 0);
#pragma unroll
        for (int i = 0; i < 8; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (t == 2) {
        // half 1 of this super-block (copies of the last k-step before; the NW weight copies of k-step 0 are younger) is there
        // and half 0 has been read, for every wavefront
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(NW) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      if (t == 6) {
        // half 0 of the next super-block and this wavefront's next weights are there, half 1 has been read
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // the raw bytes are in registers before the next copies overwrite the region
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last (unused) copies
  __syncthreads();
  float4* const h0 = reinterpret_cast<float4*>(gemm_q6w_x0);
  float4* const h1 = reinterpret_cast<float4*>(gemm_q6w_x1);
  if (kh == 0) gemm_wide_epilogue_half<0, 2>(acc, h0, h1, bias, out, out_dim, m, mt, nt, nh, j, kg, lane, bias_stride);
  else gemm_wide_epilogue_half<1, 2>(acc, h1, h0, bias, out, out_dim, m, mt, nt, nh, j, kg, lane, bias_stride);
}

extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void q6_k_gemm_wide_f16(
    const uint8_t* w, const uint4* xp, const float* bias, float* out, u32 in_dim, u32 out_dim, u32 m, u32 bias_stride) {
  u32 mt, nt;
  if (!gemm_tile_of(blockIdx.x, (m + GEMM_BM - 1) / GEMM_BM, (out_dim + GEMM_WIDE_BN - 1) / GEMM_WIDE_BN, &mt, &nt)) return;
  gemm_q6k_wide_core<T6>(w, xp, bias, out, in_dim, out_dim, m, bias_stride, mt, nt, 0, in_dim >> 8);
}

// A list of Q5_K matrices (list, xp, in_dim, m; tile_end in tiles of 256 rows; grid gemm_tiles_grid): the values of q5_k_gemm_many_f16, bit for bit.
// 30720 rows x 4096 at 256 | 512 | 1024 tokens: 77 | 151 | 298 us, 88 | 169 | 334 on the better of the four-wavefront tiles (gemm_list_rows).
extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void q5_k_gemm_many_wide_f16(const GemmManyArgs list, const uint4* xp,
                                                                                                                  u32 in_dim, u32 m) {
  u32 mt, nt, i = 0, first = 0;
  if (!gemm_tile_of(blockIdx.x, (m + GEMM_BM - 1) / GEMM_BM, list.tile_end[list.count - 1], &mt, &nt)) return;
  while (i + 1 < list.count && nt >= list.tile_end[i]) first = list.tile_end[i++];
  gemm_q6k_wide_core<T5>(list.w[i], xp, nullptr, list.out[i], in_dim, list.out_dim[i], m, 0, mt, nt - first, 0, in_dim >> 8);
}

// Two matrices with an input each (Q4_K or Q5_K, and Q4_K or Q6_K: o and down of a layer), each over all its super-blocks or split in planes out + split m out_dim:
//   q4_k|q5_k_and_q6_k|q4_k_gemm_wide_f16 (w_a, xp_a, out_a, in_dim_a, out_dim_a, splits_a, w_b, xp_b, out_b, in_dim_b, out_dim_b, splits_b, m)
//                      grid = splits x gemm_tiles_grid of both, b's first: the rows of down are the longer ones
// 512 tokens of 4096 -> 4096 beside Q6_K 12288 -> 4096, plane sums included: 90 us; 110 as launches of their own, of which o's fills half the chip and down's
// 128-row tiles reach 0.7 PFLOP/s. Splits by gemm_wide_two_plan (gemv_config.h). Q4_K in this loop instead of gemm_wide_core's because both have to share LDS.
#define GEMM_WIDE_TWO_ENTRY(PREFIX_A, WA, PREFIX_B, WB)                                                                                           \
  extern "C" __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void PREFIX_A##_and_##PREFIX_B##_gemm_wide_f16(         \
      const uint8_t* w_a, const uint4* xp_a, float* out_a, u32 in_dim_a, u32 out_dim_a, u32 splits_a, const uint8_t* w_b, const uint4* xp_b,      \
      float* out_b, u32 in_dim_b, u32 out_dim_b, u32 splits_b, u32 m) {                                                                           \
    const u32 mtiles = (m + GEMM_BM - 1) / GEMM_BM, nt_a = (out_dim_a + GEMM_WIDE_BN - 1) / GEMM_WIDE_BN;                                        \
    const u32 nt_b = (out_dim_b + GEMM_WIDE_BN - 1) / GEMM_WIDE_BN, wgs_a = gemm_tiles_grid(mtiles, nt_a), wgs_b = gemm_tiles_grid(mtiles, nt_b); \
    const u32 first_a = wgs_b * splits_b;                                                                                                         \
    u32 mt, nt;                                                                                                                                   \
    if (blockIdx.x < first_a) {                                                                                                                   \
      const u32 s = blockIdx.x / wgs_b, n = in_dim_b >> 8;                                                                                        \
      if (!gemm_tile_of(blockIdx.x % wgs_b, mtiles, nt_b, &mt, &nt)) return;                                                                      \
      gemm_q6k_wide_core<WB>(w_b, xp_b, nullptr, out_b + (size_t)s * m * out_dim_b, in_dim_b, out_dim_b, m, 0, mt, nt, s * n / splits_b,          \
                             (s + 1) * n / splits_b);                                                                                             \
    } else {                                                                                                                                      \
      const u32 id = blockIdx.x - first_a, s = id / wgs_a, n = in_dim_a >> 8;                                                                     \
      if (!gemm_tile_of(id % wgs_a, mtiles, nt_a, &mt, &nt)) return;                                                                              \
      gemm_q6k_wide_core<WA>(w_a, xp_a, nullptr, out_a + (size_t)s * m * out_dim_a, in_dim_a, out_dim_a, m, 0, mt, nt, s * n / splits_a,          \
                             (s + 1) * n / splits_a);                                                                                             \
    }                                                                                                                                             \
  }
GEMM_WIDE_TWO_ENTRY(q4_k, T4, q6_k, T6)
GEMM_WIDE_TWO_ENTRY(q4_k, T4, q4_k, T4)
GEMM_WIDE_TWO_ENTRY(q5_k, T5, q6_k, T6)
GEMM_WIDE_TWO_ENTRY(q5_k, T5, q4_k, T4)
