// Short prefills, and longer ones of small matrices, over raw Q4_K, Q5_K or Q6_K weights: out[m][n] = (add) + sum_k x[m][k] *
// deq(W[n][k]). The tile kernels (gemm_q4k.hpp, gemm_q6k.hpp) give a workgroup a compute unit and walk a row's super-blocks one
// after the other, so a matrix of few tiles is a chain of loads that most of the chip does not take part in. Here a workgroup
// is small (32 or 64 tokens x 32 or 64 rows), up to three share a compute unit, and its four wavefronts are k-slices that meet
// in LDS once, at the end: no barrier in the loop. Operands and precision are the tile kernels': x packed as fp16 by
// pack_x_f16_* (or by a producer), weights dequantized to fp16, v_mfma_f32_32x32x16_f16, fp32 sums.
//
// Kernels (list: GemmManyArgs by value, tile_end in units of 32 RT rows; block 256, grid gemm_stream_grid):
//   <type>_gemm_stream_f16_<T>x<RT>   (list, xp, add | null, add_stride, in_dim, m), grid.y = k splits: planes behind list.out[0], no add
//   q4_k_gemm_stream_swiglu_pack_q4k|q6k_f16_<T>x2   (list of the gate matrix (out may be null), w_up, xp, xq, in_dim, m): a gate
//                                     tile and the up tile of the same 32 rows per wavefront; silu(gate) * up to out and as the packed input
//                                     of the next GEMM to xq (the absent tokens of a 32-token tile as zeros)
//   q4_k|q5_k_gemm_stream_pack_f16_<T>x<RT> (list, next, xp, in_dim, m): without splits, and next.xq[i] gets out[i] as the packed input of a
//                                     following GEMM, rounded from the sums as they are stored. (q | k | v | gate | up of a layer at 48 tokens, packed for o and down: their pack launch
//                                     of 4 us is gone and the list takes no longer, the layer's projections 62.2 -> 59.2 us.)
//   <type_a>_and_<type_b>_gemm_stream_f16_<T>x1 (list_a, xp_a, in_dim_a, splits_a, list_b, xp_b, in_dim_b, splits_b, m): two matrices
//                                     with an input each (o and down of a layer) in one launch, grid = splits x gemm_stream_grid of both
//
// What bounds it: a compute unit returns loads in order, so the activations, L2 hits, wait behind weights that come from
// memory, and it keeps about 64 KB in flight: some 47 KB/us whatever the mix (Q4_K 30720 rows x 4096, 64 tokens: 250 MB of
// activations and 71 MB of weights in 27 us behind a start of 4). Hence two row tiles per wavefront where the rows suffice, loads
// for the lanes of present tokens only, and scalar-based buffer loads issued at least half a super-block ahead.
// Measured, tile kernels -> these (us, plane sums included): Q4_K 4096 -> 12288, 32 / 64 tokens 19.0 / 21.6 -> 14.0 / 16.9; 4096 ->
// 4096, 48 tokens 13.9 -> 8.9; 1024 -> 3072, 64 / 512 tokens 9.4 / 18.2 -> 5.1 / 10.1; Q6_K 12288 -> 4096, 32 tokens 22.8 -> 18.9.
#pragma once
#include "common.hpp"
#include "gemm_q4k.hpp"
#include "gemv_config.h"

#define GEMM_STREAM_WAVES 4

struct StreamQ4K {
  static constexpr u32 BS = 144, PPR = 9, STRIDE = 9, OP_VALU = 14;   // bytes of a super-block, its 16-byte pieces, pieces a row takes in LDS
  static __device__ __forceinline__ u32 piece(u32 part) { return 16u * part; }
  uint4 q[2];
  u32 S[4];
  // header, scales and codes of group 2 KH + kg of the lane's row
  template <int KH>
  __device__ __forceinline__ void take(const uint4* row, u32 kg) {
    scales<KH>(row[0], kg);
    q[0] = row[1 + 4 * KH + 2 * kg];
    q[1] = row[2 + 4 * KH + 2 * kg];
  }
  template <int KH>
  __device__ __forceinline__ void scales(const uint4& hdr, u32 kg) {
    const float d = h2f(hdr.x), dm = h2f(hdr.x >> 16);
    u32 scp, mp;
    k4_pair(hdr.y, hdr.z, hdr.w, 16u * kg, KH != 0, scp, mp);
    S[0] = h2_dup(d * ubyte_f<0>(scp));
    S[1] = h2_dup(-(dm * ubyte_f<0>(mp)));
    S[2] = h2_dup(d * ubyte_f<1>(scp));
    S[3] = h2_dup(-(dm * ubyte_f<1>(mp)));
  }
  // the eight weights of k-step 8 KH + T, T = 4 h + op (gemm_k_element)
  template <int KH, int T>
  __device__ __forceinline__ half8_t op(u32, u32 magic_lo, u32 magic_hi) const {
    constexpr int h = T >> 2, o = T & 3, hi = o >> 1;
    const u32 qa = (o & 1) ? q[h].z : q[h].x, qb = (o & 1) ? q[h].w : q[h].y;
    constexpr u32 mask = hi ? 0x00F000F0u : 0x000F000Fu, off = hi ? 0xD400D400u : 0xE400E400u;   // half2(-64) : half2(-1024)
    const u32 magic = hi ? magic_hi : magic_lo;
    const uint4 r = make_uint4(h2_fma_off((qa & mask) | magic, off, S[2 * hi], S[2 * hi + 1]),
                               h2_fma_off(((qa >> 8) & mask) | magic, off, S[2 * hi], S[2 * hi + 1]),
                               h2_fma_off((qb & mask) | magic, off, S[2 * hi], S[2 * hi + 1]),
                               h2_fma_off(((qb >> 8) & mask) | magic, off, S[2 * hi], S[2 * hi + 1]));
    return __builtin_bit_cast(half8_t, r);
  }
};
struct StreamQ5K : StreamQ4K {
  static constexpr u32 BS = 176, PPR = 11, STRIDE = 11, OP_VALU = 24;
  uint4 qh[2];
  template <int KH>
  __device__ __forceinline__ void take(const uint4* row, u32 kg) {
    scales<KH>(row[0], kg);
    qh[0] = row[1];
    qh[1] = row[2];
    q[0] = row[3 + 4 * KH + 2 * kg];
    q[1] = row[4 + 4 * KH + 2 * kg];
  }
  // (the fifth bit beside the nibble, as in gemm_k45_core)
  template <int KH, int T>
  __device__ __forceinline__ half8_t op(u32 kg, u32 magic_lo, u32 magic_hi) const {
    constexpr int h = T >> 2, o = T & 3, hi = o >> 1, up = hi ? 8 : 4;
    const u32 sh = 2 * (2 * KH + kg) + hi;
    const u32 qa = (o & 1) ? q[h].z : q[h].x, qb = (o & 1) ? q[h].w : q[h].y;
    const u32 ha = ((o & 1) ? qh[h].z : qh[h].x) >> sh, hb = ((o & 1) ? qh[h].w : qh[h].y) >> sh;
    constexpr u32 mask = hi ? 0x00F000F0u : 0x000F000Fu, off = hi ? 0xD400D400u : 0xE400E400u;
    const u32 magic = hi ? magic_hi : magic_lo;
    const uint4 r = make_uint4(h2_fma_off((qa & mask) | magic | ((ha & 0x00010001u) << up), off, S[2 * hi], S[2 * hi + 1]),
                               h2_fma_off(((qa >> 8) & mask) | magic | (((ha >> 8) & 0x00010001u) << up), off, S[2 * hi], S[2 * hi + 1]),
                               h2_fma_off((qb & mask) | magic | ((hb & 0x00010001u) << up), off, S[2 * hi], S[2 * hi + 1]),
                               h2_fma_off(((qb >> 8) & mask) | magic | (((hb >> 8) & 0x00010001u) << up), off, S[2 * hi], S[2 * hi + 1]));
    return __builtin_bit_cast(half8_t, r);
  }
};
struct StreamQ6K {   // pieces 0..12 from the block's start, the last sixteen bytes (d is their end) as piece 13
  static constexpr u32 BS = 210, PPR = 14, STRIDE = 15, OP_VALU = 22;
  static __device__ __forceinline__ u32 piece(u32 part) { return part < 13u ? 16u * part : 194u; }
  uint4 qa, qb, qh;
  u32 S[4];
  template <int KH>
  __device__ __forceinline__ void take(const uint4* row, u32 u) {
    qa = row[4 * KH + u];
    qb = row[4 * KH + 2 + u];
    qh = row[8 + 2 * KH + u];
    const uint2 sc = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(row + 12) + 8 * KH);
    const float d = h2f(*reinterpret_cast<const uint16_t*>(reinterpret_cast<const uint8_t*>(row + 13) + 14));
    const u32 lo = sc.x >> (8 * u), hi = sc.y >> (8 * u);
    S[0] = h2_dup(d * (float)(int)(signed char)(lo & 0xFFu));
    S[1] = h2_dup(d * (float)(int)(signed char)((lo >> 16) & 0xFFu));
    S[2] = h2_dup(d * (float)(int)(signed char)(hi & 0xFFu));
    S[3] = h2_dup(d * (float)(int)(signed char)((hi >> 16) & 0xFFu));
  }
  static __device__ __forceinline__ u32 mul(u32 t, u32 off, u32 s) {
    const __half2 q = __hadd2(__builtin_bit_cast(__half2, t), __builtin_bit_cast(__half2, off));
    const __half2 w = __hmul2(q, __builtin_bit_cast(__half2, s));
    return __builtin_bit_cast(u32, w);
  }
  // step T = 2 quadrant + upper eight: (code | 1024) - 1056 or, high nibbles left in place, (code / 16 + 64) - 96, times d sc
  template <int KH, int T>
  __device__ __forceinline__ half8_t op(u32, u32 magic_lo, u32 magic_hi) const {
    constexpr int qd = T >> 1, h8 = T & 1, hi = qd >> 1;
    const uint4 Q = (qd & 1) ? qb : qa;
    const u32 a = h8 ? Q.z : Q.x, b = h8 ? Q.w : Q.y, ha = h8 ? qh.z : qh.x, hb = h8 ? qh.w : qh.y;
    constexpr u32 mask = hi ? 0x00F000F0u : 0x000F000Fu, m3 = hi ? 0x03000300u : 0x00300030u, off = hi ? 0xD600D600u : 0xE420E420u;
    const u32 magic = hi ? magic_hi : magic_lo;
    // bits 2 qd, 2 qd + 1 of each qh byte to bits 4..5 (low nibbles) or 8..9 of the half
    constexpr int sl = (qd & 1) ? 2 : 4, sr = (qd & 1) ? 6 : 4;
    const uint4 r = make_uint4(mul(((a & mask) | magic) | ((ha << sl) & m3), off, S[qd]), mul((((a >> 8) & mask) | magic) | ((ha >> sr) & m3), off, S[qd]),
                               mul(((b & mask) | magic) | ((hb << sl) & m3), off, S[qd]), mul((((b >> 8) & mask) | magic) | ((hb >> sr) & m3), off, S[qd]));
    return __builtin_bit_cast(half8_t, r);
  }
};

// uint4 of LDS: the wavefronts' weights, then the k-slices' sums in their place
template <class W, int T, int RT>
constexpr u32 gemm_stream_lds() {
  constexpr u32 weights = GEMM_STREAM_WAVES * 32 * RT * W::STRIDE, sums = GEMM_STREAM_WAVES * RT * T * 256;
  return weights > sums ? weights : sums;
}
// T: token tiles of 32; RT: row tiles of 32. PACK (with SWIGLU; 12 or 14): as in gemm_epilogue_swiglu_half. bid, split, nsplits: the
// workgroup's number, its k split and their count, where they are not the launch's.
template <class W, int T, int RT, bool SWIGLU = false, int PACK = 0>
__device__ __forceinline__ void gemm_stream_core(uint4* lds, const GemmManyArgs& list, const uint4* xp, const float* add, u32 add_stride, u32 in_dim,
                                                 u32 m, const uint8_t* w_up = nullptr, uint2* xq = nullptr, u32 bid = blockIdx.x,
                                                 u32 split = blockIdx.y, u32 nsplits = gridDim.y, const GemmNextArgs* next = nullptr) {
  static_assert(!SWIGLU || RT == 2, "a gate tile and the up tile of the same rows");
  constexpr int NM = SWIGLU ? 2 : 1;                             // matrices the workgroup's row tiles come from
  constexpr u32 PIECES = 32 * RT / NM * W::PPR;                  // 16-byte pieces of a matrix's rows per super-block
  constexpr int NL = (int)((PIECES + 63) / 64);                  // loads of them per lane
  constexpr u32 ROWS = SWIGLU ? 32 : 32 * RT;                    // rows of a matrix a workgroup covers
  constexpr u32 WAVE_U4 = 32 * RT * W::STRIDE;                   // a wavefront's weights in LDS
  const u32 lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const u32 j = lane & 31, kg = lane >> 5;
  u32 mt, nt;
  gemm_terms_tile(bid, (m + 32 * T - 1) / (32 * T), &mt, &nt);
  if (nt >= list.tile_end[list.count - 1]) return;   // (the grid is rounded up to whole rows of tiles per XCD)
  u32 mi = 0, first = 0;
  while (mi + 1 < list.count && nt >= list.tile_end[mi]) first = list.tile_end[mi++];
  nt -= first;
  const uint8_t* const w = list.w[mi];
  const u32 out_dim = list.out_dim[mi];
  float* const out = list.out[mi] + (size_t)split * m * out_dim;   // one plane per k split
  const u32 nkb_all = in_dim >> 8;
  const u32 kb0 = split * nkb_all / nsplits, kb1 = (split + 1) * nkb_all / nsplits;
  const u32 n0 = nt * ROWS;
  const size_t row_bytes = (size_t)nkb_all * W::BS;
  u32 magic_lo = 0x64006400u, magic_hi = 0x54005400u;   // in registers: (q & mask) | magic is one instruction
  asm volatile("" : "+v"(magic_lo), "+v"(magic_hi));

  // Loads through buffer descriptors: scalar base, scalar offset of the super-block, a 32-bit offset per lane. Piece
  // p = 64 i + lane is 16 bytes of row p / PPR: neighbouring lanes, neighbouring bytes.
  const u32 base_row = min(n0, out_dim - 1);
  __amdgpu_buffer_rsrc_t wrsrc[NM];
  wrsrc[0] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(w + (size_t)base_row * row_bytes), 0, 0xFFFFFFFFu, 0x00027000);
  if constexpr (SWIGLU) wrsrc[1] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(w_up + (size_t)base_row * row_bytes), 0, 0xFFFFFFFFu, 0x00027000);
  u32 off[NL];
  auto piece_of = [&](int i) { return 64u * i + 64u <= PIECES ? 64u * i + lane : min(64u * i + lane, PIECES - 1u); };
  auto lds_of = [&](int i) {   // where it goes
    const u32 p = piece_of(i);
    return W::STRIDE == W::PPR ? p : p + p / W::PPR * (W::STRIDE - W::PPR);
  };
#pragma unroll
  for (int i = 0; i < NL; i++) {
    const u32 p = piece_of(i), r = p / W::PPR, part = p - W::PPR * r;
    off[i] = (min(n0 + r, out_dim - 1) - base_row) * (u32)row_bytes + W::piece(part);
  }
  uint4* const mine = lds + wave * WAVE_U4;
  // The lane's activation operand of k-step ks, token tile tt: cell 2 ks + kg of the packed super-block. The lanes of absent
  // tokens have an offset behind the descriptor's range: they read zeros and fetch nothing.
  const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(xp), 0, GEMM_STREAM_MAX_PACKED, 0x00027000);
  u32 xt[T], xlane[T];
#pragma unroll
  for (int tt = 0; tt < T; tt++) {
    const u32 i = mt * T + tt;
    xt[tt] = i < 4 * ((m + 127) / 128) ? ((i >> 2) * nkb_all * 4096 + (i & 3) * 32) * 16 : 0u;   // (the packed block has whole tiles of 128 tokens)
    xlane[tt] = 32 * i + j < m ? (kg * 128 + j) * 16 : 0xFFFFFFF0u;
  }
  float16_t acc[RT][T];
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int tt = 0; tt < T; tt++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[r][tt][v] = 0.f;

  typedef u32 u32x4 __attribute__((ext_vector_type(4)));
  u32x4 raw[NM][NL], X[8][T];
  auto load_raw = [&](u32 kb) {
#pragma unroll
    for (int n = 0; n < NM; n++)
#pragma unroll
      for (int i = 0; i < NL; i++) raw[n][i] = __builtin_amdgcn_raw_buffer_load_b128(wrsrc[n], off[i], kb * W::BS, 0);
  };
  auto load_x = [&](u32 kb, int ks) {
#pragma unroll
    for (int tt = 0; tt < T; tt++) X[ks & 7][tt] = __builtin_amdgcn_raw_buffer_load_b128(xrsrc, xlane[tt], xt[tt] + (kb * 16 + ks) * 4096, 0);
  };
  // One super-block: its raw weights go to LDS, the activation operands of its first eight k-steps are in registers. NEXT:
  // the loads of super-block kn are issued on the way. Every load is issued eight k-steps or more ahead of its use;
  // they retire in order, so the scheduling barriers keep the order of issue, in front of the loop too (the compiler's counts
  // hold for both ways into it). The weight operands of a step are built while the matrix instructions of the one before run.
  half8_t A[2][RT];
  W wt[RT];
  auto super_block = [&](u32 kc, u32 kn, auto nextc) {
    constexpr bool NEXT = decltype(nextc)::value;
#pragma unroll
    for (int n = 0; n < NM; n++)
#pragma unroll
      for (int i = 0; i < NL; i++) *reinterpret_cast<u32x4*>(&mine[n * (16 * RT) * W::STRIDE + lds_of(i)]) = raw[n][i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the lanes read what other lanes of the wavefront wrote
#pragma unroll
    for (int r = 0; r < RT; r++) wt[r].template take<0>(mine + (32 * r + j) * W::STRIDE, kg);
#pragma unroll
    for (int r = 0; r < RT; r++) A[0][r] = wt[r].template op<0, 0>(kg, magic_lo, magic_hi);
    __builtin_amdgcn_sched_barrier(0);
    auto step = [&](auto khc, auto tc) {
      constexpr int KH = decltype(khc)::value, t = decltype(tc)::value, p = t & 1;
#pragma unroll
      for (int r = 0; r < RT; r++) {
        if constexpr (t < 7) {
          A[p ^ 1][r] = wt[r].template op<KH, (t + 1) & 7>(kg, magic_lo, magic_hi);
        } else if constexpr (KH == 0) {
          wt[r].template take<1>(mine + (32 * r + j) * W::STRIDE, kg);
          A[p ^ 1][r] = wt[r].template op<1, 0>(kg, magic_lo, magic_hi);
        }
      }
#pragma unroll
      for (int r = 0; r < RT; r++)
#pragma unroll
        for (int tt = 0; tt < T; tt++)
          acc[r][tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[p][r], __builtin_bit_cast(half8_t, X[t][tt]), acc[r][tt], 0, 0, 0);
      if constexpr (KH == 0) load_x(kc, 8 + t);
      else if constexpr (NEXT) load_x(kn, t);
      if constexpr (KH == 0 && t == 7 && NEXT) load_raw(kn);
      if constexpr (KH == 0 || t < 7) {
#pragma unroll
        for (int r = 0; r < RT; r++) asm volatile("" : "+v"(A[p ^ 1][r]));   // built here, not next to its use behind the barrier
      }
      if constexpr (t < 7) {
#pragma unroll
        for (int i = 0; i < RT * T; i++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                      // one matrix instruction,
          __builtin_amdgcn_sched_group_barrier(0x002, (W::OP_VALU + T - 1) / T, 0);   // its share of the next operands
        }
      } else {
        __builtin_amdgcn_sched_group_barrier(0x008, RT * T, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x020, T + (t == 7 ? NM * NL : 0), 0);   // the loads into registers that are free now
      __builtin_amdgcn_sched_barrier(0);
    };
    auto half = [&](auto khc) {
      step(khc, std::integral_constant<int, 0>{});
      step(khc, std::integral_constant<int, 1>{});
      step(khc, std::integral_constant<int, 2>{});
      step(khc, std::integral_constant<int, 3>{});
      step(khc, std::integral_constant<int, 4>{});
      step(khc, std::integral_constant<int, 5>{});
      step(khc, std::integral_constant<int, 6>{});
      step(khc, std::integral_constant<int, 7>{});
    };
    half(std::integral_constant<int, 0>{});
    half(std::integral_constant<int, 1>{});
  };
  u32 kb = kb0 + wave;
  if (kb < kb1) {
    load_raw(kb);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 8; t++) {
      load_x(kb, t);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (; kb + GEMM_STREAM_WAVES < kb1; kb += GEMM_STREAM_WAVES) super_block(kb, kb + GEMM_STREAM_WAVES, std::true_type{});
    super_block(kb, 0, std::false_type{});
  }
  __syncthreads();   // the weights in LDS are done with: the k-slices' sums take their place
  // quad g of tile (r, tt): weight rows 8 g + 4 kg .. + 3 for token j
  float4* const part = reinterpret_cast<float4*>(lds);
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int tt = 0; tt < T; tt++)
#pragma unroll
      for (int g = 0; g < 4; g++)
        part[((wave * (RT * T) + r * T + tt) * 4 + g) * 64 + lane] =
            make_float4(acc[r][tt][4 * g], acc[r][tt][4 * g + 1], acc[r][tt][4 * g + 2], acc[r][tt][4 * g + 3]);
  __syncthreads();
  auto sum = [&](u32 i) {   // wavefront g takes quad g
    float4 s = part[(i * 4 + wave) * 64 + lane];
#pragma unroll
    for (u32 k = 1; k < GEMM_STREAM_WAVES; k++) {
      const float4 p = part[((k * (RT * T) + i) * 4 + wave) * 64 + lane];
      s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
    }
    return s;
  };
  auto store = [&](float* dst4, u32 n, float4 s, const float* a) {
    if ((out_dim & 3u) == 0) {   // n is a multiple of four: all four rows exist
      if (a) s.x += a[0], s.y += a[1], s.z += a[2], s.w += a[3];
      *reinterpret_cast<float4*>(dst4) = s;
    } else {
      const float sv[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
      for (u32 v = 0; v < 4; v++)
        if (n + v < out_dim) dst4[v] = a ? sv[v] + a[v] : sv[v];
    }
  };
  const u32 n4 = n0 + 8 * wave + 4 * kg;
  if constexpr (!SWIGLU) {
    uint2* const image = PACK ? next->xq[mi] : nullptr;   // (out_dim is whole super-blocks then)
#pragma unroll
    for (u32 i = 0; i < RT * T; i++) {
      const float4 s = sum(i);
      const u32 n = n4 + 32 * (i / T), token = 32 * (mt * T + i % T) + j;
      if (PACK && image && n < out_dim && token < 128 * ((m + 127) / 128))
        image[(((size_t)(token >> 7) * (out_dim >> 8) + (n >> 8)) * 4096 + gemm_next_cell(next->q6 >> mi & 1u, n & 248u) * 128 + (token & 127)) * 2 + kg] =
            gemm_next_half(s, token < m);
      if (n < out_dim && token < m)
        store(out + (size_t)token * out_dim + n, n, s, add ? add + (size_t)token * add_stride + n : nullptr);
    }
  } else {
#pragma unroll
    for (u32 i = 0; i < T; i++) {
      const float4 g = sum(i), u = sum(T + i);
      const u32 n = n4, token = 32 * (mt * T + i) + j;
      float4 o = make_float4(swiglu_one(g.x, u.x), swiglu_one(g.y, u.y), swiglu_one(g.z, u.z), swiglu_one(g.w, u.w));
      if (n >= out_dim) continue;
      if (list.out[0] && token < m) store(out + (size_t)token * out_dim + n, n, o, nullptr);
      if constexpr (PACK != 0) {
        if (token < 128 * ((m + 127) / 128)) {
          // rows n .. n + 3 are k values of the next matrix: half kg of the cell that eight of them fill (pack_x_core)
          const u32 kbn = n >> 8, k = n & 255u & ~7u;
          u32 ks, kgr;
          if (PACK == 14) {
            ks = 8 * (k >> 7) + 2 * ((k >> 5) & 3) + ((k >> 3) & 1);
            kgr = (k >> 4) & 1;
          } else {
            const u32 g6 = k >> 6;
            ks = 8 * (g6 >> 1) + 4 * ((k >> 4) & 1) + 2 * ((k >> 5) & 1) + ((k >> 3) & 1);
            kgr = g6 & 1;
          }
          if (token >= m) o = make_float4(0.f, 0.f, 0.f, 0.f);   // the absent tokens of the last tile are zeros
          const __half2 p0 = __floats2half2_rn(o.x, o.z), p1 = __floats2half2_rn(o.y, o.w);
          xq[(((size_t)(token >> 7) * (out_dim >> 8) + kbn) * 4096 + (ks * 2 + kgr) * 128 + (token & 127)) * 2 + kg] =
              make_uint2(__builtin_bit_cast(u32, p0), __builtin_bit_cast(u32, p1));
        }
      }
    }
  }
}

#define GEMM_STREAM_ENTRY(PREFIX, W, T, RT, OCC)                                                                                     \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void PREFIX##_gemm_stream_f16_##T##x##RT( \
      const GemmManyArgs list, const uint4* xp, const float* add, u32 add_stride, u32 in_dim, u32 m) {                                \
    __shared__ uint4 lds[gemm_stream_lds<W, T, RT>()];                                                                                \
    gemm_stream_core<W, T, RT>(lds, list, xp, add, add_stride, in_dim, m);                                                            \
  }
// a list that writes packed inputs too: PACK 1, next->xq[i] of out[i]
#define GEMM_STREAM_PACK_ENTRY(PREFIX, W, T, RT, OCC)                                                                                     \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void PREFIX##_gemm_stream_pack_f16_##T##x##RT( \
      const GemmManyArgs list, const GemmNextArgs next, const uint4* xp, u32 in_dim, u32 m) {                                             \
    __shared__ uint4 lds[gemm_stream_lds<W, T, RT>()];                                                                                     \
    gemm_stream_core<W, T, RT, false, 1>(lds, list, xp, nullptr, 0, in_dim, m, nullptr, nullptr, blockIdx.x, 0, 1, &next);                 \
  }
#define GEMM_STREAM_PACK_TYPE(PREFIX, W)    \
  GEMM_STREAM_PACK_ENTRY(PREFIX, W, 1, 1, 3) \
  GEMM_STREAM_PACK_ENTRY(PREFIX, W, 1, 2, 2) \
  GEMM_STREAM_PACK_ENTRY(PREFIX, W, 2, 1, 2) \
  GEMM_STREAM_PACK_ENTRY(PREFIX, W, 2, 2, 2)
GEMM_STREAM_PACK_TYPE(q4_k, StreamQ4K)
GEMM_STREAM_PACK_TYPE(q5_k, StreamQ5K)
#define GEMM_STREAM_TYPE(PREFIX, W)    \
  GEMM_STREAM_ENTRY(PREFIX, W, 1, 1, 3) \
  GEMM_STREAM_ENTRY(PREFIX, W, 1, 2, 2) \
  GEMM_STREAM_ENTRY(PREFIX, W, 2, 1, 2)
GEMM_STREAM_TYPE(q4_k, StreamQ4K)
GEMM_STREAM_TYPE(q5_k, StreamQ5K)
GEMM_STREAM_TYPE(q6_k, StreamQ6K)
GEMM_STREAM_ENTRY(q4_k, StreamQ4K, 2, 2, 2)
GEMM_STREAM_ENTRY(q5_k, StreamQ5K, 2, 2, 2)
#define GEMM_STREAM_SWIGLU_ENTRY(T, OCC, NEXT, PACK)                                                                                  \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void q4_k_gemm_stream_swiglu_pack_##NEXT##_f16_##T##x2( \
      const GemmManyArgs list, const uint8_t* w_up, const uint4* xp, uint2* xq, u32 in_dim, u32 m) {                                  \
    __shared__ uint4 lds[gemm_stream_lds<StreamQ4K, T, 2>()];                                                                         \
    gemm_stream_core<StreamQ4K, T, 2, true, PACK>(lds, list, xp, nullptr, 0, in_dim, m, w_up, xq);                                    \
  }
GEMM_STREAM_SWIGLU_ENTRY(1, 2, q4k, 12)
GEMM_STREAM_SWIGLU_ENTRY(2, 2, q4k, 12)
GEMM_STREAM_SWIGLU_ENTRY(1, 2, q6k, 14)
GEMM_STREAM_SWIGLU_ENTRY(2, 2, q6k, 14)

// Two matrices with an input each. b's workgroups come first: it is the one with the longer rows in a layer (down beside o), so its
// chains start at once and a's, which are shorter, fill the units in between.
// (Q4_K 4096 -> 4096 and Q6_K 12288 -> 4096 at 48 tokens are 128 and 256 workgroups of a chip that holds 512: 12 and 27 us behind a
// profiler one after the other; the projections of a layer in 63.5 us, 70.1 with two launches.)
#define GEMM_STREAM_TWO_ENTRY(PREFIX_A, WA, PREFIX_B, WB, T, OCC)                                                                      \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void PREFIX_A##_and_##PREFIX_B##_gemm_stream_f16_##T##x1( \
      const GemmManyArgs list_a, const uint4* xp_a, u32 in_dim_a, u32 splits_a, const GemmManyArgs list_b, const uint4* xp_b, u32 in_dim_b, \
      u32 splits_b, u32 m) {                                                                                                          \
    constexpr u32 LDS_A = gemm_stream_lds<WA, T, 1>(), LDS_B = gemm_stream_lds<WB, T, 1>();                                           \
    __shared__ uint4 lds[LDS_A > LDS_B ? LDS_A : LDS_B];                                                                              \
    const u32 wgs_a = gemm_stream_grid(m, T, list_a.tile_end[0]), wgs_b = gemm_stream_grid(m, T, list_b.tile_end[0]);                 \
    const u32 first_a = wgs_b * splits_b;                                                                                             \
    if (blockIdx.x < first_a) {                                                                                                       \
      gemm_stream_core<WB, T, 1>(lds, list_b, xp_b, nullptr, 0, in_dim_b, m, nullptr, nullptr, blockIdx.x % wgs_b, blockIdx.x / wgs_b, splits_b); \
    } else {                                                                                                                          \
      const u32 id = blockIdx.x - first_a;                                                                                            \
      gemm_stream_core<WA, T, 1>(lds, list_a, xp_a, nullptr, 0, in_dim_a, m, nullptr, nullptr, id % wgs_a, id / wgs_a, splits_a);     \
    }                                                                                                                                 \
  }
#define GEMM_STREAM_TWO(PREFIX_A, WA, PREFIX_B, WB)    \
  GEMM_STREAM_TWO_ENTRY(PREFIX_A, WA, PREFIX_B, WB, 1, 3) \
  GEMM_STREAM_TWO_ENTRY(PREFIX_A, WA, PREFIX_B, WB, 2, 2)
GEMM_STREAM_TWO(q4_k, StreamQ4K, q6_k, StreamQ6K)
GEMM_STREAM_TWO(q4_k, StreamQ4K, q4_k, StreamQ4K)
GEMM_STREAM_TWO(q5_k, StreamQ5K, q6_k, StreamQ6K)
GEMM_STREAM_TWO(q5_k, StreamQ5K, q4_k, StreamQ4K)
