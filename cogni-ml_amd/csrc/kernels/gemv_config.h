// Launch geometry shared by the GEMV kernels and the host code that sizes their grids.
// A workgroup is 4 wavefronts; each wavefront owns GEMV_ROWS_*(tokens) consecutive output rows.
#pragma once

#ifndef GEMV_WAVES
#define GEMV_WAVES 4
#endif
#define GEMV_BLOCK (64 * GEMV_WAVES)

// rows per wavefront. One token of a Q4_K matrix: two rows and four workgroups per compute unit (1024 resident workgroups
// that walk the row groups) measured 7.55 us against 7.9-8.0 for four rows and three workgroups at 12288 x 4096, interleaved
// runs; 896, 960 or 1088 workgroups lose that again. The one-token matrix-pair kernels keep four rows (no gain there).
#ifndef GEMV_ROWS_Q4K
#define GEMV_ROWS_Q4K(M) ((M) == 1 ? 2 : ((M) == 2 ? 4 : 2))
#endif
#define GEMV_ROWS_Q4K_PAIR 4
#ifndef GEMV_ROWS_Q5K
#define GEMV_ROWS_Q5K(M) 2
#endif
#ifndef GEMV_ROWS_Q6K
#define GEMV_ROWS_Q6K(M) 2
#endif
#ifndef GEMV_ROWS_Q80
#define GEMV_ROWS_Q80(M) 4
#endif

// rows of the weight matrix one workgroup produces
static inline int gemv_rows_per_block(unsigned type, int tokens) {
  switch (type) {
    case 12: return GEMV_WAVES * GEMV_ROWS_Q4K(tokens);
    case 13: return GEMV_WAVES * GEMV_ROWS_Q5K(tokens);
    case 14: return GEMV_WAVES * GEMV_ROWS_Q6K(tokens);
    case 8: return GEMV_WAVES * GEMV_ROWS_Q80(tokens);
    default: return 0;
  }
}

// One token of a matrix of few rows: halve the rows per wavefront until at least 256 workgroups share the matrix
// (kernels NAME_r1, Q8_0 also NAME_r2). Returns rows per wavefront; the value for many rows is the kernel's own.
#define GEMV_SHORT_MIN_GROUPS 256u
static inline int gemv_rows_m1(unsigned type, unsigned out_dim) {
  int r = gemv_rows_per_block(type, 1) / GEMV_WAVES;
  while (r > 1 && (out_dim + (unsigned)(GEMV_WAVES * r) - 1) / (unsigned)(GEMV_WAVES * r) < GEMV_SHORT_MIN_GROUPS) r >>= 1;
  return r;
}

// ---- staged activations ------------------------------------------------------------------------
// A workgroup keeps the activations of up to GEMV_LDS_BYTES in LDS: `chunk` whole column sets for the
// token group it is working on. per_set_f4 = float4 count of one column set for that token group.
#define GEMV_LDS_BYTES 49152

#if defined(__HIPCC__)
#define GEMV_HD __host__ __device__
#else
#define GEMV_HD
#endif

static inline GEMV_HD int gemv_chunk_sets(int per_set_f4, unsigned ncs) {
  // 17/16: the per-lane activation sums kept beside the staged activations never exceed 1/16 of them
  int ch = GEMV_LDS_BYTES / 17 / per_set_f4;
  if (ch < 1) ch = 1;
  if ((unsigned)ch >= ncs) return (int)ncs;
  if (ch > 1) ch &= ~1;   // a chunk boundary never splits a pair of column sets taken together
  return ch;
}

// K-quant kernels whose tokens all fit the registers at once (one token group) keep the activations in LDS in natural
// order (16 KiB per token and column set) and form the per-lane sums from the registers they are read into: no sums
// in LDS. A row of one column set is staged as just that; longer rows in chunks of as many sets as fit the budget
// (3 for one token, 1 for two), whole chunks even where the row ends inside one.
static constexpr inline GEMV_HD int gemv_chunk_sets_direct(int per_set_f4, unsigned ncs) {
  int ch = GEMV_LDS_BYTES / 16 / per_set_f4;
  if (ch < 1) ch = 1;
  return ncs <= 1 ? 1 : ch;
}
static constexpr inline GEMV_HD bool gemv_direct_x(unsigned type, int token_groups) {
  return (type == 12 || type == 13 || type == 14) && token_groups == 1;
}

// One or two tokens of a K-quant matrix (one token group): the kernel walks row groups blockIdx.x, blockIdx.x +
// gridDim.x, ... with the activations staged once, so a long matrix is launched as the workgroups that are resident
// together (256 compute units x 3 per unit at 3 wavefronts per SIMD for one token, x 2 for two), each with the same
// number of groups up to one.
#define GEMV_RESIDENT_WGS 768u
#define GEMV_RESIDENT_WGS_2 512u
// (one token of Q4_K: every resident slot is launched, 4 per compute unit, and the workgroups' group counts differ by at
// most one)
#define GEMV_RESIDENT_WGS_Q4K 1024u
// (one token of a Q6_K matrix of many groups: 5 per compute unit. The 151936 x 4096 head, interleaved runs: 93.6 us on 760,
// 768 or 1024 workgroups, 90.2 on 1280, 91.1 on 1536, 90.8 on 2048; 92.4 - 97.2 on counts that are not multiples of the 256
// compute units. With only a few groups per workgroup the even split over 768 stays: 12288 rows 10.35 us against 11.1 on
// 1280, 24576 rows 17.4 against 18.65)
#define GEMV_RESIDENT_WGS_Q6K 1280u
#define GEMV_RESIDENT_Q6K_MIN_GROUPS (8u * GEMV_RESIDENT_WGS_Q6K)
static inline unsigned gemv_grid(unsigned type, int tokens, unsigned out_dim) {
  const unsigned rows = (unsigned)gemv_rows_per_block(type, tokens);
  const unsigned groups = (out_dim + rows - 1) / rows;
  if (type == 12 && tokens == 1) return groups < GEMV_RESIDENT_WGS_Q4K ? groups : GEMV_RESIDENT_WGS_Q4K;
  if (type == 14 && tokens == 1 && groups >= GEMV_RESIDENT_Q6K_MIN_GROUPS) return GEMV_RESIDENT_WGS_Q6K;
  const unsigned resident = tokens == 1 ? GEMV_RESIDENT_WGS : GEMV_RESIDENT_WGS_2;
  if (tokens > 2 || !gemv_direct_x(type, 1) || groups <= resident) return groups;
  const unsigned per_wg = (groups + resident - 1) / resident;
  return (groups + per_wg - 1) / per_wg;
}

// column-set geometry per type: blocks per set, float4 of x per lane and set, tokens per register group
// (nsum = scale groups per lane whose activation sums are kept in LDS)
static inline void gemv_set_geometry(unsigned type, int* bps, int* nf4, int* nsum, int* mg_max, int* block_elems) {
  switch (type) {
    case 12: case 13: *bps = 16; *nf4 = 16; *nsum = 2; *mg_max = 2; *block_elems = 256; break;
    case 14: *bps = 16; *nf4 = 16; *nsum = 4; *mg_max = 2; *block_elems = 256; break;
    default: *bps = 32; *nf4 = 4; *nsum = 1; *mg_max = 4; *block_elems = 32; break;
  }
}

// dynamic shared memory (bytes) the GEMV kernel for (type, tokens) needs at this in_dim
static inline unsigned gemv_lds_bytes(unsigned type, int tokens, unsigned in_dim) {
  int bps, nf4, nsum, mg_max, be;
  gemv_set_geometry(type, &bps, &nf4, &nsum, &mg_max, &be);
  const int mg = tokens < mg_max ? tokens : mg_max;
  const int ng = (tokens + mg - 1) / mg;
  const unsigned nb = (in_dim + (unsigned)be - 1) / (unsigned)be;
  const unsigned ncs = (nb + (unsigned)bps - 1) / (unsigned)bps;
  const int per_set_f4 = mg * nf4 * 64;
  if (gemv_direct_x(type, ng)) return (unsigned)(per_set_f4 * gemv_chunk_sets_direct(per_set_f4, ncs)) * 16u;
  const int ch = ng > 1 ? 1 : gemv_chunk_sets(per_set_f4, ncs);
  return (unsigned)(per_set_f4 * ch) * 16u + (unsigned)(mg * nsum * 64 * ch) * 4u;
}

// ---- matrix-core GEMV (gemv_mfma.hpp): 8 wavefronts per workgroup ------------------------------------
#define GEMV_MFMA_WAVES 8
#define GEMV_MFMA_TMAX 3            // 16-row tiles a wavefront carries at most
#define GEMV_MFMA_MAX_TOKENS 4
// (token, super-block) pairs of activations a workgroup stages (tokens * in_dim / 256) at most
#define GEMV_MFMA_MAX_UNITS(M) ((M) >= 3 ? 64 : 96)

// log2 of the k-slices a workgroup's wavefronts form: the largest power of two <= min(8, super-blocks)
static inline GEMV_HD unsigned gemv_mfma_log2_kslices(unsigned nsb) {
  unsigned lg = 0;
  while (lg < 3 && (2u << lg) <= nsb) lg++;
  return lg;
}
// Rows too long for all their activations to be staged at once are staged a chunk at a time, which needs every
// wavefront to be a k-slice of its own: in_dim a multiple of 2048.
static inline GEMV_HD int gemv_mfma_chunked(int tokens, unsigned in_dim) {
  return (unsigned)tokens * (in_dim >> 8) > (unsigned)GEMV_MFMA_MAX_UNITS(tokens) && (in_dim & 2047u) == 0;
}
// Shapes the matrix-core kernels take: Q4_K with 1..4 tokens, Q5_K and Q6_K with 3 or 4 (its columns are laid out for four
// tokens, and two are as fast on the vector ALU); in_dim a multiple of 256, all activations staged at once or in_dim a
// multiple of 2048.
static inline int gemv_mfma_supported(unsigned type, int tokens, unsigned in_dim) {
  if ((type != 12 && type != 13 && type != 14) || tokens < (type == 12 ? 1 : 3) || tokens > GEMV_MFMA_MAX_TOKENS || in_dim == 0 ||
      (in_dim & 255u))
    return 0;
  return (unsigned)tokens * (in_dim >> 8) <= (unsigned)GEMV_MFMA_MAX_UNITS(tokens) || (in_dim & 2047u) == 0;
}
// 16-row tiles per row group and the grid: aim at one workgroup per compute unit (256 of them)
static inline unsigned gemv_mfma_tiles(int tokens, unsigned in_dim, unsigned out_dim) {
  (void)tokens;
  const unsigned nwr = GEMV_MFMA_WAVES >> gemv_mfma_log2_kslices(in_dim >> 8);
  const unsigned ntiles = (out_dim + 15) / 16, tmax = (unsigned)GEMV_MFMA_TMAX;
  unsigned t = ntiles / (nwr * 256u);
  if (t < 1) t = 1;
  if (t > tmax) t = tmax;
  return t;
}
static inline unsigned gemv_mfma_grid(int tokens, unsigned in_dim, unsigned out_dim) {
  const unsigned nwr = GEMV_MFMA_WAVES >> gemv_mfma_log2_kslices(in_dim >> 8);
  const unsigned ntiles = (out_dim + 15) / 16, per_wg = nwr * gemv_mfma_tiles(tokens, in_dim, out_dim);
  const unsigned groups = (ntiles + per_wg - 1) / per_wg;
  // more row groups of the largest size than compute units: one workgroup per unit walks them with the activations
  // staged once (not where the activations are staged in chunks)
  if (groups > 256u && per_wg == nwr * (unsigned)GEMV_MFMA_TMAX && !gemv_mfma_chunked(tokens, in_dim)) return 256u;
  return groups;
}
static inline unsigned gemv_mfma_lds_bytes(unsigned type, int tokens, unsigned in_dim) {
  const int mp = type == 14 ? 4 : (tokens <= 1 ? 1 : (tokens <= 2 ? 2 : 4));
  const unsigned nsums = type == 14 ? 16u : 8u;   // sub-block sums of the activations kept per (token, super-block)
  // (token, super-block) units the activation image holds: all of them, or one chunk per wavefront
  const unsigned per_wave = (unsigned)(GEMV_MFMA_MAX_UNITS(tokens) / GEMV_MFMA_WAVES / tokens * tokens);
  const unsigned units = gemv_mfma_chunked(tokens, in_dim) ? GEMV_MFMA_WAVES * per_wave : (unsigned)tokens * (in_dim >> 8);
  return 64u + GEMV_MFMA_WAVES * GEMV_MFMA_TMAX * 1024u + GEMV_MFMA_WAVES * GEMV_MFMA_TMAX * (unsigned)mp * 64u +
         units * (4u + 4u * nsums + 1024u);
}

// ---- several tokens in one pass over a Q4_K, Q5_K or Q6_K matrix (gemv_mt.hpp): 8 wavefronts = 8 k-slices, activations packed once
#define GEMV_MT_WAVES 8
#define GEMV_MT_TMAX 3              // 16-row tiles a wavefront carries at most (Q4_K, Q5_K; Q6_K two)
#define GEMV_MT_MAX_TOKENS 8
#define GEMV_MT_MAX_IN_DIM 12288u
// Shapes the kernels take: Q4_K, Q5_K, Q6_K or Q8_0 (eight blocks at a time), 2..8 tokens, in_dim a multiple of 256 up to 12288 (1..6 super-blocks per
// k-slice; a row whose super-blocks do not divide by 8 is worked on as if zeros filled it up, gemv_mt_padded_sb).
static inline GEMV_HD int gemv_mt_supported(unsigned type, int tokens, unsigned in_dim) {
  return (type == 12 || type == 13 || type == 14 || type == 8) && tokens >= 2 && tokens <= GEMV_MT_MAX_TOKENS && in_dim != 0 &&
         (in_dim & 255u) == 0 && in_dim <= GEMV_MT_MAX_IN_DIM;
}
// super-blocks of the activation image: the row's, rounded up to a multiple of the 8 k-slices
static inline GEMV_HD unsigned gemv_mt_padded_sb(unsigned in_dim) { return ((in_dim >> 8) + 7u) & ~7u; }
// Token count from which one matrix goes through pack + one pass rather than the per-token-group kernels (0: never): where
// the pair measures faster. Q6_K from three tokens; Q4_K and Q5_K from four on rows of 4096 values and more, else from five.
// Tall matrices of up to 4096 columns (an output head): the workgroups walk many row groups and pay their start once, which
// puts the kernel ahead earlier - Q6_K from two tokens at GEMV_MT_TALL_ROWS rows, Q4_K and Q5_K from three there and from
// two at GEMV_MT_VERY_TALL_ROWS. Q8_0 (the other way is one launch on the vector ALU for up to eight tokens, whose time
// grows with every token: 3584 -> 1024 takes 9.0 / 13.6 / 21.3 us at 2 / 4 / 8 tokens against 7.3 in one pass): from two
// tokens on rows of 3584 values and more and on tall matrices, else from three; half-filled rows (1024 values) from five.
#define GEMV_MT_TALL_ROWS 40960u
#define GEMV_MT_VERY_TALL_ROWS 98304u
static inline unsigned gemv_mt_from(unsigned type, unsigned in_dim, unsigned out_dim) {
  if (!gemv_mt_supported(type, 2, in_dim)) return 0;
  // rows that fill less than three quarters of their eight k-slices (1024 values: half of them): from five tokens, where
  // the per-token-group kernels start to read the weights twice
  const int sparse = 4u * (in_dim >> 8) < 3u * gemv_mt_padded_sb(in_dim);
  if (type == 8) {
    if (out_dim >= GEMV_MT_TALL_ROWS) return 2u;
    return sparse ? 5u : (in_dim >= 3584u ? 2u : 3u);
  }
  if (sparse) return 5u;
  if (in_dim <= 4096u && out_dim >= GEMV_MT_TALL_ROWS) return (type == 14 || out_dim >= GEMV_MT_VERY_TALL_ROWS) ? 2u : 3u;
  return type == 14 ? 3u : (in_dim >= 4096u ? 4u : 5u);
}
// The resident output head (a norm that writes the image in front, top-1 inside, with or without the logits): tokens of a group that go
// through one pass. Beside the counts above, three and four tokens of at least GEMV_MT_HEAD_ROWS rows, whatever the row length: the other kernels walk the
// weights once for the logits and once for the top-1. Two tokens never: their other kernel has activations of 32 bits, the image 22 (2-norm of the
// logits' error against 64 bits, Q4_K 1.2e-7 | 1.0e-6, Q6_K 1.9e-7 | 3.8e-7), where that of three and four has 22 as well (Q4_K 0.79e-6 to 1.46e-6 | 0.79e-6 to 1.49e-6, Q6_K 3.67e-7 to
// 4.09e-7 | 3.79e-7 to 4.09e-7). Us a step, before | one pass. Q6_K, 151936 rows of 1024 | 1280 | 2304 | 2816 values, 3 tokens with logits 132 | 64, 191 | 65, 336 | 110, 381 | 117; 32000
// rows, 3 tokens, top-1 alone 25.5 | 21.7, 34.5 | 22.2, 47.1 | 31.5, 52.6 | 32.0. Q4_K, 151936 rows with logits 68 | 48, 105 | 49, 153 | 74, 168 | 74. Not Q4_K, top-1 alone, rows of 1024 values,
// whose k-slices the matrix-core kernel fills (151936 rows 38.3 | 41.9, 32000 16.6 | 18.0), and four tokens below GEMV_MT_TALL_ROWS (2304 values, 32000 | 36000 | 40000 | 50000 rows
// 24.6 | 25.5 | 30.4 | 35.4 and 25.0 | 27.7 | 29.0 | 34.7). The line is where vocabularies start, not where the ways cross: with logits the one pass is ahead from 4096 rows on (Q6_K 1024 values,
// 3 tokens, 4096 | 16384 rows 18.1 | 23.0 and 12.2 | 17.5), with the top-1 alone from 8192 to 32000 (at 24576 Q6_K 17.2 | 19.5, 2304 values 34.8 | 26.1).
#define GEMV_MT_HEAD_ROWS 32000u
static inline int gemv_mt_head_takes(unsigned type, unsigned tokens, unsigned in_dim, unsigned out_dim, int logits) {
  if ((type != 12 && type != 14) || in_dim > 4096u || tokens > (unsigned)GEMV_MT_MAX_TOKENS || !gemv_mt_supported(type, 2, in_dim)) return 0;
  if (tokens >= gemv_mt_from(type, in_dim, out_dim)) return 1;
  if (tokens < 3u || out_dim < GEMV_MT_HEAD_ROWS) return 0;
  return logits || type != 12 || (in_dim > 1024u && (tokens == 3u || out_dim >= GEMV_MT_TALL_ROWS));
}
// The same for a pair, a list of matrices or the fused gate | up | SwiGLU: from two tokens (one pack serves all of them and
// the weights are read once), from five on rows that fill less than three quarters of their k-slices.
static inline unsigned gemv_mt_multi_from(unsigned type, unsigned in_dim) {
  if (!gemv_mt_supported(type, 2, in_dim)) return 0;
  return 4u * (in_dim >> 8) < 3u * gemv_mt_padded_sb(in_dim) ? 5u : 2u;
}
// tiles per wavefront: rows of more than 4096 values one (the operands are streamed); else the count, up to three (Q4_K, Q5_K) or
// two (Q6_K, Q8_0: their units are larger), whose rounds of 256 workgroups take least. Up to 256 tiles one. Else, in hundredths of a us fitted
// to launches of 906 to 151936 rows, weights from memory, for one | two | three tiles (one round of two | three: 755 | 950, 392 | 468, 510):
// 460 + 170 | 580 + 308 | 680 + 480 a round, rows of up to 2048 values of Q4_K and Q5_K 292 + 113 | 291 + 190 | 309 + 254, up to 1024 of Q6_K and Q8_0
// 302 + 160 | 380 + 270: the shorter a row, the more a round's start and end weigh. As many tiles as keep 256 workgroups busy, the first rule, cost up to
// 33 % more (Q4_K 4096 -> 16384 15.0 us with three tiles, 11.4 with one; -> 10240 11.0 with two, 8.9 with three), the long rows' line for all up to 19 %
// more than that where rows are short (Q4_K 1024 -> 24576 8.0 with three, 9.5 with one; Q8_0 1024 -> 13386 8.1 | 8.9). This takes at most 3 % more than
// the first rule (Q4_K 1024 -> 24576 at sixteen tokens 8.5 | 8.7), all told 5 % less. Host and kernel use the same rule.
static inline GEMV_HD unsigned gemv_mt_tiles(unsigned type, unsigned in_dim, unsigned ntiles) {
  if (in_dim > 4096u || ntiles <= 256u) return 1;
  const int two = type == 14 || type == 8;
  const unsigned r1 = (ntiles + 255u) / 256u, r2 = ((ntiles + 1u) / 2u + 255u) / 256u, r3 = ((ntiles + 2u) / 3u + 255u) / 256u;
  unsigned c1 = 460u + 170u * r1, c2 = r2 <= 1u ? 755u : 580u + 308u * r2, c3 = r3 <= 1u ? 950u : 680u + 480u * r3;
  if (two && in_dim <= 1024u) c1 = 302u + 160u * r1, c2 = r2 <= 1u ? 510u : 380u + 270u * r2;
  if (!two && in_dim <= 2048u)
    c1 = 292u + 113u * r1, c2 = r2 <= 1u ? 392u : 291u + 190u * r2, c3 = r3 <= 1u ? 468u : 309u + 254u * r3;
  return !two && c3 < c1 && c3 < c2 ? (unsigned)GEMV_MT_TMAX : (c2 < c1 ? 2u : 1u);
}
// One workgroup per compute unit at most; they walk the row groups (a workgroup that has none leaves at once).
static inline GEMV_HD unsigned gemv_mt_grid(unsigned type, unsigned in_dim, unsigned total_rows) {
  const unsigned ntiles = (total_rows + 15) / 16;
  (void)type;
  (void)in_dim;
  return ntiles < 256u ? ntiles : 256u;
}
// the k-slices' partial sums, then per wavefront the slots of its units: 6 x (16 rows x 144 B) for Q4_K, 6 x (16 rows x
// 176 B) for Q5_K, 4 x (16 rows x 240 B) for Q6_K, 4 x (16 rows x 272 B) for Q8_0
// (the sixteen-token kernels keep twice the partial sums)
#define GEMV_MT_X16_LDS_EXTRA (GEMV_MT_WAVES * GEMV_MT_TMAX * 8u * 16u * 4u)
static inline unsigned gemv_mt_lds_bytes(unsigned type) {
  return GEMV_MT_WAVES * GEMV_MT_TMAX * 8u * 16u * 4u +
         GEMV_MT_WAVES * (type == 14 ? 4u * 3840u : (type == 8 ? 4u * 4352u : (type == 13 ? 6u * 2816u : 6u * 2304u)));
}
// bytes of the activation image: per super-block (of the padded count) 8 KiB of operands, then 16 bytes per (super-block, lane) for the scales and
// the sub-block sums (one more matrix-core operand). Q4_K and Q5_K share one image, Q6_K has its own.
static inline unsigned long long gemv_mt_image_bytes(unsigned type, unsigned in_dim) {
  (void)type;
  return (unsigned long long)gemv_mt_padded_sb(in_dim) * (8192u + 1024u);
}

// ---- prefill GEMM: what a tile costs. A workgroup has a compute unit to itself, so a launch runs in rounds of 256 tiles; a round
// of 192-row tiles is 100, of 128-row tiles 75, of the 256-row tiles of the eight-wavefront kernels 131 (Q4_K; a third more work with 25 %
// fewer activation bytes copied per flop and two wavefronts per SIMD) or 107 (Q6_K, whose 192-row tile copies no raw blocks). Measured,
// Q4_K lists of 4096 columns, us a round: 47 to 53 | 37 to 39 | 61 to 69; so 30720 rows take, in 192 | 128 | 256-row tiles, 151.7 | 151.9 |
// 134.7 at 512 tokens, 94.2 | 78.1 | 69.5 at 256, 105.9 | 113.1 | 121.4 at 384, 562 | 581 | 532 at 2048. Q6_K 12288 -> 4096: 314 | 237 | 211 at
// 2048 tokens, 151 | 120 | 155 at 1024.
#define GEMM_ROUND_TILES 256u
// A single Q4_K matrix (cogni_gemm_plan) takes the 256-row tiles where they fill whole rounds and those cost less, at 124, than
// the 192- and the 128-row ones'. 4096 columns, weights from memory, us in 192 | 128 | 256-row tiles: three rounds against four and five, 12288
// rows at 2048 tokens 205 | 218 | 202, 10240 at 2048 188 | 182 | 180, 20480 at 1024 189 | 187 | 181, 32000 at 640 193 | 190 | 185; four
// against five and seven, 14336 at 2048 246 | 256 | 247, 28672 at 1024 248 | 261 | 246; seven against nine and eleven, 27648 at 2048 460 | 497 | 452.
// (12288 columns, 28672 rows at 1024: 683 | 715 | 690.) Up to 64 tokens never: 151936 rows at 64 in the 64-token kernels 153, in 256-row tiles 184.
// Lists and gate | up go by the costs above alone.
#define GEMM_Q4K_WIDE_COST 124u
static inline int gemm_q4k_use_wide(unsigned out_dim, unsigned tokens) {
  const unsigned mtiles = (tokens + 127u) / 128u;
  const unsigned narrow = mtiles * ((out_dim + 191u) / 192u), wide = mtiles * ((out_dim + 255u) / 256u);
  const unsigned rn = (narrow + GEMM_ROUND_TILES - 1) / GEMM_ROUND_TILES, rw = (wide + GEMM_ROUND_TILES - 1) / GEMM_ROUND_TILES;
  return wide >= GEMM_ROUND_TILES && rw * GEMM_Q4K_WIDE_COST < rn * 100u;
}
static inline unsigned gemm_tile_cost(unsigned type, unsigned rows) { return rows == 192u ? 100u : (rows == 128u ? 75u : (type == 14u ? 107u : (type == 13u ? 117u : 131u))); }
// knob: COGNI_GEMM_WIDE, 0 | 1 where it is set (no 256-row tiles | those wherever there is a kernel for them), else -1.
// gate | up with SwiGLU: tiles of 96 rows of both matrices (four wavefronts) or of 128 (eight). 4096 -> 12288, us: 441 | 410 at 2048
// tokens, 225 | 208 at 1024, 114 | 123 at 512, 58 | 59 at 256; 2048 -> 4096 at 1024 61.6 | 41.3; 3072 -> 8192 at 300 76.7 | 45.5.
static inline int gemm_swiglu_use_wide(unsigned out_dim, unsigned tokens, int knob) {
  const unsigned long long mtiles = (tokens + 127u) / 128u;
  const unsigned long long rn = (mtiles * ((out_dim + 95u) / 96u) + GEMM_ROUND_TILES - 1) / GEMM_ROUND_TILES;
  const unsigned long long rw = (mtiles * ((out_dim + 127u) / 128u) + GEMM_ROUND_TILES - 1) / GEMM_ROUND_TILES;
  return knob >= 0 ? knob : tokens > 64u && rw * gemm_tile_cost(12u, 256u) < rn * gemm_tile_cost(12u, 192u);
}
// Super-blocks of a row that the loop of gemm_q6k_wide.hpp takes: its offset into the activations of a token tile, 64 KiB a super-block, has 32 bits, and its
// buffers end a byte short of 4 GiB. It runs Q6_K and Q5_K tiles of 256 rows and both matrices of gemm_wide_two_plan; longer rows go to the other
// tiles, which have 64-bit addresses.
#define GEMM_Q6W_MAX_KB 65535u
// A list of Q4_K or Q5_K matrices as one launch: rows of its tiles. The 256-row ones: more tokens than the 64-token kernels take. (Q5_K, 4096 columns, weights
// from memory, us, 192 | 128 | 256 rows: 30720 rows at 256 tokens 107.8 | 87.7 | 77.3, 384 120.9 | 128.3 | 135.8, 512 169 | 170 | 151, 1024 341 | 334 | 298; 65536 rows at 128
// 126.5 | 105.3 | 89.0, 81920 129.9 | 142.4 | 150; 19456 x 2048 at 300 61.4 | 49.7 | 44.2, at 512 66.4 | 73.2 | 77.5: the costs pick the fastest of each.)
static inline unsigned gemm_list_rows(unsigned type, unsigned in_dim, const unsigned* out_dims, unsigned count, unsigned tokens, int knob) {
  const unsigned of[3] = {192u, 128u, 256u};
  unsigned long long least = ~0ull;
  unsigned best = 192u, k, i;
  const int can = type == 12u || in_dim / 256u <= GEMM_Q6W_MAX_KB;
  if (knob == 1 && can) return 256u;
  for (k = 0; k < (tokens > 64u && knob != 0 && can ? 3u : 2u); k++) {
    unsigned long long tiles = 0, cost;
    for (i = 0; i < count; i++) tiles += ((unsigned long long)out_dims[i] + of[k] - 1u) / of[k];
    cost = ((tokens + 127u) / 128u * tiles + GEMM_ROUND_TILES - 1) / GEMM_ROUND_TILES * gemm_tile_cost(type, of[k]);
    if (cost < least) least = cost, best = of[k];
  }
  return best;
}

// The kernels of 256 tokens x 256 rows (gemm_q4k_tall.hpp; Q4_K lists and gate | up, whose tile is 128 rows of both): where their tiles take less
// time than those of the kernel the rules above pick. A last round that is not full is charged 0.6 + 0.4 fill^2 of a round: the fewer compute units
// work, the higher the chip's clock. One launch of 64 | 128 | 192 | 256 | 320 | 512 tiles, 4096 columns, us: 192 rows 42.6 | 45.9 | 49.5 | 57.7 | 92.0 |
// 111.5, 128 rows 31.5 | 34.0 | 36.6 | 42.4 | 67.7 | 78.9, 256 rows 50.7 | 54.8 | 61.4 | 74.5 | 116.7 | 147.5, these 82 | 87.5 | 99.9 | 122.9 | 193 | 242; gate | up
// with 96 rows 48.4 | 51.4 | 55.5 | 63.8 | 103 | 121, with 128 50.6 | 54.0 | 64.2 | 77.3 | 121 | 154, these 90 | 96 | 112.5 | 135.6 | 217 | 266: a round is 213 in lists
// and 217 to 232 in gate | up. Weights from memory, what the rules above take | these: lists of 30720 rows x 4096 at 512 tokens 139 to 149 | 116, 1024
// 270 | 224, 2048 522 | 438, at 256 72 | 82 (not taken); 30720 x 512 | 2048 | 8192 at 512 tokens 40 | 81 | 261 and 31 | 67 | 217; gate | up 4096 -> 12288 at 512 tokens
// 121 | 110, 2048 431 | 380, 1024 217 | 226 (not taken); 2048 -> 6144 at 1024 75 | 66.
#define GEMM_TALL_COST 213u
#define GEMM_TALL_SWIGLU_COST 232u
static inline unsigned long long gemm_fill_cost(unsigned long long tiles, unsigned cost) {
  const unsigned long long full = tiles / GEMM_ROUND_TILES, rest = tiles % GEMM_ROUND_TILES;
  return cost * (256ull * full + (rest ? 154ull + 102ull * rest * rest / 65536ull : 0ull));
}
static inline unsigned long long gemm_list_tiles(const unsigned* out_dims, unsigned count, unsigned rows) {
  unsigned long long n = 0;
  unsigned i;
  for (i = 0; i < count; i++) n += ((unsigned long long)out_dims[i] + rows - 1u) / rows;
  return n;
}
static inline int gemm_tall_takes(unsigned type, unsigned in_dim, const unsigned* out_dims, unsigned count, unsigned tokens) {
  const unsigned long long mt = (tokens + 127ull) / 128ull;
  if (type != 12u || tokens <= 128u || (in_dim & 255u) != 0 || in_dim == 0) return 0;
  const unsigned rows = gemm_list_rows(type, in_dim, out_dims, count, tokens, -1);
  return gemm_fill_cost((mt + 1u) / 2u * gemm_list_tiles(out_dims, count, 256u), GEMM_TALL_COST) <
         gemm_fill_cost(mt * gemm_list_tiles(out_dims, count, rows), gemm_tile_cost(type, rows));
}
static inline int gemm_tall_swiglu_takes(unsigned type, unsigned in_dim, unsigned out_dim, unsigned tokens) {
  const unsigned long long mt = (tokens + 127ull) / 128ull;
  if (type != 12u || tokens <= 128u || (in_dim & 255u) != 0 || in_dim == 0) return 0;
  const int wide = gemm_swiglu_use_wide(out_dim, tokens, -1);
  return gemm_fill_cost((mt + 1u) / 2u * gemm_list_tiles(&out_dim, 1u, 128u), GEMM_TALL_SWIGLU_COST) <
         gemm_fill_cost(mt * gemm_list_tiles(&out_dim, 1u, wide ? 128u : 96u), gemm_tile_cost(12u, wide ? 256u : 192u));
}

// Two matrices with an input each in one launch of 128-token x 256-row tiles, each with its own k splits (gemm_q6k_wide.hpp; a: Q4_K or Q5_K, b:
// Q4_K or Q6_K: o and down of a layer): the two share the chip where one alone would leave half of it idle, and the splits even their chains out. The plan is the
// cheapest of those whose tiles fit one round of the chip: start and end 11 us, the longer chain at 3.7 (Q4_K) or 4.2 us (Q5_K, Q6_K) a super-block, a split
// matrix's planes at 5 TB/s and a launch (within a tenth of what 36 shapes measured). Taken from 1300 tile super-blocks in all, below which the
// launches of their own do better, and where the plan's time is less than what those reach at their best, 19.5 ns a tile super-block and
// 36 us of starts, ends and sums. Weights from memory, us, launches of their own | this: o 4096 -> 4096 and Q6_K down 12288 -> 4096 at 256 | 384 | 512 | 640 tokens 59.9 |
// 94 | 110 | 159 and 59.0 | 73.5 | 90 | 115 (1024: 162 | 180, not taken: chains of 48), Q4_K down at 512 90.5 | 83.6; 2560 -> 2560 and 9728 -> 2560 at 300 | 700
// tokens 78.5 | 130 and 50 | 72.5; 2048 and 11008 at 700 85.6 | 64; 1536 and 8448 at 546 (1170 super-blocks) 36.5 | 40.6, 2048 and 10240 at 290 (1152) 35.4 | 39.7: not taken. Q5_K o: 4096 and Q6_K
// 12288 -> 4096 at 256 | 512 63.6 | 117 and 58.8 | 91.4, Q4_K down at 640 118 | 99.5; 2560 and 9728 at 300 78.3 | 49.
#define GEMM_WIDE_TWO_SCRATCH (256ull * 128ull * 256ull * 4ull)   // the planes of a launch of one round at most
static inline int gemm_wide_two_plan(unsigned type_a, unsigned in_a, unsigned out_a, unsigned type_b, unsigned in_b, unsigned out_b, unsigned tokens,
                                     unsigned* splits_a, unsigned* splits_b) {
  const unsigned long long mt = (tokens + 127ull) / 128ull, ta = mt * ((out_a + 255ull) / 256ull), tb = mt * ((out_b + 255ull) / 256ull);
  const unsigned na = in_a >> 8, nb = in_b >> 8;
  const unsigned long long work = ta * na + tb * nb;
  unsigned long long least = ~0ull;   // ns
  unsigned sa, sb;
  if ((type_a != 12u && type_a != 13u) || (type_b != 12u && type_b != 14u) || ((in_a | in_b) & 255u) != 0 || na > GEMM_Q6W_MAX_KB || nb > GEMM_Q6W_MAX_KB || tokens <= 192u ||
      ta + tb > 256u || work < 1300u)
    return 0;
  for (sa = 1; sa == 1u || (sa <= 4u && 2u * sa <= na); sa++)
    for (sb = 1; sb == 1u || (sb <= 8u && 2u * sb <= nb); sb++) {
      const unsigned long long ca = ((na + sa - 1u) / sa) * (type_a == 13u ? 4200ull : 3700ull), cb = ((nb + sb - 1u) / sb) * (type_b == 14u ? 4200ull : 3700ull);
      unsigned long long c = 11000ull + (ca > cb ? ca : cb);
      if (ta * sa + tb * sb > 256u) break;
      if (sa > 1u) c += 2000ull + (sa + 1ull) * tokens * out_a / 1250ull;
      if (sb > 1u) c += 2000ull + (sb + 1ull) * tokens * out_b / 1250ull;
      if (c < least) least = c, *splits_a = sa, *splits_b = sb;
    }
  return least < work * 195ull / 10ull + 36000ull;
}

// ---- prefill GEMM: which tile a workgroup takes. Workgroups go to the 8 XCDs round-robin (id % 8), each XCD has its own
// L2 and 32 compute units, and a GEMM workgroup has a compute unit to itself, so the workgroups id = 8 l + x with the
// same l / 32 run side by side on XCD x. Every XCD gets an equal share of the tiles (they are numbered in one line and it takes
// a contiguous piece of it), so that none has a round of workgroups more than the others, and the line winds through the
// matrix so that 32 neighbours on it are a compact block: gn weight tiles of one token tile after each other, then the
// same of the next token tile, then the next gn weight tiles. A weight tile is then fetched into that L2 once for the token tiles
// of its block and an x tile once for gn weight tiles. (Whole blocks of 4 token tiles x 8 weight tiles dealt round-robin, as this was
// before, left XCDs idle where the token tiles do not divide by four; us before -> now: Q4_K 4096 -> 30720 in 192-row tiles, 384 tokens
// 140.9 -> 105.9, 640 tokens 269 -> 197; Q6_K 12288 -> 4096 in 128-row tiles, 640 tokens 190 -> 97.5; 512, 1024, 2048 tokens level.)
#define GEMM_XCD_COUNT 8u
#define GEMM_XCD_UNITS 32u
// weight tiles of a block: 32 tiles of up to 4 token tiles where there are enough of them, fewer when the launch has fewer
// than 256 tiles
static inline GEMV_HD unsigned gemm_block_mt(unsigned mtiles) { return mtiles >= 4u ? 4u : (mtiles >= 2u ? 2u : 1u); }
static inline GEMV_HD unsigned gemm_block_nt(unsigned mtiles, unsigned ntiles) {
  const unsigned bmt = gemm_block_mt(mtiles);
  const unsigned per_xcd = (mtiles * ntiles + GEMM_XCD_COUNT - 1u) / GEMM_XCD_COUNT;
  const unsigned want = (per_xcd + bmt - 1u) / bmt, cap = GEMM_XCD_UNITS / bmt;
  return want < 1u ? 1u : (want > cap ? cap : want);
}
// The workgroups the library launches: one per tile, rounded up to equal shares.
static inline GEMV_HD unsigned gemm_tiles_grid(unsigned mtiles, unsigned ntiles) {
  return GEMM_XCD_COUNT * ((mtiles * ntiles + GEMM_XCD_COUNT - 1u) / GEMM_XCD_COUNT);
}
// The grid cogni_gemm_plan gives hosts that launch by name: rounded up to whole blocks for every XCD, as it always was (any grid of
// gemm_tiles_grid or more is valid: the surplus workgroups leave).
static inline GEMV_HD unsigned gemm_grid_x(unsigned mtiles, unsigned ntiles) {
  if (mtiles < 2u) return gemm_tiles_grid(mtiles, ntiles);
  const unsigned bmt = gemm_block_mt(mtiles), bnt = gemm_block_nt(mtiles, ntiles);
  const unsigned nb = ((ntiles + bnt - 1u) / bnt) * ((mtiles + bmt - 1u) / bmt);
  return GEMM_XCD_COUNT * bmt * bnt * ((nb + GEMM_XCD_COUNT - 1u) / GEMM_XCD_COUNT);
}
// false: this workgroup has no tile
static inline GEMV_HD bool gemm_tile_of(unsigned id, unsigned mtiles, unsigned ntiles, unsigned* mt, unsigned* nt) {
  const unsigned total = mtiles * ntiles, per = (total + GEMM_XCD_COUNT - 1u) / GEMM_XCD_COUNT;
  const unsigned l = id / GEMM_XCD_COUNT, vt = (id % GEMM_XCD_COUNT) * per + l;
  if (l >= per || vt >= total) return false;
  const unsigned gn = gemm_block_nt(mtiles, ntiles), g = vt / (gn * mtiles), i = vt - g * gn * mtiles;
  const unsigned left = ntiles - g * gn, n = left < gn ? left : gn;   // (the last group of weight tiles may be a smaller one)
  *mt = i / n;
  *nt = g * gn + i % n;
  return true;
}

// ---- several tokens of F32, F16, IQ4_NL or Q8_0 weights (gemm_terms.hpp): eight wavefronts = eight k-slices per tile.
// Workgroups go to the XCDs round-robin: the token tiles of one row of weight tiles follow each other on one XCD, so that
// its L2 fetches the weights once.
#define GEMM_TERMS_WAVES 8
static inline GEMV_HD void gemm_terms_tile(unsigned id, unsigned mtiles, unsigned* mt, unsigned* nt) {
  const unsigned x = id % GEMM_XCD_COUNT, l = id / GEMM_XCD_COUNT;
  *mt = l % mtiles;
  *nt = (l / mtiles) * GEMM_XCD_COUNT + x;
}
// Which calls take these kernels. F16 and F32: the row kernels re-read a row per four tokens and are level for the first few
// of a short row (F16, weights from memory, us, row kernel | tile: 512 -> 512 at 4 tokens 3.3 | 3.6, at 8 4.7 | 3.6; 2048 -> 2048 at 2
// tokens 7.8 | 7.0, from the cache level, at 3 9.7 | 7.1; 4096 -> 4096 at 2 16.1 | 11.9; F32 512 -> 512 at 4 3.4 | 3.8, at 5 4.1 | 3.9).
// IQ4_NL: always (one token of 1024 -> 3584 11.5 | 4.5). Q8_0: what the one-pass kernels leave - more than eight tokens (9 of 1024 ->
// 3584: 9.6 | 5.0), and rows that are no multiple of 256 from three (at 2 tokens 4000 -> 4096 11.1 | 10.2, 1000 -> 2041 4.7 | 5.2; a third
// costs the row kernels 2.3 and 0.8 more, the tiles nothing).
#define GEMM_TERMS_Q80_FROM 3u
static inline int gemm_terms_take(unsigned type, unsigned tokens, unsigned in_dim) {
  if (type == 20) return 1;
  if (type == 0 || type == 1) return tokens >= 5u || (tokens >= 3u && tokens * (unsigned long long)in_dim >= 4096u) || (tokens == 2u && in_dim >= 4096u);
  if (type != 8) return 0;
  return tokens > 8u || (tokens >= GEMM_TERMS_Q80_FROM && ((in_dim & 255u) != 0 || in_dim > GEMV_MT_MAX_IN_DIM));
}
// The tile (16 tm tokens x 16 tn rows) that takes the least time when the launch runs in rounds of 256 workgroups: a round
// of 1 x 1 tiles is the unit, the others measured against it (4096 columns of Q8_0, one round each: 6.4 / 8.8 / 13.9 / 21.2 /
// 34.6 us above an empty launch). By LDS and registers two or three of the smaller tiles share a compute unit, but a second round
// still costs a tile its time (Q8_0 4096 columns, 1 x 1: 256 workgroups 10.2 us, 448 15.7, 896 28.0). Of all five tiles, timed for the
// four types at 1024 / 2048 / 4096 columns, 1024 / 3584 rows and 17 / 33 / 64 / 100 / 200 / 256 tokens, this picks the fastest one 144
// times out of 144 (Q8_0 4096 -> 3584 at 100 tokens: 44.8 / 36.9 / 28.7 / 23.5 / 38.8 us).
static inline unsigned gemm_terms_plan(unsigned tokens, unsigned out_dim, unsigned* tm, unsigned* tn) {
  static const unsigned shape[5][3] = {{1, 1, 100}, {1, 2, 140}, {2, 2, 220}, {2, 4, 335}, {4, 4, 545}};
  unsigned best = 0;
  unsigned long long cost = ~0ull;
  for (unsigned i = 0; i < 5; i++) {
    const unsigned long long mt = (tokens + 16ull * shape[i][0] - 1) / (16ull * shape[i][0]), nt = (out_dim + 16ull * shape[i][1] - 1) / (16ull * shape[i][1]);
    const unsigned long long c = ((mt * nt + 255ull) / 256ull) * shape[i][2];
    if (c < cost) cost = c, best = i;
  }
  *tm = shape[best][0];
  *tn = shape[best][1];
  const unsigned mt = (tokens + 16 * *tm - 1) / (16 * *tm), nt = (out_dim + 16 * *tn - 1) / (16 * *tn);
  return mt * ((nt + GEMM_XCD_COUNT - 1u) / GEMM_XCD_COUNT) * GEMM_XCD_COUNT;
}

// Whether a tile's kernel for rows of in_dim values is a second one whose steps are interleaved (gemm_terms.hpp), "<name>_i"; the sums are the same bits. The
// kernels alone, weights from memory, one round of 160 to 240 workgroups, us, row tile by row tile | interleaved. 2 x 2 at 1024, 1184, 1408, 2048 and 3072 columns: Q8_0 7.67 | 7.78,
// 9.40 | 9.15, 9.57 | 9.45, 12.8 | 12.7, 16.2 | 16.2; F32 10.77 | 10.82, 11.98 | 11.96, 12.85 | 12.82, 16.2 | 15.7, 21.6 | 21.4; IQ4_NL 7.54 | 7.86, 8.42 | 8.71, 9.71 | 9.60, 12.2 | 12.3, 17.0 | 16.6;
// F16 8.79 | 9.05, 10.3 | 10.4, 10.7 | 10.8, 13.2 | 13.0, 17.7 | 17.5. 2 x 4 at 1184, 1536, 2592 and 3488: Q8_0 11.8 | 12.0, 13.9 | 13.8 (calls of 1632 11.7 | 12.0), 20.6 | 19.5, 28.9 | 26.1; F16 13.4 | 13.6, 16.7 | 16.1, 22.2 | 22.3,
// 30.2 | 30.1 (4096 32.7 | 31.5); IQ4_NL 11.5 | 12.0, 13.9 | 14.3, level at 2592, 26.8 | 25.8. One order is the better one at (nearly) every length, and has the name, for 1 x 1 (no other sum to
// go to); 1 x 2 of F32 (interleaved, 8.35 | 8.17, 18.7 | 18.1), F16 (level), Q8_0 and IQ4_NL (not, 768 columns 5.18 | 5.31, 5.73 | 5.77, long rows level); 2 x 4 of F32 (not, 12.5 | 13.4,
// 39.3 | 40.4); 4 x 4 (interleaved, 1024 and 4096 columns, Q8_0 15.2 | 14.7, 40.0 | 38.3, the others alike).
static inline int gemm_terms_interleaved(unsigned type, unsigned tm, unsigned tn, unsigned in_dim) {
  if (tm != 2u) return 0;
  if (tn == 2u) return in_dim >= (type == 1u ? 1536u : (type == 20u ? 1408u : 1152u));
  return type != 0u && in_dim >= (type == 1u ? 1536u : (type == 20u ? 2560u : 1696u));
}

// ---- short prefills of Q4_K, Q5_K and Q6_K (gemm_stream.hpp): a workgroup takes 32 t tokens x 32 rt rows
#define GEMM_STREAM_MAX_SPLITS 8u
#define GEMM_STREAM_MAX_PACKED 0x7FFFFFFFu   // bytes of packed activations the kernels can address
typedef struct {
  unsigned t, rt, splits;
} GemmStreamPlan;
static inline unsigned gemm_stream_tokens(unsigned tokens) { return tokens <= 32u ? 1u : 2u; }
// Rows of a workgroup and k splits: the cheapest of (super-blocks a wavefront walks) x (time of one, by type and tile) x
// (load), plus the plane sum. The load is what workgroups that share a compute unit cost each other, charged as 1 up to 180
// workgroups and 1.7 more for every 256 from there: steeper than it measures (Q4_K, 64 tokens x 32 rows, 4096 columns, 128 / 256 / 384 /
// 960 workgroups: 9.2 / 10.0 / 19.5 / 39.1 us = 1 / 1.09 / 2.1 / 4.3, charged 1 / 1.5 / 2.4 / 6.2); the plane sum counts 3 us (4.0 to 6.4
// behind a profiler). So the picks were checked, every tile and split by name, 12 shapes of 1024 to 12288 columns and 17 to 512 tokens
// with weights from memory, us: Q4_K picks the fastest but once (12288 -> 4096 at 32 tokens 15.2, fastest 14.6), Q6_K is at most 5 % off
// (4096 -> 12288 at 24 tokens 19.5 | 18.5), Q5_K takes 64 rows too early: 4096 -> 4096 at 48 tokens 12.0 where 32 rows without a split
// take 10.0, 4096 -> 12288 at 24 tokens 16.7 | 15.4, 12288 -> 4096 at 32 and 48 tokens 6 % off, the rest level. (Its 64 tokens x 64
// rows need more than the 256 registers and spill three; Q6_K has no such kernel.)
static inline GemmStreamPlan gemm_stream_plan(unsigned type, unsigned tokens, unsigned in_dim, unsigned long long rows, unsigned planes_max) {
  static const unsigned us100[3][2][2] = {{{100, 160}, {150, 260}}, {{170, 260}, {200, 320}}, {{200, 420}, {260, 0}}};   // [type][t][rt]
  const unsigned ty = type == 14u ? 2u : (type == 13u ? 1u : 0u), t = gemm_stream_tokens(tokens), nkb = in_dim >> 8;
  const unsigned long long mt = (tokens + 32u * t - 1u) / (32u * t);
  GemmStreamPlan best;
  unsigned long long least = ~0ull;
  unsigned rt, s;
  best.t = t;
  best.rt = best.splits = 1;
  for (rt = 1; rt <= 2u; rt++)
    for (s = 1; s <= planes_max && (s == 1u || 4u * s <= nkb); s *= 2u) {
      const unsigned step = us100[ty][t - 1u][rt - 1u];
      const unsigned long long wgs = mt * ((rows + 32u * rt - 1u) / (32u * rt)) * s;
      const unsigned long long load = wgs <= 180u ? 256u : (wgs * 17u) / 10u - 50u;   // in 256ths
      const unsigned long long cost = ((nkb + 4u * s - 1u) / (4u * s)) * step * (load < 256u ? 256u : load) / 256u + (s > 1u ? 300u : 0u);
      if (step && cost < least) least = cost, best.rt = rt, best.splits = s;
    }
  return best;
}
static inline GEMV_HD unsigned gemm_stream_grid(unsigned tokens, unsigned t, unsigned ntiles) {
  const unsigned mt = (tokens + 32u * t - 1u) / (32u * t);
  return mt * ((ntiles + GEMM_XCD_COUNT - 1u) / GEMM_XCD_COUNT) * GEMM_XCD_COUNT;
}
// Which launches take these kernels: more tokens than the sixteen-token one-pass kernels have, and no more weights x groups of
// 64 tokens (in values) than the line up to which they measured ahead of the tile kernels (us, tile | stream). One group, Q4_K
// 4096 -> 12288 at 32 tokens 19.0 | 14.0, 64 21.6 | 16.9; 12288 -> 12288 at 24 37.1 | 31.7, at 48 40.3 | 39.8; Q6_K 12288 ->
// 4096 at 32 22.8 | 18.9, at 64 23.9 | 23.0. More: Q4_K 1024 -> 3072 at 512 18.2 | 10.1, 2048 -> 2048 at 1024 25.5 | 16.9, 2048 ->
// 4096 at 512 24.6 | 15.8, at 1024 24.2 | 29.4; rows of 4096 and more hold on longer (4096 -> 4096 at 512 29.9 | 26.4, at 1024
// 40.5 | 53.2; 4096 -> 12288 at 128 31.7 | 25.8). Q6_K 4096 -> 4096 at 256 23.9 | 21.8, at 512 33.5 | 39.8.
static inline int gemm_stream_take(unsigned type, unsigned tokens, unsigned in_dim, unsigned long long rows) {
  const unsigned long long groups = (tokens + 63ull) / 64ull, values = groups * in_dim * rows;
  unsigned long long most = 1ull << 26;
  if (tokens <= 16u || 256ull * ((tokens + 127ull) / 128ull) * in_dim > GEMM_STREAM_MAX_PACKED) return 0;
  if (type == 14u) most = tokens <= 32u ? 100000000ull : 1ull << 26;
  else if (tokens <= 64u) most = 160000000ull;
  else if (in_dim >= 4096u) most = 140000000ull;
  return values <= most;
}

// ---- one-pass kernel, rows above 4096 values: what a streamed unit waits for (gemv_mt.hpp)
// vmcnt value that says "operand set i and unit i of a streamed row group have landed" (T = 1, S super-blocks per
// k-slice, NSLOT units in LDS). Issue order: set 0, unit 0, set 1, unit 1, units 2 .. min(S, NSLOT) - 1 up front; behind unit
// i's arithmetic: set i + 2, then unit i + NSLOT. NA loads per set, NC copies per unit. The answer is the number of loads
// issued, by the time of the wait, behind the later of the two.
static inline GEMV_HD constexpr int mt_stream_wait(int S, int NSLOT, int NS, int NA, int NC, int i) {
  int pos = 0, end_set[8] = {}, end_unit[8] = {};
  const int up = S < NSLOT ? S : NSLOT;
  for (int u = 0; u < up; u++) {
    if (u < NS) end_set[u] = (pos += NA);
    end_unit[u] = (pos += NC);
  }
  for (int j = 0; j < i; j++) {   // what was issued behind the units before i
    if (j + NS < S) end_set[j + NS] = (pos += NA);
    if (j + NSLOT < S) end_unit[j + NSLOT] = (pos += NC);
  }
  const int need = end_set[i] > end_unit[i] ? end_set[i] : end_unit[i];
  return pos - need;
}
