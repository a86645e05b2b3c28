// Numbers that the product kernels (gemm.hip) and the rule for K ranges (engine.hip) share.
#pragma once

// Steps of more than KAPPAI_ROWS32_MIN_ROWS and up to KAPPAI_ROWS32_MAX_ROWS rows over a W in fragment order, K in runs
// of KAPPAI_ROWS32_RUN: the smallest block products from K = 1,024 on, else the kernel with 32 x 32 tiles and the
// rows through LDS (gemm_bf16_rows32).  Below, the kernels with 16 x 16 tiles, which give a matrix kept as rows the
// same bits (24 rows of 9216 x 1024 gated 7.8 us by them, 6.3 in blocks; 1024 x 4608 in eight ranges 4.4, in six 4.7).
#define KAPPAI_ROWS32_MIN_ROWS 24
#define KAPPAI_ROWS32_MAX_ROWS 128
// K of a block of that kernel comes in runs of this many
#define KAPPAI_ROWS32_RUN 256

// The blocks of a product of more rows whose W lies in fragment order (gemm_bf16_direct, gemm_bf16_staged),
// and a model of what each takes, in us: a tile of 64 of K costs `tile` in every round of blocks over the
// 256 CUs and `fill` more when the round is full, a round `round`, a megabyte of results `mb`.  Least squares
// of relative errors over 5,289 products (128 to 4,400 rows, 512 to 16,384 columns, K from 512 to 10,752, one
// to eight ranges, float, bfloat16 and gated results), good to 5 to 10 % each.  Over the same products the
// form that the model likes best takes 0.6 % more than the fastest of the five in sum; a fifth of the products
// each are best in the first, fourth and fifth, two fifths in the third.  Over 366 others, measured later on
// another card: errors of 6 to 10 %, and 0.6 % again.
// The last three are for products of at most a block a CU (beyond, a larger block is the faster: 2048 x 1024 of
// 1040 rows 9.3 us in 128 x 128 and 10.7 in 64 x 128) and for ranges of up to 2,048 of K, 1,536 where the sums are
// float planes (2048 x 8192 of 417 rows 21.8 us with the norm's share in four ranges of 128 x 128, 23.0 in two of
// 128 x 64).  Fitted to 185 products of 160 to 1,040 rows on a card that is 4 % slower than the model, good to 4 to
// 8 %.  Over 240 products, ranges among them, the form that the model likes best takes 0.2 % more than the fastest
// of the six up to 256 x 128; without these three 17 % more.
struct kappai_block_form {
  int shape, rows, cols;           // (shape: gemm.hip, launch_tile)
  double tile, fill, round, mb, start;
};
static const kappai_block_form KAPPAI_BLOCK_FORMS[8] = {
    {5, 256, 256, 0.95, 0.40, 6.0, 0.112, 2.9},  {9, 256, 192, 0.81, 0.30, 5.5, 0.111, 3.0},
    {12, 256, 128, 0.51, 0.25, 1.9, 0.158, 3.2}, {11, 192, 128, 0.42, 0.22, 0.7, 0.198, 3.2},
    {8, 128, 128, 0.32, 0.18, 0.1, 0.244, 3.1},  {13, 64, 128, 0.180, 0.131, 0.0, 0.095, 3.7},
    {14, 128, 64, 0.196, 0.062, 0.0, 0.151, 3.7}, {15, 64, 64, 0.147, 0.036, 0.0, 0.165, 2.8}};
// The shape of the blocks for M rows, N rows of W, K in `split` ranges; `time`: what the model says.
static inline int kappai_block_shape(int M, int N, int K, int split, double result_mb, bool gated,
                                     double* time) {
  int best = 8;
  double best_t = -1.0;
  const int longest = result_mb > 3e-6 * M * N * split ? 1536 : 2048;
  for (const kappai_block_form& f : KAPPAI_BLOCK_FORMS) {
    if (gated && f.shape == 9) continue;       // (its waves' columns are no whole pairs of 64)
    const double blocks = (double)((M + f.rows - 1) / f.rows) * ((N + f.cols - 1) / f.cols) * split;
    if (f.rows * f.cols < 128 * 128 && (blocks > 256 || K / split > longest)) continue;
    const double rounds = (double)(((long)blocks + 255) / 256), tiles = (double)K / split / 64.0;
    const double t = tiles * (f.tile * rounds + f.fill * blocks / 256) + f.round * rounds +
                     f.mb * result_mb + f.start;
    if (best_t < 0 || t < best_t) {
      best = f.shape;
      best_t = t;
    }
  }
  if (time) *time = best_t;
  return best;
}

// The same for a W that lies as rows (gemm_bf16_block256).
//
// 256 x 256 blocks, one a CU, against 128 x 128 blocks, two a CU: from 140 blocks on when one round
// does it, and with more rounds when the last one is not mostly idle (idle CU-rounds under a third
// of the blocks).  From sweeps over the layer shapes at 160 to 8192 rows; gate/up 14336 x 2048 of 1759
// rows, 392 blocks: 109 against 118 us; 16384 x 2048 of 1500 rows, 384 blocks: 111 against 110.
static inline bool kappai_use_256_form(long blocks256) {
  if (blocks256 <= 256) return blocks256 >= 140;
  const long rem = blocks256 % 256;
  return rem == 0 || (256 - rem) * 3 < blocks256;
}
// 128 x 128 blocks that would each have a CU to themselves anyway: the form with four LDS buffers
// (0.45 to 0.6 against 0.7 to 0.8 us per 64 of K) unless K is too short for its start (2 us more).
// 3072 x 2048 in two ranges, 417 rows: 14.6 against 18.0 us; gate/up 9216 x 1024, 256 rows: 13.7 against
// 17.5; ranges of 512 and less: equal or 5 % slower.
static inline bool kappai_deep_form(long blocks128, int k_range) {
  return blocks128 <= 256 && k_range >= 768;
}

