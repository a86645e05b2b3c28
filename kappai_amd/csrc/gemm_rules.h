// Numbers that the product kernels (gemm.hip) and the rule for K ranges (engine.hip) share.
#pragma once

// Steps of more than KAPPAI_ROWS32_MIN_ROWS and up to KAPPAI_ROWS32_MAX_ROWS rows over a W in fragment order, K in runs
// of KAPPAI_ROWS32_RUN: the block products (the forms below), or the kernel with 32 x 32 tiles and the rows through LDS
// (gemm_bf16_rows32, where kappai_rows32_takes says so).  Below, the kernels with 16 x 16 tiles, which give a matrix
// kept as rows the same bits (24 rows of 9216 x 1024 gated 7.8 us by them, 6.3 in blocks; 1024 x 4608 in eight ranges
// 4.4, in six 4.7).
#define KAPPAI_ROWS32_MIN_ROWS 24
#define KAPPAI_ROWS32_MAX_ROWS 128
// K of a block of that kernel comes in runs of this many
#define KAPPAI_ROWS32_RUN 256
// M rows in `split` ranges of K, n_rows rows of W.  A K below 1,024, where that kernel is at a dependent kernel's own
// time as it is; and of up to 32 rows, of which it wastes none, the very wide products of a short K (65536 x 1024 28.5
// us, in blocks 29.6 to 32) and the smallest (256 x 1024 in four ranges 3.3 and 3.4, 64 x 1024 4.4 and 4.7; 512 x 1024
// in four 3.5 both).  Else the blocks, us by that kernel and by them: 64 rows of 16384 x 2048 gated 17.4 and 15.5, of
// 6144 x 2048 in two ranges 9.9 and 8.7, of 8192 x 4096 gated 24.7 and 20.2, 100 rows of 1024 x 4608 in six 8.0 and 5.1.
static inline bool kappai_rows32_takes(int M, int n_rows, int K, int split) {
  return K < 1024 || (M <= 32 && ((K < 2048 && n_rows > 16384) || (long)n_rows * (K / split) < 131072));
}

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
// Up to 128 rows the blocks of 64 rows or columns are the faster at every K (97 rows of 4096 x 4096 gated 17.4 and
// 32.6 us in 128 x 128), and 64 x 64 of up to 64 rows also in more blocks than CUs, two to a CU (32 rows of 40960 x
// 2048 gated 34.4 and 41.9).  There W's stream bounds them and the model's times are 15 to 25 % short, but over 657
// products (25 to 128 rows, 256 to 65,536 columns, K from 1,024 to 16,384, up to eight ranges, float, bfloat16 and
// gated results) the form that it likes best, with kappai_rows32_takes, takes 0.2 % more than the fastest in sum; with
// the limits of more rows 19 % more.
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
  const bool few = M <= KAPPAI_ROWS32_MAX_ROWS;
  const int longest = result_mb > 3e-6 * M * N * split ? 1536 : 2048;
  for (const kappai_block_form& f : KAPPAI_BLOCK_FORMS) {
    if (gated && f.shape == 9) continue;       // (its waves' columns are no whole pairs of 64)
    const double blocks = (double)((M + f.rows - 1) / f.rows) * ((N + f.cols - 1) / f.cols) * split;
    if (f.rows * f.cols < 128 * 128 && !(few && f.shape == 15 && M <= 64) &&
        (blocks > 256 || (!few && K / split > longest)))
      continue;
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
// The same for results of `elem` bytes each, float planes if there are ranges.
static inline int kappai_block_shape_for(int M, int N, int K, int split, int elem, bool gated) {
  return kappai_block_shape(M, N, K, split, (double)M * N * split * elem * (gated ? 0.5e-6 : 1e-6), gated, nullptr);
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

