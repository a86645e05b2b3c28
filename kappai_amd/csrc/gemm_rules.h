// Numbers that the product kernels (gemm.hip) and the rule for K ranges (engine.hip) share.
#pragma once

// The kernel with 32 x 32 tiles and the rows through LDS (gemm_bf16_rows32) takes steps of more
// than KAPPAI_ROWS32_MIN_ROWS and up to KAPPAI_ROWS32_MAX_ROWS rows.  Below, the kernels with
// 16 x 16 tiles are as fast or faster (up to 24 rows they read the rows of A straight from L2);
// above, the block kernels.  Measured on one box, decode steps of the LFM2-1.2B shape: 64 rows
// 38.95 k against 37.63 k tok/s with the kernel for 17 to 64 rows, 32 rows 26.0 k against 25.1 k;
// the LFM2-350M serving workload 35.1 k against 34.2 k generated tok/s.
#define KAPPAI_ROWS32_MIN_ROWS 24
#define KAPPAI_ROWS32_MAX_ROWS 128
// K of a block of that kernel comes in runs of this many
#define KAPPAI_ROWS32_RUN 256

// The forms of the block kernel (gemm_bf16_block256) for more than 128 rows.
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
