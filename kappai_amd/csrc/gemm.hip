// Matrix products  C[M,N] = A[M,K] * W[N,K]^T (+ bias[N])  for every projection and the
// output head.  W is a weight matrix [out, in] with `in` contiguous, as stored in the
// checkpoint (kappai: y[n] = sum_k W[n,k] x[k], src/backend/cpu/scalar/quants.c:1398-1414).
//
//   gemm_f32         true 32-bit: float products and sums on the matrix cores
//                    (v_mfma_f32_16x16x4_f32) in an order that K alone decides, so a row's result
//                    does not depend on M; a kernel for up to 64 rows and one for more.
//   gemm_bf16_direct, gemm_bf16_staged  large products over a W in fragment order (K a multiple of
//                    128 per K range): bf16 inputs, fp32 accumulation on the matrix cores
//                    (v_mfma_f32_32x32x16_bf16), 256x256 to 64x64 blocks, tiles of 64 of K loaded
//                    straight into LDS (in the largest blocks W's straight into registers).
//   gemm_bf16_block256  the same over a W that lies as rows.
//   gemm_bf16_tile   any K that is a multiple of 8: 256x128 or 128x128 blocks staged through
//                    registers into LDS.
//   gemm_bf16_skinny M <= 64 (decode): every block streams 16 or 32 rows of W once, its 4 to 16
//                    waves split K and meet in LDS (v_mfma_f32_16x16x32_bf16).
//   gemm_bf16_shared_rows  17 <= M <= 64 and a W with many rows: as above, but two waves that
//                    stream different rows of W share the rows of A through LDS.
//   gemm_bf16_rows32 25 <= M <= 128 where the block products do not fit or are the slower: the same idea with
//                    32 x 32 tiles (v_mfma_f32_32x32x16_bf16), W from its fragment-order copy.
//   gemm_bf16_any    K or a row stride that is no multiple of 8: a plain kernel, so that no
//                    width is refused.
#include "common.h"
#include "gemm_rules.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

#define KAPPAI_GPTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define KAPPAI_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

#define SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)
// (nothing that touches memory is moved across, by any pass of the compiler)
#define ORDER_FENCE()                  \
  do {                                 \
    asm volatile("" ::: "memory");     \
    __builtin_amdgcn_sched_barrier(0); \
  } while (0)
// waits until at most `behind` loads are under way (_AND_LDS: and no LDS access is)
#define WAIT_LOADS(behind) __builtin_amdgcn_s_waitcnt(0x0F70 | ((behind) & 15) | ((behind) >> 4 << 14))
#define WAIT_LOADS_AND_LDS(behind) \
  __builtin_amdgcn_s_waitcnt(0x0070 | ((behind) & 15) | ((behind) >> 4 << 14))

// A buffer of `bytes` bytes from p on: loads whose lane's and scalar offset together lie outside it read
// nothing and give zeros, so a loop's last loads need no branch.  (The type is the device compiler's; the host
// pass sees neither it nor the loads.)
#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t raw_buffer(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
#endif

// ---------------------------------------------------------------------------------------
// true fp32
// ---------------------------------------------------------------------------------------
#if !defined(GATE_ACT) || GATE_ACT == 0     // (the builds with another gate hold gated products only)
// Both kernels multiply on the matrix cores in 32 bits (v_mfma_f32_16x16x4_f32: float products
// and float sums, 256 flops a clock and CU against 128 for a float FMA on the vector units) and add
// in ONE order that K alone decides, so a row's result depends neither on M nor on which of them
// runs: K is cut into chunks of 128, the chunks into 8 or 32 runs; the products of a chunk are
// added 16 of K after 16 (lane group q of a load holds k = 4 q .. 4 q + 3 of the 16, step e takes
// the e-th of every group), then chunk after chunk into the run's sum, then run after run.  A single
// running sum over K = 8192 would lose about sqrt(K) roundings; this way it is sqrt(128) + a few.
//
// LOADS: F32_WHOLE, K is a multiple of 128 and everything is aligned to 16 bytes; F32_FOURS, K is a
// multiple of 4 and everything is aligned; F32_ELEMENTS, any other K from 4 on; F32_FEW, less.  Where
// K ends the row's last four places are read again and what lies behind counts as 0, so that no load
// stands in a branch that asks how far K goes (such a branch has the compiler wait for one load before
// it asks for the next), and 16s of K that are all behind it are left out.  4096 columns over K = 16, 1,000
// rows: 21.4 us with such branches and all 128 multiplied, 12.8 now; 1024 x 1030 of 64 rows 34.4 and
// 19.6, of 1,000 46.5 and 31.8.
#define F32_CHUNK 128
#define F32_STEPS (F32_CHUNK / 16)
enum { F32_FEW, F32_ELEMENTS, F32_FOURS, F32_WHOLE };

__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__host__ __device__ __forceinline__ int f32_runs(int chunks) { return chunks <= 16 ? 8 : 32; }
__device__ __forceinline__ int f32_run_start(int run, int runs, int chunks) {
  return run * chunks / runs;
}

// The gate as kappai_swiglu computes it.
__device__ __forceinline__ float f32_gate(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// Four values of a row from k on; zeros from K on.
template <int LOADS>
__device__ __forceinline__ f32x4_t load4_f32(const float* __restrict__ row, int k, int K) {
  if (LOADS == F32_WHOLE) return *reinterpret_cast<const f32x4_t*>(row + k);
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
  if (LOADS == F32_FEW) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (k + e < K) v[e] = row[k + e];
    return v;
  }
  const int from = min(k, K - 4), behind = k - from;
  if (LOADS == F32_FOURS) {
    const f32x4_t x = *reinterpret_cast<const f32x4_t*>(row + from);
    return behind ? v : x;
  }
  float x[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = row[from + e];
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int back = 0; e + back < 4; ++back) v[e] = behind == back ? x[e + back] : v[e];
  return v;
}

// A lane's share of a chunk (its q-th four of every 16).
template <int LOADS>
__device__ __forceinline__ void load_chunk_f32(const float* __restrict__ row, int chunk, int q, int K,
                                               f32x4_t (&v)[F32_STEPS]) {
  const int k = chunk * F32_CHUNK + 4 * q;
#pragma unroll
  for (int j = 0; j < F32_STEPS; ++j) v[j] = load4_f32<LOADS>(row, k + 16 * j, K);
}

// M rows of the stream, normed, to LDS (F32_ROW_PAD floats between rows): x * 1/sqrt(mean(x^2) + eps) * w with the
// bits of add_rmsnorm_row_kernel, whose wave of 64 times eight values is a turn here; a wave takes the turns
// number wave, wave + NW, ..  `behind_loads` is called once a wave's loads are on their way.
#define F32_ROW_PAD 16
#define F32_NORM_TURNS 16                  // turns of all rows, at most
template <int NW, typename F>
__device__ __forceinline__ void f32_normed_rows(const float* __restrict__ x, const float* __restrict__ w, float eps,
                                                int M, int D, int ldx, float* __restrict__ rows, F behind_loads) {
  constexpr int PER = F32_NORM_TURNS / NW;
  __shared__ __attribute__((aligned(16))) float sums[F32_NORM_TURNS][4];     // (M <= 16)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int a_row = (D + 511) / 512, turns = M * a_row;
  float v[PER][8], w8[PER][8];
#pragma unroll
  for (int t = 0; t < PER; ++t) {
    const int turn = wave + t * NW, m = turn / a_row, j = (turn - m * a_row) * 512 + lane * 8;
    if (turn >= turns) break;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[t][e] = 0.f;
    if (j < D) {
      load8(x + (size_t)m * ldx + j, v[t]);
      load8(w + j, w8[t]);
    }
  }
  ORDER_FENCE();
  behind_loads();
  ORDER_FENCE();
#pragma unroll
  for (int t = 0; t < PER; ++t) {
    const int turn = wave + t * NW, m = turn / a_row;
    if (turn >= turns) break;
    const float ss = wave_sum(sum_of_squares8(v[t]));
    if (lane == 0) sums[m][turn - m * a_row] = ss;
    if (lane > 0 && lane < 4 && turn == m * a_row && lane >= a_row) sums[m][lane] = 0.f;
  }
  // (bare barriers: the loads of W stay under way)
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  ORDER_FENCE();
#pragma unroll
  for (int t = 0; t < PER; ++t) {
    const int turn = wave + t * NW, m = turn / a_row, j = (turn - m * a_row) * 512 + lane * 8;
    if (turn >= turns) break;
    const float4 s = *reinterpret_cast<const float4*>(sums[m]);
    const float scale = 1.0f / sqrtf((((s.x + s.y) + s.z) + s.w) / (float)D + eps);
    if (j < D) {
#pragma unroll
      for (int e = 0; e < 8; ++e) w8[t][e] = v[t][e] * scale * w8[t][e];
      store8(rows + m * (D + F32_ROW_PAD) + j, w8[t]);
    }
  }
  ORDER_FENCE();
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  ORDER_FENCE();
}

// 1 to 64 rows: bound by the stream of W, in small matrices by what one block has under way.  A
// block owns COLS rows of W, a wave one or several runs of K, and the waves meet in LDS.  COLS = 16: a
// wave walks its RUNS / 8 runs one after the other.  COLS = 8 (up to 8 rows; matrices of few rows, so
// that twice the blocks stream them): places 0-7 of both operands hold the wave's first run and 8-15
// its second, and the product's two diagonal quarters are the two runs' sums.  COLS = 4 (up to 4 rows and 1,024
// columns, a block for every CU): four runs and the four squares on the diagonal; three rows in a decode step, with
// 8 and 4 columns a block: 1024 x 4608 11.0 and 9.0 us, 1024 x 1024 4.9 and 4.1.  The next chunk's share
// of W is under way while a chunk is multiplied.  Three rows, W from memory: 9216 x 1024 12 us
// (3.1 TB/s), 65536 x 1024 51 us (5.3 TB/s); the vector kernel before took 100 to
// 1,500 us, a block a 64 x 64 tile of which three rows were real.
//
// GATED: W holds 2 N rows, gate rows and behind them the up rows; a block's 16 columns are the gates of 8
// results and their up rows, C[m, n] = silu(gate) up, the bits of the product and kappai_swiglu behind it.
// (Three rows, 4,608 gates: a kernel of 4.4 us less a layer; 825 rows in blocks: 9.3 us less.)
//
// NORM (decode steps of few rows): A is the residual stream and every block norms its rows itself, with the bits of
// the norm's row kernel (f32_normed_rows), its first W under way meanwhile; add: the product is added to C, which is
// that stream, so the norm has no sum left to make.  A norm kernel between two products is 4.8 us of a trace;
// norming inside costs 9216 x 1024 gated of three rows 1.5 of its 11.2 us, 2048 x 1024 and 3072 x 1024 half a us.
//
// ONE: no run has more than a chunk (8 runs, K up to 1,024) and no more than 4 rows: nothing is under way beside the
// chunk, and with the registers of three blocks a CU instead of two, 576 blocks of gate/up run at once (13.1 -> 12.7
// us).  With more rows to hold it is the slower (a decode step of the 350M shape, 5 to 9 rows 798 to 930 us with it and
// 788 to 924 without).
template <int MT, int COLS, int RUNS, int LOADS, bool GATED = false, bool NORM = false, bool ONE = false>
__global__ __launch_bounds__((COLS < 16 ? RUNS * COLS / 16 : 8) * WAVE) __attribute__((amdgpu_waves_per_eu(ONE ? 6 : 1)))
void gemm_f32_skinny_kernel(
    const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
    float* __restrict__ C, int M, int N, int K, int lda, int ldc, int add, const float* __restrict__ norm_w,
    float eps) {
  constexpr bool SIDE = COLS < 16;               // two or four runs side by side
  constexpr int NW = SIDE ? RUNS * COLS / 16 : 8, ROWS = SIDE ? COLS : 16;
  static_assert(!NORM || (MT == 1 && LOADS == F32_WHOLE), "few rows of whole chunks");
  static_assert(!SIDE || MT == 1, "runs side by side leave room for as many rows as columns");
  __shared__ float red[RUNS][MT][ROWS][COLS];
  extern __shared__ __attribute__((aligned(16))) float f32_rows[];      // NORM: M rows
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int r = lane % 16, q = lane / 16;
  static_assert(!GATED || COLS == 16, "eight gates and their up rows");
  const int n0 = blockIdx.x * (GATED ? 8 : COLS);
  const float* w = W + (GATED ? (size_t)(r / 8) * N + min(n0 + r % 8, N - 1)
                              : (size_t)min(n0 + r % COLS, N - 1)) * K;
  const float* a[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    a[mt] = A + (size_t)min(mt * 16 + r % ROWS, M - 1) * lda;

  const int chunks = (K + F32_CHUNK - 1) / F32_CHUNK;
  // this lane's chunks c0 .. c0 + len - 1; the wave takes `most` steps, a chunk each
  constexpr int per = RUNS / NW;
  const int run0 = wave * per;
  int c0 = f32_run_start(run0, RUNS, chunks);
  int len = f32_run_start(run0 + per, RUNS, chunks) - c0, most = len;
  if (SIDE) {
    most = 0;
#pragma unroll
    for (int i = 0, from = c0; i < per; ++i) {
      const int to = f32_run_start(run0 + i + 1, RUNS, chunks);
      most = max(most, to - from);
      if (r / COLS == i) {
        c0 = from;
        len = to - from;
      }
      from = to;
    }
  }
  f32x4_t tot[MT], wv[F32_STEPS], av[MT][F32_STEPS];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) tot[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int run = run0;                                // (one after the other) the run that `tot` is of
  const auto write_run = [&]() {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        red[run][mt][(4 * q + i) % ROWS][r % COLS] = tot[mt][i];
        tot[mt][i] = 0.f;
      }
    ++run;
  };
  // (a chunk behind a lane's last is read again from the last of all and not added)
  const auto load_w = [&](int c, f32x4_t (&v)[F32_STEPS]) {
    load_chunk_f32<LOADS>(w, min(c0 + c, chunks - 1), q, K, v);
  };
  // (lanes without a row stay out: a masked load costs what its live lanes do)
  const int live = r % ROWS;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < F32_STEPS; ++j) av[mt][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const auto load_a = [&](int c) {
    if constexpr (NORM) {
      const float* row = f32_rows + live * (K + F32_ROW_PAD) + min(c0 + c, chunks - 1) * F32_CHUNK + 4 * q;
      if (live < M)
#pragma unroll
        for (int j = 0; j < F32_STEPS; ++j) av[0][j] = *reinterpret_cast<const f32x4_t*>(row + 16 * j);
      return;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      if (mt * 16 + live < M) load_chunk_f32<LOADS>(a[mt], min(c0 + c, chunks - 1), q, K, av[mt]);
  };
  const auto multiply = [&](int c) {
    if (!SIDE)
      while (f32_run_start(run + 1, RUNS, chunks) <= c0 + c) write_run();
    f32x4_t acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < F32_STEPS; ++j) {
      if (LOADS != F32_WHOLE && 16 * j >= K) break;      // (a K of less than one chunk)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma_f32(av[mt][j][e], wv[j][e], acc[mt]);
    }
    // (side by side, a lane's results belong to the run that its column's part holds)
    if (!SIDE || c < len)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) tot[mt] += acc[mt];
  };
  // (the value that the thread's first result is added to)
  constexpr int OUT = GATED ? 8 : COLS;
  float old = 0.f;
  if (add && threadIdx.x < MT * ROWS * OUT) {
    const int m = threadIdx.x / OUT, n = n0 + threadIdx.x % OUT;
    if (m < M && n < N) old = C[(size_t)m * ldc + n];
  }
  if constexpr (NORM) {
    f32_normed_rows<NW>(A, norm_w, eps, M, K, lda, f32_rows, [&]() { if (most > 0) load_w(0, wv); });
  } else if (most > 0) {
    load_w(0, wv);
  }
  if (ONE && most > 0) {
    load_a(0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
  } else if (most > 0) {
    int c = 0;
    for (; c + 1 < most; ++c) {
      f32x4_t wn[F32_STEPS];
      load_a(c);
      load_w(c + 1, wn);
      __builtin_amdgcn_sched_barrier(0);       // (left alone, the loads sink to their use)
      multiply(c);
#pragma unroll
      for (int j = 0; j < F32_STEPS; ++j) wv[j] = wn[j];
    }
    load_a(c);
    __builtin_amdgcn_sched_barrier(0);
    multiply(c);
  }
  if (SIDE) {
    run += r / COLS;
    if (r / COLS == 4 * q / COLS) write_run();
  } else {
    while (run < run0 + per) write_run();
  }
  __syncthreads();
  const auto whole = [&](int m, int col, int row) {
    float s = red[0][m / 16][m % 16][col];
#pragma unroll
    for (int g = 1; g < RUNS; ++g) s += red[g][m / 16][m % 16][col];
    return s + (bias ? bias[row] : 0.f);
  };
  for (int at = threadIdx.x; at < MT * ROWS * OUT; at += NW * WAVE) {
    const int m = at / OUT, n = n0 + at % OUT;
    if (m >= M || n >= N) continue;
    const float s = whole(m, at % OUT, n);
    float* to = C + (size_t)m * ldc + n;
    if (add) *to = (at < NW * WAVE ? old : *to) + s;
    else *to = GATED ? f32_gate(s, whole(m, at % OUT + 8 * GATED, N + n)) : s;
  }
}

// More rows: bound by the matrix cores.  Blocks of WY x WX waves with wave tiles of 16 TY x 16 TX;
// K tiles of BK in two LDS buffers whose 16-byte places are XOR-permuted by the row, so that the 16 rows of
// a read hit all banks.  An XCD takes every eighth column of tiles and walks its rows of tiles, so W
// is read into one L2 only.  Two waves a SIMD: a wave's chunk, run and whole sums stay in
// vector registers, and one wave multiplies while the other waits for LDS.
//
// DIRECT (K a multiple of 128, everything aligned): a tile goes straight into LDS as soon as everybody has
// the last fragments of the tile that lay there in registers, a whole tile's products ahead of its use,
// and the next tile's first fragments are read while those last ones are multiplied.  Else the next tile's
// loads are under way in registers while this one is multiplied, and are written behind its products, where
// both waves of a SIMD wait (a third of the time: 99 TFLOP/s at 2048 x 9216 x 1024, the instruction alone
// reaches 153).  825 rows, through registers / straight: 9216 x 1024 158.7 / 139.4 us (112 TFLOP/s), 3072 x 1024
// 63.8 / 52.1, 2048 x 1024 43.2 / 36.7, 1024 x 4608 95.4 / 80.6; 65 rows of 9216 x 1024 43.3 / 37.1; the same bits.
// (With four waves a block of 64 x 64, one a SIMD, 13 % slower.)
//
// GATED (wave tiles of two 16s of columns): the second 16 of every 32 columns are the up rows of the first.
template <int WY, int WX, int TY, int TX, int BK, int LOADS, bool GATED = false, bool DIRECT = false>
__global__ __launch_bounds__(WY * WX * WAVE) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_f32_block_kernel(
    const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
    float* __restrict__ C, int M, int N, int K, int lda, int ldc, int tiles_m) {
  constexpr int BM = 16 * WY * TY, BN = 16 * WX * TX, SLOTS = BK / 4, NT = WY * WX * WAVE;
  constexpr int PER = BM * SLOTS / NT;                         // 16-byte places a thread and operand
  static_assert(BM == BN && PER * NT == BM * SLOTS && F32_CHUNK % BK == 0, "a tile");
  static_assert(!DIRECT || LOADS == F32_WHOLE, "tiles without a remainder");
  constexpr int MIX = SLOTS - 1;                               // places a row's number turns
  __shared__ __attribute__((aligned(1024))) f32x4_t lds[2][2][BM * SLOTS];
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int r = lane % 16, q = lane / 16;
  const int wm = wave / WX * 16 * TY, wn = wave % WX * 16 * TX;
  const int m0 = (int)(blockIdx.x / 8) % tiles_m * BM;
  static_assert(!GATED || TX == 2, "a wave has the gates and the up rows of its results");
  const int n0 = ((int)(blockIdx.x / 8) / tiles_m * 8 + (int)(blockIdx.x % 8)) * (GATED ? BN / 2 : BN);
  if (n0 >= N) return;

  const float* src[2][PER];
  int at[PER];
  const int slot = tid % SLOTS;
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int row = (tid + NT * p) / SLOTS;
    src[0][p] = A + (size_t)min(m0 + row, M - 1) * lda;
    src[1][p] = W + (GATED ? (size_t)(row / 16 % 2) * N + min(n0 + row / 32 * 16 + row % 16, N - 1)
                           : (size_t)min(n0 + row, N - 1)) * K;
    at[p] = row * SLOTS + (slot ^ (row & MIX));
  }
  // DIRECT: a load of a wave brings 64 / SLOTS rows of a tile straight into LDS, 16 bytes a lane in the
  // order of the lanes, so that the lane turns what it asks for; half of the waves bring A, half W.
  constexpr int ROWS_A_LOAD = 64 / SLOTS, LOADS_A_WAVE = 2 * BM / ROWS_A_LOAD / (NT / WAVE);
  static_assert(LOADS_A_WAVE < 16 && LOADS_A_WAVE * (NT / WAVE) * ROWS_A_LOAD == 2 * BM, "a wave's loads");
  const int uw = __builtin_amdgcn_readfirstlane(wave);
  const int operand = uw / (NT / WAVE / 2), first_row = uw % (NT / WAVE / 2) * LOADS_A_WAVE * ROWS_A_LOAD;
  uint32_t off[LOADS_A_WAVE];
  if constexpr (DIRECT) {
#pragma unroll
    for (int i = 0; i < LOADS_A_WAVE; ++i) {
      const int row = first_row + i * ROWS_A_LOAD + lane / SLOTS;
      const uint32_t from = operand == 0 ? (uint32_t)min(m0 + row, M - 1) * (uint32_t)lda
          : (GATED ? (uint32_t)(row / 16 % 2) * (uint32_t)N + min(n0 + row / 32 * 16 + row % 16, N - 1)
                   : (uint32_t)min(n0 + row, N - 1)) * (uint32_t)K;
      off[i] = (from + ((lane % SLOTS) ^ (row & MIX)) * 4) * 4u;
    }
  }
  // (buffer loads: of a global load into LDS the compiler holds that it may be any access to LDS, and waits for
  // all reads under way where it should wait for the oldest)
#if defined(__HIP_DEVICE_COMPILE__)
  const __amdgpu_buffer_rsrc_t from = raw_buffer(operand ? W : A, 0xFFFFFFFFu);
  const auto bring = [&](int t) {
#pragma unroll
    for (int i = 0; i < LOADS_A_WAVE; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          from, KAPPAI_LPTR(&lds[t & 1][operand][(first_row + i * ROWS_A_LOAD) * SLOTS]), 16, off[i],
          t * (int)(BK * sizeof(float)), 0, 0);
  };
#else
  const auto bring = [&](int) {};
#endif
  f32x4_t next[2][PER];
  const auto fetch = [&](int t) {
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int p = 0; p < PER; ++p)
        next[o][p] = load4_f32<LOADS>(src[o][p], t * BK + 4 * slot, K);
  };
  const auto keep = [&](int t) {
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int p = 0; p < PER; ++p) lds[t & 1][o][at[p]] = next[o][p];
  };
  f32x4_t tot[TY][TX], fin[TY][TX];
#pragma unroll
  for (int i = 0; i < TY; ++i)
#pragma unroll
    for (int j = 0; j < TX; ++j) tot[i][j] = fin[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int chunks = (K + F32_CHUNK - 1) / F32_CHUNK, runs = f32_runs(chunks);
  const int tiles = (K + BK - 1) / BK;
  int run = 0;
  // a chunk's sums into its run's, and the run's into the whole when it ends
  const auto add_chunk = [&](int chunk, const f32x4_t (&acc)[TY][TX]) {
#pragma unroll
    for (int i = 0; i < TY; ++i)
#pragma unroll
      for (int j = 0; j < TX; ++j) tot[i][j] += acc[i][j];
    while (run < runs && f32_run_start(run + 1, runs, chunks) <= chunk) ++run;
    if (f32_run_start(run + 1, runs, chunks) == chunk + 1) {   // the run ends with this chunk
#pragma unroll
      for (int i = 0; i < TY; ++i)
#pragma unroll
        for (int j = 0; j < TX; ++j) {
          fin[i][j] += tot[i][j];
          tot[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
  };
  f32x4_t av[2][TY], wv[2][TX];
  // the fragments of the 16 of K number s of the tile in buffer b
  const auto read = [&](int b, int s) {
#pragma unroll
    for (int i = 0; i < TY; ++i) {
      const int ra = wm + 16 * i + r;
      av[s & 1][i] = lds[b][0][ra * SLOTS + ((4 * s + q) ^ (ra & MIX))];
    }
#pragma unroll
    for (int j = 0; j < TX; ++j) {
      const int rw = wn + 16 * j + r;
      wv[s & 1][j] = lds[b][1][rw * SLOTS + ((4 * s + q) ^ (rw & MIX))];
    }
  };
  const auto multiply = [&](int s, f32x4_t (&acc)[TY][TX]) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < TY; ++i)
#pragma unroll
        for (int j = 0; j < TX; ++j)
          acc[i][j] = mfma_f32(av[s & 1][i][e], wv[s & 1][j][e], acc[i][j]);
  };
  if constexpr (DIRECT) {
    constexpr int STEPS = BK / 16;
    static_assert(F32_CHUNK == 2 * BK, "a chunk is a tile in either buffer");
    bring(0);
    bring(1);
    WAIT_LOADS_AND_LDS(LOADS_A_WAVE);                          // tile 0 is there
    __builtin_amdgcn_s_barrier();
    ORDER_FENCE();
    read(0, 0);
    for (int chunk = 0; chunk < chunks; ++chunk) {
      f32x4_t acc[TY][TX];
#pragma unroll
      for (int i = 0; i < TY; ++i)
#pragma unroll
        for (int j = 0; j < TX; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int t = 2 * chunk + u;
#pragma unroll
        for (int s = 0; s + 1 < STEPS; ++s) {
          read(u, s + 1);
          __builtin_amdgcn_sched_barrier(0);
          multiply(s, acc);
          __builtin_amdgcn_sched_barrier(0);
        }
        // The tile's last fragments are in registers: its buffer takes the tile after the next, and the
        // next one's first fragments come while the last of this one are multiplied.  (Behind the last tile
        // too: what is read there is not used, but a branch would have the products wait for it.)
        ORDER_FENCE();
        WAIT_LOADS_AND_LDS(0);
        __builtin_amdgcn_s_barrier();
        ORDER_FENCE();
        if (t + 2 < tiles) bring(t + 2);
        read(u ^ 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(STEPS - 1, acc);
        __builtin_amdgcn_sched_barrier(0);
      }
      add_chunk(chunk, acc);
    }
  } else {
    fetch(0);
    keep(0);
    __syncthreads();
    for (int chunk = 0; chunk < chunks; ++chunk) {
      f32x4_t acc[TY][TX];
#pragma unroll
      for (int i = 0; i < TY; ++i)
#pragma unroll
        for (int j = 0; j < TX; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < F32_CHUNK / BK; ++u) {
        const int t = chunk * (F32_CHUNK / BK) + u;
        if (LOADS != F32_WHOLE && t >= tiles) break;
        fetch(min(t + 1, tiles - 1));                  // (the last tile once more, unused)
        __builtin_amdgcn_sched_barrier(0);             // (left alone, the loads sink to their use)
        read(t & 1, 0);
#pragma unroll
        for (int s = 0; s < BK / 16; ++s) {
          if (LOADS != F32_WHOLE && t * BK + 16 * s >= K) break;
          if (s + 1 < BK / 16) read(t & 1, s + 1);
          __builtin_amdgcn_sched_barrier(0);
          multiply(s, acc);
          __builtin_amdgcn_sched_barrier(0);
        }
        keep(t + 1);
        __syncthreads();
      }
      add_chunk(chunk, acc);
    }
  }
  if constexpr (GATED) {
    const int n = n0 + wn / 2 + r;
    if (n >= N) return;
    const float bg = bias ? bias[n] : 0.f, bu = bias ? bias[N + n] : 0.f;
#pragma unroll
    for (int i = 0; i < TY; ++i)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int m = m0 + wm + 16 * i + 4 * q + x;
        if (m < M) C[(size_t)m * ldc + n] = f32_gate(fin[i][0][x] + bg, fin[i][TX - 1][x] + bu);
      }
    return;
  }
#pragma unroll
  for (int j = 0; j < TX; ++j) {
    const int n = n0 + wn + 16 * j + r;
    if (n >= N) continue;
    const float b = bias ? bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < TY; ++i)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int m = m0 + wm + 16 * i + 4 * q + x;
        if (m < M) C[(size_t)m * ldc + n] = fin[i][j][x] + b;
      }
  }
}

template <int LOADS, int TY, int TX, bool GATED = false>
static void launch_f32_blocks(const float* A, const float* W, const float* bias, float* C, int M,
                              int N, int K, int lda, int ldc, hipStream_t stream) {
  constexpr int B = 32 * TY;
  const int tm = (M + B - 1) / B, tn = ((GATED ? 2 : 1) * N + B - 1) / B;
  const dim3 grid((tn + 7) / 8 * 8 * tm);
  // (offsets of 32 bits within either operand)
  if constexpr (LOADS == F32_WHOLE)
    if ((size_t)M * lda < 1u << 30 && (size_t)(GATED ? 2 : 1) * N * K < 1u << 30) {
      hipLaunchKernelGGL((gemm_f32_block_kernel<2, 4, TY, TX, 64, LOADS, GATED, true>), grid, dim3(512), 0, stream,
                         A, W, bias, C, M, N, K, lda, ldc, tm);
      return;
    }
  hipLaunchKernelGGL((gemm_f32_block_kernel<2, 4, TY, TX, 64, LOADS, GATED>), grid, dim3(512), 0, stream, A, W, bias,
                     C, M, N, K, lda, ldc, tm);
}

static bool f32_large_blocks(int M, int N) {
  const auto tiles = [](int n, int b) { return (n + b - 1) / b; };
  const long big = (long)tiles(M, 128) * tiles(N, 128), small = (long)tiles(M, 64) * tiles(N, 64);
  return (big + 255) / 256 * 4 * 8 <= (small + 255) / 256 * 9;
}

static bool f32_one(int M, int K) { return M <= 4 && K <= 8 * F32_CHUNK; }

template <int LOADS>
static void launch_f32_gated(const float* A, const float* W, const float* bias, float* C, int M, int F, int K,
                             int lda, int ldc, hipStream_t stream) {
  if (M > 64) {
    launch_f32_blocks<LOADS, 4, 2, true>(A, W, bias, C, M, F, K, lda, ldc, stream);
    return;
  }
  const bool many = f32_runs((K + F32_CHUNK - 1) / F32_CHUNK) == 32, one = f32_one(M, K);
#define F32_GATED(MT, RUNS, ...)                                                                     \
  hipLaunchKernelGGL((gemm_f32_skinny_kernel<MT, 16, RUNS, LOADS, true, ##__VA_ARGS__>), dim3((F + 7) / 8), \
                     dim3(8 * WAVE), 0, stream, A, W, bias, C, M, F, K, lda, ldc, 0, (const float*)nullptr, 0.f)
  if (M <= 16) {
    if (many) F32_GATED(1, 32);
    else if (LOADS == F32_WHOLE && one) F32_GATED(1, 8, false, LOADS == F32_WHOLE);
    else F32_GATED(1, 8);
  } else if (M <= 32) {
    if (many) F32_GATED(2, 32);
    else F32_GATED(2, 8);
  } else {
    if (many) F32_GATED(4, 32);
    else F32_GATED(4, 8);
  }
#undef F32_GATED
}

// add (up to 64 rows): to what C holds
template <int LOADS>
static void launch_f32(const float* A, const float* W, const float* bias, float* C, int M, int N,
                       int K, int lda, int ldc, hipStream_t stream, int add = 0) {
  if (M <= 64) {
    const bool many = f32_runs((K + F32_CHUNK - 1) / F32_CHUNK) == 32, one = f32_one(M, K);
#define F32_SKINNY(MT, COLS, RUNS, ...)                                                           \
  hipLaunchKernelGGL((gemm_f32_skinny_kernel<MT, COLS, RUNS, LOADS, false, ##__VA_ARGS__>), dim3((N + COLS - 1) / COLS), \
                     dim3((COLS < 16 ? RUNS * COLS / 16 : 8) * WAVE), 0, stream, A, W, bias, C, M, N, K,   \
                     lda, ldc, add, (const float*)nullptr, 0.f)
    if (M <= 4 && N <= 256 * 4) {
      if (many) F32_SKINNY(1, 4, 32);
      else F32_SKINNY(1, 4, 8);
    } else if (M <= 8 && N <= 256 * 8) {
      if (many) F32_SKINNY(1, 8, 32);
      else F32_SKINNY(1, 8, 8);
    } else if (M <= 16) {
      if (many) F32_SKINNY(1, 16, 32);
      else if (LOADS == F32_WHOLE && one) F32_SKINNY(1, 16, 8, false, LOADS == F32_WHOLE);
      else F32_SKINNY(1, 16, 8);
    } else if (M <= 32) {
      if (many) F32_SKINNY(2, 16, 32);
      else F32_SKINNY(2, 16, 8);
    } else {
      if (many) F32_SKINNY(4, 16, 32);
      else F32_SKINNY(4, 16, 8);
    }
#undef F32_SKINNY
    return;
  }
  if (f32_large_blocks(M, N))
    launch_f32_blocks<LOADS, 4, 2>(A, W, bias, C, M, N, K, lda, ldc, stream);
  else
    launch_f32_blocks<LOADS, 2, 1>(A, W, bias, C, M, N, K, lda, ldc, stream);
}

// Rows and columns of any number and any K.
extern "C" int kappai_gemm_f32(const float* A, const float* W, const float* bias, float* C, int M,
                               int N, int K, int lda, int ldc, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  const bool fours = K % 4 == 0 && lda % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
  if (K < 4) launch_f32_blocks<F32_FEW, 2, 1>(A, W, bias, C, M, N, K, lda, ldc, stream);  // (0 too)
  else if (fours && K % F32_CHUNK == 0) launch_f32<F32_WHOLE>(A, W, bias, C, M, N, K, lda, ldc, stream);
  else if (fours) launch_f32<F32_FOURS>(A, W, bias, C, M, N, K, lda, ldc, stream);
  else launch_f32<F32_ELEMENTS>(A, W, bias, C, M, N, K, lda, ldc, stream);
  KAPPAI_RETURN_LAUNCH_STATUS();
}

extern "C" int kappai_gemm_f32_gates(int M, int F, int K);
// The two ends of a decode step's products that save the norm's kernel between them.
// kappai_gemm_f32_add: C += A W^T (+ bias), up to 64 rows, the bits of the product and a sum behind it.
extern "C" int kappai_gemm_f32_add(const float* A, const float* W, const float* bias, float* C, int M, int N, int K,
                                   int lda, int ldc, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || K < 4) return (int)hipErrorInvalidValue;
  const bool fours = K % 4 == 0 && lda % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
  if (fours && K % F32_CHUNK == 0) launch_f32<F32_WHOLE>(A, W, bias, C, M, N, K, lda, ldc, stream, 1);
  else if (fours) launch_f32<F32_FOURS>(A, W, bias, C, M, N, K, lda, ldc, stream, 1);
  else launch_f32<F32_ELEMENTS>(A, W, bias, C, M, N, K, lda, ldc, stream, 1);
  KAPPAI_RETURN_LAUNCH_STATUS();
}
// kappai_gemm_f32_normed: the product, or with `gated` silu(gate) up over 2 N rows of W, of the RMS-normed rows of x
// [M, K], the bits of the norm's kernel and the product behind it.  For rows that kappai_gemm_f32_norms takes: up to
// 8 and 16 turns of 512 values (8 rows of 1,024, 4 of 2,048; every block norms all of them), whole chunks of K.
extern "C" int kappai_gemm_f32_norms(int M, int K) {
  return M >= 1 && M <= 8 && K >= F32_CHUNK && K <= 16 * F32_CHUNK && K % F32_CHUNK == 0 &&
         M * ((K + 511) / 512) <= F32_NORM_TURNS;
}
extern "C" int kappai_gemm_f32_normed(const float* x, const float* norm_w, float eps, const float* W,
                                      const float* bias, float* C, int M, int N, int K, int ldc, int gated,
                                      hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (!kappai_gemm_f32_norms(M, K) || ((uintptr_t)x | (uintptr_t)W | (uintptr_t)norm_w) % 16 ||
      (gated && !kappai_gemm_f32_gates(M, N, K)))
    return (int)hipErrorInvalidValue;
  const size_t lds = (size_t)M * (K + F32_ROW_PAD) * sizeof(float);       // (up to 33 KB)
#define F32_NORMED(COLS, GATED, BLOCK, ONE)                                                             \
  hipLaunchKernelGGL((gemm_f32_skinny_kernel<1, COLS, 8, F32_WHOLE, GATED, true, ONE>),                 \
                     dim3((N + BLOCK - 1) / BLOCK), dim3((COLS == 8 ? 4 : 8) * WAVE), lds, stream, x, W, \
                     bias, C, M, N, K, K, ldc, 0, norm_w, eps)
  const bool one = f32_one(M, K);
  if (gated && one) F32_NORMED(16, true, 8, true);
  else if (gated) F32_NORMED(16, true, 8, false);
  else if (N <= 256 * 8) F32_NORMED(8, false, 8, false);
  else if (one) F32_NORMED(16, false, 16, true);
  else F32_NORMED(16, false, 16, false);
#undef F32_NORMED
  KAPPAI_RETURN_LAUNCH_STATUS();
}

// C[m, f] = silu(A W_f) (A W_{F + f}) over the 2 F rows of W: the bits of kappai_gemm_f32 and kappai_swiglu,
// whose results of 2 F columns neither are written nor read again.  For the sizes whose plain product takes
// kernels with both rows of a result in one wave (kappai_gemm_f32_gates; else hipErrorInvalidValue): up to 64
// rows wherever a block owns 16 rows of W, beyond wherever the 128 x 128 blocks run.
extern "C" int kappai_gemm_f32_gates(int M, int F, int K) {
  if (M <= 0 || F <= 0 || K < 4) return 0;
  return M <= 64 ? (M > 8 || F > 128 * 8) : f32_large_blocks(M, 2 * F);
}
extern "C" int kappai_gemm_f32_swiglu(const float* A, const float* W, const float* bias, float* C, int M,
                                      int F, int K, int lda, int ldc, hipStream_t stream) {
  if (M <= 0 || F <= 0) return 0;
  if (!kappai_gemm_f32_gates(M, F, K)) return (int)hipErrorInvalidValue;
  const bool fours = K % 4 == 0 && lda % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
  if (fours && K % F32_CHUNK == 0) launch_f32_gated<F32_WHOLE>(A, W, bias, C, M, F, K, lda, ldc, stream);
  else if (fours) launch_f32_gated<F32_FOURS>(A, W, bias, C, M, F, K, lda, ldc, stream);
  else launch_f32_gated<F32_ELEMENTS>(A, W, bias, C, M, F, K, lda, ldc, stream);
  KAPPAI_RETURN_LAUNCH_STATUS();
}
#endif  // GATE_ACT == 0

// ---------------------------------------------------------------------------------------
// bf16 on the matrix cores
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ u32x4_t load16(const bf16_t* p) {
  return *reinterpret_cast<const u32x4_t*>(p);
}
__device__ __forceinline__ bf16x8_t as_bf16x8(u32x4_t v) {
  return __builtin_bit_cast(bf16x8_t, v);
}
__device__ __forceinline__ void store_out(float* p, float v) { *p = v; }
__device__ __forceinline__ void store_out(bf16_t* p, float v) { *p = f32_to_bf16(v); }

// silu(g) = g / (1 + e^-g) for the epilogues that store bfloat16: the hardware's 2^x and reciprocal
// (each good to about an ulp of float, far below a bfloat16's rounding) instead of expf and a
// division, which were 9 of the 132 us of gate/up at 2048 rows.  e^-g overflows to infinity for
// g < -88: the reciprocal is then 0 and the result -0, as it should be.
// GATE_ACT (a constant of the build) chooses what the gated epilogues pass the gate through:
// 0 silu; 1 the tanh form of gelu, 0.5 g (1 + tanh(a)) with a = sqrt(2/pi) (g + 0.044715 g^3),
// which is g * sigmoid(2 a) and so the same two instructions; 2 the clamped gate, g = min(g, limit),
// u = clamp(u, -limit, limit), g sigmoid(slope g) (u + shift), whose three constants the gated
// epilogues read where the others find a bias; 3 silu behind biases, one float a row of W in W's own
// order, which are added to both sums first and rounded as a product with biases stores its results (the
// silu is then the two instructions of the other gates, a few 32-bit units off the division of the
// kernel of its own, before it is rounded to bfloat16)
// (with the gate a kernel of its own behind the product, a decode step of two rows paid 4.6 us more a
// layer at 9,216 rows of W, a prompt step of 1,900 rows 30).
#ifndef GATE_ACT
#define GATE_ACT 0
#endif
__device__ __forceinline__ float silu_f(float g) {
#if GATE_ACT == 1
  const float a2 = 1.5957691216057308f * (g + 0.044715f * g * g * g);
  return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * a2));
#else
  return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * g));
#endif
}

// What a gated epilogue makes of the sums of a gate row and an up row.
// `row`: the gate row's number in W (the up row stands 16 further).
__device__ __forceinline__ float gated_f(float g, float u, const float* __restrict__ consts,
                                         int row) {
#if GATE_ACT == 3
  // (rounded as a product with biases stores its results)
  g = to_f32(f32_to_bf16(g + consts[row]));
  u = to_f32(f32_to_bf16(u + consts[row + 16]));
#endif
#if GATE_ACT == 2
  const float limit = consts[0], slope = consts[1], shift = consts[2];
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * slope * g)) *
         (u + shift);
#else
  return silu_f(g) * u;
#endif
}

// Block = WAVES_M x WAVES_N waves, each owning (WM*32) x (WN*32) of the result as WM*WN
// accumulator tiles of 32x32: per 16 of K a wave reads WM+WN fragments from LDS for WM*WN
// matrix instructions, so large wave tiles keep LDS traffic below what the matrix cores
// consume.  Tiles of A (BM x BK) and W (BN x BK) go global -> registers -> LDS,
// double-buffered: the loads of tile k+1 are in flight while tile k is multiplied, one
// barrier a tile.
// Blocks are renumbered so that the blocks that run on one XCD (every eighth) work on
// neighbouring tiles and share their L2.
//
// EPI 1 (SwiGLU): W holds gate and up rows interleaved in groups of 16 (16 gate rows, the 16 up
// rows of the same columns, ...); the kernel writes silu(gate) * up, N/2 columns wide
// (kappai: src/backend/cpu/quants.h:369-371, src/recipe/builders.c:344-370).
// Block number -> (row tile, column tile).  Consecutive block numbers go to the 8 XCDs in
// turn, each with an L2 of its own.  An XCD is given a band of column tiles (an eighth of W, so
// that W is fetched from memory once) and walks it in groups of up to 8 x 8 tiles, row tiles
// fastest: the blocks that run on it at one time then share both their rows of A and their
// rows of W in its L2.
__device__ __forceinline__ int2 xcd_tile(int b, int tiles_m, int tiles_n) {
  constexpr int XCDS = 8, GROUP = 8;
  if (tiles_n % XCDS != 0) return make_int2(b / tiles_n, b % tiles_n);
  const int band = tiles_n / XCDS;             // column tiles of one XCD
  const int xcd = b % XCDS;
  int j = b / XCDS;                            // position in the XCD's own order
  const int per_group = GROUP * band;
  const int groups = (tiles_m + GROUP - 1) / GROUP;
  const int g = min(j / per_group, groups - 1);
  j -= g * per_group;
  const int gm = min(GROUP, tiles_m - g * GROUP);
  return make_int2(g * GROUP + j % gm, xcd * band + j / gm);
}

// The same for blocks over a W in fragment order, K ranges among the things to be placed, on a grid of one
// dimension: an XCD is given an equal run of the list of all blocks, ranges slowest, then groups of `group` row
// tiles, then columns, the rows of a group fastest.  What an XCD reads of A and W comes to it once over its
// link (0.7 to 0.8 TB/s) and then out of its L2, so its run should lie in as few ranges as it can and be as
// square as it can within them (xcd_group).  With a band of column tiles for each XCD, every range among
// them, each XCD took in all of A: down, 2048 x 8192, 417 rows in four ranges 88 MB over the links, 47 so.  us so
// and with bands, W from memory: that product 22.6 and 23.9, 2048 x 10752 26.3 and 28.9; 1024 x 4608 of 575
// rows in six ranges 11.9 and 13.9, of 1900 in four 24.0 and 28.9; 2048 x 8192 of 2048 rows in two 62.1 and 63.2;
// whole products 1 to 3 % less (gate/up 9216 x 1024 of 1900 rows 42.4 and 44.9).  `cut`: group + 65536 * ranges.
struct BlockPlace {
  int m, n, range;
};
__device__ __forceinline__ BlockPlace xcd_place(int tiles_m, int tiles_n, uint32_t cut) {
  constexpr uint32_t XCDS = 8;
  const uint32_t plane = tiles_m * tiles_n, ranges = cut >> 16, group = cut & 0xffff, total = plane * ranges;
  const uint32_t b = blockIdx.x, xcd = b % XCDS, tail = total % XCDS;
  uint32_t j = xcd * (total / XCDS) + (xcd < tail ? xcd : tail) + b / XCDS, g = 0;
  BlockPlace at;
  at.range = 0;
  if (ranges > 1) {
    at.range = j / plane;
    j -= at.range * plane;
  }
  if (group < (uint32_t)tiles_m) {
    g = j / (group * tiles_n);
    j -= g * (group * tiles_n);
  }
  const uint32_t left = tiles_m - g * group, gm = group < left ? group : left;
  at.n = j / gm;
  at.m = g * group + j - at.n * gm;
  return at;
}
// Row tiles of a group: the blocks that an XCD runs at one time read the fewest rows of A and W between them (even
// groups; of equals the larger, which reads W in fewer XCDs).  Over 118 products of 300 to 2,048 rows the group
// chosen so takes 1 % more than the best of all groups in sum.
static int xcd_group(int tiles_m, int tiles_n, int ranges, int rows, int cols) {
  const int share = (tiles_m * tiles_n * ranges + 7) / 8, at_once = share < 32 ? share : 32;
  int best = 1, best_cost = -1;
  for (int g = tiles_m < 32 ? tiles_m : 32; g > 0; --g) {
    const int groups = (tiles_m + g - 1) / g, even = (tiles_m + groups - 1) / groups;
    if (even != g) continue;
    const int cost = g * rows + (at_once + g - 1) / g * cols;
    if (best_cost < 0 || cost < best_cost) {
      best = g;
      best_cost = cost;
    }
  }
  return best;
}

template <typename TO, int EPI, int WAVES_M, int WAVES_N, int WM, int WN, int BK, int NBUF,
          int OCC>
__global__ __launch_bounds__(WAVES_M * WAVES_N * WAVE)
    __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void gemm_bf16_tile_kernel(
        const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
        const float* __restrict__ bias, TO* __restrict__ C, int M, int N, int K, int lda, int ldc,
        int tiles_n, int w_frag) {
  constexpr int BM = WAVES_M * WM * 32, BN = WAVES_N * WN * 32;
  constexpr int LDS_STRIDE = BK + 8;   // in bf16: rows stay 16-byte aligned, banks are spread
  constexpr int THREADS = WAVES_M * WAVES_N * WAVE;
  constexpr int CPR = BK / 8;                              // 16-byte chunks a row
  constexpr int A_CHUNKS = BM * CPR / THREADS;             // chunks a thread stages
  constexpr int W_CHUNKS = BN * CPR / THREADS;
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
  // LDS: the A tiles of the NBUF buffers, then their W tiles
  constexpr int A_TILE = BM * LDS_STRIDE, W_TILE = BN * LDS_STRIDE;
  const int tid = threadIdx.x;
  const int lane = tid % WAVE, wave = tid / WAVE;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  // block -> tile, XCD-aware
  const int2 tile = xcd_tile(blockIdx.x, gridDim.x / tiles_n, tiles_n);
  const int m0 = tile.x * BM, n0 = tile.y * BN;
  // gridDim.y > 1 splits K over blocks: block y writes its partial sums to C + y * M * ldc
  const int kblk = ((K + BK * (int)gridDim.y - 1) / (BK * (int)gridDim.y)) * BK;
  const int kbeg = blockIdx.y * kblk, kend = min(K, kbeg + kblk);
  C += (size_t)blockIdx.y * M * ldc;

  f32x16_t acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // Staging: a thread copies 16-byte chunks; consecutive lanes take consecutive chunks of a
  // row, so that a row's bytes are asked for by neighbouring lanes and coalesce.
  const u32x4_t zero = {0u, 0u, 0u, 0u};
  u32x4_t ra[A_CHUNKS], rw[W_CHUNKS];
  auto chunk_row = [&](int idx) { return idx / CPR; };
  auto chunk_col = [&](int idx) { return (idx % CPR) * 8; };
  auto fetch = [&](int k0) {
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) {
      const int idx = tid + c * THREADS;
      const int r = chunk_row(idx), gk = k0 + chunk_col(idx);
      ra[c] = (m0 + r < M && gk < kend) ? load16(A + (size_t)(m0 + r) * lda + gk) : zero;
    }
#pragma unroll
    for (int c = 0; c < W_CHUNKS; ++c) {
      const int idx = tid + c * THREADS;
      const int r = chunk_row(idx), gk = k0 + chunk_col(idx);
      // (w_frag: W in fragment order, see gemm_bf16_skinny_kernel: the chunk of row n0 + r at gk)
      const size_t wr = (size_t)(n0 + r);
      const bf16_t* wp = w_frag ? W + (wr / 16) * 16 * K + (size_t)(gk / 32) * 512 +
                                      (((gk % 32) / 8) * 16 + wr % 16) * 8
                                : W + wr * K + gk;
      rw[c] = (n0 + r < N && gk < kend) ? load16(wp) : zero;
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) {
      const int idx = tid + c * THREADS;
      *reinterpret_cast<u32x4_t*>(lds + buf * A_TILE + chunk_row(idx) * LDS_STRIDE +
                                  chunk_col(idx)) = ra[c];
    }
#pragma unroll
    for (int c = 0; c < W_CHUNKS; ++c) {
      const int idx = tid + c * THREADS;
      *reinterpret_cast<u32x4_t*>(lds + NBUF * A_TILE + buf * W_TILE +
                                  chunk_row(idx) * LDS_STRIDE + chunk_col(idx)) = rw[c];
    }
  };
  // While tile k is multiplied out of LDS, the loads of tile k+1 are in flight into registers;
  // after the products they are written to LDS: into the other buffer (NBUF 2, one barrier a
  // tile) or, after a barrier, into the same one (NBUF 1: half the LDS, so that two blocks fit
  // a CU even with long tiles, whose products give the loads more time to arrive).
  fetch(kbeg);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = kbeg; k0 < kend; k0 += BK) {
    const bool more = k0 + BK < kend;
    if (more) fetch(k0 + BK);
    const bf16_t* as =
        lds + buf * A_TILE + (wm * WM * 32 + lane % 32) * LDS_STRIDE + (lane / 32) * 8;
    const bf16_t* ws = lds + NBUF * A_TILE + buf * W_TILE +
                       (wn * WN * 32 + lane % 32) * LDS_STRIDE + (lane / 32) * 8;
    bf16x8_t a[2][WM], w[2][WN];
    auto frags = [&](int fb, int ks) {
#pragma unroll
      for (int i = 0; i < WM; ++i)
        a[fb][i] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(as + i * 32 * LDS_STRIDE + ks));
#pragma unroll
      for (int j = 0; j < WN; ++j)
        w[fb][j] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(ws + j * 32 * LDS_STRIDE + ks));
    };
    frags(0, 0);
#pragma unroll
    for (int s2 = 0; s2 < BK / 16; ++s2) {
      if (s2 + 1 < BK / 16) frags((s2 + 1) & 1, (s2 + 1) * 16);
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s2 & 1][i], w[s2 & 1][j],
                                                              acc[i][j], 0, 0, 0);
    }
    if (NBUF == 1) {
      __syncthreads();
      if (more) stage(0);
    } else {
      if (more) stage(buf ^ 1);
      buf ^= 1;
    }
    __syncthreads();
  }
  // D[m][n] of a 32x32 tile: lane holds column lane%32, rows 8*(v/4) + 4*(lane/32) + v%4
  if (EPI == 1) {
    // a 32-column tile is 16 gate columns and their 16 up columns: lane c < 16 holds gate,
    // lane c + 16 the matching up
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        const int c = lane % 32;
        const int gcol = n0 + (wn * WN + j) * 32;        // first interleaved column of the tile
        const int on = gcol / 2 + c;                     // output column for c < 16
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const float other = __shfl_xor(acc[i][j][v], 16, WAVE);
          const int gm = m0 + (wm * WM + i) * 32 + 8 * (v / 4) + 4 * (lane / 32) + v % 4;
          if (c < 16 && gm < M && gcol + c < N)
            store_out(C + (size_t)gm * ldc + on, gated_f(acc[i][j][v], other, bias, gcol + c));
        }
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int gn = n0 + (wn * WN + j) * 32 + lane % 32;
      if (gn >= N) continue;
      const float bv = (bias && blockIdx.y == 0) ? bias[gn] : 0.f;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int gm = m0 + (wm * WM + i) * 32 + 8 * (v / 4) + 4 * (lane / 32) + v % 4;
        if (gm < M) store_out(C + (size_t)gm * ldc + gn, acc[i][j][v] + bv);
      }
    }
}

template <typename TO, int EPI, int WAVES_M, int WAVES_N, int WM, int WN, int BK, int NBUF,
          int OCC>
static void launch_tile_cfg(const bf16_t* A, const bf16_t* W, const float* bias, TO* C, int M,
                            int n_rows_w, int K, int lda, int ldc, int ksplit,
                            hipStream_t stream, int w_frag = 0) {
  constexpr int BM = WAVES_M * WM * 32, BN = WAVES_N * WN * 32;
  constexpr size_t lds_bytes = (size_t)NBUF * (BM + BN) * (BK + 8) * sizeof(bf16_t);
  auto kern = gemm_bf16_tile_kernel<TO, EPI, WAVES_M, WAVES_N, WM, WN, BK, NBUF, OCC>;
  static bool attr_set = false;       // more than 64 KB of LDS has to be asked for once
  if (!attr_set) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds_bytes);
    attr_set = true;
  }
  const int tn = (n_rows_w + BN - 1) / BN, tm = (M + BM - 1) / BM;
  hipLaunchKernelGGL(kern, dim3(tm * tn, ksplit), dim3(WAVES_M * WAVES_N * WAVE), lds_bytes,
                     stream, A, W, bias, C, M, n_rows_w, K, lda, ldc, tn, w_frag);
}

// ---------------------------------------------------------------------------------------
// 256 x 256 blocks for large products (prefill)
// ---------------------------------------------------------------------------------------
// Four waves, one on each SIMD, each owning 128 x 128 of the result as 4 x 4 accumulator tiles
// (256 accumulator registers): per 16 of K a wave reads 8 fragments from LDS for 16 matrix
// instructions.  Tiles of 64 of K (128-byte rows, whole cache lines) go from global memory
// straight into LDS (global_load_lds), two buffers; the 16-byte chunks of a row are permuted
// by (chunk ^ (row / 2) % 8) on the way in, so that the 16 lanes of a fragment read (16 rows,
// one chunk each) fall on 16 different 16-byte bank groups without padding.  The order of LDS reads, loads and matrix instructions is written out slot by slot
// and fenced, one wave has to hide every latency by itself: while the products of one 16 of K
// run, the fragments of the next are read; the loads of tile k+2 are issued as soon as the
// barrier of tile k has shown that everybody is done with its buffer.
//
// The matrix instruction takes the W fragment as its first operand: a lane then holds one row
// of C and 4 consecutive columns per register group, which the epilogue packs, transposes
// through LDS and stores as whole 16-byte chunks of rows (the SwiGLU pairs gate and up in one
// lane: registers v and v + 8).
//
// Host side guarantees: K / gridDim.y is a multiple of 128, rows of W a multiple of 8 (32 with
// SwiGLU), C and its row stride 16-byte aligned, M * lda and N * K below 2^31 elements.
template <int N> struct IntC { static constexpr int value = N; };

// The block products' epilogue: a wave turns 32 rows of its tile at a time through its own piece of LDS.
// acc[i][j][4g + e] is C[row (wm*WTM+i)*32 + lane%32][column (wn*WTN+j)*32 + 8g + 4*(lane/32) + e].
template <typename TO, int EPI, int WTM, int WTN>
__device__ __forceinline__ void block_epilogue(const f32x16_t (&acc)[WTM][WTN], bf16_t* lds,
                                               const float* bias, TO* C, int M, int N, int ldc, int m0,
                                               int n0, int range, int wave, int lane) {
  const int wm = wave / 2, wn = wave % 2, r_in = lane % 32, hh = lane / 32;
  constexpr int WROWS_N = WTN * 32;
  constexpr int OUT_COLS = EPI == 1 ? WROWS_N / 2 : WROWS_N;   // columns a wave writes
  constexpr int ROW_BYTES = OUT_COLS * (int)sizeof(TO) + 16;
  char* mine = reinterpret_cast<char*>(lds) + wave * 32 * ROW_BYTES;
  const int out_n = EPI == 1 ? N / 2 : N;
  const int col0 = EPI == 1 ? (n0 + wn * WROWS_N) / 2 : n0 + wn * WROWS_N;
#pragma unroll
  for (int i = 0; i < WTM; ++i) {
    char* wrow = mine + r_in * ROW_BYTES;
#pragma unroll
    for (int j = 0; j < WTN; ++j) {
#pragma unroll
      for (int g = 0; g < (EPI == 1 ? 2 : 4); ++g) {
        float v4[4];
        int c;                                   // first of the 4 columns, within the wave's
        if (EPI == 1) {
          c = j * 16 + 8 * g + 4 * hh;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            // (columns past the end are not stored: any row that is there)
            v4[e] = gated_f(acc[i][j][4 * g + e], acc[i][j][4 * g + 8 + e], bias,
                            min(n0 + wn * WROWS_N + j * 32 + 8 * g + 4 * hh + e, N - 17));
        } else {
          c = j * 32 + 8 * g + 4 * hh;
#pragma unroll
          for (int e = 0; e < 4; ++e) v4[e] = acc[i][j][4 * g + e];
          if (bias && range == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (col0 + c + e < out_n) v4[e] += bias[col0 + c + e];
          }
        }
        if (sizeof(TO) == 2) {
          uint2 pk;
          pk.x = pack_bf16x2(v4[0], v4[1]);
          pk.y = pack_bf16x2(v4[2], v4[3]);
          *reinterpret_cast<uint2*>(wrow + c * 2) = pk;
        } else {
          *reinterpret_cast<float4*>(wrow + c * 4) = make_float4(v4[0], v4[1], v4[2], v4[3]);
        }
      }
    }
    // rows back out, 16 bytes a lane
    constexpr int CHUNKS = OUT_COLS * (int)sizeof(TO) / 16;   // per row
    constexpr int ROWS_PER = WAVE / CHUNKS;                   // (lanes left over sit out)
    constexpr int PER = 16 / (int)sizeof(TO);                 // columns a chunk
    constexpr bool EVEN = WAVE % CHUNKS == 0 && 32 % ROWS_PER == 0;
#pragma unroll
    for (int it = 0; it < (32 + ROWS_PER - 1) / ROWS_PER; ++it) {
      const int rr = it * ROWS_PER + lane / CHUNKS, ch = lane % CHUNKS;
      if (!EVEN && (lane >= ROWS_PER * CHUNKS || rr >= 32)) continue;
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(mine + rr * ROW_BYTES + ch * 16);
      const int gm = m0 + (wm * WTM + i) * 32 + rr, gn = col0 + ch * PER;
      if (gm < M && gn < out_n) *reinterpret_cast<u32x4_t*>(C + (size_t)gm * ldc + gn) = v;
    }
  }
}

template <typename TO, int EPI, int WT, bool DEEP = false, int WN_ = 0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4 / WT, 4 / WT)))
void gemm_bf16_block256_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                               const float* __restrict__ bias, TO* __restrict__ C, int M, int N,
                               int K, int lda, int ldc, int tiles_n) {
  // WTM x WTN accumulator tiles of 32 x 32 a wave (WTN = WT unless WN_ is given): 4 x 4 ->
  // 256 x 256 blocks, 2 x 2 -> 128 x 128, 4 x 3 -> 256 rows x 192 columns (for a product whose
  // 256 x 256 blocks would leave a quarter of the chip without one)
  constexpr int WTM = WT, WTN = WN_ ? WN_ : WT;
  static_assert(!DEEP || (WTM == 2 && WTN == 2), "four LDS buffers: the 128 x 128 form only");
  static_assert(WTN <= WTM && 2 * WTN >= WTM, "the load slots are laid out for the rows' side");
  constexpr int BM = WTM * 64, BN = WTN * 64, BK = 64;
  constexpr int WROWS_M = WTM * 32, WROWS_N = WTN * 32;        // rows, columns of a wave's tile
  constexpr int NPROD = WTM * WTN, NREAD = WTM + WTN;          // per 16 of K
  // load instructions a wave and tile: the waves that bring A issue NLOAD, those that bring W
  // the first NLOAD_W of the same slots
  constexpr int NLOAD = 4 * WTM, NLOAD_W = 4 * WTN, HALF = NLOAD / 2;
  constexpr int A_TILE = BM * BK, BUF = (BM + BN) * BK;        // in bf16
  extern __shared__ __attribute__((aligned(1024))) bf16_t lds[];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wm = wave / 2, wn = wave % 2;
  const int2 tile = xcd_tile(blockIdx.x, gridDim.x / tiles_n, tiles_n);
  const int m0 = tile.x * BM, n0 = tile.y * BN;
  const int kblk = K / (int)gridDim.y;
  const int nk = kblk / BK;
  C += (size_t)blockIdx.y * M * ldc;

  f32x16_t acc[WTM][WTN];
#pragma unroll
  for (int i = 0; i < WTM; ++i)
#pragma unroll
    for (int j = 0; j < WTN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // One load instruction = 8 rows x 128 bytes: lane -> (row lane/8, LDS chunk lane%8), which
  // receives the row's chunk (lane%8) ^ ((row/2)%8).  Waves 0, 1 bring the A tile, waves 2, 3 the W
  // tile, NLOAD instructions each; rows past the end of the matrix repeat its last row (their
  // products are never stored).
  const bool brings_a = wave < 2;
  const char* gk = reinterpret_cast<const char*>(brings_a ? A : W) +
                   (size_t)blockIdx.y * kblk * sizeof(bf16_t);
  const int ld = brings_a ? lda : K;
  const int last_row = (brings_a ? M : N) - 1;
  const int row0 = brings_a ? m0 + wave * WROWS_M : n0 + (wave - 2) * WROWS_N;
  const int lds_row0 = brings_a ? wave * WROWS_M : BM + (wave - 2) * WROWS_N;   // in the buffer
  const int my_loads = brings_a ? NLOAD : NLOAD_W;
  const int lrow = lane / 8;
  uint32_t roff[NLOAD];
#pragma unroll
  for (int i = 0; i < NLOAD; ++i) {
    const int lchunk = (lane % 8) ^ (((i * 8 + lrow) >> 1) & 7);
    roff[i] = (uint32_t)(min(row0 + i * 8 + lrow, last_row) * ld + lchunk * 8) *
              (uint32_t)sizeof(bf16_t);
  }
  constexpr uint32_t kstep = BK * sizeof(bf16_t);    // bytes from one tile of 64 of K to the next
  // the address of a load is a wave-uniform 64-bit base (the tile's first column) plus the
  // lane's 32-bit row offset; pinning the base into scalar registers keeps the compiler from
  // folding the two into sixteen 64-bit per-lane pointers
  auto tile_base = [&](int kt) {
    const uint64_t p = reinterpret_cast<uint64_t>(gk) + (uint64_t)kt * kstep;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)p);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
    return reinterpret_cast<const char*>(((uint64_t)hi << 32) | lo);
  };
  auto load_one = [&](int buf, const char* base, int i) {
    if (NLOAD_W < NLOAD && i >= my_loads) return;       // (uniform over the wave)
    __builtin_amdgcn_global_load_lds(KAPPAI_GPTR(base + roff[i]),
                                     KAPPAI_LPTR(lds + buf * BUF + (lds_row0 + i * 8) * BK), 16,
                                     0, 0);
  };
  // fragments of the 16 of K number s: chunks 2s and 2s+1; lane -> (row lane%32, chunk 2s+lane/32)
  const int r_in = lane % 32, hh = lane / 32;
  int aoff[4], woff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    aoff[s] = (wm * WROWS_M + r_in) * BK + (((s * 2 + hh) ^ ((r_in >> 1) & 7)) * 8);
    woff[s] = A_TILE + (wn * WROWS_N + r_in) * BK + (((s * 2 + hh) ^ ((r_in >> 1) & 7)) * 8);
  }
  bf16x8_t fa[2][WTM], fw[2][WTN];
  // in the order the products ask for them: w0 a0, the other w, the other a
  auto read_one = [&](int fb, int buf, int s, int idx) {
    const bool is_w = idx == 0 || (idx >= 2 && idx <= WTN);
    const int n = idx <= 1 ? 0 : idx <= WTN ? idx - 1 : idx - WTN;
    if (is_w)
      fw[fb][n] = as_bf16x8(
          *reinterpret_cast<const u32x4_t*>(lds + buf * BUF + woff[s] + n * 32 * BK));
    else
      fa[fb][n] = as_bf16x8(
          *reinterpret_cast<const u32x4_t*>(lds + buf * BUF + aoff[s] + n * 32 * BK));
  };
  auto product = [&](int fb, int t) {
    const int i = t / WTN, j = t % WTN;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[fb][j], fa[fb][i], acc[i][j], 0, 0, 0);
  };
  // One tile of K out of buffer U.  next: there is a tile kt+1 (its second half is loaded
  // here, its first fragments are read at the end); next2: there is a tile kt+2 (its first
  // half is loaded into this tile's buffer once the barrier has passed).  Both are uniform.
  auto tile_step = [&](auto u_c, int kt, bool next, bool next2) {
    constexpr int U = decltype(u_c)::value;
    const char* base1 = tile_base(kt + 1);
    const char* base2 = tile_base(kt + 2);
#pragma unroll
    for (int s = 0; s < 3; ++s) {
#pragma unroll
      for (int t = 0; t < NPROD; ++t) {
        if (t < NREAD) read_one((s + 1) & 1, U, s + 1, t);
        if (s == 0 && t >= NPROD - HALF && next) load_one(U ^ 1, base1, HALF + t - (NPROD - HALF));
        product(s & 1, t);
        SCHED_FENCE();
      }
    }
    // the last 16 of K: a few products first, so that the matrix cores have work while the
    // wave waits at the barrier
    constexpr int PRE = WTM == 4 ? 4 : 1;
    constexpr int REST = NPROD - PRE;
    constexpr int SPREAD = REST < 8 ? REST : 8;         // slots that also read and load
    constexpr int READS_PER = (NREAD + SPREAD - 1) / SPREAD;
    constexpr int LOADS_PER = (HALF + SPREAD - 1) / SPREAD;
#pragma unroll
    for (int t = 0; t < PRE; ++t) {
      product(1, t);
      SCHED_FENCE();
    }
    if (next) {
      __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0): tile kt+1 has landed
      __builtin_amdgcn_s_barrier();
    }
    SCHED_FENCE();
#pragma unroll
    for (int t = PRE; t < NPROD; ++t) {
      const int k = t - PRE;
#pragma unroll
      for (int q = 0; q < READS_PER; ++q)
        if (k * READS_PER + q < NREAD && next) read_one(0, U ^ 1, 0, k * READS_PER + q);
#pragma unroll
      for (int q = 0; q < LOADS_PER; ++q)
        if (k * LOADS_PER + q < HALF && next2) load_one(U, base2, k * LOADS_PER + q);
      product(1, t);
      SCHED_FENCE();
    }
  };

  if constexpr (DEEP) {
    // Four LDS buffers, the block alone on its CU (128 KB): a 128 x 128 block's products of one
    // tile take about 0.2 us, far less than a tile's way from memory, so with two buffers a
    // block that has no neighbour on its CU waits for every tile (0.62 us each).  Here the loads
    // of tile kt+3 are issued while tile kt is multiplied: three tiles are under way.
    // Buffer of tile kt: kt % 4.  After the barrier of step kt-1 nobody reads tile kt-1's
    // buffer any more, which is where tile kt+3 goes.
    auto load_deep = [&](int kt, const char* base, int i) {
      __builtin_amdgcn_global_load_lds(
          KAPPAI_GPTR(base + roff[i]),
          KAPPAI_LPTR(lds + (kt & 3) * BUF + (lds_row0 + i * 8) * BK), 16, 0, 0);
    };
    auto read_deep = [&](int fb, const bf16_t* buf, int s, int idx) {
      const bool is_w = idx == 0 || (idx >= 2 && idx <= WTN);
      const int n = idx <= 1 ? 0 : idx <= WTN ? idx - 1 : idx - WTN;
      if (is_w)
        fw[fb][n] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(buf + woff[s] + n * 32 * BK));
      else
        fa[fb][n] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(buf + aoff[s] + n * 32 * BK));
    };
    const int pre = min(nk, 3);
    for (int p = 0; p < pre; ++p) {
      const char* base = tile_base(p);
#pragma unroll
      for (int i = 0; i < NLOAD; ++i) load_deep(p, base, i);
    }
    // tile 0 has landed when only the loads of the tiles after it are outstanding
    if (pre == 3)
      __builtin_amdgcn_s_waitcnt(0x4F70);         // vmcnt(16)
    else if (pre == 2)
      __builtin_amdgcn_s_waitcnt(0x0F78);         // vmcnt(8)
    else
      __builtin_amdgcn_s_waitcnt(0x0F70);         // vmcnt(0)
    __builtin_amdgcn_s_barrier();
    SCHED_FENCE();
#pragma unroll
    for (int t = 0; t < NREAD; ++t) read_deep(0, lds, 0, t);
    static_assert(NLOAD == 2 * NPROD, "one load a slot over the first two 16s of K");
    for (int kt = 0; kt < nk; ++kt) {
      const bf16_t* cur = lds + (kt & 3) * BUF;
      const bf16_t* nxt = lds + ((kt + 1) & 3) * BUF;
      const bool has1 = kt + 1 < nk, has2 = kt + 2 < nk, has3 = kt + 3 < nk;
      const char* base3 = tile_base(kt + 3);
#pragma unroll
      for (int s = 0; s < 3; ++s) {
#pragma unroll
        for (int t = 0; t < NPROD; ++t) {
          if (t < NREAD) read_deep((s + 1) & 1, cur, s + 1, t);
          if (s < 2 && has3) load_deep(kt + 3, base3, s * NPROD + t);
          product(s & 1, t);
          SCHED_FENCE();
        }
      }
      product(1, 0);
      SCHED_FENCE();
      if (has1) {
        // tile kt+1 has landed when only the loads of tiles kt+2 and kt+3 are outstanding
        if (has3)
          __builtin_amdgcn_s_waitcnt(0x4F70);     // vmcnt(16)
        else if (has2)
          __builtin_amdgcn_s_waitcnt(0x0F78);     // vmcnt(8)
        else
          __builtin_amdgcn_s_waitcnt(0x0F70);     // vmcnt(0)
        __builtin_amdgcn_s_barrier();
      }
      SCHED_FENCE();
#pragma unroll
      for (int t = 1; t < NPROD; ++t) {
        if (has1) {
          if (t == 1) {
            read_deep(0, nxt, 0, 0);
            read_deep(0, nxt, 0, 1);
          } else if (t == 2) {
            read_deep(0, nxt, 0, 2);
            read_deep(0, nxt, 0, 3);
          }
        }
        product(1, t);
        SCHED_FENCE();
      }
    }
  } else {
#pragma unroll
  for (int i = 0; i < NLOAD; ++i) load_one(0, tile_base(0), i);
#pragma unroll
  for (int i = 0; i < HALF; ++i) load_one(1, tile_base(1), i);
  __builtin_amdgcn_s_waitcnt(0x0F70 | HALF);    // vmcnt(HALF): tile 0 has landed
  __builtin_amdgcn_s_barrier();
  SCHED_FENCE();
#pragma unroll
  for (int t = 0; t < NREAD; ++t) read_one(0, 0, 0, t);

  // nk is even: the loop body is straight-line code for the accumulators (a conditional
  // second tile would merge two versions of all 256 of them)
  for (int kt = 0; kt < nk; kt += 2) {
    const bool more = kt + 2 < nk;
    tile_step(IntC<0>{}, kt, true, more);
    tile_step(IntC<1>{}, kt + 1, more, more);
  }
  }

  __syncthreads();                               // everybody is done with the last tile
  block_epilogue<TO, EPI, WTM, WTN>(acc, lds, bias, C, M, N, ldc, m0, n0, blockIdx.y, wave, lane);
}

// Block products whose W lies in fragment order ([rows / 16][K / 32] pieces of 16 rows x 32 of K, 1 KB
// each, the lane's 16 bytes at lane = (k % 32) / 8 * 16 + row % 16; see gemm_bf16_skinny_kernel).  Two
// kernels, four waves each, one a SIMD.  Rows of A and of W past the end are not stored; their offsets lie
// behind the buffer, or, where 32 bits run over, at some other row of it.
//
// The large blocks (256 x 256, 256 x 192) are bound by LDS and by the rate at which a CU takes in tiles
// (about 60 GB/s from memory, 85 from L2) more than by the matrix cores: with both operands in LDS a tile
// of 64 of K reads 128 KB from LDS and writes 64 KB into it, at 64 bytes a clock about 2,500 clocks beside
// 2,048 of matrix instructions.  Here W's fragments go from memory straight into registers, seven 16s of K
// ahead, and only A goes through LDS, three tiles ahead: 96 KB of LDS traffic a tile, at the price of 32 KB
// more taken in (two waves ask for the same pieces).  gate/up 16384 x 2048 of 2048 rows 112.4 us against
// 117.0 with both operands in LDS (1.22 PFLOP/s; the loop without loads takes 91.6: matrix instructions on
// real values run at 1.7 PFLOP/s), 9216 x 1024 of 1024 rows 26.4 against 29.2, in_proj 6144 x 2048 of 2048
// rows in 256 x 192 blocks 45.6 against 50.2.
//
// Loads return in order, so the waits count those behind the one that is waited for.  Per tile a wave
// issues WTN loads of W in each 16 of K and NA of A in the first two.  The wait for the next tile of A before
// the barrier is a formality: the products before it have waited for pieces of W that were asked for after it.
//
// Host side guarantees for both: K / gridDim.y is a multiple of 128, rows of W a multiple of 16 (32 with
// the gated epilogue), C and its row stride 16-byte aligned, M * lda and N * K below 2^31 elements.
template <typename TO, int EPI, int WTM, int WTN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_bf16_direct_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                             const float* __restrict__ bias, TO* __restrict__ C, int M, int N,
                             int K, int lda, int ldc, int tiles_m, int tiles_n, uint32_t cut) {
  constexpr int BM = WTM * 64, BN = WTN * 64, BK = 64, NB = 4, SLOTS = 8;
  constexpr int NPROD = WTM * WTN, NA = BM / 32;               // loads of A a wave and tile
  constexpr int A_TILE = BM * BK;                              // in bf16
  extern __shared__ __attribute__((aligned(1024))) bf16_t lds[];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wm = wave / 2, wn = wave % 2;
  const BlockPlace place = xcd_place(tiles_m, tiles_n, cut);
  const int m0 = place.m * BM, n0 = place.n * BN;
  const int kblk = cut >> 17 ? (int)((uint32_t)K / (cut >> 16)) : K;
  const int nk = kblk / BK;
  const int k0 = place.range * kblk;
  C += (size_t)place.range * M * ldc;

  f32x16_t acc[WTM][WTN];
#pragma unroll
  for (int i = 0; i < WTM; ++i)
#pragma unroll
    for (int j = 0; j < WTN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const bf16_t* a_from = A + k0;
  const bf16_t* w_from = W + (size_t)k0 * 16;
  const uint32_t a_bytes = (uint32_t)(M - 1) * (uint32_t)lda * 2u + (uint32_t)kblk * 2u;
  const uint32_t w_bytes = (uint32_t)N * (uint32_t)K * 2u - (uint32_t)k0 * 32u;
  const int lrow = lane / 8;
  uint32_t a_at[NA], w_at[WTN];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int lchunk = (lane % 8) ^ (((i * 8 + lrow) >> 1) & 7);
    a_at[i] = (uint32_t)(m0 + wave * (BM / 4) + i * 8 + lrow) * (uint32_t)lda * 2u + lchunk * 16u;
  }
  const int r_in = lane % 32, hh = lane / 32;
#pragma unroll
  for (int j = 0; j < WTN; ++j)
    w_at[j] = (uint32_t)((n0 + wn * WTN * 32 + j * 32) / 16 + r_in / 16) * 16u * (uint32_t)K * 2u +
              hh * 256u + (r_in % 16) * 16u;
  // (the fragments of the s-th 16 of K: chunks 2s and 2s + 1)
  const int aoff = (wm * WTM * 32 + r_in) * BK + ((hh ^ ((r_in >> 1) & 7)) * 8);

  auto load_a = [&](int kt, int i) {           // tile kt; nothing is read of a tile that is not there
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        raw_buffer(a_from, kt < nk ? a_bytes : 0u),
        KAPPAI_LPTR(lds + (kt & (NB - 1)) * A_TILE + (wave * (BM / 4) + i * 8) * BK), 16, a_at[i],
        kt * 128, 0, 0);
#endif
  };
  u32x4_t fw[SLOTS][WTN];
  auto load_w = [&](int slot, int kt, int s, int j) {
#if defined(__HIP_DEVICE_COMPILE__)
    fw[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(
        raw_buffer(w_from, kt < nk ? w_bytes : 0u), w_at[j] + s * 512, kt * 2048, 0);
#endif
  };
  bf16x8_t fa[2][WTM];
  auto read_a = [&](int fb, int kt, int s, int i) {
    fa[fb][i] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(lds + (kt & (NB - 1)) * A_TILE +
                                                            (aoff ^ (s * 16)) + i * 32 * BK));
  };
  auto product = [&](int fb, int slot, int t) {
    const int i = t / WTN, j = t % WTN;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(fw[slot][j]), fa[fb][i],
                                                        acc[i][j], 0, 0, 0);
  };
  constexpr int PRE = WTN > 2 ? 4 : 2;
  constexpr int OUT = 10 * WTN + 2 * NA;       // loads behind those of the next tile of A
  static_assert(OUT < 64 && PRE >= WTN, "");
  auto tile_step = [&](auto u_c, int kt) {
    constexpr int U = decltype(u_c)::value;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int ahead = s - 1 + SLOTS;           // the stage that the last stage's slot is for
#pragma unroll
      for (int t = 0; t < NPROD; ++t) {
        if (s == 3 && t == PRE) {
          WAIT_LOADS_AND_LDS(OUT);
          __builtin_amdgcn_s_barrier();
          SCHED_FENCE();
        }
        if (t < WTN) load_w((U * 4 + ahead) % SLOTS, kt + ahead / 4, ahead % 4, t);
        if (s < 2 && t >= NPROD - NA / 2) load_a(kt + 3, s * (NA / 2) + t - (NPROD - NA / 2));
        if (s < 3) {
          if (t < WTM) read_a((s + 1) & 1, kt, s + 1, t);
        } else if (t >= PRE && t < PRE + WTM) {
          read_a(0, kt + 1, 0, t - PRE);
        }
        product(s & 1, U * 4 + s, t);
        SCHED_FENCE();
      }
    }
  };
#pragma unroll
  for (int i = 0; i < NA; ++i) load_a(0, i);
  ORDER_FENCE();
#pragma unroll
  for (int i = 0; i < NA; ++i) load_a(1, i);
  ORDER_FENCE();
#pragma unroll
  for (int s = 0; s < SLOTS - 1; ++s) {
    if (s == 4) {
#pragma unroll
      for (int i = 0; i < NA; ++i) load_a(2, i);
      ORDER_FENCE();
    }
#pragma unroll
    for (int j = 0; j < WTN; ++j) load_w(s, s / 4, s % 4, j);
    ORDER_FENCE();
  }
  constexpr int FIRST = 2 * NA + (SLOTS - 1) * WTN;          // loads behind those of tile 0 of A
  WAIT_LOADS(FIRST);
  __builtin_amdgcn_s_barrier();
  ORDER_FENCE();
#pragma unroll
  for (int i = 0; i < WTM; ++i) read_a(0, 0, 0, i);
  int kt = 0;
  do {
    tile_step(IntC<0>{}, kt);
    tile_step(IntC<1>{}, kt + 1);
    kt += 2;
  } while (kt < nk);
#if defined(__HIP_DEVICE_COMPILE__)
  // (the sums stay in accumulation registers to the end of the loop: without this the gated form keeps
  // some of W's pieces in scratch memory)
#pragma unroll
  for (int i = 0; i < WTM; ++i)
#pragma unroll
    for (int j = 0; j < WTN; ++j) asm volatile("" : "+a"(acc[i][j]));
#endif
  // (the loads of tiles that are not there have ended too: the epilogue uses their LDS)
  WAIT_LOADS_AND_LDS(0);
  __syncthreads();
  block_epilogue<TO, EPI, WTM, WTN>(acc, lds, bias, C, M, N, ldc, m0, n0, place.range, wave, lane);
}

// The same product with both operands in LDS, NB buffers, for blocks whose tile is small beside what it
// has under way: 128 x 128, 192 x 128, 256 x 128.  A block has its CU to itself, the loads of tile
// kt + NB - 1 are spread over the first three 16s of tile kt (no branches: see raw_buffer), so NB - 1 tiles
// are under way.  These are bound by what a CU takes in, so the block that covers the product in one round
// with the fewest bytes wins (gemm_rules.h).  Against the forms before (128 x 128, two blocks a CU or four
// buffers), W from memory: gate/up 16384 x 2048 of 417 rows 31.2 us against 36.8, 9216 x 1024 of 575 rows
// 14.3 against 18.7; 3072 x 1024 of 575 rows 9.7 against 12.1; 2048 x 2048 of 417 rows in four ranges 9.6
// against 12.2, 2048 x 8192 in four 21.2 against 24.0; 3072 x 2048 of 2048 rows 27.6 against 32.3.
// Products that leave CUs without a block of 128 x 128 take 64 x 128, 128 x 64 or 64 x 64 (a wave's tile 32 rows or
// columns, six and five buffers): more CUs take in less each.  128 x 128 and the best of the three, us: 3072 x 1024
// of 575 rows 9.0 and 7.4 (216 blocks), 3072 x 2048 of 417 rows 15.4 and 11.6 (192), 1024 x 1024 of 575 rows 8.5 and
// 5.4 (144), 1024 x 4608 of 417 rows in two ranges 15.2 and 8.9 (224).  Of more blocks than CUs they are slower (2048 x
// 1024 of 1040 rows 9.3 and 10.6), with three buffers and two blocks a CU too (10.7).
template <typename TO, int EPI, int WTM, int WTN, int NB>
__global__ __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(1, NB * (WTM + WTN) * 8192 <= 80 * 1024 ? 2 : 1)))   // (as LDS has room for)
void gemm_bf16_staged_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                             const float* __restrict__ bias, TO* __restrict__ C, int M, int N,
                             int K, int lda, int ldc, int tiles_m, int tiles_n, uint32_t cut) {
  constexpr int BM = WTM * 64, BN = WTN * 64, BK = 64;
  constexpr int NPROD = WTM * WTN, NREAD = WTM + WTN;
  constexpr int NA = BM / 32, NW = BN / 32, NLOAD = NA + NW;   // loads a wave and tile
  constexpr int A_TILE = BM * BK, TILE = (BM + BN) * BK;       // in bf16
  extern __shared__ __attribute__((aligned(1024))) bf16_t lds[];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wm = wave / 2, wn = wave % 2;
  const BlockPlace place = xcd_place(tiles_m, tiles_n, cut);
  const int m0 = place.m * BM, n0 = place.n * BN;
  const int kblk = cut >> 17 ? (int)((uint32_t)K / (cut >> 16)) : K;
  const int nk = kblk / BK;
  const int k0 = place.range * kblk;
  C += (size_t)place.range * M * ldc;
  f32x16_t acc[WTM][WTN];
#pragma unroll
  for (int i = 0; i < WTM; ++i)
#pragma unroll
    for (int j = 0; j < WTN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  const bf16_t* a_from = A + k0;
  const bf16_t* w_from = W + (size_t)k0 * 16;
  const uint32_t a_bytes = (uint32_t)(M - 1) * (uint32_t)lda * 2u + (uint32_t)kblk * 2u;
  const uint32_t w_bytes = (uint32_t)N * (uint32_t)K * 2u - (uint32_t)k0 * 32u;
  const int lrow = lane / 8;
  uint32_t a_at[NA], w_at[NW];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int lchunk = (lane % 8) ^ (((i * 8 + lrow) >> 1) & 7);
    a_at[i] = (uint32_t)(m0 + wave * (BM / 4) + i * 8 + lrow) * (uint32_t)lda * 2u + lchunk * 16u;
  }
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int p = wave * NW + i;
    w_at[i] = (uint32_t)(n0 / 16 + p / 2) * 16u * (uint32_t)K * 2u + (p % 2) * 1024u + lane * 16u;
  }
  const int r_in = lane % 32, hh = lane / 32;
  const int aoff = (wm * WTM * 32 + r_in) * BK + ((hh ^ ((r_in >> 1) & 7)) * 8);
  const int woff = A_TILE + (wn * WTN * 4 + (r_in / 16) * 2) * 512 + (hh * 16 + r_in % 16) * 8;
  auto load = [&](int at, int kt, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
    if (i < NA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          raw_buffer(a_from, kt < nk ? a_bytes : 0u),
          KAPPAI_LPTR(lds + at + (wave * (BM / 4) + i * 8) * BK), 16, a_at[i < NA ? i : 0], kt * 128, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          raw_buffer(w_from, kt < nk ? w_bytes : 0u),
          KAPPAI_LPTR(lds + at + A_TILE + (wave * NW + i - NA) * 512), 16, w_at[i < NA ? 0 : i - NA],
          kt * 2048, 0, 0);
#endif
  };
  bf16x8_t fa[2][WTM], fw[2][WTN];
  auto read = [&](int fb, int at, int s, int n) {       // w0 a0, the other w, the other a
    const bool is_w = n == 0 || (n >= 2 && n <= WTN);
    const int x = n <= 1 ? 0 : n <= WTN ? n - 1 : n - WTN;
    if (is_w)
      fw[fb][x] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(
          lds + at + woff + (s / 2) * 512 + (s % 2) * 256 + x * 2048));
    else
      fa[fb][x] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(lds + at + (aoff ^ (s * 16)) + x * 32 * BK));
  };
  auto product = [&](int fb, int t) {
    const int i = t / WTN, j = t % WTN;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[fb][j], fa[fb][i], acc[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int b = 0; b < NB - 1; ++b)
#pragma unroll
    for (int i = 0; i < NLOAD; ++i) load(b * TILE, b, i);
  constexpr int BEHIND = (NB - 2) * NLOAD;
  static_assert(BEHIND < 64, "");
  WAIT_LOADS(BEHIND);
  __builtin_amdgcn_s_barrier();
  ORDER_FENCE();
#pragma unroll
  for (int n = 0; n < NREAD; ++n) read(0, 0, 0, n);
  constexpr int PRE = NPROD > 4 ? 2 : NPROD > 1 ? 1 : 0;
  constexpr int LOADS_AT = 3 * NPROD;                       // slots of the first three 16s of K
  int cur = 0, kt = 0;
  do {
    const int nxt = cur == (NB - 1) * TILE ? 0 : cur + TILE;
    const int into = cur == 0 ? (NB - 1) * TILE : cur - TILE;   // where the tile before this one lay
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int t = 0; t < NPROD; ++t) {
        if (s == 3 && t == PRE) {
          WAIT_LOADS_AND_LDS(BEHIND);
          __builtin_amdgcn_s_barrier();
          SCHED_FENCE();
        }
        if (s < 3) {
          constexpr int AT_ONCE = (NREAD + NPROD - 1) / NPROD;
#pragma unroll
          for (int q = 0; q < AT_ONCE; ++q)
            if (t * AT_ONCE + q < NREAD) read((s + 1) & 1, cur, s + 1, t * AT_ONCE + q);
          const int slot = s * NPROD + t;
          // NLOAD loads spread over the slots
#pragma unroll
          for (int i = slot * NLOAD / LOADS_AT; i < (slot + 1) * NLOAD / LOADS_AT; ++i) load(into, kt + NB - 1, i);
        } else if (t >= PRE) {
          constexpr int PER = (NREAD + NPROD - PRE - 1) / (NPROD - PRE);
#pragma unroll
          for (int q = 0; q < PER; ++q)
            if ((t - PRE) * PER + q < NREAD) read(0, nxt, 0, (t - PRE) * PER + q);
        }
        product(s & 1, t);
        SCHED_FENCE();
      }
    }
    cur = nxt;
    ++kt;
  } while (kt < nk);
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int i = 0; i < WTM; ++i)
#pragma unroll
    for (int j = 0; j < WTN; ++j) asm volatile("" : "+a"(acc[i][j]));   // (see the kernel above)
#endif
  WAIT_LOADS_AND_LDS(0);
  __syncthreads();
  block_epilogue<TO, EPI, WTM, WTN>(acc, lds, bias, C, M, N, ldc, m0, n0, place.range, wave, lane);
}

template <typename TO, int EPI>
static bool block256_fits(const bf16_t* A, const bf16_t* W, TO* C, int M, int n_rows_w, int K,
                          int lda, int ldc, int ksplit) {
  const long long limit = 1ll << 31;
  return K % (128 * ksplit) == 0 && n_rows_w % (EPI == 1 ? 32 : 8) == 0 &&
         ((uintptr_t)C % 16) == 0 && ((size_t)ldc * sizeof(TO)) % 16 == 0 &&
         (long long)M * lda < limit && (long long)n_rows_w * K < limit;
}

template <typename TO, int EPI, int WT, bool DEEP = false, int WN_ = 0>
static void launch_block256(const bf16_t* A, const bf16_t* W, const float* bias, TO* C, int M,
                            int n_rows_w, int K, int lda, int ldc, int ksplit,
                            hipStream_t stream) {
  constexpr int B = WT * 64, BN = (WN_ ? WN_ : WT) * 64;       // block: B rows x BN columns
  constexpr size_t lds_bytes = (DEEP ? 4 : 2) * (B + BN) * 64 * sizeof(bf16_t);
  auto kern = gemm_bf16_block256_kernel<TO, EPI, WT, DEEP, WN_>;
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds_bytes);
    attr_set = true;
  }
  const int tn = (n_rows_w + BN - 1) / BN, tm = (M + B - 1) / B;
  hipLaunchKernelGGL(kern, dim3(tm * tn, ksplit), dim3(256), lds_bytes, stream, A, W, bias, C, M,
                     n_rows_w, K, lda, ldc, tn);
}

template <typename TO, int EPI, int WTM, int WTN, int NB>
static void launch_fragment_block(const bf16_t* A, const bf16_t* Wf, const float* bias, TO* C, int M,
                                  int n_rows_w, int K, int lda, int ldc, int ksplit,
                                  hipStream_t stream) {
  constexpr int BM = WTM * 64, BN = WTN * 64;
  constexpr bool DIRECT = WTN > 2;
  // the tiles of A (and W), or what the epilogue turns its rows in
  constexpr size_t lds_bytes = NB * (BM + (DIRECT ? 0 : BN)) * 64 * sizeof(bf16_t);
  static_assert(4 * 32 * (WTN * 32 * 4 + 16) <= lds_bytes && lds_bytes <= 160 * 1024, "LDS");
  void (*kern)(const bf16_t*, const bf16_t*, const float*, TO*, int, int, int, int, int, int, int, uint32_t);
  if constexpr (DIRECT) kern = gemm_bf16_direct_kernel<TO, EPI, WTM, WTN>;
  else kern = gemm_bf16_staged_kernel<TO, EPI, WTM, WTN, NB>;
  static bool attr_set = false;       // more than 64 KB of LDS has to be asked for once
  if (!attr_set) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds_bytes);
    attr_set = true;
  }
  const int tn = (n_rows_w + BN - 1) / BN, tm = (M + BM - 1) / BM;
  const uint32_t cut = (uint32_t)xcd_group(tm, tn, ksplit, BM, BN) + 65536u * ksplit;
  hipLaunchKernelGGL(kern, dim3(tm * tn * ksplit), dim3(256), lds_bytes, stream, A, Wf, bias, C, M,
                     n_rows_w, K, lda, ldc, tm, tn, cut);
}

// shape: 0 = chosen by size, 1 = 128x128 blocks of two waves, 2 = 256x128 blocks (tiles of 32
// of K, two LDS buffers), 3 = 256x128 blocks (tiles of 64 of K, one LDS buffer), 4 = 256x256
// blocks of the same kernel (tiles of 64 of K), 5 = the 256x256 kernel with one wave a SIMD, 6 = its
// 128x128 form (when the sizes fit them, else 3), 8 = the 128x128 form with four LDS buffers, one
// block a CU, 9 = the one-wave-a-SIMD kernel with blocks of 256 rows x 192 columns, 11 = 192x128, 12 =
// 256x128, 13 = 64x128, 14 = 128x64, 15 = 64x64 (11 to 15 only with W in fragment order, else 6).  With W in
// fragment order 6 and 8 are one kernel, one block a CU with four buffers.
template <typename TO, int EPI>
static void launch_tile(const bf16_t* A, const bf16_t* W, const float* bias, TO* C, int M,
                        int n_rows_w, int K, int lda, int ldc, int ksplit, int shape,
                        hipStream_t stream, const bf16_t* Wf = nullptr) {
  const bool fits = EPI != 2 && block256_fits<TO, EPI>(A, W, C, M, n_rows_w, K, lda, ldc, ksplit);
  // Wf: W in fragment order (W may then be null)
  if constexpr (EPI != 2) {
    if (Wf != nullptr && fits && (shape == 0 || shape >= 5)) {
      if (shape == 0)
        shape = kappai_block_shape_for(M, n_rows_w, K, ksplit, sizeof(TO), EPI == 1);
#define KAPPAI_BLOCKS(...)                                                                         \
  launch_fragment_block<TO, EPI, __VA_ARGS__>(A, Wf, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream)
      if (shape == 9 && EPI != 0) shape = 5;
      if (shape == 5) KAPPAI_BLOCKS(4, 4, 4);
      else if (shape == 11) KAPPAI_BLOCKS(3, 2, 3);
      else if (shape == 12) KAPPAI_BLOCKS(4, 2, 3);
      else if (shape == 13) KAPPAI_BLOCKS(1, 2, 6);
      else if (shape == 14) KAPPAI_BLOCKS(2, 1, 6);
      else if (shape == 15) KAPPAI_BLOCKS(1, 1, 5);
      else if (shape != 9) KAPPAI_BLOCKS(2, 2, 4);
      else if constexpr (EPI == 0) KAPPAI_BLOCKS(4, 3, 4);
#undef KAPPAI_BLOCKS
      return;
    }
  }
  if (shape >= 11 && shape <= 15) shape = 6;
  if (shape == 0) {
    const int big = ((M + 255) / 256) * ((n_rows_w + 127) / 128) * ksplit;
    const int blocks256 = ((M + 255) / 256) * ((n_rows_w + 255) / 256) * ksplit;
    // the one-wave-a-SIMD kernel when its 256 x 256 blocks fill most of the chip, its
    // 128 x 128 forms below that (gemm_rules.h)
    const long blocks128 = (long)((M + 127) / 128) * ((n_rows_w + 127) / 128) * ksplit;
    const bool deep = kappai_deep_form(blocks128, K / ksplit);
    // (up to 128 rows a block of 256 rows would be half empty)
    shape = !fits ? (big >= 128 ? 3 : 1) : (M > 128 && kappai_use_256_form(blocks256)) ? 5 : deep ? 8 : 6;
    if (shape == 5 && EPI == 0) {
      // blocks of 256 rows x 192 columns when they fill their rounds and come to fewer rounds'
      // worth of work than 256 x 256 (in_proj of 2048 rows: 192 blocks of 256 x 256 leave 64 CUs
      // idle, 256 blocks of 256 x 192 none: 49 against 55 us).  Only against the 256 x 256 form:
      // where the 128 x 128 form was chosen (rows or columns that fill their last tiles badly, K
      // split into ranges) the 192 form was measured slower (2063 x 2048 x 7168: 88 against 74 us).
      const long blocks192 = (long)((M + 255) / 256) * ((n_rows_w + 191) / 192) * ksplit;
      const long r256 = (blocks256 + 255) / 256, r192 = (blocks192 + 255) / 256;
      if (kappai_use_256_form(blocks192) && r192 * (192 + 16) < r256 * (256 + 16)) shape = 9;
    }
  }
  if ((shape == 5 || shape == 6 || shape == 8 || shape == 9) && !fits) shape = 3;
  if (shape == 9 && EPI != 0) shape = 5;
  // The tile kernel reads fragment order a little slower than rows (47 against 43 us), so it takes the
  // rows when there are any.
  const int w_frag = Wf != nullptr && W == nullptr;
  if (w_frag) W = Wf;
  switch (shape) {
    case 5:
      if constexpr (EPI != 2)
        launch_block256<TO, EPI, 4>(A, W, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream);
      break;
    case 6:
      if constexpr (EPI != 2)
        launch_block256<TO, EPI, 2>(A, W, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream);
      break;
    case 8:
      if constexpr (EPI != 2)
        launch_block256<TO, EPI, 2, true>(A, W, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream);
      break;
    case 9:
      if constexpr (EPI == 0)
        launch_block256<TO, EPI, 4, false, 3>(A, W, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream);
      break;
    case 1:
      launch_tile_cfg<TO, EPI, 1, 2, 4, 2, 32, 2, 2>(A, W, bias, C, M, n_rows_w, K, lda, ldc, ksplit,
                                                  stream, w_frag);
      break;
    case 2:
      launch_tile_cfg<TO, EPI, 2, 2, 4, 2, 32, 2, 2>(A, W, bias, C, M, n_rows_w, K, lda, ldc, ksplit,
                                                  stream, w_frag);
      break;
    case 3:
      launch_tile_cfg<TO, EPI, 2, 2, 4, 2, 64, 1, 2>(A, W, bias, C, M, n_rows_w, K, lda, ldc, ksplit,
                                                  stream, w_frag);
      break;
    default:
      launch_tile_cfg<TO, EPI, 2, 2, 4, 4, 64, 2, 1>(A, W, bias, C, M, n_rows_w, K, lda, ldc, ksplit,
                                                  stream, w_frag);
      break;
  }
}

// M <= 16*MT (decode).  Bound by reading W once: a block owns 16 columns of the result and
// streams their 16 rows of W; its NW waves split K into contiguous ranges and meet in LDS.
// Every wave issues SK_UNROLL independent 16-byte loads of W per lane before it consumes
// them, so that enough bytes are in flight to keep HBM busy.  A fragment: lane holds row
// lane%16, k-group lane/16; W fragment: lane holds column lane%16, k-group lane/16; result:
// lane holds column lane%16, rows 4*(lane/16) + v.
#define SK_UNROLL 8

// FRAG (W in fragment order): what such a kernel takes beside the stream of W is what stands ahead of its
// first load and behind its last.  So a wave's loads are buffer loads at one lane offset and scalar steps,
// without conditions (what a lane must not read lies outside its buffer), the first loads need only
// arguments that are handed over in registers, and the row scales are summed by the waves that stream.  us
// of a product alone, W from memory, with conditions and an extra wave for the scales / so: 9216 x 1024
// gated 1 row 7.1 / 5.7, 16 rows 9.3 / 6.7, behind a folded norm 8.4 / 6.7 and 9.9 / 7.2 (8 rows); 16384 x 2048
// gated 8 rows 15.0 / 14.1; 6144 x 2048 8 rows 8.4 / 7.1; the conv step of 2048 channels 9.1 / 8.4; 24 rows of
// 9216 x 1024 gated 9.9 / 7.5.  Into the stream, 8 rows: 1024 x 1024 4.8 / 4.3, 2048 x 8192 13.5 / 11.3, 1 row of
// 2048 x 10752 13.6 / 11.9.  Not FRAG: W as rows, and offsets of more than 31 bits.

// EPI 1 (SwiGLU, see the tile kernel): a block owns 16 output columns = 16 gate rows and
// their 16 up rows of the interleaved W; N is the number of output columns.
// gridDim.y > 1 splits K over blocks as well: block (x, y) writes its partial sums to
// C + y * M * ldc (float), which the consumer adds up in a fixed order.
// EPI 2 (gated short convolution, one decoded row a request; kappai:
// src/backend/cpu/common.c:2393-2431): W is the conv layer's in_proj [3N, K]; a block owns 16
// channels and streams their B, C and x rows (N rows apart), then bx = B*x meets the request's
// state, the taps give s, the kernel writes C*s and shifts the state.
struct ConvStep {
  const float* taps;       // [N, L]
  const float* conv_bias;  // [N] or null
  float* state;            // [slots, N, L-1]
  const int* seg_pos0;     // [M]: position of the row (0: no history)
  const int* seg_slot;     // [M]
  int L;
};

// Two ways of saving the RMSNorm kernel between two products of a decode step (one row tile,
// at most 16 rows).  RMSNorm(x) W^T = (x * w) W^T / rms(x) row by row (kappai:
// src/backend/cpu/scalar/quants.c:1507-1512 for the norm), so the product can run on x * w and
// be scaled afterwards:
//   ResidOut (a product whose result is added to the residual stream, plain epilogue, float, K
//     not split over blocks): resid[m][n] += sum (+ bias) in place, in float; and when `rows` is
//     set the block also writes what the next product reads, rows[m][n] = bf16(resid[m][n] *
//     norm_w[n]) (row order, or the fragment order of add_rmsnorm when rows_frag), and
//     ss[blockIdx.x][m] = the sum of resid[m][n]^2 over its 8 columns (gemm_bf16_into_resid);
//   RowScale (the product that follows): its rows are such x * w, and every result is
//     multiplied by 1 / sqrt(sum_p ss[p][m] / K + eps) before bias and epilogue.
struct RowScale {
  const float* ss;   // [n_parts][16] (a row's value at [p][m]), or null: rows are used as they are
  int n_parts;
  float eps;
};
struct ResidOut {
  float* resid;          // [M, ldr], or null: the result goes to C
  int ldr;
  const float* norm_w;   // [N]; null: no rows for a next product
  bf16_t* rows;          // [M, N] or 16 rows in fragment order
  int rows_frag;
  float* ss;             // [gridDim.x][16]: a part holds one value a row, rows beyond M unwritten
};

template <typename TO, int MT, int NW, int EPI, int NT, bool FRAG>
__global__ __launch_bounds__(NW * WAVE) __attribute__((amdgpu_waves_per_eu(MT == 1 && EPI < 2 ? 4 : 1)))
void gemm_bf16_skinny_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, const float* __restrict__ ss, int M,
    int N, int K, int kblk, int lda, int a_frag, int w_frag, int ss_count, TO* __restrict__ C,
    const float* __restrict__ bias, int ldc, ConvStep cs, float ss_eps, int c_frag) {
  // (the arguments that the first loads need come first: the hardware hands over the first 14 words in
  // registers, the rest costs a load.  All of them together are a multiple of eight bytes: with an int less here
  // and in the kernel below, a step of 2 rows of 79 kernels, 65 of them these, took 478 us instead of 458.)
  static_assert(NT == 1 || EPI == 0, "several column tiles a wave: plain products only");
  // c_frag (one row tile, the SwiGLU and conv epilogues): the result is written as 16 rows in
  // fragment order, which is how the product that follows likes to read it (see a_frag)
  auto out_at = [&](int gm, int gn_) {
    return c_frag ? ((size_t)(gn_ / 8) * 16 + gm) * 8 + gn_ % 8 : (size_t)gm * ldc + gn_;
  };
  // row groups of W a block streams: gate/up, the three conv gates, or NT column tiles
  constexpr int NG = EPI == 1 ? 2 : (EPI == 2 ? 3 : (EPI == 3 ? 2 : NT));
  __shared__ f32x4_t red[NW][NG * MT][WAVE];
  const int tid = threadIdx.x;
  const int lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int n0 = blockIdx.x * (EPI == 3 ? 8 : 16 * NT);
  const int col = lane % 16, kg = (lane / 16) * 8;
  // EPI 3: columns 0-7 and 8-15 are the same 8 channels (of two different gates)
  const int gn = n0 + (EPI == 3 ? col % 8 : col);
  const u32x4_t zero = {0u, 0u, 0u, 0u};
  f32x4_t acc[NG * MT];
#pragma unroll
  for (int t = 0; t < NG * MT; ++t) acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  // plain: row gn (and 16 further for the next column tile).  SwiGLU: gate row 32*block + col, up
  // row 16 further.  Conv: rows gn, N + gn, 2N + gn.
  // EPI 3 (the conv step with 8 channels a block, twice as many blocks for narrow models): row
  // group 0 is the B gate's rows in columns 0-7 and the C gate's in columns 8-15, row group 1 the
  // x gate's rows in columns 0-7 (columns 8-15 stay zero).
  const size_t wr0 = EPI == 1 ? (size_t)blockIdx.x * 32 + col
                              : (EPI == 3 && col >= 8 ? (size_t)N + gn : (size_t)gn);
  const size_t group_rows = EPI == 2 ? (size_t)N : (EPI == 3 ? 2 * (size_t)N : 16);
  // W as it is stored ([rows, K]), or its copy in fragment order (w_frag): [rows / 16][K / 32]
  // pieces of 1 KB, each what one load instruction of a wave wants, lane by lane (lane =
  // (k % 32) / 8 * 16 + row % 16, 8 values a lane).  A wave's loads then touch every cache line
  // once instead of twice, and neighbouring lines: the products with 1-16 rows are bound by the
  // number of lines asked for as much as by bytes (gate/up at 8 rows: 14.7 against 18.2 us).
  // One step of 32 along K is 32 elements here and 512 there.
  const size_t wr1 = gn < N ? wr0 : 0;
  const int kmul = w_frag ? 16 : 1;
  const bf16_t* wrow = w_frag ? W + (wr1 / 16) * 16 * K + ((size_t)(kg / 8) * 16 + wr1 % 16) * 8
                              : W + wr1 * K + kg;
  auto group_ok = [&](int r) { return EPI == 3 ? (r == 0 || col < 8) : true; };
  const bf16_t* arow[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int gm = t * 16 + col;
    // a_frag (at most 16 rows): the rows lie in fragment order too, [K / 32][(k % 32) / 8][16 rows]
    // [8 values] (add_rmsnorm writes them so): a load then takes whole lines of neighbouring rows
    arow[t] = a_frag ? A + ((size_t)(kg / 8) * 16 + (gm < M ? gm : 0)) * 8
                     : A + (size_t)(gm < M ? gm : 0) * lda + kg;
  }
  // The row scales: a part is 16 floats, one a row, so a load takes 16 parts whole, a lane the four rows
  // lane % 4 of one.  The waves deal the loads among themselves, ask for them behind their first of W and meet in LDS.
  // (An extra wave that did this while the others streamed left room for one block a CU instead of two.)
  __shared__ f32x4_t row_ss[NW][4];
  f32x4_t ss_pre[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#if defined(__HIP_DEVICE_COMPILE__)
  const auto ask_for_parts = [&](int c) {
    // (rows behind M and parts behind the last lie outside the buffer: zeros, nothing read)
    const __amdgpu_buffer_rsrc_t parts = raw_buffer(ss, ss != nullptr ? (uint32_t)ss_count * 64u : 0u);
    return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
        parts, 4 * (lane % 4) < M ? lane * 16u : 0x7FFFFF00u, c * 1024, 0));
  };
  const auto ask_for_first_parts = [&]() {
    ss_pre[0] = ask_for_parts(wave);
    ss_pre[1] = ask_for_parts(wave + NW);
  };
  const auto add_parts = [&](bool asked) {
    if (!asked) ask_for_first_parts();
    asm volatile("" : "+v"(ss_pre[0]), "+v"(ss_pre[1]));       // (added here, not ahead of W)
    f32x4_t q = ss_pre[0] + ss_pre[1];
    for (int c = wave + 2 * NW; c * 16 < ss_count; c += NW) q += ask_for_parts(c);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      q[i] += dpp_move<0x124>(q[i]);             // row_ror 4
      q[i] += dpp_move<0x128>(q[i]);             // row_ror 8
      q[i] += lane_xor16(q[i]);
      q[i] += lane_xor32(q[i]);
    }
    if (lane < 4) row_ss[wave][lane] = q;
  };
#else
  const auto ask_for_first_parts = [&]() {};
  const auto add_parts = [&](bool) {};
#endif
  // The conv step's epilogue (EPI 2, 3) needs the rows' state, the channel's taps and the biases, asked for
  // by the waves that will use them so that they have arrived when W has gone through: the rows' slots
  // before the first loads of W, the state that they name behind those.  Up to CONV_PRE taps are held this
  // way; a longer filter reads the rest when it gets there.
  constexpr int CONV_PRE = 4;
  constexpr bool CONV = EPI == 2 || EPI == 3;
  float st_pre[4][CONV_PRE], tap_pre[CONV_PRE + 1], conv_bias_pre = 0.f;
  float gate_bias_pre[3] = {0.f, 0.f, 0.f};
  int pos_pre[4], slot_pre[4];
  float* st_ptr[4] = {nullptr, nullptr, nullptr, nullptr};
  const bool channel = gn < N && (EPI != 3 || col < 8);
#if defined(__HIP_DEVICE_COMPILE__)
  if (CONV && wave < MT) {
    // (buffer loads: an offset outside the buffer, or a buffer of no bytes, gives 0 and needs no branch.  The
    // taps' buffer begins with the block's first channel: there may be 4 GiB of them, and less than that of the rest.)
    constexpr int OUT = 0x7FFFFF00;
    const auto word = [](const void* p, uint32_t bytes, int at) {
      return __builtin_amdgcn_raw_buffer_load_b32(raw_buffer(p, bytes), at, 0, 0);
    };
    const auto number = [&](const void* p, uint32_t bytes, int at) {
      return __builtin_bit_cast(float, word(p, bytes, at));
    };
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int gm = wave * 16 + 4 * (lane / 16) + v;
      slot_pre[v] = (int)word(cs.seg_slot, M * 4u, channel ? gm * 4 : OUT);
      pos_pre[v] = (int)word(cs.seg_pos0, M * 4u, channel ? gm * 4 : OUT);
    }
#pragma unroll
    for (int k = 0; k <= CONV_PRE; ++k)
      tap_pre[k] = number(cs.taps + (size_t)n0 * cs.L, 16u * cs.L * 4u,
                          channel && k < cs.L ? ((gn - n0) * cs.L + k) * 4 : OUT);
    conv_bias_pre = number(cs.conv_bias, cs.conv_bias ? N * 4u : 0u, channel ? gn * 4 : OUT);
#pragma unroll
    for (int g = 0; g < 3; ++g)
      gate_bias_pre[g] = number(bias, bias ? N * 12u : 0u, channel ? (int)(((uint32_t)g * N + gn) * 4u) : OUT);
  }
#endif
  const auto ask_for_state = [&]() {
    const int H = cs.L - 1;
#pragma unroll
    for (int v = 0; v < 4; ++v) st_ptr[v] = cs.state + ((size_t)slot_pre[v] * N + (channel ? gn : 0)) * H;
#pragma unroll
    for (int k = 0; k < CONV_PRE; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) st_pre[v][k] = st_ptr[v][min(k, H - 1)];   // (H >= 1)
  };
  const int kb0 = blockIdx.y * kblk, kb1 = min(K, kb0 + kblk);     // the block's K
  const int kper = ((kb1 - kb0 + 32 * NW - 1) / (32 * NW)) * 32;
  const int k0 = kb0 + wave * kper;
  const int k1 = min(kb1, k0 + kper);
  C += (size_t)blockIdx.y * M * ldc;
  // loads in flight a lane: U * (NG + MT)
  constexpr int U = (NG + MT) <= 3 ? SK_UNROLL : ((NG + MT) <= 6 ? 4 : 2);
  if constexpr (FRAG) {
#if defined(__HIP_DEVICE_COMPILE__)
    // One buffer a row group of W, from the wave's first piece on and as long as its pieces; a lane's
    // offset, the same for every step but for a constant.  Lanes without a row of A (or, with EPI 3, of W)
    // stand behind every buffer's end and read nothing.
    constexpr uint32_t OUT = 0x7FFFFF00u;
    const int steps = max(k1 - k0, 0) / 32;
    __amdgpu_buffer_rsrc_t wbuf[NG], abuf;
    uint32_t woff[NG], aoff[MT];
    const size_t group = (size_t)16 * K;                 // of 16 rows, in values
#pragma unroll
    for (int r = 0; r < NG; ++r) {
      const int first = EPI == 0 ? (int)blockIdx.x * NT + r
                      : EPI == 1 ? (int)blockIdx.x * 2 + r
                      : EPI == 2 ? (int)blockIdx.x + r * (N / 16) : n0 / 16 + 2 * r * (N / 16);
      const bool there = EPI != 0 || first * 16 < N;
      // (EPI 3: the C gate's rows lie N rows behind the B gate's)
      const uint32_t bytes = there ? (uint32_t)steps * 1024u + (EPI == 3 && r == 0 ? (uint32_t)N * K * 2u : 0u) : 0u;
      wbuf[r] = raw_buffer(W + (size_t)first * group + (size_t)max(k0, 0) * 16, bytes);
      woff[r] = (uint32_t)lane * 16u;
      if (EPI == 3) {
        woff[r] = (uint32_t)((lane / 16) * 16 + n0 % 16 + col % 8) * 16u;
        if (col >= 8) woff[r] = r == 0 ? woff[r] + (uint32_t)N * K * 2u : OUT;
      }
    }
    abuf = raw_buffer(A + (size_t)k0 * (a_frag ? 16 : 1), OUT);
    const uint32_t astep = a_frag ? 1024u : 64u;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int gm = t * 16 + col;
      aoff[t] = gm >= M ? OUT : a_frag ? (uint32_t)lane * 16u : (uint32_t)gm * lda * 2u + kg * 2u;
    }
    const auto run = [&](auto count, int from) {
      constexpr int S = decltype(count)::value;
      u32x4_t wv[S][NG], av[S][MT];
#pragma unroll
      for (int u = 0; u < S; ++u) {
#pragma unroll
        for (int r = 0; r < NG; ++r)
          wv[u][r] = __builtin_amdgcn_raw_buffer_load_b128(wbuf[r], woff[r], (from + u) * 1024, 0);
#pragma unroll
        for (int t = 0; t < MT; ++t)
          av[u][t] = __builtin_amdgcn_raw_buffer_load_b128(abuf, aoff[t], (from + u) * astep, 0);
      }
      __builtin_amdgcn_sched_barrier(0);                 // (left alone, loads sink to their use)
      if (CONV && from == 0 && wave < MT) ask_for_state();
      if (MT == 1 && from == 0 && ss != nullptr) ask_for_first_parts();
#pragma unroll
      for (int u = 0; u < S; ++u)
#pragma unroll
        for (int r = 0; r < NG; ++r)
#pragma unroll
          for (int t = 0; t < MT; ++t)
            acc[r * MT + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                as_bf16x8(av[u][t]), as_bf16x8(wv[u][r]), acc[r * MT + t], 0, 0, 0);
    };
    int s = 0;
    if (CONV && steps == 0 && wave < MT) ask_for_state();        // (a wave of the epilogue without pieces)
    for (; s + U <= steps; s += U) run(IntC<U>{}, s);
    switch (steps - s) {
      case 1: run(IntC<1>{}, s); break;
      case 2: if constexpr (U > 2) run(IntC<2>{}, s); break;
      case 3: if constexpr (U > 2) run(IntC<3>{}, s); break;
      case 4: if constexpr (U > 4) run(IntC<4>{}, s); break;
      case 5: if constexpr (U > 4) run(IntC<5>{}, s); break;
      case 6: if constexpr (U > 4) run(IntC<6>{}, s); break;
      case 7: if constexpr (U > 4) run(IntC<7>{}, s); break;
      default: break;
    }
#endif
  } else {
    if (CONV && wave < MT) ask_for_state();
    if (MT == 1 && ss != nullptr) ask_for_first_parts();
    for (int k = k0; k < k1; k += 32 * U) {
      // the loads of W and of A alternate, in the order of K
      u32x4_t wv[U][NG], av[U][MT];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int gk = k + 32 * u;
        const bool kin = gk + kg < k1;
#pragma unroll
        for (int r = 0; r < NG; ++r)
          wv[u][r] = (kin && gn + (EPI == 0 ? r * 16 : 0) < N && group_ok(r))
                         ? load16(wrow + r * group_rows * K + (size_t)gk * kmul)
                         : zero;
#pragma unroll
        for (int t = 0; t < MT; ++t)
          av[u][t] = (kin && t * 16 + col < M) ? load16(arow[t] + (size_t)gk * (a_frag ? 16 : 1)) : zero;
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < NG; ++r)
#pragma unroll
          for (int t = 0; t < MT; ++t)
            acc[r * MT + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                as_bf16x8(av[u][t]), as_bf16x8(wv[u][r]), acc[r * MT + t], 0, 0, 0);
    }
  }
  if (MT == 1 && ss != nullptr) add_parts(!FRAG || k0 < k1);
#pragma unroll
  for (int t = 0; t < NG * MT; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
  // a tile's sums over the waves, in a fixed order
  auto whole = [&](int tile, int from) {
    f32x4_t sum = red[0][tile][from];
#pragma unroll(NW < 16 ? NW : 4)
    for (int w = 1; w < NW; ++w) sum += red[w][tile][from];
    return sum;
  };
  // of the lane's rows 4 (lane / 16) ..
  f32x4_t scale = {1.f, 1.f, 1.f, 1.f};
  if (MT == 1 && wave < NG && ss != nullptr) {
    f32x4_t q = row_ss[0][lane / 16];
#pragma unroll
    for (int w = 1; w < NW; ++w) q += row_ss[w][lane / 16];
#pragma unroll
    for (int v = 0; v < 4; ++v) scale[v] = 1.0f / sqrtf(q[v] / (float)K + ss_eps);
  }
  // the first MT waves each sum one row tile over the NW partial results, in a fixed order
  if (EPI == 0 && NT > 1) {
    // waves take the NT * MT tiles in turn
    for (int tile = wave; tile < NT * MT; tile += NW) {
      const int r = tile / MT, t = tile % MT;
      const int gnr = gn + r * 16;
      if (gnr >= N) continue;
      const float bv = (bias && blockIdx.y == 0) ? bias[gnr] : 0.f;
      const f32x4_t sum = whole(tile, lane);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gm = t * 16 + 4 * (lane / 16) + v;
        if (gm >= M) continue;
        store_out(C + (size_t)gm * ldc + gnr, sum[v] * scale[v] + bv);
      }
    }
  } else if (wave < MT && channel) {
    const int t = wave;
    const float bv = (EPI != 1 && bias && blockIdx.y == 0) ? bias[gn] : 0.f;
    const f32x4_t sums = whole(t, lane);
    // the up row; or where the other two gates of this channel lie: EPI 2 in row groups 1 and 2 of this
    // lane, EPI 3 the C gate 8 columns further in group 0 and the x gate in group 1
    f32x4_t second = sums, third = sums;
    if (EPI == 1 || EPI == 2) second = whole(MT + t, lane);
    if (EPI == 3) second = whole(t, lane + 8);
    if (EPI == 2) third = whole(2 * MT + t, lane);
    if (EPI == 3) third = whole(MT + t, lane);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int gm = t * 16 + 4 * (lane / 16) + v;
      if (gm < M) {
        const float rs = scale[v];
        const float sum = sums[v] * rs;
        if (EPI == 1) {
          store_out(C + out_at(gm, gn), gated_f(sum, second[v] * rs, bias, (int)blockIdx.x * 32 + col));
        } else if (EPI == 2 || EPI == 3) {
          float cg = second[v] * rs, xg = third[v] * rs;
          const float bg = sum + gate_bias_pre[0];
          cg += gate_bias_pre[1];
          xg += gate_bias_pre[2];
          // the three gates are rounded as the unfused path stores them
          const float bx = to_f32(f32_to_bf16(bg)) * to_f32(f32_to_bf16(xg));
          const int H = cs.L - 1;
          int pos = pos_pre[v];
          asm volatile("" : "+v"(pos));          // (compared here, not where it was asked for)
          const bool fresh = pos == 0;
          float* st = st_ptr[v];
          const float* wc = cs.taps + (size_t)gn * cs.L;
          float s = conv_bias_pre;
          if (H <= CONV_PRE) {
            // everything is in registers already
            float prev = fresh ? 0.f : st_pre[v][0];
#pragma unroll
            for (int k = 0; k < CONV_PRE; ++k) {
              if (k < H) {
                s += tap_pre[k] * prev;
                const float next = (k + 1 < H) ? (fresh ? 0.f : st_pre[v][k + 1 < CONV_PRE ? k + 1 : 0]) : bx;
                st[k] = next;
                prev = next;
              }
            }
            float last = tap_pre[0];
#pragma unroll
            for (int k = 1; k <= CONV_PRE; ++k) last = k == H ? tap_pre[k] : last;
            s += last * bx;
          } else {
            float prev = fresh ? 0.f : st[0];
            for (int k = 0; k < H; ++k) {
              s += wc[k] * prev;
              const float next = (k + 1 < H) ? (fresh ? 0.f : st[k + 1]) : bx;
              st[k] = next;
              prev = next;
            }
            s += wc[H] * bx;
          }
          store_out(C + out_at(gm, gn), to_f32(f32_to_bf16(cg)) * s);
        } else {
          store_out(C + (size_t)gm * ldc + gn, sum + bv);
        }
      }
    }
  }
}

// A product whose result joins the residual stream (ResidOut; at most 16 rows, K in one piece).
// Such products have few columns (the model's width), so a block owns 8 of them, and the two
// halves of the matrix tile's 16 columns take the two halves of K: column j < 8 is row n0 + j of
// W over K's first half, column j + 8 the same row over the second half.  The rows of A of the
// two halves meet the one fragment of W in two matrix instructions, whose valid halves are added
// at the end.  Twice as many blocks stream W as with 16 columns a block, and K needs no split
// over blocks, so the residual sum can be made here, in a fixed order.
// ROWS8 (up to 8 rows, FRAG): the rows of A of the two halves share a fragment as well, row r of the first half in
// place r, of the second in place r + 8, so that one instruction makes both halves' sums (the tile's two quarters
// on its diagonal; the same sums in the same order) from one load of A where there were two.  A load takes its
// clocks at the CU's door whether its lanes need anything or not, and these blocks have the CU to themselves: one row
// of 1024 x 4608 7.0 -> 6.5 us.  In the form with 16 waves: with 8, whose waves have two to four steps, there is no
// line of loads to wait in (1024 x 1024: 23 us more over 256 products).
template <int NW, bool FRAG, bool ROWS8>
__global__ __launch_bounds__(NW * WAVE) void gemm_bf16_into_resid_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, float* __restrict__ resid, int M, int N,
    int K, int lda, int frags, int ldr, const float* __restrict__ norm_w, const float* __restrict__ bias,
    bf16_t* __restrict__ rows, float* __restrict__ ss, int rows_frag, int spare) {
  // frags: the rows' order, and where not FRAG as the second bit that of W; spare: see above
  const int a_frag = FRAG ? frags : frags & 1, w_frag = FRAG ? 1 : frags & 2;
  static_assert(FRAG || !ROWS8, "");
  constexpr int HI = ROWS8 ? 0 : 1, ACROSS = ROWS8 ? 40 : 8;   // where a lane's columns 8 further are, and whose
  __shared__ f32x4_t red[NW][1 + HI][WAVE];
  const int tid = threadIdx.x;
  const int lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int col = lane % 16, kg = (lane / 16) * 8;
  const int half = col / 8;
  const int gn = blockIdx.x * 8 + col % 8;               // the lane's row of W
  const int khalf = ((K / 2 + 31) / 32) * 32;            // the second half starts here
  const u32x4_t zero = {0u, 0u, 0u, 0u};
  // What the epilogue needs, asked for before the stream of W: offsets outside the buffers for lanes that
  // need nothing, since of loads in branches the compiler waits for the first before it asks for the next.
  // (FRAG: the residual's offsets have 31 bits, see the launch.)
  float resid_in[4] = {0.f, 0.f, 0.f, 0.f};
  float norm_w_in = 0.f;
#if defined(__HIP_DEVICE_COMPILE__)
  const bool near = FRAG || ((uint64_t)(M - 1) * ldr + N) * 4 < 0x7FFFFF00u;
  if (wave == 0 && near) {
    const bool mine = half == 0 && gn < N;
    const __amdgpu_buffer_rsrc_t res = raw_buffer(resid, 0x7FFFFF00u);
    const __amdgpu_buffer_rsrc_t nw = raw_buffer(norm_w, rows != nullptr ? (uint32_t)N * 4u : 0u);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int gm = 4 * (lane / 16) + v;
      resid_in[v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
          res, mine && gm < M ? (gm * ldr + gn) * 4 : 0x7FFFFF00, 0, 0));
    }
    norm_w_in = __builtin_bit_cast(
        float, __builtin_amdgcn_raw_buffer_load_b32(nw, mine ? gn * 4 : 0x7FFFFF00, 0, 0));
  }
  if (wave == 0 && !near && half == 0 && gn < N) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int gm = 4 * (lane / 16) + v;
      if (gm < M) resid_in[v] = resid[(size_t)gm * ldr + gn];
    }
    if (rows != nullptr) norm_w_in = norm_w[gn];
  }
#endif
  const size_t wr = gn < N ? gn : 0;
  const int kmul = w_frag ? 16 : 1;                      // see the kernel above for the two orders
  const bf16_t* wrow = (w_frag ? W + (wr / 16) * 16 * K + ((size_t)(kg / 8) * 16 + wr % 16) * 8
                               : W + wr * K + kg) + (size_t)half * khalf * kmul;
  const int am = col < M ? col : 0;                      // the lane's row of A
  const int amul = a_frag ? 16 : 1;
  const bf16_t* arow = a_frag ? A + ((size_t)(kg / 8) * 16 + am) * 8 : A + (size_t)am * lda + kg;
  const int kper = ((khalf + 32 * NW - 1) / (32 * NW)) * 32;
  const int k0 = wave * kper, k1 = min(khalf, k0 + kper);
  f32x4_t acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
  constexpr int U = SK_UNROLL;
  if constexpr (FRAG) {
#if defined(__HIP_DEVICE_COMPILE__)
    // as in the kernel above; K is a multiple of 64, so that both halves have as many steps
    constexpr uint32_t OUT = 0x7FFFFF00u;
    const int steps = max(k1 - k0, 0) / 32;
    const __amdgpu_buffer_rsrc_t wbuf =
        raw_buffer(W + ((size_t)(blockIdx.x / 2) * K + k0) * 16, (uint32_t)(khalf + 32 * steps) * 32u);
    const uint32_t woff =
        ((lane / 16) * 16 + blockIdx.x % 2 * 8 + col % 8) * 16u + (half ? (uint32_t)khalf * 32u : 0u);
    const __amdgpu_buffer_rsrc_t abuf = raw_buffer(A + (size_t)k0 * (a_frag ? 16 : 1), OUT);
    const uint32_t astep = a_frag ? 1024u : 64u, second = (uint32_t)khalf * (a_frag ? 32u : 2u);
    const uint32_t aoff =
        ROWS8 ? (col % 8 >= M ? OUT
                              : (a_frag ? (uint32_t)(lane - half * 8) * 16u : (uint32_t)(col % 8) * lda * 2u + kg * 2u) +
                                    (half ? second : 0u))
              : col >= M ? OUT : a_frag ? (uint32_t)lane * 16u : (uint32_t)col * lda * 2u + kg * 2u;
    const auto run = [&](auto count, int from) {
      constexpr int S = decltype(count)::value;
      u32x4_t wv[S], a0[S], a1[ROWS8 ? 1 : S];
#pragma unroll
      for (int u = 0; u < S; ++u) {
        wv[u] = __builtin_amdgcn_raw_buffer_load_b128(wbuf, woff, (from + u) * 1024, 0);
        a0[u] = __builtin_amdgcn_raw_buffer_load_b128(abuf, aoff, (from + u) * astep, 0);
        if constexpr (!ROWS8)
          a1[u] = __builtin_amdgcn_raw_buffer_load_b128(abuf, aoff, (from + u) * astep + second, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < S; ++u) {
        acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a0[u]), as_bf16x8(wv[u]), acc0, 0, 0, 0);
        if constexpr (!ROWS8)
          acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a1[u]), as_bf16x8(wv[u]), acc1, 0, 0, 0);
      }
    };
    int s = 0;
    for (; s + U <= steps; s += U) run(IntC<U>{}, s);
    switch (steps - s) {
      case 1: run(IntC<1>{}, s); break;
      case 2: run(IntC<2>{}, s); break;
      case 3: run(IntC<3>{}, s); break;
      case 4: run(IntC<4>{}, s); break;
      case 5: run(IntC<5>{}, s); break;
      case 6: run(IntC<6>{}, s); break;
      case 7: run(IntC<7>{}, s); break;
      default: break;
    }
#endif
  } else
  for (int k = k0; k < k1; k += 32 * U) {
    u32x4_t wv[U], a0[U], a1[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int gk = k + 32 * u;
      const bool in0 = gk + kg < k1 && gk + kg < K;       // within the wave's range of a half
      const bool in1 = in0 && khalf + gk + kg < K;        // and, for the second half, within K
      wv[u] = ((half ? in1 : in0) && gn < N) ? load16(wrow + (size_t)gk * kmul) : zero;
      a0[u] = (in0 && col < M) ? load16(arow + (size_t)gk * amul) : zero;
      a1[u] = (in1 && col < M) ? load16(arow + (size_t)(khalf + gk) * amul) : zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a0[u]), as_bf16x8(wv[u]), acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a1[u]), as_bf16x8(wv[u]), acc1, 0, 0, 0);
    }
  }
  red[wave][0][lane] = acc0;
  if constexpr (!ROWS8) red[wave][HI][lane] = acc1;
  __syncthreads();
  if (wave != 0) return;
  f32x4_t lo = red[0][0][lane], hi = red[0][HI][lane ^ ACROSS];
#pragma unroll 4
  for (int w = 1; w < NW; ++w) {
    lo += red[w][0][lane];
    hi += red[w][HI][lane ^ ACROSS];
  }
  // columns 0-7: the first half's sums of this lane and the second half's of the lane 8 further
  const bool mine = half == 0 && gn < N;
  const float bv = (bias && mine) ? bias[gn] : 0.f;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int gm = 4 * (lane / 16) + v;
    float q = 0.f;
    if (mine && gm < M) {
      const float x = resid_in[v] + ((lo[v] + hi[v]) + bv);
      resid[(size_t)gm * ldr + gn] = x;
      if (rows != nullptr) {
        const size_t at = rows_frag ? ((size_t)(gn / 8) * 16 + gm) * 8 + gn % 8
                                       : (size_t)gm * N + gn;
        rows[at] = f32_to_bf16(x * norm_w_in);
      }
      q = x * x;
    }
    if (rows != nullptr) {
      // the sum of squares over the block's 8 columns, row by row
      q += __shfl_xor(q, 1, WAVE);
      q += __shfl_xor(q, 2, WAVE);
      q += __shfl_xor(q, 4, WAVE);
      if (col == 0 && gm < M) ss[(size_t)blockIdx.x * 16 + gm] = q;
    }
  }
}

static void launch_into_resid(const bf16_t* A, const bf16_t* W, const float* bias, int M, int N,
                              int K, int lda, const ResidOut& ro, hipStream_t stream,
                              const bf16_t* Wf, int a_frag) {
  const int frags = a_frag ? 1 : 0;
  const int w_order = Wf ? 2 : 0;
  if (Wf) W = Wf;
  const dim3 grid((N + 7) / 8);
  // (both halves of K whole pieces and offsets of 31 bits, into the stream too: the loads without conditions)
  const bool pieces = Wf != nullptr && K % 64 == 0 && ((size_t)M * lda + K) * 2 < 0x7FFFFF00u &&
                      (size_t)K * 32 < 0x7FFFFF00u && ((size_t)(M - 1) * ro.ldr + N) * 4 < 0x7FFFFF00u;
#define INTO_RESID(NW)                                                                                 \
  do {                                                                                                 \
    if (pieces && M <= 8)                                                                              \
      hipLaunchKernelGGL((gemm_bf16_into_resid_kernel<NW, true, NW == 16>), grid, dim3(NW * WAVE), 0,  \
                         stream, A, W, ro.resid, M, N, K, lda, frags, ro.ldr, ro.norm_w, bias,         \
                         ro.rows, ro.ss, ro.rows_frag, 0);                                             \
    else if (pieces)                                                                                   \
      hipLaunchKernelGGL((gemm_bf16_into_resid_kernel<NW, true, false>), grid, dim3(NW * WAVE), 0,     \
                         stream, A, W, ro.resid, M, N, K, lda, frags, ro.ldr, ro.norm_w, bias,         \
                         ro.rows, ro.ss, ro.rows_frag, 0);                                             \
    else                                                                                               \
      hipLaunchKernelGGL((gemm_bf16_into_resid_kernel<NW, false, false>), grid, dim3(NW * WAVE), 0, stream,   \
                         A, W, ro.resid, M, N, K, lda, frags | w_order, ro.ldr, ro.norm_w, bias,       \
                         ro.rows, ro.ss, ro.rows_frag, 0);                                             \
  } while (0)
  // K a wave: 128 or more where K allows it
  if (K >= 4096) INTO_RESID(16);
  else if (K >= 1024) INTO_RESID(8);
  else INTO_RESID(4);
#undef INTO_RESID
}

struct Fuse {
  RowScale rsc;
  ResidOut ro;
  int c_frag = 0;
};

template <typename TO, int MT, int NW, int EPI, int NT = 1>
static void launch_skinny(const bf16_t* A, const bf16_t* W, const float* bias, TO* C, int M, int N,
                          int K, int lda, int ldc, int ksplit, ConvStep cs, hipStream_t stream,
                          const Fuse& fuse = Fuse{}, const bf16_t* Wf = nullptr, int a_frag = 0) {
  // Wf: the copy of W in fragment order (see the kernel), or null
  const dim3 grid(EPI == 3 ? (N + 7) / 8 : (N + 16 * NT - 1) / (16 * NT), ksplit);
  const int c_frag = (MT == 1 && EPI != 0) ? fuse.c_frag : 0;
  const int kblk = (K + 32 * ksplit - 1) / (32 * ksplit) * 32;
  // (fragment order and offsets of 31 bits within A, a group of W and the gates of EPI 3: the loads
  // without conditions)
  const bool pieces = Wf != nullptr && ((size_t)M * lda + K) * 2 < 0x7FFFFF00u && (size_t)K * 32 < 0x7FFFFF00u &&
                      (EPI != 3 || (size_t)(N + 16) * K * 2 < 0x7FFFFF00u);
#define SKINNY(FRAG)                                                                                   \
  hipLaunchKernelGGL((gemm_bf16_skinny_kernel<TO, MT, NW, EPI, NT, FRAG>), grid, dim3(NW * WAVE), 0,    \
                     stream, A, Wf ? Wf : W, fuse.rsc.ss, M, N, K, kblk, lda, a_frag, Wf ? 1 : 0,       \
                     fuse.rsc.n_parts, C, bias, ldc, cs, fuse.rsc.eps, c_frag)
  if (pieces) SKINNY(true);
  else SKINNY(false);
#undef SKINNY
}

// more waves a block when there are few blocks, so that about 2048 waves or more stream W
template <typename TO, int MT, int EPI>
static void launch_skinny_mt(const bf16_t* A, const bf16_t* W, const float* bias, TO* C, int M,
                             int N, int K, int lda, int ldc, int ksplit, ConvStep cs,
                             hipStream_t stream, const Fuse& fuse = Fuse{},
                             const bf16_t* Wf = nullptr, int a_frag = 0) {
  // several row tiles and a plain product: a wave takes two column tiles for every fragment
  // of A it loads, which halves the reads of A (every block reads all of it)
  if constexpr (EPI == 0 && MT >= 2) {
    if (N >= 64) {
      launch_skinny<TO, MT, 4, EPI, 2>(A, W, bias, C, M, N, K, lda, ldc, ksplit, cs, stream,
                                       Fuse{}, Wf, a_frag);
      return;
    }
  }
  // 8 to 16 rows and columns enough (the output head): four column tiles for every fragment of
  // A (58 against 62 us for 65,536 columns at 8 rows, 62 against 74 at 16; slower below 8 rows).
  // With W in fragment order one tile a wave is the faster up to 11 rows (50 against 56 us at 8
  // rows, 56 either way at 12, 62 against 56 at 16).
  if constexpr (EPI == 0 && MT == 1) {
    if (M >= (Wf ? 12 : 8) && (long)(N / 64) * ksplit >= 512) {
      launch_skinny<TO, MT, 4, EPI, 4>(A, W, bias, C, M, N, K, lda, ldc, ksplit, cs, stream,
                                       fuse, Wf, a_frag);
      return;
    }
  }
  const int blocks = (EPI == 3 ? (N + 7) / 8 : (N + 15) / 16) * ksplit;
  const int kb = K / ksplit;                              // K a block
  constexpr int NG = EPI == 1 ? 2 : (EPI == 2 ? 3 : (EPI == 3 ? 2 : 1));
  // 1 KB of LDS a wave, group and row tile; the conv step's 16 waves would have no room for what its
  // epilogue waits with
  constexpr int MAXW = EPI >= 2 && MT == 1 ? 8 : 48 / (MT * NG);
  if (blocks * 4 >= 2048 || kb <= 512 || MAXW < 8)
    launch_skinny<TO, MT, 4, EPI>(A, W, bias, C, M, N, K, lda, ldc, ksplit, cs, stream, fuse, Wf, a_frag);
  else if (blocks * 8 >= 2048 || kb <= 1024 || MAXW < 16)
    launch_skinny<TO, MT, (MAXW >= 8 ? 8 : 4), EPI>(A, W, bias, C, M, N, K, lda, ldc, ksplit, cs,
                                                    stream, fuse, Wf, a_frag);
  else
    launch_skinny<TO, MT, (MAXW >= 16 ? 16 : 4), EPI>(A, W, bias, C, M, N, K, lda, ldc, ksplit, cs,
                                                      stream, fuse, Wf, a_frag);
}

// ---------------------------------------------------------------------------------------
// 17 to 64 rows (decode at larger batches): the activations go through LDS
// ---------------------------------------------------------------------------------------
// With several row tiles every wave of the kernel above reads all rows of A for its K range
// from L2 again, which at 64 rows is twice the bytes of W it streams.  Here a block is
// NWN x NWK waves: wave (wn, wk) owns 32 rows of W (two column tiles, or the gate and up rows
// of 16 SwiGLU columns) and the wk-th part of the block's K range, and the NWN waves with the
// same wk share the rows of A: chunk by chunk of KC of K they are loaded once, straight into
// LDS (global_load_lds, two buffers, 16-byte chunks permuted so that a fragment read is free of
// bank conflicts), while W goes from global memory into registers, one chunk ahead.  The waves
// meet in LDS at the end to add their K parts in a fixed order.
//
// Host side guarantees: K / gridDim.y is a multiple of NWK * KC, M * lda < 2^31.  Rows of A
// past M and rows of W past the end repeat the last row (their products are not stored).
template <int MT, int NWN, int NWK, int KC>
struct SharedRows {
  static constexpr int NW = NWN * NWK, ROWS = 16 * MT, CH = KC / 8, UK = KC / 32;
  static constexpr int RPI = 64 / CH;                        // rows a load instruction brings
  static constexpr int INSTR = NWK * ROWS / RPI;             // load instructions a chunk
  static constexpr int PER_WAVE = (INSTR + NW - 1) / NW;
  static constexpr int BUF = NWK * ROWS * KC;                // bf16 elements a buffer
  static constexpr size_t stage_bytes = 2 * (size_t)BUF * sizeof(bf16_t);
  static constexpr size_t red_bytes = (size_t)NW * 2 * MT * WAVE * sizeof(f32x4_t);
  static constexpr size_t lds_bytes = stage_bytes > red_bytes ? stage_bytes : red_bytes;
  __device__ static int swz(int row) { return CH == 16 ? (row & 15) : ((row >> 1) & 7); }
};

template <typename TO, int MT, int EPI, int NWN, int NWK, int KC, int NSETS>
__global__ __launch_bounds__(NWN * NWK * WAVE) void gemm_bf16_shared_rows_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, const float* __restrict__ bias,
    TO* __restrict__ C, int M, int n_rows_w, int K, int lda, int ldc, int w_frag) {
  static_assert(NSETS % 2 == 0 && 2 * (KC / 32) * (NSETS - 1) < 64, "register sets");
  using S = SharedRows<MT, NWN, NWK, KC>;
  constexpr int NW = S::NW, UK = S::UK, CH = S::CH;
  extern __shared__ __attribute__((aligned(1024))) bf16_t lds[];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wn = wave / NWK, wk = wave % NWK;
  const int col = lane % 16, kgi = lane / 16;
  const int kblk = K / (int)gridDim.y;               // K of the block
  const int kper = kblk / NWK;                       // K of a wave
  const int nchunks = kper / KC;
  const int kb0 = blockIdx.y * kblk;
  C += (size_t)blockIdx.y * M * ldc;

  // rows of W of this wave: group r = rows wrow0 + 16 r + (0..15)
  const int wrow0 = (blockIdx.x * NWN + wn) * 32;
  const bf16_t* wptr[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    // W as stored, or its copy in fragment order (see gemm_bf16_skinny_kernel): a step of 32
    // along K is 32 elements here and 512 there
    const size_t row = (size_t)min(wrow0 + 16 * r + col, n_rows_w - 1);
    const size_t kbase = (size_t)kb0 + (size_t)wk * kper;
    wptr[r] = w_frag ? W + (row / 16) * 16 * K + kbase * 16 + ((size_t)kgi * 16 + row % 16) * 8
                     : W + row * K + kbase + kgi * 8;
  }
  const int kmul = w_frag ? 16 : 1;

  // the block's load instructions for a chunk of A, dealt round the waves: instruction j
  // brings rows (j % (ROWS / RPI)) * RPI + lane / CH of K part j / (ROWS / RPI)
  uint32_t aoff[S::PER_WAVE];
#pragma unroll
  for (int i = 0; i < S::PER_WAVE; ++i) {
    const int j = i * NW + wave;
    const int part = j / (S::ROWS / S::RPI), row = (j % (S::ROWS / S::RPI)) * S::RPI + lane / CH;
    const int chunk = (lane % CH) ^ S::swz(row);
    aoff[i] = (uint32_t)(min(row, M - 1) * lda + kb0 + part * kper + chunk * 8) *
              (uint32_t)sizeof(bf16_t);
  }
  auto stage = [&](int buf, int c) {
    const uint64_t p = reinterpret_cast<uint64_t>(A) + (uint64_t)c * (KC * sizeof(bf16_t));
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)p);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
    const char* base = reinterpret_cast<const char*>(((uint64_t)hi << 32) | lo);
#pragma unroll
    for (int i = 0; i < S::PER_WAVE; ++i) {
      const int j = i * NW + wave;
      if (S::INSTR % NW == 0 || j < S::INSTR)
        __builtin_amdgcn_global_load_lds(KAPPAI_GPTR(base + aoff[i]),
                                         KAPPAI_LPTR(lds + buf * S::BUF + j * 512), 16, 0, 0);
    }
  };
  auto load_w = [&](u32x4_t (&wv)[UK][2], int c) {
#pragma unroll
    for (int u = 0; u < UK; ++u)
#pragma unroll
      for (int r = 0; r < 2; ++r) wv[u][r] = load16(wptr[r] + (size_t)(c * KC + 32 * u) * kmul);
  };
  f32x4_t acc[2 * MT];
#pragma unroll
  for (int t = 0; t < 2 * MT; ++t) acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  // fragment of A: lane holds row 16 t + col, the 8 of K number 4 u + kgi of the chunk
  int roff[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) roff[t] = (wk * S::ROWS + 16 * t + col) * KC;
  auto products = [&](const u32x4_t (&wv)[UK][2], int buf) {
#pragma unroll
    for (int u = 0; u < UK; ++u) {
      u32x4_t av[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t)
        av[t] = *reinterpret_cast<const u32x4_t*>(
            lds + buf * S::BUF + roff[t] + (((4 * u + kgi) ^ S::swz(16 * t + col)) * 8));
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[r * MT + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              as_bf16x8(av[t]), as_bf16x8(wv[u][r]), acc[r * MT + t], 0, 0, 0);
    }
  };

  // W is loaded NSETS - 1 chunks ahead into register sets used in turn; A one chunk ahead.  In
  // every pass of the loop the loads of A are issued before those of W, and loads come back in
  // the order they were issued: waiting until only the latest pass's loads of W are out means that
  // the chunk of A issued before them has landed.  NSETS is even, so that the LDS buffer of a pass
  // is known at compile time (else the compiler waits for every load before it reads LDS).
  u32x4_t wv[NSETS][UK][2];
  stage(0, 0);
#pragma unroll
  for (int s = 0; s < NSETS - 1; ++s)
    if (s < nchunks) load_w(wv[s], s);
  constexpr int VM_ROUND = 0x0F70 | ((2 * UK) & 15) | (((2 * UK) >> 4) << 14);
  constexpr int VM_FIRST = 0x0F70 | ((2 * UK * (NSETS - 1)) & 15) | (((2 * UK * (NSETS - 1)) >> 4) << 14);
  for (int c = 0; c < nchunks; c += NSETS) {
#pragma unroll
    for (int s = 0; s < NSETS; ++s) {
      const int cc = c + s;
      if (cc >= nchunks) break;
      // chunk cc of A was issued in round cc - 1 and after it that round's chunk of W, if there
      // was one left to load (before the loop: chunk 0 of A, then NSETS - 1 chunks of W)
      if (cc == 0 && nchunks >= NSETS - 1)
        __builtin_amdgcn_s_waitcnt(VM_FIRST);
      else if (cc > 0 && cc + NSETS - 2 < nchunks)
        __builtin_amdgcn_s_waitcnt(VM_ROUND);
      else
        __builtin_amdgcn_s_waitcnt(0x0F70);
      // everybody's part of chunk cc is there and nobody reads the other buffer any more (a
      // bare barrier: a fence would wait for the loads of W that are meant to stay in flight)
      __builtin_amdgcn_s_barrier();
      SCHED_FENCE();
      if (cc + 1 < nchunks) stage((s + 1) & 1, cc + 1);
      if (cc + NSETS - 1 < nchunks) load_w(wv[(s + NSETS - 1) % NSETS], cc + NSETS - 1);
      products(wv[s], s & 1);
    }
  }
  __syncthreads();
  // the K parts meet: wave (wn, wk) adds up and stores row tiles wk, wk + NWK, ...
  f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);
#pragma unroll
  for (int t = 0; t < 2 * MT; ++t) red[(wave * 2 * MT + t) * WAVE + lane] = acc[t];
  __syncthreads();
  for (int t = wk; t < MT; t += NWK) {
    f32x4_t sum[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      sum[r] = red[((wn * NWK) * 2 * MT + r * MT + t) * WAVE + lane];
#pragma unroll
      for (int w = 1; w < NWK; ++w) sum[r] += red[((wn * NWK + w) * 2 * MT + r * MT + t) * WAVE + lane];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int gm = 16 * t + 4 * kgi + v;
      if (gm >= M) continue;
      if (EPI == 1) {
        const int on = wrow0 / 2 + col;                 // 16 output columns a wave
        if (wrow0 + 16 + col < n_rows_w)
          store_out(C + (size_t)gm * ldc + on, gated_f(sum[0][v], sum[1][v], bias, wrow0 + col));
      } else {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const int gn = wrow0 + 16 * r + col;
          if (gn < n_rows_w)
            store_out(C + (size_t)gm * ldc + gn,
                      sum[r][v] + ((bias && blockIdx.y == 0) ? bias[gn] : 0.f));
        }
      }
    }
  }
}

template <int NWK, int KC>
static bool shared_rows_fits(int M, int K, int lda, int ksplit) {
  return M > 16 && M <= 64 && ksplit >= 1 && K % (ksplit * NWK * KC) == 0 &&
         (long)M * lda < (1L << 31) - 8 * (long)KC;
}

template <typename TO, int MT, int EPI, int NWN, int NWK, int KC, int NSETS>
static void launch_shared_rows_cfg(const bf16_t* A, const bf16_t* W, const float* bias, TO* C,
                                   int M, int n_rows_w, int K, int lda, int ldc, int ksplit,
                                   hipStream_t stream, const bf16_t* Wf) {
  using S = SharedRows<MT, NWN, NWK, KC>;
  auto kern = gemm_bf16_shared_rows_kernel<TO, MT, EPI, NWN, NWK, KC, NSETS>;
  static bool attr_set = false;       // more than 64 KB of LDS has to be asked for once
  if (!attr_set) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)S::lds_bytes);
    attr_set = true;
  }
  hipLaunchKernelGGL(kern, dim3((n_rows_w + 32 * NWN - 1) / (32 * NWN), ksplit),
                     dim3(S::NW * WAVE), S::lds_bytes, stream, A, Wf ? Wf : W, bias, C, M, n_rows_w, K,
                     lda, ldc, Wf ? 1 : 0);
}

// 2 x 4 waves, chunks of 128 of K, two register sets of W.  (4 x 4 waves leave half the CUs
// without a block on the layer shapes; more register sets or 16 waves with chunks of 64 gain
// nothing.)  Returns false when the shape does not fit.
#define SR_NWN 2
#define SR_NWK 4
#define SR_KC 128
template <typename TO, int EPI>
static bool launch_shared_rows(const bf16_t* A, const bf16_t* W, const float* bias, TO* C, int M,
                               int n_rows_w, int K, int lda, int ldc, int ksplit,
                               hipStream_t stream, const bf16_t* Wf) {
  if (!shared_rows_fits<SR_NWK, SR_KC>(M, K, lda, ksplit)) return false;
  if (M <= 32)
    launch_shared_rows_cfg<TO, 2, EPI, SR_NWN, SR_NWK, SR_KC, 2>(A, W, bias, C, M, n_rows_w, K, lda,
                                                                 ldc, ksplit, stream, Wf);
  else if (M <= 48)
    launch_shared_rows_cfg<TO, 3, EPI, SR_NWN, SR_NWK, SR_KC, 2>(A, W, bias, C, M, n_rows_w, K, lda,
                                                                 ldc, ksplit, stream, Wf);
  else
    launch_shared_rows_cfg<TO, 4, EPI, SR_NWN, SR_NWK, SR_KC, 2>(A, W, bias, C, M, n_rows_w, K, lda,
                                                                 ldc, ksplit, stream, Wf);
  return true;
}

// ---------------------------------------------------------------------------------------
// 25 to 128 rows (decode at batches of that size, short prompt portions): 32 x 32 tiles, rows
// via LDS
// ---------------------------------------------------------------------------------------
// The block kernels above need hundreds of rows to fill their tiles, and the kernel for 17 to 64
// rows reads every fragment of A once per 16 x 16 tile (it still runs where this one does not
// fit: a matrix kept as rows, a K range that is no multiple of 256).  Here a block is 2 x 4 waves: wave
// (wn, wk) owns 32 rows of W (one 32 x 32 tile of the result for each 32 rows of A,
// v_mfma_f32_32x32x16_bf16: half the LDS reads per product of the 16 x 16 form) and, of every
// run of 256 of the block's K range, the 64 number wk.  The block's rows of A go through LDS run
// by run (global_load_lds, two buffers of rows x 256, rows of 128 bytes per 64 of K permuted as
// in the block kernel: a fragment read is free of bank conflicts), W comes from its
// fragment-order copy straight into registers, one run ahead: a load instruction takes the two
// pieces of the wave's 32 rows, 256 bytes of each of two groups of 8 of K.  The waves meet in LDS
// at the end to add their K parts in a fixed order.  K can be cut over blocks as well (float
// partial sums), which is what fills the chip for the products with few rows of W.
// It takes what the block products do not (launch_rows32): what kappai_rows32_takes names, and results that are not
// laid out in sixteens of bytes.
//
// Host side guarantees: W in fragment order, K / gridDim.y a multiple of 256, lda a multiple of
// 8, M * lda < 2^31.  Rows of A past M repeat the last row, pieces of W past the end the last
// piece (their products are not stored).
#define R32_NWN 2
#define R32_NWK 4
static_assert(R32_NWK * 64 == KAPPAI_ROWS32_RUN, "the rule for K ranges counts in runs");
template <typename TO, int MT, int EPI>
__global__ __launch_bounds__(R32_NWN * R32_NWK * WAVE) void gemm_bf16_rows32_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ Wf, const float* __restrict__ bias,
    TO* __restrict__ C, int M, int n_rows_w, int K, int lda, int ldc) {
  constexpr int NWN = R32_NWN, NWK = R32_NWK, NW = NWN * NWK, ROWS = 32 * MT, RUN = NWK * 64;
  constexpr int BUF = ROWS * RUN;                       // bf16 elements a buffer
  constexpr int INSTR = ROWS * NWK / 8;                 // load instructions a run (8 rows x 128 B)
  constexpr int PER_WAVE = INSTR / NW;
  static_assert(INSTR % NW == 0, "the loads of a run are dealt round the waves evenly");
  extern __shared__ __attribute__((aligned(1024))) bf16_t lds[];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wn = wave / NWK, wk = wave % NWK;
  const int r_in = lane % 32, hh = lane / 32;
  const int kblk = K / (int)gridDim.y;
  const int nruns = kblk / RUN;
  const int kb0 = blockIdx.y * kblk;
  C += (size_t)blockIdx.y * M * ldc;

  // W: lane -> row wrow0 + r_in, the 8 of K number hh (+ 2 for the second 16) of a piece of 16
  // rows x 32 of K; step s of a run (16 of K) lies in piece s / 2, half s % 2
  const int wrow0 = (blockIdx.x * NWN + wn) * 32;
  const int piece_row = min((wrow0 + r_in) / 16, n_rows_w / 16 - 1);
  const bf16_t* wbase = Wf + ((size_t)piece_row * (K / 32) + (kb0 + wk * 64) / 32) * 512 +
                        (hh * 16 + r_in % 16) * 8;
  auto load_w = [&](u32x4_t (&wv)[4], int run) {
    const bf16_t* p = wbase + (size_t)run * (RUN / 32) * 512;
#pragma unroll
    for (int s = 0; s < 4; ++s) wv[s] = load16(p + (s / 2) * 512 + (s % 2) * 256);
  };

  // A: instruction j of a run brings rows (j % (ROWS / 8)) * 8 + lane / 8 of the 64 number
  // j / (ROWS / 8) of the run; in LDS: the four 64s one after the other, rows of 128 bytes
  uint32_t aoff[PER_WAVE];
#pragma unroll
  for (int i = 0; i < PER_WAVE; ++i) {
    const int j = i * NW + wave;
    const int slice = j / (ROWS / 8), row = (j % (ROWS / 8)) * 8 + lane / 8;
    const int chunk = (lane % 8) ^ ((row >> 1) & 7);
    aoff[i] = (uint32_t)(min(row, M - 1) * lda + kb0 + slice * 64 + chunk * 8) *
              (uint32_t)sizeof(bf16_t);
  }
  auto stage = [&](int buf, int run) {
    const uint64_t p = reinterpret_cast<uint64_t>(A) + (uint64_t)run * (RUN * sizeof(bf16_t));
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)p);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
    const char* base = reinterpret_cast<const char*>(((uint64_t)hi << 32) | lo);
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) {
      const int j = i * NW + wave;
      const int slice = j / (ROWS / 8), rowblk = j % (ROWS / 8);
      __builtin_amdgcn_global_load_lds(
          KAPPAI_GPTR(base + aoff[i]),
          KAPPAI_LPTR(lds + buf * BUF + (slice * ROWS + rowblk * 8) * 64), 16, 0, 0);
    }
  };

  f32x16_t acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;
  // fragment of A: lane -> row 32 t + r_in, chunk 2 s + hh of the wave's 64
  int roff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
    roff[s] = (wk * ROWS + r_in) * 64 + (((2 * s + hh) ^ ((r_in >> 1) & 7)) * 8);
  auto products = [&](const u32x4_t (&wv)[4], int buf) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      u32x4_t av[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t)
        av[t] = *reinterpret_cast<const u32x4_t*>(lds + buf * BUF + roff[s] + t * 32 * 64);
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(wv[s]), as_bf16x8(av[t]), acc[t],
                                                         0, 0, 0);
    }
  };

  // W one run ahead in two register sets used in turn, A one run ahead in the other LDS buffer.
  // In every pass of the loop the loads of A are issued before those of W, and loads come back in
  // the order they were issued: waiting until only the latest pass's four loads of W are out means
  // that the run of A issued before them has landed (and the run of W before that).
  u32x4_t wv[2][4];
  stage(0, 0);
  load_w(wv[0], 0);
  for (int c = 0; c < nruns; c += 2) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int cc = c + s;
      if (cc >= nruns) break;
      // run cc of A was issued before the four loads of run cc of W, which may stay out
      __builtin_amdgcn_s_waitcnt(0x0F70 | 4);       // vmcnt(4)
      // everybody's part of run cc is there and nobody reads the other buffer any more (a bare
      // barrier: a fence would wait for the loads of W that are meant to stay in flight)
      __builtin_amdgcn_s_barrier();
      SCHED_FENCE();
      if (cc + 1 < nruns) {
        stage((s + 1) & 1, cc + 1);
        load_w(wv[(s + 1) & 1], cc + 1);
      }
      products(wv[s], s & 1);
    }
  }
  // the K parts meet: wave (wn, wk) adds up and stores row tiles wk, wk + 4, ...
  // acc[t][v] is C[row 32 t + r_in][column wrow0 + 8 (v / 4) + 4 hh + v % 4]
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
  constexpr int RSTRIDE = MT * 16 * WAVE;               // floats a wave
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) red[wave * RSTRIDE + (t * 16 + v) * WAVE + lane] = acc[t][v];
  __syncthreads();
  for (int t = wk; t < MT; t += NWK) {
    float sum[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      sum[v] = red[(wn * NWK) * RSTRIDE + (t * 16 + v) * WAVE + lane];
#pragma unroll
      for (int w = 1; w < NWK; ++w)
        sum[v] += red[(wn * NWK + w) * RSTRIDE + (t * 16 + v) * WAVE + lane];
    }
    const int gm = 32 * t + r_in;
    if (gm >= M) continue;
    if (EPI == 1) {
      // rows 0..15 of the wave's W are gate rows, 16..31 the up rows of the same 16 columns:
      // registers v and v + 8 of a lane
      if (wrow0 + 16 < n_rows_w) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          uint2 pk;
          const int row = wrow0 + 8 * g + 4 * hh;
          pk.x = pack_bf16x2(gated_f(sum[4 * g], sum[4 * g + 8], bias, row),
                             gated_f(sum[4 * g + 1], sum[4 * g + 9], bias, row + 1));
          pk.y = pack_bf16x2(gated_f(sum[4 * g + 2], sum[4 * g + 10], bias, row + 2),
                             gated_f(sum[4 * g + 3], sum[4 * g + 11], bias, row + 3));
          if constexpr (sizeof(TO) == 2)
            *reinterpret_cast<uint2*>(C + (size_t)gm * ldc + wrow0 / 2 + 8 * g + 4 * hh) = pk;
        }
      }
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int gn = wrow0 + 8 * g + 4 * hh;
        if (gn >= n_rows_w) continue;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = sum[4 * g + e] + ((bias && blockIdx.y == 0) ? bias[gn + e] : 0.f);
        TO* dst = C + (size_t)gm * ldc + gn;
        if constexpr (sizeof(TO) == 2) {
          uint2 pk;
          pk.x = pack_bf16x2(o[0], o[1]);
          pk.y = pack_bf16x2(o[2], o[3]);
          *reinterpret_cast<uint2*>(dst) = pk;
        } else {
          *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
        }
      }
    }
  }
}

template <typename TO, int MT, int EPI>
static void launch_rows32_cfg(const bf16_t* A, const bf16_t* Wf, const float* bias, TO* C, int M,
                              int n_rows_w, int K, int lda, int ldc, int ksplit,
                              hipStream_t stream) {
  constexpr int NW = R32_NWN * R32_NWK, ROWS = 32 * MT, RUN = R32_NWK * 64;
  constexpr size_t stage_bytes = 2 * (size_t)ROWS * RUN * sizeof(bf16_t);
  constexpr size_t red_bytes = (size_t)NW * MT * 16 * WAVE * sizeof(float);
  constexpr size_t lds_bytes = stage_bytes > red_bytes ? stage_bytes : red_bytes;
  static_assert(lds_bytes <= 160 * 1024, "a block's LDS");
  auto kern = gemm_bf16_rows32_kernel<TO, MT, EPI>;
  static bool attr_set = false;       // more than 64 KB of LDS has to be asked for once
  if (!attr_set) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds_bytes);
    attr_set = true;
  }
  hipLaunchKernelGGL(kern, dim3((n_rows_w + 32 * R32_NWN - 1) / (32 * R32_NWN), ksplit),
                     dim3(NW * WAVE), lds_bytes, stream, A, Wf, bias, C, M, n_rows_w, K, lda, ldc);
}

// Returns false when the shape does not fit (the caller then takes a block kernel).  The output
// must allow the kernel's stores of four values (8 or 16 bytes).  itself: no block product in its place.
template <typename TO, int EPI>
static bool launch_rows32(const bf16_t* A, const bf16_t* Wf, const float* bias, TO* C, int M,
                          int n_rows_w, int K, int lda, int ldc, int ksplit, bool itself, hipStream_t stream) {
  const int out_cols = EPI == 1 ? n_rows_w / 2 : n_rows_w;
  if (Wf == nullptr || M < 1 || M > KAPPAI_ROWS32_MAX_ROWS || ksplit < 1 || K % (ksplit * R32_NWK * 64) ||
      n_rows_w % (EPI == 1 ? 32 : 16) || (lda % 8) || (long)M * lda >= (1L << 31) - 2048 ||
      (out_cols % 4) || (ldc % 4) || ((uintptr_t)C % 16) || (EPI == 1 && sizeof(TO) != 2))
    return false;
  if (!itself && !kappai_rows32_takes(M, n_rows_w, K, ksplit) &&
      block256_fits<TO, EPI>(A, Wf, C, M, n_rows_w, K, lda, ldc, ksplit)) {
    launch_tile<TO, EPI>(A, nullptr, bias, C, M, n_rows_w, K, lda, ldc, ksplit, 0, stream, Wf);
    return true;
  }
  switch ((M + 31) / 32) {
    case 1: launch_rows32_cfg<TO, 1, EPI>(A, Wf, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream); break;
    case 2: launch_rows32_cfg<TO, 2, EPI>(A, Wf, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream); break;
    case 3: launch_rows32_cfg<TO, 3, EPI>(A, Wf, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream); break;
    default: launch_rows32_cfg<TO, 4, EPI>(A, Wf, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream); break;
  }
  return true;
}

template <typename TO, int EPI>
static int launch_bf16(const bf16_t* A, const bf16_t* W, const float* bias, TO* C, int M, int N,
                       int K, int lda, int ldc, int force_kernel, int ksplit, hipStream_t stream,
                       ConvStep cs = ConvStep{}, const bf16_t* Wf = nullptr, int a_frag = 0,
                       const Fuse& fuse = Fuse{}) {
  // a_frag: the rows of A lie in fragment order, which only the kernel for 1 to 16 rows reads
  if (a_frag && (M > 16 || force_kernel == 1 || force_kernel >= 3)) return (int)hipErrorInvalidValue;
  // so are the row scale and the residual epilogue (and the latter only with K in one piece)
  const bool fused = fuse.rsc.ss != nullptr || fuse.ro.resid != nullptr || fuse.c_frag;
  if (fuse.c_frag && (EPI == 0 || (N % 32))) return (int)hipErrorInvalidValue;
  if (fused && (M > 16 || force_kernel == 1 || force_kernel >= 3)) return (int)hipErrorInvalidValue;
  if (fuse.ro.resid != nullptr) {
    if (EPI != 0 || ksplit != 1 || fuse.rsc.ss != nullptr) return (int)hipErrorInvalidValue;
    launch_into_resid(A, W, bias, M, N, K, lda, fuse.ro, stream, Wf, a_frag);
    KAPPAI_RETURN_LAUNCH_STATUS();
  }
  if (fuse.rsc.ss != nullptr && ksplit != 1) return (int)hipErrorInvalidValue;
  // Wf: W in fragment order (see the kernel for 1 to 16 rows); W may be null when Wf is there
  // N counts output columns; with the SwiGLU epilogue W has 2N rows
  // a very wide plain product (the output head) with more than 32 rows streams faster through
  // the 128 x 128 blocks than through the decode kernel, which reads the rows once per 32 columns
  const bool wide_head = EPI == 0 && M > 32 && N >= 16384 && force_kernel == 0 && ksplit == 1 &&
                         block256_fits<TO, EPI>(A, W, C, M, N, K, lda, ldc, ksplit);
  // 25 to 128 rows: the block products, or 32 x 32 tiles with the rows through LDS, when W is there in
  // fragment order and the shape fits (else the kernels below)
  if constexpr (EPI != 2) {
    const bool forced = force_kernel == 12 || force_kernel == 18;
    if (forced || (force_kernel == 0 && M > KAPPAI_ROWS32_MIN_ROWS && M <= KAPPAI_ROWS32_MAX_ROWS &&
                   Wf != nullptr && !wide_head)) {
      if (launch_rows32<TO, EPI>(A, Wf, bias, C, M, EPI == 1 ? 2 * N : N, K, lda, ldc, ksplit,
                                 force_kernel == 18, stream))
        KAPPAI_RETURN_LAUNCH_STATUS();
      if (forced) return (int)hipErrorInvalidValue;
    }
  } else if (force_kernel == 12 || force_kernel == 18) {
    return (int)hipErrorInvalidValue;
  }
  // 17 to 64 rows and blocks enough to fill half the chip: the rows go through LDS
  if constexpr (EPI != 2) {
    const int n_rows_w = EPI == 1 ? 2 * N : N;
    const long sr_blocks = (long)((n_rows_w + 32 * SR_NWN - 1) / (32 * SR_NWN)) * ksplit;
    // (with W in fragment order the kernel for few rows keeps up to 24 rows: gate/up 16.6
    // against 17.5 us at 24 rows, 15.7 against 17.6 at 17)
    if (force_kernel == 9 ||
        (force_kernel == 0 && M > (Wf ? 24 : 16) && M <= 64 && sr_blocks >= 128 && !wide_head)) {
      if (launch_shared_rows<TO, EPI>(A, W, bias, C, M, n_rows_w, K, lda, ldc, ksplit, stream, Wf))
        KAPPAI_RETURN_LAUNCH_STATUS();
      if (force_kernel == 9) return (int)hipErrorInvalidValue;
    }
  } else if (force_kernel == 9) {
    return (int)hipErrorInvalidValue;
  }
  if (M <= 64 && force_kernel != 1 && force_kernel < 3 && !wide_head) {
    const int mt = (M + 15) / 16;
    switch (mt) {
      case 1:
        launch_skinny_mt<TO, 1, EPI>(A, W, bias, C, M, N, K, lda, ldc, ksplit, cs, stream, fuse,
                                     Wf, a_frag);
        break;
      case 2:
        launch_skinny_mt<TO, 2, EPI>(A, W, bias, C, M, N, K, lda, ldc, ksplit, cs, stream, Fuse{},
                                     Wf);
        break;
      case 3:
        launch_skinny_mt<TO, 3, EPI>(A, W, bias, C, M, N, K, lda, ldc, ksplit, cs, stream, Fuse{},
                                     Wf);
        break;
      default:
        launch_skinny_mt<TO, 4, EPI>(A, W, bias, C, M, N, K, lda, ldc, ksplit, cs, stream, Fuse{},
                                     Wf);
        break;
    }
  } else {
    // rows of W = columns the tiles run over
    launch_tile<TO, EPI>(A, W, bias, C, M, EPI == 1 ? 2 * N : N, K, lda, ldc, ksplit,
                         force_kernel >= 3 ? force_kernel - 2 : (wide_head && M <= 64 ? 6 : 0),
                         stream, Wf);
  }
  KAPPAI_RETURN_LAUNCH_STATUS();
}

// K, lda must be multiples of 8 and A, W 16-byte aligned (checked by the caller).
// force_kernel: 0 = by M, 1 = tile kernel, 2 = skinny kernel (M <= 64 only), 3..8 = tile kernel
// with block shape 1..6 (see launch_tile), 9 = shared-rows kernel (17 to 64 rows, K / ksplit a
// multiple of 512), 10 = block shape 8, 11 = block shape 9, 12 = what steps of 25 to 128 rows take
// (1 to 128 rows, W in fragment order, K / ksplit a multiple of 256), 13 to 17 = block shapes 11 to
// 15, 18 = gemm_bf16_rows32 wherever 12 is taken; for tests and tuning.
// ksplit > 1 (float output only): C is [ksplit][M][ldc] partial sums over K ranges.
// W_frag: null, or W in fragment order (K a multiple of 32, rows a multiple of 16); W may then
// be null: every kernel reads the fragment order (only kappai_gemm_bf16_any needs rows).
static bool frag_ok(const void* W_frag, int rows, int K) {
  return W_frag == nullptr || (K % 32 == 0 && rows % 16 == 0 && ((uintptr_t)W_frag % 16) == 0);
}

// The fused forms (at most 16 rows, see RowScale and ResidOut in the kernel for 1 to 16 rows):
// scale_ss [scale_parts][16] (or null) scales every result row by 1 / sqrt(sum of its parts / K +
// scale_eps); resid [M, ldr] (or null; float output, ksplit 1) receives the result added in place
// instead of C, and with norm_w also rows_out (bf16(resid * norm_w), [M, N] or fragment order)
// and ss_out [(N + 7) / 8][16].
static bool fuse_ok(const Fuse& f, int M, int N, int K, int out_is_f32, int ksplit) {
  if (f.rsc.ss != nullptr && (M > 16 || f.rsc.n_parts < 1 || ksplit != 1)) return false;
  if (f.c_frag && M > 16) return false;
  if (f.ro.resid != nullptr) {
    if (M > 16 || !out_is_f32 || ksplit != 1 || f.ro.ldr < N) return false;
    if (f.ro.norm_w != nullptr && (f.ro.rows == nullptr || f.ro.ss == nullptr)) return false;
    if (f.ro.rows_frag && (N % 32)) return false;
  } else if (f.ro.norm_w != nullptr || f.ro.rows != nullptr) {
    return false;
  }
  return true;
}

extern "C" int kappai_gemm_bf16(const void* A, const void* W, const void* W_frag, const float* bias,
                                void* C, int M, int N, int K, int lda, int ldc, int out_is_f32,
                                int force_kernel, int ksplit, int a_frag, const float* scale_ss,
                                int scale_parts, float scale_eps, float* resid, int ldr,
                                const float* norm_w, void* rows_out, int rows_frag, float* ss_out,
                                hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if ((K % 8) || (lda % 8) || ksplit < 1 || ksplit > 64) return (int)hipErrorInvalidValue;
  if (!frag_ok(W_frag, N, K) || (a_frag && (K % 32))) return (int)hipErrorInvalidValue;
  if (force_kernel == 2 && M > 64) return (int)hipErrorInvalidValue;
  if (ksplit > 1 && !out_is_f32) return (int)hipErrorInvalidValue;
  Fuse fuse{RowScale{scale_ss, scale_parts, scale_eps},
            ResidOut{resid, ldr, resid && rows_out ? norm_w : nullptr,
                     resid ? (bf16_t*)rows_out : nullptr, rows_frag, ss_out}};
  if (!fuse_ok(fuse, M, N, K, out_is_f32, ksplit)) return (int)hipErrorInvalidValue;
  if (out_is_f32)
    return launch_bf16<float, 0>((const bf16_t*)A, (const bf16_t*)W, bias, (float*)C, M, N, K, lda,
                                 ldc, force_kernel, ksplit, stream, ConvStep{},
                                 (const bf16_t*)W_frag, a_frag, fuse);
  return launch_bf16<bf16_t, 0>((const bf16_t*)A, (const bf16_t*)W, bias, (bf16_t*)C, M, N, K, lda,
                                ldc, force_kernel, 1, stream, ConvStep{}, (const bf16_t*)W_frag,
                                a_frag, fuse);
}

// C[M, F] = silu(A Wg^T) * (A Wu^T) with W = gate and up rows interleaved in groups of 16,
// [2F, K]; F must be a multiple of 16.  `consts`: the gate's constants, where GATE_ACT has any.
extern "C" int kappai_gemm_bf16_gated(const void* A, const void* W, const void* W_frag, void* C,
                                      int M, int F, int K, int lda, int ldc, int force_kernel,
                                      int a_frag, const float* scale_ss, int scale_parts,
                                      float scale_eps, int c_frag, const float* consts,
                                      hipStream_t stream) {
  if (M <= 0 || F <= 0) return 0;
  if ((consts != nullptr) != (GATE_ACT >= 2)) return (int)hipErrorInvalidValue;
  if ((K % 8) || (lda % 8) || (F % 16)) return (int)hipErrorInvalidValue;
  if (force_kernel == 2 && M > 64) return (int)hipErrorInvalidValue;
  if (!frag_ok(W_frag, 2 * F, K) || (a_frag && (K % 32))) return (int)hipErrorInvalidValue;
  Fuse fuse{RowScale{scale_ss, scale_parts, scale_eps}, ResidOut{}, c_frag};
  if (!fuse_ok(fuse, M, F, K, 0, 1)) return (int)hipErrorInvalidValue;
  return launch_bf16<bf16_t, 1>((const bf16_t*)A, (const bf16_t*)W, consts, (bf16_t*)C, M, F, K,
                                lda, ldc, force_kernel, 1, stream, ConvStep{},
                                (const bf16_t*)W_frag, a_frag, fuse);
}

extern "C" int kappai_gemm_bf16_swiglu(const void* A, const void* W, const void* W_frag, void* C,
                                       int M, int F, int K, int lda, int ldc, int force_kernel,
                                       int a_frag, const float* scale_ss, int scale_parts,
                                       float scale_eps, int c_frag, hipStream_t stream) {
  return kappai_gemm_bf16_gated(A, W, W_frag, C, M, F, K, lda, ldc, force_kernel, a_frag, scale_ss,
                                scale_parts, scale_eps, c_frag, nullptr, stream);
}

// Conv layer decode step in one kernel: C[M, D] = Cgate * conv(Bgate * x | state) from A [M, K]
// and the in_proj matrix W [3D, K]; M <= 64, one row a request; D a multiple of 16.
extern "C" int kappai_gemm_bf16_shortconv_step(const void* A, const void* W, const void* W_frag,
                                               const float* bias,
                                               void* C, int M, int D, int K, int lda,
                                               const float* taps, const float* conv_bias,
                                               float* state, const int* seg_pos0,
                                               const int* seg_slot, int L, int a_frag,
                                               const float* scale_ss, int scale_parts,
                                               float scale_eps, int c_frag, hipStream_t stream) {
  if (M <= 0 || D <= 0) return 0;
  if ((K % 8) || (lda % 8) || (D % 16) || M > 64 || L < 2) return (int)hipErrorInvalidValue;
  if (!frag_ok(W_frag, 3 * D, K) || (a_frag && ((K % 32) || M > 16)))
    return (int)hipErrorInvalidValue;
  Fuse fuse{RowScale{scale_ss, scale_parts, scale_eps}, ResidOut{}, c_frag};
  if (!fuse_ok(fuse, M, D, K, 0, 1) || (c_frag && (D % 32))) return (int)hipErrorInvalidValue;
  const bf16_t* wf = (const bf16_t*)W_frag;
  ConvStep cs{taps, conv_bias, state, seg_pos0, seg_slot, L};
  if (D / 16 < 256) {
    // too few blocks of 16 channels for the chip: 8 channels a block
    const bf16_t* a = (const bf16_t*)A;
    const bf16_t* w = (const bf16_t*)W;
    bf16_t* c = (bf16_t*)C;
    switch ((M + 15) / 16) {
      case 1:
        launch_skinny_mt<bf16_t, 1, 3>(a, w, bias, c, M, D, K, lda, D, 1, cs, stream, fuse, wf,
                                       a_frag);
        break;
      case 2:
        launch_skinny_mt<bf16_t, 2, 3>(a, w, bias, c, M, D, K, lda, D, 1, cs, stream, Fuse{}, wf);
        break;
      case 3:
        launch_skinny_mt<bf16_t, 3, 3>(a, w, bias, c, M, D, K, lda, D, 1, cs, stream, Fuse{}, wf);
        break;
      default:
        launch_skinny_mt<bf16_t, 4, 3>(a, w, bias, c, M, D, K, lda, D, 1, cs, stream, Fuse{}, wf);
        break;
    }
    KAPPAI_RETURN_LAUNCH_STATUS();
  }
  return launch_bf16<bf16_t, 2>((const bf16_t*)A, (const bf16_t*)W, bias, (bf16_t*)C, M, D, K, lda,
                                D, 2, 1, stream, cs, wf, a_frag, fuse);
}

// ---------------------------------------------------------------------------------------
// bf16 at any size and alignment (K or a row stride that is no multiple of 8): one wave per
// row and four output columns, lanes stride over K with 2-byte loads, float sums added up
// across the wave.  Slow, and only there so that no width is refused.
// ---------------------------------------------------------------------------------------
template <typename TO>
__global__ __launch_bounds__(WAVE) void gemm_bf16_any_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, const float* __restrict__ bias,
    TO* __restrict__ C, int M, int N, int K, int lda, int ldc) {
  const int m = blockIdx.y, n0 = blockIdx.x * 4, lane = threadIdx.x;
  const bf16_t* a = A + (size_t)m * lda;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k = lane; k < K; k += WAVE) {
    const float x = bf16_to_f32(a[k]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n0 + j < N) acc[j] = fmaf(x, bf16_to_f32(W[(size_t)(n0 + j) * K + k]), acc[j]);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float sum = wave_sum(acc[j]);
    if (lane == 0 && n0 + j < N)
      store_out(C + (size_t)m * ldc + n0 + j, sum + (bias ? bias[n0 + j] : 0.f));
  }
}

extern "C" int kappai_gemm_bf16_any(const void* A, const void* W, const float* bias, void* C,
                                    int M, int N, int K, int lda, int ldc, int out_is_f32,
                                    hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K < 1 || M > 65535) return (int)hipErrorInvalidValue;
  const dim3 grid((N + 3) / 4, M);
  if (out_is_f32)
    hipLaunchKernelGGL(gemm_bf16_any_kernel<float>, grid, dim3(WAVE), 0, stream, (const bf16_t*)A,
                       (const bf16_t*)W, bias, (float*)C, M, N, K, lda, ldc);
  else
    hipLaunchKernelGGL(gemm_bf16_any_kernel<bf16_t>, grid, dim3(WAVE), 0, stream,
                       (const bf16_t*)A, (const bf16_t*)W, bias, (bf16_t*)C, M, N, K, lda, ldc);
  KAPPAI_RETURN_LAUNCH_STATUS();
}
