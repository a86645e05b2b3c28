// bfloat16 attention over the paged cache on the matrix cores, for one head size
// (HEAD_DIM, a multiple of 16, set when the file is compiled).
//
// Both kernels keep "one query per lane column".  For a tile of keys they compute
//     S^T = K Q^T        A = K rows (a key per lane row, 8 consecutive d per lane)
//                        B = Q     (a query per lane column)
//     O^T += V^T P^T     A = V^T   (a d index per lane row, 8 key slots per lane)
//                        B = P^T   (the lane's own values of S^T, no data movement)
// so that a lane holds, for ITS query, scores of several keys and later outputs of several d
// indices: the running maximum, the running sum and the rescaling are per lane, in float.
// The value pool is stored transposed, [page][kv_head][head_dim][page_size], which makes the
// 8 key slots of the A operand two 8-byte loads.  page_size must be a multiple of 16.
//
//   attn_prefill   v_mfma_f32_32x32x16_bf16; one block per (tile of 32 rows of a segment, head),
//                  its waves sharing out the key tiles
//   attn_decode    v_mfma_f32_16x16x32_bf16; one wave per (row, kv head, split of the keys): the
//                  query heads that share the kv head are the columns; partial results are
//                  merged by attn_merge.
// Formulas: softmax(q.k/sqrt(d)) v over keys lo..pos (kappai: src/backend/cpu/scalar/core.c:383-433,
// 623-666), online softmax as in its flash form (:386-413).
#include "common.h"
#include "no_alloc.h"
#include "score_mods.h"
#include <stdio.h>

#ifndef HEAD_DIM
#error "compile with -DHEAD_DIM=<multiple of 16>"
#endif
static_assert(HEAD_DIM % 16 == 0 && HEAD_DIM >= 16 && HEAD_DIM <= 256, "unsupported head size");

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_any_t;   // at any float
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

__device__ __forceinline__ bf16x8_t as_frag(u32x4_t v) { return __builtin_bit_cast(bf16x8_t, v); }
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) { return pack_bf16x2(lo, hi); }
// 2^x for x <= 0 straight from the hardware (v_exp_f32); results below the normal range flush
// to zero, which is what a softmax weight that small is worth
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// keep the j-th of four bf16 values only if keep bit j is set
__device__ __forceinline__ u32x2_t mask4(u32x2_t v, int keep) {
  const uint32_t m0 = ((keep & 1) ? 0x0000ffffu : 0u) | ((keep & 2) ? 0xffff0000u : 0u);
  const uint32_t m1 = ((keep & 4) ? 0x0000ffffu : 0u) | ((keep & 8) ? 0xffff0000u : 0u);
  return (u32x2_t){v.x & m0, v.y & m1};
}

#define LOG2E 1.4426950408889634f

// the value that lane ^ 32 holds, by one swap of the wave's halves (no trip through LDS)
__device__ __forceinline__ float other_half(float x) {
  const uint32_t u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  // r[0] = the lower half's values in both halves, r[1] = the upper half's
  return __uint_as_float((threadIdx.x & 32) ? r[0] : r[1]);
}

// four key slots of V^T for d index `dd`, keys key0..key0+3 (one 16-key group: one page);
// keys outside [lo, hi] read as zero
__device__ __forceinline__ u32x2_t load_vt4(const bf16_t* __restrict__ vt_pool,
                                            const int* __restrict__ bt, int G, int g, int ps,
                                            int dd, int key0, int lo, int hi) {
  u32x2_t z = {0u, 0u};
  if (dd >= HEAD_DIM || key0 > hi || key0 + 3 < lo) return z;
  const int page = bt[key0 / ps];
  if (page < 0) return z;
  const bf16_t* p = vt_pool + (((size_t)page * G + g) * HEAD_DIM + dd) * ps + key0 % ps;
  u32x2_t v = *reinterpret_cast<const u32x2_t*>(p);
  int keep = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (key0 + i >= lo && key0 + i <= hi) keep |= 1 << i;
  return keep == 15 ? v : mask4(v, keep);
}

// the same with the page already looked up.  The load itself is unconditional (from the pool's
// first page when the keys are not wanted) and its result is masked, so that the compiler
// keeps it in straight-line code and can leave it in flight across other work.
__device__ __forceinline__ u32x2_t load_vt4_pg(const bf16_t* __restrict__ vt_pool, int page, int G,
                                               int g, int ps, int dd, int key0, int lo, int hi) {
  const bool want = dd < HEAD_DIM && key0 <= hi && key0 + 3 >= lo && page >= 0;
  const size_t off =
      want ? (((size_t)page * G + g) * HEAD_DIM + dd) * ps + key0 % ps : (size_t)0;
  u32x2_t v = *reinterpret_cast<const u32x2_t*>(vt_pool + off);
  int keep = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (want && key0 + i >= lo && key0 + i <= hi) keep |= 1 << i;
  return mask4(v, keep);
}

// eight key slots of V^T for d index `dd`, keys key0..key0+7 (half a 16-key group: one page),
// the page already looked up; keys outside [lo, hi] read as zero
__device__ __forceinline__ u32x4_t load_vt8_pg(const bf16_t* __restrict__ vt_pool, int page, int G,
                                               int g, int ps, int dd, int key0, int lo, int hi) {
  const bool want = dd < HEAD_DIM && key0 <= hi && key0 + 7 >= lo && page >= 0;
  const size_t off =
      want ? (((size_t)page * G + g) * HEAD_DIM + dd) * ps + key0 % ps : (size_t)0;
  const u32x4_t v = *reinterpret_cast<const u32x4_t*>(vt_pool + off);
  uint32_t m[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool k0 = want && key0 + 2 * i >= lo && key0 + 2 * i <= hi;
    const bool k1 = want && key0 + 2 * i + 1 >= lo && key0 + 2 * i + 1 <= hi;
    m[i] = (k0 ? 0x0000ffffu : 0u) | (k1 ? 0xffff0000u : 0u);
  }
  return (u32x4_t){v.x & m[0], v.y & m[1], v.z & m[2], v.w & m[3]};
}

__device__ __forceinline__ u32x4_t load_k8_pg(const bf16_t* __restrict__ k_pool, int page, int G,
                                              int g, int ps, int key, int d0, int lo, int hi) {
  const bool want = d0 < HEAD_DIM && key >= lo && key <= hi && page >= 0;
  const size_t off = want ? (((size_t)page * G + g) * ps + key % ps) * HEAD_DIM + d0 : (size_t)0;
  u32x4_t v = *reinterpret_cast<const u32x4_t*>(k_pool + off);
  const uint32_t m = want ? 0xffffffffu : 0u;
  return (u32x4_t){v.x & m, v.y & m, v.z & m, v.w & m};
}

// eight consecutive d of key `key` starting at d0; zero outside [lo, hi] or beyond the head
__device__ __forceinline__ u32x4_t load_k8(const bf16_t* __restrict__ k_pool,
                                           const int* __restrict__ bt, int G, int g, int ps,
                                           int key, int d0, int lo, int hi) {
  u32x4_t z = {0u, 0u, 0u, 0u};
  if (d0 >= HEAD_DIM || key < lo || key > hi) return z;
  const int page = bt[key / ps];
  if (page < 0) return z;
  return *reinterpret_cast<const u32x4_t*>(
      k_pool + (((size_t)page * G + g) * ps + key % ps) * HEAD_DIM + d0);
}

// ---------------------------------------------------------------------------------------
// prefill: q_tiles[tile] = (segment, first row, rows <= 32, unused)
// ---------------------------------------------------------------------------------------
#define P_KS (HEAD_DIM / 16)            // k-steps of S^T over d
#define P_MT ((HEAD_DIM + 31) / 32)     // row tiles of O^T over d

// (decode) keys whose loads a wave has in flight at once (their registers: keys * HEAD_DIM / 64)
#define D_KPW (HEAD_DIM <= 64 ? 128 : (HEAD_DIM <= 128 ? 64 : 32))
// What the shares of a row's keys over blocks are whole numbers of.  A block costs a place in a second kernel:
// 96 keys a block for 128 are 3 to 9 % more at head sizes 80 to 128, where 96 are three parts for two (4 rows of
// up to 8,000 keys, 32 heads of 128 on 8: 28.5 us against 26.2), and equal at 64.
#define D_SPLIT_SHARE (HEAD_DIM == 64 ? 32 : D_KPW)
// ... and over the waves of a block in a decode step: 64 keys for 32 are 2 to 4 % more at head sizes 64 and 128.  At
// the others whole chunks, as the kernel had them: one measure of the differential attention's maps of 16,
// whose difference leaves little but the rounding of either, hangs on the order of their sums.  (A decoded
// row beside portions takes shares of 32 at every head size.)
#define D_BLOCK_SHARE (HEAD_DIM == 64 || HEAD_DIM == 128 ? 32 : D_KPW)

// One row and one kv head by a block of NW waves, which take equal shares of the keys and meet in `sh`
// (NW (rep HEAD_DIM + 32) floats of LDS; rep <= 16): defined with the decode kernels.
// (FUSED: with the prologue of `qk` in the waves that have keys)
struct QkFuse;
template <bool MODS, bool FUSED = false, int SHARE = 32>
__device__ __forceinline__ void attn_one_row(const bf16_t* q, int q_stride, const bf16_t* k_pool,
                                             const bf16_t* vt_pool, bf16_t* out, int out_stride,
                                             const int* bt, int max_blocks, int t, int pos, int g, int H,
                                             int G, int ps, int window, float scale,
                                             const kappai_score_mods& mods, float* sh, int NW,
                                             const QkFuse* qk = nullptr);

// waves of a block: they share one q tile and take its key tiles in turn, which shortens the
// longest chain of dependent work fourfold; their partial results meet in LDS
#define P_NW (HEAD_DIM <= 128 ? 4 : 1)

// MODS: the scores pass a cap and a bias by distance between the scaled product and the softmax
// (score_mods.h).  The head's row of the bias table lies in LDS (tables of up to P_BIAS_MAX
// columns; longer ones are read where they are), and a key tile that is further from every query
// of the block than the table reaches takes the table's last column without looking.  With kept
// first positions the tiles that hold them stand in front of the window's first tile
// (kappai_key_at).  A sink may join the denominator with or without MODS.
#define P_BIAS_MAX 2048
#define P_BIAS_EDGE 64
// waves a SIMD that the registers are held down to (2,048 rows of 32 heads of 64: 132 us with one
// wave, which is what the compiler settles on by itself, 76 us with two)
#define P_MIN_WAVES (HEAD_DIM <= 96 ? 2 : 1)
template <bool MODS>
__global__ __launch_bounds__(P_NW * WAVE, P_MIN_WAVES) void attn_prefill_kernel(
    const int* __restrict__ q_tiles, const int* __restrict__ row_pos,
    const int* __restrict__ block_tables, int max_blocks, int H, int G, int ps, int q_stride, int window,
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ vt_pool,
    bf16_t* __restrict__ out, int out_stride, float scale, kappai_score_mods mods) {
  // later tiles of a segment have more keys: they are started first
  const int tile = gridDim.x - 1 - blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x % WAVE;
  // the wave's number in scalar registers: everything that depends only on the key tile (its
  // pages, its base addresses, whether it is masked) is then scalar work
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int seg = q_tiles[4 * tile], r0 = q_tiles[4 * tile + 1], nr = q_tiles[4 * tile + 2];
  const int g = h / (H / G);
  const int col = lane % 32, hh = lane / 32;
  const int* bt = block_tables + (size_t)seg * max_blocks;
  const int pos_first = row_pos[r0], pos_last = pos_first + nr - 1;
  // what waves 1.. hand to wave 0
  constexpr int SH_O = P_NW > 1 ? (P_NW - 1) * P_MT * 16 * WAVE : 1;
  __shared__ float sh_o[SH_O];
  if constexpr (!MODS && P_NW > 1) {
    // A decoded token beside portions: all query heads of its kv head at once and an equal share of the keys
    // a wave, as in a decode step.  Walked like a portion's tile, head by head and 32 keys at a time, a
    // row's keys were read rep times and a chain of up to 12 round trips to memory held the kernel: 63 rows
    // of up to 1,500 keys beside a portion of 512, 16 heads on 8: 43.9 us, now 30.6; 32 heads on 8 in
    // the kernel below 62.4, now 29.2; 8 rows of up to 500 keys 11.0, now 10.3.
    static_assert(P_NW * (16 * HEAD_DIM + 32) <= SH_O || HEAD_DIM < 32, "LDS of a lone row");
    const int rep = H / G;
    if (nr == 1 && P_NW * (rep * HEAD_DIM + 32) <= SH_O && rep <= 16) {
      if (h % rep == 0)
        attn_one_row<false>(q, q_stride, k_pool, vt_pool, out, out_stride, bt, max_blocks, r0, pos_first,
                            g, H, G, ps, window, scale, mods, sh_o, P_NW);
      return;
    }
  }
  const bool row_ok = col < nr;
  const int my_pos = row_ok ? pos_first + col : -1;
  const int my_lo = kappai_first_key(my_pos, window);
  const int lo_tile = kappai_first_key(pos_first, window);

  bf16x8_t qf[P_KS];
  {
    const bf16_t* qr = q + (size_t)(r0 + (row_ok ? col : 0)) * q_stride + (size_t)h * HEAD_DIM;
#pragma unroll
    for (int ks = 0; ks < P_KS; ++ks) {
      u32x4_t v = {0u, 0u, 0u, 0u};
      if (row_ok) v = *reinterpret_cast<const u32x4_t*>(qr + 16 * ks + 8 * hh);
      qf[ks] = as_frag(v);
    }
  }
  f32x16_t o[P_MT];
#pragma unroll
  for (int mt = 0; mt < P_MT; ++mt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[mt][v] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  // MODS, where the registers suffice: the sums of the weights come from the matrix cores (a V^T
  // fragment of ones), of the same rounded weights that the output is made of
  constexpr bool MFMA_SUM = MODS && HEAD_DIM <= 64;
  f32x16_t o_sum;
#pragma unroll
  for (int v = 0; v < 16; ++v) o_sum[v] = 0.f;
  const bf16x8_t ones = as_frag((u32x4_t){0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
  // (with MODS the scores are scaled, worked on and brought to units of log 2 one by one)
  const float sc = MODS ? 1.0f : scale * LOG2E;
  // the head's biases in units of log 2, the far ones first, with room for the distances that only
  // masked scores and the block's spread of rows reach: place bias_top - dist
  __shared__ float sh_bias[MODS ? P_BIAS_MAX + 2 * P_BIAS_EDGE : 1];
  const bool has_bias = MODS && mods.dist_bias != nullptr;
  const bool bias_in_lds = has_bias && mods.dist_cols <= P_BIAS_MAX;
  const float* bias_row = has_bias ? kappai_bias_row(mods, h) : nullptr;
  const float far_bias = has_bias ? bias_row[mods.dist_cols - 1] * LOG2E : 0.f;
  const int bias_top = MODS ? mods.dist_cols - 1 + P_BIAS_EDGE : 0;
  const int bias_pos = row_ok ? my_pos : pos_first;
  if (MODS) {
    if (bias_in_lds)
      for (int i = threadIdx.x; i < mods.dist_cols + 2 * P_BIAS_EDGE; i += P_NW * WAVE)
        sh_bias[i] = bias_row[max(0, min(bias_top - i, mods.dist_cols - 1))] * LOG2E;
    __syncthreads();
  }

  // A tile of 32 keys is "whole" when every row of the q tile sees all of its keys: then nothing
  // is masked, and addresses are a base that is the same for all lanes of a 16-key group (its
  // page) plus an offset that a lane computes once.  The tiles at the window's lower edge and at
  // the diagonal take the general path.  Either way the loads of the next tile are issued
  // before the current one is worked on.
  const int lo_last = kappai_first_key(pos_last, window);
  const int keep = MODS ? mods.keep_first : 0;
  const int lo32 = (lo_tile / 32) * 32;
  const int kept = MODS ? kappai_kept_places(keep, lo32) : 0;
  auto whole = [&](int kb) {
    return (kb >= lo_last || (MODS && kb + 31 < keep)) && kb + 31 <= pos_first;
  };
  const int k_lane = (col % 16) * HEAD_DIM + 8 * hh;       // + 16*ks
  const int v_lane = col * ps + 4 * hh;                    // + 32*mt*ps (+ 8)
  constexpr bool P_AHEAD = HEAD_DIM <= 128;      // beyond that the registers do not suffice
  constexpr int P_NB = P_AHEAD ? 2 : 1;
  u32x4_t kfr[P_NB][P_KS];
  u32x2_t vfa[P_NB][2][P_MT], vfb[P_NB][2][P_MT];
  auto fetch = [&](int buf, int kb) {
    const int g0 = min(kb / ps, max_blocks - 1), g1 = min((kb + 16) / ps, max_blocks - 1);
    const int pg0 = kb <= pos_last ? bt[g0] : -1;
    const int pg1 = kb + 16 <= pos_last ? bt[g1] : -1;
    if (whole(kb)) {
      const bf16_t* kb0p = k_pool + (((size_t)pg0 * G + g) * ps + kb % ps) * HEAD_DIM;
      const bf16_t* kb1p = k_pool + (((size_t)pg1 * G + g) * ps + (kb + 16) % ps) * HEAD_DIM;
      const bf16_t* kp = (col < 16 ? kb0p : kb1p) + k_lane;
#pragma unroll
      for (int ks = 0; ks < P_KS; ++ks)
        kfr[buf][ks] = *reinterpret_cast<const u32x4_t*>(kp + 16 * ks);
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bf16_t* vp = vt_pool + ((size_t)(st == 0 ? pg0 : pg1) * G + g) * HEAD_DIM * ps +
                           (kb + 16 * st) % ps + v_lane;
#pragma unroll
        for (int mt = 0; mt < P_MT; ++mt) {
          const bool dok = HEAD_DIM % 32 == 0 || 32 * mt + col < HEAD_DIM;
          const bf16_t* vq = vp + (dok ? 32 * mt * ps : -v_lane);
          u32x2_t a = *reinterpret_cast<const u32x2_t*>(vq);
          u32x2_t b = *reinterpret_cast<const u32x2_t*>(vq + 8);
          if (!dok) a = b = (u32x2_t){0u, 0u};
          vfa[buf][st][mt] = a;
          vfb[buf][st][mt] = b;
        }
      }
      return;
    }
    // what no query of the block sees reads as zero
    const int f_lo = MODS && kb < keep ? kb : lo_tile;
    const int f_hi = MODS && kb < lo32 ? keep - 1 : pos_last;
    const int my_key = kb + col;
    const int my_pg = col < 16 ? pg0 : pg1;
#pragma unroll
    for (int ks = 0; ks < P_KS; ++ks)
      kfr[buf][ks] =
          load_k8_pg(k_pool, my_pg, G, g, ps, my_key, 16 * ks + 8 * hh, f_lo, f_hi);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const int key0 = kb + 16 * st + 4 * hh;
      const int pg = st == 0 ? pg0 : pg1;
#pragma unroll
      for (int mt = 0; mt < P_MT; ++mt) {
        const int dd = 32 * mt + col;
        vfa[buf][st][mt] = load_vt4_pg(vt_pool, pg, G, g, ps, dd, key0, f_lo, f_hi);
        vfb[buf][st][mt] = load_vt4_pg(vt_pool, pg, G, g, ps, dd, key0 + 8, f_lo, f_hi);
      }
    }
  };
  auto work = [&](int buf, int kb) {
    // ---- S^T tile: 32 keys x 32 queries -------------------------------------------------
    f32x16_t s;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
    for (int ks = 0; ks < P_KS; ++ks)
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(kfr[buf][ks]), qf[ks], s, 0, 0, 0);
    // lane holds, for query `col`, keys kb + 8*(v/4) + 4*hh + v%4
    if (MODS) {
      const bool capped = mods.softcap > 0.f;
      const float by = capped ? LOG2E : scale * LOG2E;
      if (capped)
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = kappai_fast_cap(s[v] * scale, mods.softcap);
      if (!has_bias || pos_first - (kb + 31) >= mods.dist_cols - 1) {
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = fmaf(s[v], by, far_bias);
      } else if (bias_in_lds) {
        // (a distance here is at most dist_cols - 2 + 62 and at least -62)
        const float* at0 = sh_bias + (bias_top - (bias_pos - kb - 4 * hh));
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = fmaf(s[v], by, at0[8 * (v / 4) + v % 4]);
      } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int dist = bias_pos - (kb + 8 * (v / 4) + 4 * hh + v % 4);
          s[v] = fmaf(s[v], by, bias_row[max(0, min(dist, mods.dist_cols - 1))] * LOG2E);
        }
      }
    }
    float mloc = -INFINITY;
    if (whole(kb)) {
#pragma unroll
      for (int v = 0; v < 16; ++v) mloc = fmaxf(mloc, s[v]);
      mloc *= sc;           // sc > 0: scaling commutes with the maximum
    } else {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int key = kb + 8 * (v / 4) + 4 * hh + v % 4;
        const bool ok = key <= my_pos && (key >= my_lo || (MODS && key < keep));
        s[v] = ok ? s[v] : -INFINITY;
        mloc = fmaxf(mloc, s[v] * sc);
      }
    }
    mloc = fmaxf(mloc, other_half(mloc));
    // MODS: the reference that the weights are taken against moves only when a tile's maximum lies
    // more than 2^8 above it (or there is none yet): most tiles leave the output accumulators alone
    const bool move = !MODS || mloc > m_run + 8.0f;
    if (!MODS || __builtin_amdgcn_ballot_w64(move) != 0) {
      const float m_new = move ? fmaxf(m_run, mloc) : m_run;
      const float corr = move ? fast_exp2(m_run - (m_new == -INFINITY ? 0.f : m_new)) : 1.0f;
      l_run *= corr;
      if (MFMA_SUM)
#pragma unroll
        for (int v = 0; v < 16; ++v) o_sum[v] *= corr;
#pragma unroll
      for (int mt = 0; mt < P_MT; ++mt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[mt][v] *= corr;
      m_run = m_new;
    }
    const float m_safe = m_run == -INFINITY ? 0.f : m_run;
    float lsum = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = fast_exp2(fmaf(s[v], sc, -m_safe));
      if (!MFMA_SUM) lsum += s[v];
    }
    if (!MFMA_SUM) {
      lsum += other_half(lsum);
      l_run += lsum;
    }
    // ---- O^T += V^T P^T, two k-steps of 16 keys ---------------------------------------
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const u32x4_t pw = {pack_bf16(s[8 * st + 0], s[8 * st + 1]),
                          pack_bf16(s[8 * st + 2], s[8 * st + 3]),
                          pack_bf16(s[8 * st + 4], s[8 * st + 5]),
                          pack_bf16(s[8 * st + 6], s[8 * st + 7])};
      const bf16x8_t pf = as_frag(pw);
      if (MFMA_SUM) o_sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pf, o_sum, 0, 0, 0);
#pragma unroll
      for (int mt = 0; mt < P_MT; ++mt) {
        const u32x4_t vw = {vfa[buf][st][mt].x, vfa[buf][st][mt].y, vfb[buf][st][mt].x,
                            vfb[buf][st][mt].y};
        o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(vw), pf, o[mt], 0, 0, 0);
      }
    }
  };
  // wave w takes the key tiles kb0 + 32 * (w + P_NW * i)
  const int kb0 = lo32 - kept + 32 * wave;
  constexpr int KSTEP = 32 * P_NW;
  auto at = [&](int place) { return MODS ? kappai_key_at(place, lo32, kept) : place; };
  if (P_AHEAD) {
    if (kb0 <= pos_last) fetch(0, at(kb0));
    for (int kb = kb0; kb <= pos_last; kb += 2 * KSTEP) {
      if (kb + KSTEP <= pos_last) fetch(P_NB - 1, at(kb + KSTEP));
      work(0, at(kb));
      if (kb + KSTEP <= pos_last) {
        if (kb + 2 * KSTEP <= pos_last) fetch(0, at(kb + 2 * KSTEP));
        work(P_NB - 1, at(kb + KSTEP));
      }
    }
  } else {
    for (int kb = kb0; kb <= pos_last; kb += KSTEP) {
      fetch(0, at(kb));
      work(0, at(kb));
    }
  }
  if (MFMA_SUM) l_run = o_sum[0];
  if (P_NW > 1) {
    // merge: every wave rescales to the common maximum; waves 1.. hand their sums to wave 0
    __shared__ float sh_m[P_NW][32], sh_l[P_NW][32];
    if (hh == 0) sh_m[wave][col] = m_run;
    __syncthreads();
    float M = sh_m[0][col];
#pragma unroll
    for (int w = 1; w < P_NW; ++w) M = fmaxf(M, sh_m[w][col]);
    const float f = m_run == -INFINITY ? 0.f : fast_exp2(m_run - M);
    l_run *= f;
    if (hh == 0) sh_l[wave][col] = l_run;
    if (wave > 0) {
#pragma unroll
      for (int mt = 0; mt < P_MT; ++mt)
#pragma unroll
        for (int v = 0; v < 16; ++v) sh_o[((wave - 1) * P_MT * 16 + mt * 16 + v) * WAVE + lane] = o[mt][v] * f;
    }
    __syncthreads();
    if (wave > 0) return;
    l_run = sh_l[0][col];
#pragma unroll
    for (int w = 1; w < P_NW; ++w) l_run += sh_l[w][col];
    if (mods.sink != nullptr && M != -INFINITY)
      l_run += fast_exp2(mods.sink[h] * LOG2E - M);
#pragma unroll
    for (int mt = 0; mt < P_MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        float acc = o[mt][v] * f;
#pragma unroll
        for (int w = 1; w < P_NW; ++w) acc += sh_o[((w - 1) * P_MT * 16 + mt * 16 + v) * WAVE + lane];
        o[mt][v] = acc;
      }
  }
  if (!row_ok) return;
  if (P_NW == 1 && mods.sink != nullptr && m_run != -INFINITY)
    l_run += fast_exp2(mods.sink[h] * LOG2E - m_run);
  const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
  bf16_t* orow = out + (size_t)(r0 + col) * out_stride + (size_t)h * HEAD_DIM;
#pragma unroll
  for (int mt = 0; mt < P_MT; ++mt)
#pragma unroll
    for (int v4 = 0; v4 < 4; ++v4) {
      const int dd = 32 * mt + 8 * v4 + 4 * hh;     // four consecutive d: v = 4*v4 .. 4*v4+3
      if (dd < HEAD_DIM) {
        u32x2_t w = {pack_bf16(o[mt][4 * v4] * inv, o[mt][4 * v4 + 1] * inv),
                     pack_bf16(o[mt][4 * v4 + 2] * inv, o[mt][4 * v4 + 3] * inv)};
        *reinterpret_cast<u32x2_t*>(orow + dd) = w;
      }
    }
}

// ---------------------------------------------------------------------------------------
// prefill, key tiles shared by the query heads of a kv head
// ---------------------------------------------------------------------------------------
// One block = two q tiles (32 rows each) of one segment x four query heads of one kv head, a
// wave each.  The eight waves walk the same key tiles, so a tile of K (32 keys x d) and of V^T
// (d x 32 keys) is brought from global memory once, straight into LDS (buffer loads, three
// buffers, two tiles ahead), and every wave reads its matrix operands from there.  Pairing an
// early q tile with a late one gives every block the same number of keys to walk.  K rows keep their 16-byte chunks permuted (chunk ^ f(key)) so that the
// 16 keys of a fragment read fall on different banks; V^T lies as [16-key group][d][16 keys],
// every other 8 rows with their two halves of 8 keys swapped, for the same reason.
// The running maximum is only moved when a tile's maximum exceeds it by more than 2^8: most
// tiles then leave the output accumulators alone (no rescaling), and the weights stay <= 256.
//
// Bound by the issue of vector instructions: a step (two tiles) of two waves is about 2,000 cycles of them,
// 32 exponentials of 16 cycles a wave among them, beside 1,280 of products; it takes 2,400.  2,048 rows are
// 256 blocks, two waves a SIMD, so the chip has no more waves to fill gaps with, and each gap of a wave had
// to be closed by itself.  2,048 rows, 32 heads of 64 on 8, without past / behind 4,096 keys / behind 9,900:
//   values put together from two reads, one loop for masked and whole steps      54.1 / 156.5 / 307.5 us
//   16-byte reads of values, a loop of its own for whole steps                    44 / 130 / 246
//   tiles by buffer loads, page numbers from a register (see there), half of the
//   scalar work in front of a tile's loads, LDS asked for ahead of it             40 / 122 / 230
//   next step's scores among this step's exponentials                             37 / 116 / 217 (0.81 PFLOP/s)
// At head size 128 (behind 4,096 keys, 16 heads on 4) 176 -> 154 us without the last.  Priorities for the
// waves of one tile, for the products or for the exponentials: within 3 %.
#if HEAD_DIM == 64 || HEAD_DIM == 128
#define PG_OK 1
#define PG_NBUF 3
#define PG_SUB 2
template <int N> struct PgBuf { static constexpr int value = N; };
#define PG_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

__global__ __launch_bounds__(8 * WAVE) void attn_prefill_shared_kernel(
    const int* __restrict__ q_tiles, const int* __restrict__ row_pos,
    const int* __restrict__ block_tables, int max_blocks, int H, int G, int ps, int q_stride, int window,
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ vt_pool,
    bf16_t* __restrict__ out, int out_stride, float scale, const float* __restrict__ sink) {
  constexpr int ROWB = HEAD_DIM * 2;                // bytes of a key's row
  constexpr int KTILE = 32 * ROWB, VGROUP = HEAD_DIM * 32, BUF = KTILE + 2 * VGROUP;   // bytes
  constexpr int CPR = ROWB / 16;                    // 16-byte chunks a K row
  constexpr int K_ROWS_PER = 1024 / ROWB;           // K rows one load instruction brings
  constexpr int NL = 8 / K_ROWS_PER;                // loads a wave issues per tile: a K wave
                                                    // brings 8 keys, a V wave half a 16-key group
  static_assert(NL == (HEAD_DIM / 2) / 32, "K and V waves issue the same number of loads");
  // a buffer holds PG_SUB key tiles: one barrier for that many tiles
  __shared__ __attribute__((aligned(1024))) char lds[PG_NBUF * PG_SUB * BUF];
  const int t_a = gridDim.x - 1 - blockIdx.x;
  // The block's second q tile.  q_tiles[t][3] = (index of the tile within its segment) |
  // (tiles of the segment << 16), 0 if unknown.  Without a window tile j is paired with tile
  // n-1-j, so that every block walks about the same number of keys; with a window, with its
  // neighbour, whose keys are nearly the same.  The later tile of a pair has no block of its own.
  int t_b = -1;
  {
    const int info = q_tiles[4 * t_a + 3];
    const int j = info & 0xffff, n = info >> 16;
    if (n > 0) {
      if (window == 0) {
        if (2 * j > n - 1) return;
        if (2 * j < n - 1) t_b = t_a + (n - 1 - 2 * j);
      } else {
        if (j & 1) return;
        if (j + 1 < n) t_b = t_a + 1;
      }
    }
  }
  const int rep = H / G, quads = rep / 4;
  const int g = blockIdx.y / quads;
  // a decoded token beside portions (see the kernel above): eight waves share its keys
  if (t_b < 0 && q_tiles[4 * t_a + 2] == 1 && rep <= 16 &&
      8 * (rep * HEAD_DIM + 32) * (int)sizeof(float) <= (int)sizeof lds) {
    const int t = q_tiles[4 * t_a + 1];
    if (blockIdx.y % quads == 0)
      attn_one_row<false>(q, q_stride, k_pool, vt_pool, out, out_stride,
                          block_tables + (size_t)q_tiles[4 * t_a] * max_blocks, max_blocks, t, row_pos[t],
                          g, H, G, ps, window, scale, kappai_score_mods{0.f, nullptr, 0, sink, 0},
                          reinterpret_cast<float*>(lds), 8);
    return;
  }
  const int lane = threadIdx.x % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int grp = wave / 4;                         // 0: tile a, 1: tile b
  const int h = g * rep + (blockIdx.y % quads) * 4 + wave % 4;
  const int tile = grp == 0 ? t_a : t_b;
  const bool has_tile = tile >= 0;
  const int seg = q_tiles[4 * t_a];                 // both tiles are of one segment
  const int r0 = has_tile ? q_tiles[4 * tile + 1] : 0, nr = has_tile ? q_tiles[4 * tile + 2] : 0;
  const int col = lane % 32, hh = lane / 32;
  const int* bt = block_tables + (size_t)seg * max_blocks;
  const int pos_first = row_pos[r0], pos_last = pos_first + nr - 1;
  const bool row_ok = col < nr;
  const int my_pos = row_ok ? pos_first + col : -1;
  const int my_lo = kappai_first_key(my_pos, window);
  const int lo_tile = kappai_first_key(pos_first, window);
  const int lo_last = kappai_first_key(pos_last, window);
  // the keys the block walks: from the first key of either tile to the last key of either
  int blk_first, blk_last;
  {
    const int ra = q_tiles[4 * t_a + 1], pa0 = row_pos[ra], pa1 = pa0 + q_tiles[4 * t_a + 2] - 1;
    blk_first = kappai_first_key(pa0, window);
    blk_last = pa1;
    if (t_b >= 0) {
      const int rb = q_tiles[4 * t_b + 1], pb0 = row_pos[rb], pb1 = pb0 + q_tiles[4 * t_b + 2] - 1;
      blk_first = min(blk_first, kappai_first_key(pb0, window));
      blk_last = max(blk_last, pb1);
    }
  }

  bf16x8_t qf[P_KS];
  {
    const bf16_t* qr = q + (size_t)(r0 + (row_ok ? col : 0)) * q_stride + (size_t)h * HEAD_DIM;
#pragma unroll
    for (int ks = 0; ks < P_KS; ++ks) {
      u32x4_t v = {0u, 0u, 0u, 0u};
      if (row_ok) v = *reinterpret_cast<const u32x4_t*>(qr + 16 * ks + 8 * hh);
      qf[ks] = as_frag(v);
    }
  }
  f32x16_t o[P_MT];
#pragma unroll
  for (int mt = 0; mt < P_MT; ++mt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[mt][v] = 0.f;
  // The sums of the weights come from the matrix cores too: a V^T fragment of ones gives a
  // tile whose every row is the sum over the keys, of the same rounded weights the output is made
  // of.  (The kernel is bound by the issue of vector instructions: 16 additions and an exchange
  // between half waves less per tile.)  Only at head size 64: at 128 the 16 registers more spill.
  constexpr bool MFMA_SUM = HEAD_DIM == 64;
  float l_add = 0.f;
  f32x16_t o_sum;
#pragma unroll
  for (int v = 0; v < 16; ++v) o_sum[v] = 0.f;
  const bf16x8_t ones = as_frag((u32x4_t){0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
  float m_ref = -INFINITY;
  const float sc = scale * LOG2E;

  const int kbase = (blk_first / 32) * 32;
  const int n_tiles = (blk_last - kbase) / 32 + 1;
  auto swz = [](int key) { return HEAD_DIM == 64 ? (key >> 1) & 7 : key & 15; };
  // what this lane brings: waves 0-3 eight rows of K each, waves 4-7 half a 16-key group of V^T
  const int k_row_in = lane / CPR, k_slot = lane % CPR;
  const int vw = wave - 4, v_st = vw / 2, v_d0 = (vw % 2) * (HEAD_DIM / 2) + lane / 2;
  const int v_half = lane % 2;
  // The buffer of a tile is a compile-time constant (the tile loop is unrolled three times):
  // only then can the compiler tell that the loads it issues into one buffer do not touch
  // the buffer it reads from, and leave them in flight across the reads.
  // Tiles are issued in order, so the wave keeps the place of its next keys (block table
  // index, offset in the page) and looks the next page up one tile ahead; a group past the
  // last key (or given back by the window) is read from the pool's first page instead and
  // masked when it is used.  A wave's keys (8 of K, 16 of V^T) lie in one page.
  // All of this is scalar work that a wave does at every tile before its own products, with one other wave to
  // fill the gap, so it is kept short: a page of K and one of V^T are the same number of bytes, a wave brings
  // one of the two, and what differs is chosen once.
  int nx_key = kbase + (wave < 4 ? 8 * wave : 16 * v_st);
  int nx_pidx = nx_key / ps, nx_off = nx_key % ps;
  const int step_pages = 32 / ps, step_off = 32 % ps;
  const char* const mine =
      reinterpret_cast<const char*>(wave < 4 ? k_pool : vt_pool) + (size_t)g * ps * HEAD_DIM * sizeof(bf16_t);
  const size_t page_bytes = (size_t)G * ps * HEAD_DIM * sizeof(bf16_t);
  const int key_bytes = (int)sizeof(bf16_t) * (wave < 4 ? HEAD_DIM : 1);
  // 64 of the segment's pages, a lane each, and the number of the first: a scalar load a tile would have every
  // wait for LDS wait for it too
  int pages_from = min(nx_pidx, max_blocks - 1), pages = bt[min(pages_from + lane, max_blocks - 1)];
  auto lookup = [&]() {
    const int at = min(nx_pidx, max_blocks - 1);
    if (__builtin_expect(at - pages_from >= WAVE, 0)) {
      pages_from = at;
      pages = bt[min(at + lane, max_blocks - 1)];
      asm volatile("" : "+v"(pages));      // (waits here, and not at every tile for a load that may be under way)
    }
    const int page = __builtin_amdgcn_readlane(pages, at - pages_from);
    return nx_key <= blk_last ? max(page, 0) : 0;
  };
  // (the first by a scalar load beside those 64, which it does not wait for: two portions of 16 tiles gain 0.3 us)
  int nx_page = nx_key <= blk_last ? max(bt[pages_from], 0) : 0;
  // (buffer loads: of a global load into LDS the compiler holds that it may be any access to LDS, and waits for
  // all reads under way where it should wait for the oldest)
  uint32_t from[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int row = i * K_ROWS_PER + k_row_in;                 // 0..7 within the wave's keys
    // (V^T: rows 8 apart would meet on the same banks: every other group of 8 rows keeps its two 16-byte halves
    // swapped)
    const int dd = v_d0 + 32 * i;
    from[i] = 2u * (uint32_t)(wave < 4 ? row * HEAD_DIM + (k_slot ^ swz(8 * wave + row)) * 8
                                       : dd * ps + 8 * (v_half ^ ((dd >> 3) & 1)));
  }
  const int to = wave < 4 ? 8 * wave * ROWB : KTILE + v_st * VGROUP + (vw % 2) * (HEAD_DIM / 2) * 32;
  static_assert(K_ROWS_PER * ROWB == 32 * 32, "a load's bytes, of K and of V^T");
  auto issue_one = [&](char* buf) {
#if defined(__HIP_DEVICE_COMPILE__)
    const __amdgpu_buffer_rsrc_t keys = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(mine + (size_t)(uint32_t)nx_page * page_bytes), 0, 0x7FFFFF00, 0x00020000);
#pragma unroll
    for (int i = 0; i < NL; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(keys, PG_LPTR(buf + to + i * 1024), 16, from[i], nx_off * key_bytes,
                                               0, 0);
#endif
    nx_key += 32;
    nx_off += step_off;
    nx_pidx += step_pages + (nx_off >= ps ? 1 : 0);
    nx_off -= nx_off >= ps ? ps : 0;
    nx_page = lookup();
  };
  auto issue = [&](auto buf_c) {
#pragma unroll
    for (int sub = 0; sub < PG_SUB; ++sub)
      issue_one(lds + (decltype(buf_c)::value * PG_SUB + sub) * BUF);
  };
  // Row i of a score tile is key (i with its bits 2 and 3 exchanged): a lane's weights are then those of
  // the keys 16 st + 8 hh .. + 7 in order, and their values ONE 16-byte piece of a V^T row.
  const int krow = (col & 19) | (col & 4) << 1 | (col & 8) >> 1;
  // this lane's piece of a V^T row in a 16-key group (every other 8 rows have their halves swapped)
  const int v_at = col * 32 + 16 * (hh ^ ((col >> 3) & 1));
  auto whole = [&](int kb) { return kb >= lo_last && kb + 31 <= pos_first; };
  auto work = [&](auto buf_c, auto sub_c, int it) {
    const int kb = kbase + 32 * it;
    const char* buf = lds + (decltype(buf_c)::value * PG_SUB + decltype(sub_c)::value) * BUF;
    const bool full = whole(kb);
    // ---- S^T tile: 32 keys x 32 queries -------------------------------------------------
    f32x16_t s;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
    for (int ks = 0; ks < P_KS; ++ks) {
      const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(
          buf + krow * ROWB + (((2 * ks + hh) ^ swz(krow)) * 16));
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(kf), qf[ks], s, 0, 0, 0);
    }
    // V^T operands: d index 32*mt + col, keys 16*st + 8*hh .. +7
    u32x4_t vv[2][P_MT];
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int mt = 0; mt < P_MT; ++mt)
        vv[st][mt] = *reinterpret_cast<const u32x4_t*>(buf + KTILE + st * VGROUP + 32 * 32 * mt + v_at);
    // lane holds, for query `col`, keys kb + 16*(v/8) + 8*hh + v%8
    float mloc = -INFINITY;
    if (full) {
#pragma unroll
      for (int v = 0; v < 16; ++v) mloc = fmaxf(mloc, s[v]);
      mloc *= sc;           // sc > 0: scaling commutes with the maximum
    } else {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int key = kb + 16 * (v / 8) + 8 * hh + v % 8;
        const bool ok = key <= my_pos && key >= my_lo;
        s[v] = ok ? s[v] : -INFINITY;
        mloc = fmaxf(mloc, s[v] * sc);
      }
      // what lies in LDS for keys outside the tile's range is not cache content: zero it
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        int keep = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int key = kb + 16 * st + 8 * hh + i;
          if (key >= lo_tile && key <= pos_last) keep |= 1 << i;
        }
#pragma unroll
        for (int mt = 0; mt < P_MT; ++mt) {
          const u32x2_t a = mask4(u32x2_t{vv[st][mt].x, vv[st][mt].y}, keep & 15);
          const u32x2_t b = mask4(u32x2_t{vv[st][mt].z, vv[st][mt].w}, keep >> 4);
          vv[st][mt] = u32x4_t{a.x, a.y, b.x, b.y};
        }
      }
    }
    mloc = fmaxf(mloc, other_half(mloc));
    // move the reference only when it is far off (or unset): uniform for the wave's branch
    const bool move = mloc > m_ref + 8.0f;
    if (__builtin_amdgcn_ballot_w64(move) != 0) {
      const float m_new = move ? mloc : m_ref;
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;
      const float corr = move ? fast_exp2(m_ref - m_safe) : 1.0f;
      if (MFMA_SUM) {
#pragma unroll
        for (int v = 0; v < 16; ++v) o_sum[v] *= corr;
      } else {
        l_add *= corr;
      }
#pragma unroll
      for (int mt = 0; mt < P_MT; ++mt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[mt][v] *= corr;
      m_ref = m_new;
    }
    const float m_safe = m_ref == -INFINITY ? 0.f : m_ref;
    float lsum = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = fast_exp2(fmaf(s[v], sc, -m_safe));
      if (!MFMA_SUM) lsum += s[v];
    }
    if (!MFMA_SUM) {
      lsum += other_half(lsum);
      l_add += lsum;
    }
    // ---- O^T += V^T P^T, two k-steps of 16 keys ---------------------------------------
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const u32x4_t pw = {pack_bf16(s[8 * st + 0], s[8 * st + 1]),
                          pack_bf16(s[8 * st + 2], s[8 * st + 3]),
                          pack_bf16(s[8 * st + 4], s[8 * st + 5]),
                          pack_bf16(s[8 * st + 6], s[8 * st + 7])};
      const bf16x8_t pf = as_frag(pw);
      if (MFMA_SUM) o_sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pf, o_sum, 0, 0, 0);
#pragma unroll
      for (int mt = 0; mt < P_MT; ++mt)
        o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(vv[st][mt]), pf, o[mt], 0, 0, 0);
    }
  };

  // Both tiles of a buffer when neither needs a mask (most steps of a long history), a step behind the
  // scores: `s` holds this step's, and the products of the next step's stand among this step's
  // exponentials (two waves a SIMD leave a barrier together, so that without this both do products while
  // the vector unit idles, then both exponentials while the matrix cores do).  All of LDS is asked for
  // first, and the loads of a later step (`ask`) go out while it answers.
  f32x16_t s[2];
  auto keys_of = [&](auto buf_c, u32x4_t (&kf)[2][P_KS]) {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int ks = 0; ks < P_KS; ++ks)
        kf[sub][ks] = *reinterpret_cast<const u32x4_t*>(
            lds + (decltype(buf_c)::value * PG_SUB + sub) * BUF + krow * ROWB +
            (((2 * ks + hh) ^ swz(krow)) * 16));
  };
  auto scores = [&](const u32x4_t (&kf)[P_KS]) {
    f32x16_t r;
#pragma unroll
    for (int v = 0; v < 16; ++v) r[v] = 0.f;
#pragma unroll
    for (int ks = 0; ks < P_KS; ++ks)
      r = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(kf[ks]), qf[ks], r, 0, 0, 0);
    return r;
  };
  auto work2 = [&](auto buf_c, auto next_c, auto ask) {
    u32x4_t kf[2][P_KS], vv[2][2][P_MT];
    keys_of(next_c, kf);
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int mt = 0; mt < P_MT; ++mt)
          vv[sub][st][mt] = *reinterpret_cast<const u32x4_t*>(
              lds + (decltype(buf_c)::value * PG_SUB + sub) * BUF + KTILE + st * VGROUP + 32 * 32 * mt + v_at);
    __builtin_amdgcn_sched_barrier(0);
    ask();
    // the running reference moves only when a tile's maximum is far above it (rare: a branch)
    auto update_reference = [&](const f32x16_t& s) {
      float mloc = -INFINITY;
#pragma unroll
      for (int v = 0; v < 16; ++v) mloc = fmaxf(mloc, s[v]);
      mloc *= sc;
      mloc = fmaxf(mloc, other_half(mloc));
      const bool move = mloc > m_ref + 8.0f;
      if (__builtin_amdgcn_ballot_w64(move) != 0) {
        const float m_new = move ? mloc : m_ref;
        const float m_safe = m_new == -INFINITY ? 0.f : m_new;
        const float corr = move ? fast_exp2(m_ref - m_safe) : 1.0f;
        if (MFMA_SUM) {
#pragma unroll
          for (int v = 0; v < 16; ++v) o_sum[v] *= corr;
        } else {
          l_add *= corr;
        }
#pragma unroll
        for (int mt = 0; mt < P_MT; ++mt)
#pragma unroll
          for (int v = 0; v < 16; ++v) o[mt][v] *= corr;
        m_ref = m_new;
      }
    };
    auto weights_and_output = [&](const u32x4_t (&vv)[2][P_MT], f32x16_t s) {
      const float m_safe = m_ref == -INFINITY ? 0.f : m_ref;
      float lsum = 0.f;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        s[v] = fast_exp2(fmaf(s[v], sc, -m_safe));
        if (!MFMA_SUM) lsum += s[v];
      }
      if (!MFMA_SUM) {
        lsum += other_half(lsum);
        l_add += lsum;
      }
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const u32x4_t pw = {pack_bf16(s[8 * st + 0], s[8 * st + 1]),
                            pack_bf16(s[8 * st + 2], s[8 * st + 3]),
                            pack_bf16(s[8 * st + 4], s[8 * st + 5]),
                            pack_bf16(s[8 * st + 6], s[8 * st + 7])};
        const bf16x8_t pf = as_frag(pw);
        if (MFMA_SUM) o_sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pf, o_sum, 0, 0, 0);
#pragma unroll
        for (int mt = 0; mt < P_MT; ++mt)
          o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(vv[st][mt]), pf, o[mt], 0, 0, 0);
      }
    };
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      update_reference(s[sub]);
      const f32x16_t now = s[sub];
      s[sub] = scores(kf[sub]);
      weights_and_output(vv[sub], now);
    }
  };

  // `it` counts buffers' worth of tiles (PG_SUB each)
  const int n_steps = (n_tiles + PG_SUB - 1) / PG_SUB;
  // the tiles of step `it` have landed (this wave's part; the barrier makes it everybody's), and at head
  // size 64 those of the next step too, which a wave a step ahead with its scores reads: all waves of a
  // block pass one barrier a step, whichever way they go.  At 128 the next step's may still be on their way.
  auto arrive = [&](int it) {
    // Everything read of LDS is in registers too: the tiles of step it - 1 are written over behind the barrier.
    // (No fence: a fence would wait for the loads in flight.)
    if (HEAD_DIM != 64 && it + 1 < n_steps) __builtin_amdgcn_s_waitcnt(0x0070 | (PG_SUB * NL));
    else __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto step = [&](auto buf_c, int it) {
    constexpr int B = decltype(buf_c)::value;
    arrive(it);
    // step it+2 goes into the buffer of step it-1: everybody is done with it
    if (it + 2 < n_steps) issue(PgBuf<(B + 2) % PG_NBUF>{});
    const int kb = kbase + 32 * PG_SUB * it;
    if (has_tile && kb + 31 >= lo_tile && kb <= pos_last) work(buf_c, PgBuf<0>{}, PG_SUB * it);
    if (has_tile && kb + 63 >= lo_tile && kb + 32 <= pos_last)
      work(buf_c, PgBuf<1>{}, PG_SUB * it + 1);
  };
  static_assert(PG_SUB == 2, "the step works on two tiles");
  issue(PgBuf<0>{});
  if (n_steps > 1) issue(PgBuf<1>{});
  // (the queries have arrived: where this is not said, every step waits for all loads but its own first)
#pragma unroll
  for (int ks = 0; ks < P_KS; ++ks) asm volatile("" : "+v"(qf[ks]));
  // The steps whose tiles need no mask, in whole rounds of the buffers, are a loop of their own: where the
  // two ways through a step meet again, 48 accumulators are copied (a sixth of the step's vector work).
  int it = 0, fast_from = 0, fast_to = 0;
  if (HEAD_DIM == 64 && has_tile) {                                    // (128: registers spill)
    fast_from = (max(lo_last - kbase, 0) + 32 * PG_SUB - 1) / (32 * PG_SUB);
    fast_from = (fast_from + PG_NBUF - 1) / PG_NBUF * PG_NBUF;
    fast_to = max(pos_first + 1 - kbase, 0) / (32 * PG_SUB);
    fast_from = __builtin_amdgcn_readfirstlane(fast_from);
    fast_to = __builtin_amdgcn_readfirstlane(min(fast_to, n_steps));
  }
  const auto steps_to = [&](int end) {
    for (; it < end; it += PG_NBUF) {
      step(PgBuf<0>{}, it);
      if (it + 1 < n_steps) step(PgBuf<1>{}, it + 1);
      if (it + 2 < n_steps) step(PgBuf<2>{}, it + 2);
    }
  };
  steps_to(fast_to - fast_from >= PG_NBUF ? fast_from : n_steps);
  if constexpr (HEAD_DIM == 64) {
    if (it + PG_NBUF <= fast_to) {
      auto fast = [&](auto buf_c, int at) {
        constexpr int B = decltype(buf_c)::value;
        work2(buf_c, PgBuf<(B + 1) % PG_NBUF>{}, [&]() {
          if (at + 2 < n_steps) issue(PgBuf<(B + 2) % PG_NBUF>{});
        });
      };
      arrive(it);
      {
        u32x4_t kf[2][P_KS];
        keys_of(PgBuf<0>{}, kf);
        s[0] = scores(kf[0]);
        s[1] = scores(kf[1]);
      }
      for (;;) {
        fast(PgBuf<0>{}, it);
        arrive(it + 1);
        fast(PgBuf<1>{}, it + 1);
        arrive(it + 2);
        fast(PgBuf<2>{}, it + 2);             // (the scores of a step behind the last whole one go unused)
        it += PG_NBUF;
        if (it + PG_NBUF > fast_to) break;
        arrive(it);
      }
    }
  }
  steps_to(n_steps);
  if (!row_ok) return;
  float l_run = MFMA_SUM ? o_sum[0] : l_add;
  if (sink != nullptr && m_ref != -INFINITY) l_run += fast_exp2(sink[h] * LOG2E - m_ref);
  const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
  bf16_t* orow = out + (size_t)(r0 + col) * out_stride + (size_t)h * HEAD_DIM;
#pragma unroll
  for (int mt = 0; mt < P_MT; ++mt)
#pragma unroll
    for (int v4 = 0; v4 < 4; ++v4) {
      const int dd = 32 * mt + 8 * v4 + 4 * hh;     // four consecutive d: v = 4*v4 .. 4*v4+3
      u32x2_t w = {pack_bf16(o[mt][4 * v4] * inv, o[mt][4 * v4 + 1] * inv),
                   pack_bf16(o[mt][4 * v4 + 2] * inv, o[mt][4 * v4 + 3] * inv)};
      *reinterpret_cast<u32x2_t*>(orow + dd) = w;
    }
}
#else
#define PG_OK 0
#endif

// ---------------------------------------------------------------------------------------
// prefill at head size 256, key tiles shared by four query heads of a kv head
// ---------------------------------------------------------------------------------------
// One block = one q tile (32 rows) x four query heads of one kv head, two waves a head: both make the
// scores, each half of the output's columns (with all of them in one wave the registers spill and a
// SIMD has no second wave to work while the first is at its exponentials).  A tile of K (32 keys x d)
// and of V^T comes from global memory once, straight into LDS (buffer loads, three buffers, two
// tiles ahead), in the places the kernel above gives them.  A wave alone with its head, which is the other way, reads
// every operand from the caches itself and has no registers to ask ahead: it waits about 3 us for a
// tile, whatever else runs.  Two portions of 1,900 rows in all, 16 heads on one kv head: 127 -> 79 us;
// what bounds it now is a wave's own chain over a tile (scores, exponentials, output), two waves a
// SIMD, about 2 us for each of the longest portion's 38 tiles.  The arithmetic is that wave's to the bit: the accumulators are only
// left alone where they would have been multiplied by one.
#if HEAD_DIM == 256
#define PH_NBUF 3
template <int N> struct PhBuf { static constexpr int value = N; };
__global__ __launch_bounds__(8 * WAVE) void attn_prefill_heads_kernel(
    const int* __restrict__ q_tiles, const int* __restrict__ row_pos,
    const int* __restrict__ block_tables, int max_blocks, int H, int G, int ps, int q_stride, int window,
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ vt_pool,
    bf16_t* __restrict__ out, int out_stride, float scale, const float* __restrict__ sink) {
  constexpr int ROWB = HEAD_DIM * 2;                                              // bytes of a key's row
  constexpr int KTILE = 32 * ROWB, VGROUP = HEAD_DIM * 32, BUF = KTILE + 2 * VGROUP;   // bytes
  constexpr int NL = 4, MT = P_MT / 2;       // loads a wave issues a tile; row tiles of its half of O^T
  __shared__ __attribute__((aligned(1024))) char lds[PH_NBUF * BUF];
  const int tile = gridDim.x - 1 - blockIdx.x;      // (later tiles have more keys: they go first)
  const int lane = threadIdx.x % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int rep = H / G, quads = rep / 4;
  const int g = blockIdx.y / quads, h = g * rep + (blockIdx.y % quads) * 4 + wave % 4;
  const int mt0 = wave / 4 * MT;
  const int seg = q_tiles[4 * tile], r0 = q_tiles[4 * tile + 1], nr = q_tiles[4 * tile + 2];
  const int col = lane % 32, hh = lane / 32;
  const int* bt = block_tables + (size_t)seg * max_blocks;
  const int pos_first = row_pos[r0], pos_last = pos_first + nr - 1;
  const bool row_ok = col < nr;
  const int my_pos = row_ok ? pos_first + col : -1;
  const int my_lo = kappai_first_key(my_pos, window);
  const int lo_tile = kappai_first_key(pos_first, window);
  const int lo_last = kappai_first_key(pos_last, window);

  bf16x8_t qf[P_KS];
  {
    const bf16_t* qr = q + (size_t)(r0 + (row_ok ? col : 0)) * q_stride + (size_t)h * HEAD_DIM;
#pragma unroll
    for (int ks = 0; ks < P_KS; ++ks) {
      u32x4_t v = {0u, 0u, 0u, 0u};
      if (row_ok) v = *reinterpret_cast<const u32x4_t*>(qr + 16 * ks + 8 * hh);
      qf[ks] = as_frag(v);
    }
  }
  f32x16_t o[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[mt][v] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const float sc = scale * LOG2E;
  const int kbase = (lo_tile / 32) * 32, n_steps = (pos_last - kbase) / 32 + 1;
  // what this lane brings: waves 0 to 3 eight rows of K each (two a load), waves 4 to 7 half a 16-key
  // group of V^T (32 rows a load); a wave's keys lie in one page.  A group past the last key (or given
  // back by the window) is read from the pool's first page and masked when it is used.
  const int part = wave % 4, half = part % 2, v_half = lane % 2;
  int nx_key = kbase + 16 * (part / 2);
  // a lane's first place behind the page's address in bytes; the others follow from it
  const unsigned k_chunk = lane % 32, k_row = 8 * half + lane / 32, v_row = 128 * half + lane / 2;
  const unsigned at0 = wave < 4 ? k_row * ROWB
                                : v_row * ps * 2 + 16 * (v_half ^ ((v_row >> 3) & 1));
  // (a tile's page is asked for before the barrier in front of its loads: behind it, among the reads of LDS, the
  // wait for a scalar load is one for all of them)
  int nx_page = 0;
  auto lookup = [&]() { nx_page = bt[min(min(nx_key, pos_last) / ps, max_blocks - 1)]; };
  auto issue = [&](auto buf_c) {
    char* buf = lds + decltype(buf_c)::value * BUF;
#if defined(__HIP_DEVICE_COMPILE__)
    const size_t head = (size_t)(nx_key <= pos_last ? max(nx_page, 0) : 0) * G + g;
    const int off = nx_key % ps;
    // (rows 32 apart have the same swapped halves)
    const bf16_t* from = wave < 4 ? k_pool + (head * ps + off) * HEAD_DIM : vt_pool + head * HEAD_DIM * ps + off;
    const __amdgpu_buffer_rsrc_t keys =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(from), 0, 0x7FFFFF00, 0x00020000);
    const unsigned step = wave < 4 ? 2 * ROWB : 64 * ps;
    unsigned first = at0;
    asm volatile("" : "+v"(first));                  // (four places kept over the loop: registers there are not)
    char* to = wave < 4 ? buf + 8 * part * ROWB : buf + KTILE + (part / 2) * VGROUP + half * 128 * 32;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const unsigned swap = wave < 4 ? 16 * (k_chunk ^ ((k_row + 2 * i) & 15)) : 0;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(keys, (__attribute__((address_space(3))) void*)(to + 1024 * i), 16,
                                               first + swap, i * step, 0, 0);
    }
#endif
    nx_key += 32;
  };
  auto work = [&](auto buf_c, int kb) {
    const char* buf = lds + decltype(buf_c)::value * BUF;
    // (a lane's places in LDS are made anew for every tile: kept over the loop for three buffers they
    // are more registers than there are)
    int at = col;
    asm volatile("" : "+v"(at));
    f32x16_t s;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
    for (int ks = 0; ks < P_KS; ++ks) {
      const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(
          buf + at * ROWB + (((2 * ks + hh) ^ (at & 15)) * 16));
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(kf), qf[ks], s, 0, 0, 0);
      // (fences here and below: left to itself the compiler reads a whole tile ahead and spills, and
      // a reload waits for the tiles on their way)
      if (ks % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    const bool full = kb >= lo_last && kb + 31 <= pos_first;
    // lane holds, for query `col`, keys kb + 8*(v/4) + 4*hh + v%4
    float mloc = -INFINITY;
    if (full) {
#pragma unroll
      for (int v = 0; v < 16; ++v) mloc = fmaxf(mloc, s[v]);
      mloc *= sc;           // sc > 0: scaling commutes with the maximum
    } else {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int key = kb + 8 * (v / 4) + 4 * hh + v % 4;
        s[v] = key <= my_pos && key >= my_lo ? s[v] : -INFINITY;
        mloc = fmaxf(mloc, s[v] * sc);
      }
    }
    mloc = fmaxf(mloc, other_half(mloc));
    const float m_new = fmaxf(m_run, mloc);
    float corr = 1.0f;
    if (__builtin_amdgcn_ballot_w64(m_new != m_run) != 0) {
      corr = fast_exp2(m_run - (m_new == -INFINITY ? 0.f : m_new));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[mt][v] *= corr;
      m_run = m_new;
    }
    const float m_safe = m_run == -INFINITY ? 0.f : m_run;
    float lsum = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = fast_exp2(fmaf(s[v], sc, -m_safe));
      lsum += s[v];
    }
    lsum += other_half(lsum);
    l_run = fmaf(l_run, corr, lsum);
    auto output = [&](auto masked_c) {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const u32x4_t pw = {pack_bf16(s[8 * st + 0], s[8 * st + 1]),
                            pack_bf16(s[8 * st + 2], s[8 * st + 3]),
                            pack_bf16(s[8 * st + 4], s[8 * st + 5]),
                            pack_bf16(s[8 * st + 6], s[8 * st + 7])};
        const bf16x8_t pf = as_frag(pw);
        int keep_a = 0, keep_b = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int ka = kb + 16 * st + 4 * hh + i, kbb = ka + 8;
          if (ka >= lo_tile && ka <= pos_last) keep_a |= 1 << i;
          if (kbb >= lo_tile && kbb <= pos_last) keep_b |= 1 << i;
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const int sw = ((at >> 3) & 1) * 16;      // (this row's halves are swapped)
          const char* vp = buf + KTILE + st * VGROUP + (32 * (mt0 + mt) + at) * 32 + 8 * hh;
          u32x2_t va = *reinterpret_cast<const u32x2_t*>(vp + sw);
          u32x2_t vb = *reinterpret_cast<const u32x2_t*>(vp + (16 - sw));
          // what lies in LDS for keys outside the tile's range is not cache content: zero it
          if (decltype(masked_c)::value) {
            va = mask4(va, keep_a);
            vb = mask4(vb, keep_b);
          }
          o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              as_frag((u32x4_t){va.x, va.y, vb.x, vb.y}), pf, o[mt], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (full) output(PhBuf<0>{});
    else output(PhBuf<1>{});
  };
  auto step = [&](auto buf_c, int it) {
    __builtin_amdgcn_sched_barrier(0);
    constexpr int B = decltype(buf_c)::value;
    if (it + 2 < n_steps) lookup();
    // this step's tile has landed (this wave's part; the barrier makes it everybody's), and what was read of
    // the step before (no fence: a fence would wait for the loads in flight)
    if (it + 1 < n_steps) __builtin_amdgcn_s_waitcnt(0x0070 | NL);
    else __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // step it + 2 goes into the buffer of step it - 1: everybody is done with it
    if (it + 2 < n_steps) issue(PhBuf<(B + 2) % PH_NBUF>{});
    work(buf_c, kbase + 32 * it);
  };
  lookup();
  issue(PhBuf<0>{});
  lookup();
  if (n_steps > 1) issue(PhBuf<1>{});
  // (the queries have arrived: where this is not said, every step waits for all loads but its own first)
#pragma unroll
  for (int ks = 0; ks < P_KS; ++ks) asm volatile("" : "+v"(qf[ks]));
  for (int it = 0; it < n_steps; it += PH_NBUF) {
    step(PhBuf<0>{}, it);
    if (it + 1 < n_steps) step(PhBuf<1>{}, it + 1);
    if (it + 2 < n_steps) step(PhBuf<2>{}, it + 2);
  }
  if (!row_ok) return;
  if (sink != nullptr && m_run != -INFINITY) l_run += fast_exp2(sink[h] * LOG2E - m_run);
  const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
  bf16_t* orow = out + (size_t)(r0 + col) * out_stride + (size_t)h * HEAD_DIM;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int v4 = 0; v4 < 4; ++v4) {
      const int dd = 32 * (mt0 + mt) + 8 * v4 + 4 * hh;   // four consecutive d: v = 4*v4 .. 4*v4+3
      u32x2_t w = {pack_bf16(o[mt][4 * v4] * inv, o[mt][4 * v4 + 1] * inv),
                   pack_bf16(o[mt][4 * v4 + 2] * inv, o[mt][4 * v4 + 3] * inv)};
      *reinterpret_cast<u32x2_t*>(orow + dd) = w;
    }
}
#endif

// ---------------------------------------------------------------------------------------
// decode: one row a request; columns are the query heads of one kv head (at most 16)
// ---------------------------------------------------------------------------------------
#define D_KS ((HEAD_DIM + 31) / 32)     // k-steps of S^T over d (32 each)
#define D_MT (HEAD_DIM / 16)            // row tiles of O^T over d

// head sizes whose decode kernel can take the prologue below: the rotation's partner d / 2 further
// must lie in the same lane, and the registers must hold it beside a chunk of keys
#define D_QK_FUSABLE (HEAD_DIM % 64 == 0 && HEAD_DIM <= 128)

// The per-head RMSNorm, the rotation and the storing of a decoded row's own key and value, done in
// the attention kernel's prologue instead of a kernel of their own (kappai: QK-norm, then RoPE,
// then the cache write, src/models/lfm.c:36-44).  For head sizes of 64 and 128; rotate-half over
// the whole head.
struct QkFuse {
  int on;                   // 0: q is ready and the row's key and value are in the pools
  int kv;                   // the row's own key and value come from the projection beside q (k of
                            // kv head g at column (H + g) d, v at (H + G + g) d) and go to the pools
  const float* q_norm_w;    // [d] or null
  const float* k_norm_w;
  float eps;
  const float* cos_tab;     // [positions][d / 2], or null: no rotation
  const float* sin_tab;
  bf16_t* k_pool_w;         // the pools once more, to be written
  bf16_t* vt_pool_w;
};

// What the prologue reads beside the projection, asked for before the first keys so that it has
// arrived when they have: the lane's norm weights at d = 32 ks + 8 kg and, for the first half of
// the head, the cosines and sines of its position.
struct QkTables {
  float wq[(HEAD_DIM + 31) / 32][8], wk[(HEAD_DIM + 31) / 32][8];
  float cs[(HEAD_DIM + 63) / 64][8], sn[(HEAD_DIM + 63) / 64][8];
};

__device__ __forceinline__ void load8f(const float* __restrict__ p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

__device__ __forceinline__ void qk_load_tables(const QkFuse& qk, int pos, int kg, QkTables& tb) {
  constexpr int KS = (HEAD_DIM + 31) / 32, HALF = HEAD_DIM / 2;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    if (qk.q_norm_w != nullptr) load8f(qk.q_norm_w + 32 * ks + 8 * kg, tb.wq[ks]);
    if (qk.k_norm_w != nullptr && qk.kv) load8f(qk.k_norm_w + 32 * ks + 8 * kg, tb.wk[ks]);
  }
  if (qk.cos_tab != nullptr) {
#pragma unroll
    for (int ks = 0; ks < KS / 2; ++ks) {
      load8f(qk.cos_tab + (size_t)pos * HALF + 32 * ks + 8 * kg, tb.cs[ks]);
      load8f(qk.sin_tab + (size_t)pos * HALF + 32 * ks + 8 * kg, tb.sn[ks]);
    }
  }
}

// raw[ks] = the lane's eight values at d = 32 ks + 8 kg of one head; returns them normalised over
// the head (the four lanes kg = 0..3 with the same lane % 16 hold a head together), weighted
// (w: the lane's weights, when has_w) and rotated (cs, sn, when rotate), rounded to bfloat16
__device__ __forceinline__ void qk_norm_rotate(u32x4_t (&raw)[(HEAD_DIM + 31) / 32], bool has_w,
                                               const float (&w)[(HEAD_DIM + 31) / 32][8], float eps,
                                               bool rotate,
                                               const float (&cs)[(HEAD_DIM + 63) / 64][8],
                                               const float (&sn)[(HEAD_DIM + 63) / 64][8]) {
  constexpr int KS = (HEAD_DIM + 31) / 32;
  float x[KS][8];
  float ss = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const uint32_t r[4] = {raw[ks].x, raw[ks].y, raw[ks].z, raw[ks].w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[ks][2 * i] = __uint_as_float(r[i] << 16);
      x[ks][2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = fmaf(x[ks][i], x[ks][i], ss);
  }
  ss += __shfl_xor(ss, 16, WAVE);
  ss += other_half(ss);
  if (has_w) {
    const float sc = 1.0f / sqrtf(ss / (float)HEAD_DIM + eps);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < 8; ++i) x[ks][i] = x[ks][i] * sc * w[ks][i];
  }
  if (rotate) {
#pragma unroll
    for (int ks = 0; ks < KS / 2; ++ks)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float lo = x[ks][i], hi = x[ks + KS / 2][i];
        x[ks][i] = lo * cs[ks][i] - hi * sn[ks][i];
        x[ks + KS / 2][i] = lo * sn[ks][i] + hi * cs[ks][i];
      }
  }
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    raw[ks] = (u32x4_t){pack_bf16(x[ks][0], x[ks][1]), pack_bf16(x[ks][2], x[ks][3]),
                        pack_bf16(x[ks][4], x[ks][5]), pack_bf16(x[ks][6], x[ks][7])};
}

// One wave's share of a row's attention: the query heads of kv head g (columns) against the keys first ..
// k_end - 1 (`first` a multiple of 32), with a running maximum and sum per column.  Leaves the unnormalised
// output in o (lane: column lane % 16, d rows 16 mt + 4 (lane / 16) + v), the maximum (in units of log 2) in
// m_run, the sum in l_run.
//
// Bound by the stream of keys and values.  The keys go by in parts of 32 whose loads (16 bytes a lane) are
// asked for D_AHEAD parts ahead: a part's registers are filled again as soon as it is worked on, so that
// loads stay under way from the first key to the last.  The page ids are read 64 at a time, the next 64
// ahead of their use, and handed out as scalars.  A part whose keys are not all seen is loaded like any
// other and cut when it is worked on (loads of its own for it were half the kernel's code).  Against chunks
// of 128 keys, each asked for, waited for and worked on by itself, 32 heads on 8: head size 64, 8 rows of
// 300 keys in a block 6.3 us against 7.9, 64 rows of up to 2,000 keys 33.9 against 38.3 (135 MB: 4.0 TB/s,
// the kernel's start and the three lookups before its first key among it), 1 row of 8,000 keys and the
// merge 9.7 against 11.9; head size 128, 8 rows of 300 keys 8.1 against 9.1.  Head size 32 has registers for
// two blocks a CU with three parts ahead, not with four (128 rows of 300 keys 13.3 us; with one block a CU 22.8).
#define D_AHEAD (HEAD_DIM == 32 ? 3 : (HEAD_DIM <= 64 ? 4 : (HEAD_DIM <= 128 ? 2 : 1)))
template <bool FUSABLE>
__device__ __forceinline__ void attn_decode_wave(
    const bf16_t* __restrict__ q, int q_stride, const bf16_t* __restrict__ k_pool,
    const bf16_t* __restrict__ vt_pool, const int* __restrict__ bt, int max_blocks, int t, int g,
    int H, int G, int ps, float scale, int lo, int first, int k_end, f32x4_t (&o)[D_MT], float& m_run,
    float& l_run, const QkFuse& qk, int pos) {
  const int lane = threadIdx.x % WAVE;
  const int rep = H / G;
  const int col = lane % 16, kg = lane / 16;
  const bool head_ok = col < rep;
  const int h = g * rep + (head_ok ? col : 0);
  const int hi = k_end - 1;
  // Page ids 64 at a time: asked for before anything else, those behind the last key's page as that page's
  // (a load under a condition is waited for where the two ways meet).
  const int page0 = first / ps, page_last = min(hi / ps, max_blocks - 1);
  auto ask_pages = [&](int from) { return bt[min(from + lane, page_last)]; };
  int pages = ask_pages(page0), pages_next = ask_pages(page0 + WAVE), page_at = 0, page_off = first % ps;
  int pages_from = page0;
  // (what is in the register has arrived: else every part's ids would wait for the loads of the part before)
  auto pages_are_here = [&] {
    pages = pages_from + lane <= page_last ? pages : -1;
    asm volatile("" : "+v"(pages));
  };

  bf16x8_t qf[D_KS];
  u32x4_t qraw[D_KS];
  u32x4_t k_new[D_KS];                 // the row's own key, in the K fragment's order of d
  uint32_t v_new[D_MT];                // its value at d = 16 mt + col
  QkTables tb;
  const bool fused = FUSABLE && D_QK_FUSABLE && qk.on;
  const bool own_kv = fused && qk.kv;
  {
    const bf16_t* row = q + (size_t)t * q_stride;
    const bf16_t* qr = row + (size_t)h * HEAD_DIM;
#pragma unroll
    for (int ks = 0; ks < D_KS; ++ks) {
      u32x4_t v = {0u, 0u, 0u, 0u};
      const int d0 = 32 * ks + 8 * kg;
      if (head_ok && d0 < HEAD_DIM) v = *reinterpret_cast<const u32x4_t*>(qr + d0);
      qraw[ks] = v;
    }
    if constexpr (FUSABLE && D_QK_FUSABLE) {
      if (fused) {
        // everything the prologue needs is asked for here; it is worked on when the first keys
        // have been asked for as well
        if (own_kv) {
          const bf16_t* kr = row + (size_t)(H + g) * HEAD_DIM;
          const bf16_t* vr = row + (size_t)(H + G + g) * HEAD_DIM;
#pragma unroll
          for (int ks = 0; ks < D_KS; ++ks)
            k_new[ks] = *reinterpret_cast<const u32x4_t*>(kr + 32 * ks + 8 * kg);
#pragma unroll
          for (int mt = 0; mt < D_MT; ++mt) v_new[mt] = vr[16 * mt + col];
        }
        qk_load_tables(qk, pos, kg, tb);
      }
    }
    if (!fused) {
#pragma unroll
      for (int ks = 0; ks < D_KS; ++ks) qf[ks] = as_frag(qraw[ks]);
    }
  }
#pragma unroll
  for (int mt = 0; mt < D_MT; ++mt) o[mt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  m_run = -INFINITY;
  float l_lane = 0.f;                  // of the lane's own keys
  const float sc = scale * LOG2E;

  struct Part {
    u32x4_t k[2][D_KS], v[D_MT];
    int missing;             // bit i: the i-th 16 keys have no page
  };
  // (scalars) the page of the next 16 keys and their place in it
  auto next16 = [&](int& page, int& off) {
    page = __builtin_amdgcn_readlane(pages, page_at);
    off = page_off;
    page_off += 16;
    if (page_off >= ps) {
      page_off = 0;
      if (++page_at == WAVE) {
        page_at = 0;
        pages = pages_next;
        pages_from += WAVE;
        pages_are_here();
        pages_next = ask_pages(pages_from + WAVE);
      }
    }
  };
  // Row r of the key tile tt (of the 32 keys from kb) is key kb + 8 (r / 4) + 4 tt + r % 4:
  // the lane that holds rows 4 kg .. 4 kg + 3 of both tiles' scores then holds the keys
  // kb + 8 kg .. + 7 in order, and their values are ONE 16-byte piece of a V^T row.
  const int k_lane = (8 * (col / 4 % 2) + col % 4) * HEAD_DIM + 8 * kg;     // + 4 tt rows, + 32 ks
  const int v_lane = col * ps + 8 * (kg % 2);                               // + 16 mt ps
  auto ask = [&](int kb, Part& p) {
    int pg[2], off[2];
    next16(pg[0], off[0]);
    next16(pg[1], off[1]);
    // (a key that no row sees lies in a page that is there, or page 0 stands in for the one that is not:
    // what comes of it is left out when the part is worked on)
    p.missing = (pg[0] < 0 ? 1 : 0) | (pg[1] < 0 ? 2 : 0);
    const size_t a0 = ((size_t)max(pg[0], 0) * G + g) * ps, a1 = ((size_t)max(pg[1], 0) * G + g) * ps;
    const bf16_t* kp = k_pool + (col < 8 ? (a0 + off[0]) * HEAD_DIM : (a1 + off[1]) * HEAD_DIM) + k_lane;
    const bf16_t* vp = vt_pool + (kg < 2 ? a0 * HEAD_DIM + off[0] : a1 * HEAD_DIM + off[1]) + v_lane;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int ks = 0; ks < D_KS; ++ks) {
        const bool there = HEAD_DIM % 32 == 0 || 32 * ks + 8 * kg < HEAD_DIM;
        const u32x4_t x = *reinterpret_cast<const u32x4_t*>(there ? kp + 4 * tt * HEAD_DIM + 32 * ks : k_pool);
        p.k[tt][ks] = there ? x : (u32x4_t){0u, 0u, 0u, 0u};
      }
#pragma unroll
    for (int mt = 0; mt < D_MT; ++mt) p.v[mt] = *reinterpret_cast<const u32x4_t*>(vp + 16 * mt * ps);
  };
  // the part's keys that the row does not see, or whose page is missing: their values read as zero, and so
  // do the keys of a missing page (the others' scores are dropped, whatever they are)
  auto leave_out = [&](int kb, Part& p) {
    const int key0 = kb + 8 * kg;
    const bool there = !(p.missing >> (kg / 2) & 1);
    uint32_t m[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      m[i] = (there && key0 + 2 * i >= lo && key0 + 2 * i <= hi ? 0x0000ffffu : 0u) |
             (there && key0 + 2 * i + 1 >= lo && key0 + 2 * i + 1 <= hi ? 0xffff0000u : 0u);
#pragma unroll
    for (int mt = 0; mt < D_MT; ++mt)
      p.v[mt] = (u32x4_t){p.v[mt].x & m[0], p.v[mt].y & m[1], p.v[mt].z & m[2], p.v[mt].w & m[3]};
    if (p.missing) {
      const uint32_t mk = p.missing >> (col / 8) & 1 ? 0u : 0xffffffffu;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int ks = 0; ks < D_KS; ++ks)
          p.k[tt][ks] = (u32x4_t){p.k[tt][ks].x & mk, p.k[tt][ks].y & mk, p.k[tt][ks].z & mk, p.k[tt][ks].w & mk};
    }
  };
  // the pools do not hold the row's own key and value yet (or only just): the part that holds
  // the row's position takes them from the registers
  auto own = [&](int kb, Part& p) {
    if (!(own_kv && pos >= kb && pos < kb + 32)) return;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      if (kb + 8 * (col / 4) + 4 * tt + col % 4 == pos) {
#pragma unroll
        for (int ks = 0; ks < D_KS; ++ks) p.k[tt][ks] = k_new[ks];
      }
    }
    const int e = pos - (kb + 8 * kg);
    if (e >= 0 && e < 8) {
      const uint32_t keep = (e & 1) ? 0x0000ffffu : 0xffff0000u;
#pragma unroll
      for (int mt = 0; mt < D_MT; ++mt) {
        const uint32_t put = (v_new[mt] & 0xffffu) << ((e & 1) * 16);
        uint32_t w[4] = {p.v[mt].x, p.v[mt].y, p.v[mt].z, p.v[mt].w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (i == e / 2) w[i] = (w[i] & keep) | put;
        p.v[mt] = (u32x4_t){w[0], w[1], w[2], w[3]};
      }
    }
  };
  auto work = [&](int kb, Part& p) {
    const bool whole = kb >= lo && kb + 31 <= hi;
    if (!whole || p.missing) leave_out(kb, p);
    own(kb, p);
    f32x4_t s[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      s[tt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < D_KS; ++ks)
        s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(p.k[tt][ks]), qf[ks], s[tt], 0, 0, 0);
    }
    // lane holds, for head `col`, keys kb + 8*kg + 4*tt + v
    float mloc = -INFINITY;
    if (whole) {
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          s[tt][v] *= sc;
          mloc = fmaxf(mloc, s[tt][v]);
        }
    } else {
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int key = kb + 8 * kg + 4 * tt + v;
          s[tt][v] = key >= lo && key <= hi ? s[tt][v] * sc : -INFINITY;
          mloc = fmaxf(mloc, s[tt][v]);
        }
    }
    mloc = fmaxf(mloc, lane_xor16(mloc));
    mloc = fmaxf(mloc, other_half(mloc));
    const float m_new = fmaxf(m_run, mloc);
    const float m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float corr = fast_exp2(m_run - m_safe);
    float lsum = 0.f;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s[tt][v] = fast_exp2(s[tt][v] - m_safe);
        lsum += s[tt][v];
      }
    l_lane = l_lane * corr + lsum;
    m_run = m_new;
    const u32x4_t pw = {pack_bf16(s[0][0], s[0][1]), pack_bf16(s[0][2], s[0][3]),
                        pack_bf16(s[1][0], s[1][1]), pack_bf16(s[1][2], s[1][3])};
    const bf16x8_t pf = as_frag(pw);
#pragma unroll
    for (int mt = 0; mt < D_MT; ++mt) {
      o[mt] = o[mt] * corr;
      o[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(p.v[mt]), pf, o[mt], 0, 0, 0);
    }
  };
  // (what the row's own position needs: the norm, the rotation, the store)
  auto prologue = [&] {
    if constexpr (FUSABLE && D_QK_FUSABLE) {
      if (fused) {
        if (own_kv) qk_norm_rotate(k_new, qk.k_norm_w != nullptr, tb.wk, qk.eps,
                                   qk.cos_tab != nullptr, tb.cs, tb.sn);
        qk_norm_rotate(qraw, qk.q_norm_w != nullptr, tb.wq, qk.eps, qk.cos_tab != nullptr, tb.cs,
                       tb.sn);
#pragma unroll
        for (int ks = 0; ks < D_KS; ++ks)
          qf[ks] = as_frag(head_ok ? qraw[ks] : (u32x4_t){0u, 0u, 0u, 0u});
        // the wave whose keys hold the row's own position puts its key and value into the pools
        if (own_kv && pos >= first && pos < k_end) {
          const size_t pg = (size_t)bt[pos / ps] * G + g;
          if (col == 0) {
#pragma unroll
            for (int ks = 0; ks < D_KS; ++ks)
              *reinterpret_cast<u32x4_t*>(qk.k_pool_w + (pg * ps + pos % ps) * HEAD_DIM + 32 * ks +
                                          8 * kg) = k_new[ks];
          }
          if (kg == 0) {
#pragma unroll
            for (int mt = 0; mt < D_MT; ++mt)
              qk.vt_pool_w[(pg * HEAD_DIM + 16 * mt + col) * ps + pos % ps] = (bf16_t)v_new[mt];
          }
        }
      }
    }
  };
  // A wait counts the loads that may stay under way, the fewest over all ways that lead to it.  Hence a loop
  // of whole rounds without conditions, left at its end only, for waves with D_AHEAD parts or more; what is
  // left to ask for behind it, and the parts of a wave that has fewer, stand by themselves.
  Part part[D_AHEAD];
  const int n_parts = (k_end - first + 31) / 32;
  int kb = first, kb_ask = first + 32 * D_AHEAD;
  int left = n_parts;                        // parts to be worked on behind everything else
  pages_are_here();
  if (n_parts >= D_AHEAD) {
#pragma unroll
    for (int i = 0; i < D_AHEAD; ++i) {
      ask(first + 32 * i, part[i]);
      __builtin_amdgcn_sched_barrier(0);      // (in this order)
    }
    prologue();
    for (left = n_parts - D_AHEAD; left >= D_AHEAD; left -= D_AHEAD) {
#pragma unroll
      for (int i = 0; i < D_AHEAD; ++i) {
        work(kb, part[i]);
        ask(kb_ask, part[i]);
        kb += 32;
        kb_ask += 32;
      }
    }
#pragma unroll
    for (int i = 0; i < D_AHEAD; ++i) {
      work(kb, part[i]);
      if (i < left) ask(kb_ask, part[i]);
      kb += 32;
      kb_ask += 32;
    }
  } else {
#pragma unroll
    for (int i = 0; i < D_AHEAD - 1; ++i)
      if (i < left) ask(first + 32 * i, part[i]);
    prologue();
  }
#pragma unroll
  for (int i = 0; i < D_AHEAD - 1; ++i) {
    if (i < left) work(kb, part[i]);
    kb += 32;
  }
  l_lane += lane_xor16(l_lane);
  l_run = l_lane + other_half(l_lane);
}

// One wave's share of a row's attention: the query heads of kv head g (columns) against the keys
// of the chunks c0 = first, first + stride, ... below k_end (D_KPW keys each), with a running
// maximum and sum per column.  Leaves the unnormalised output in o (lane: column lane % 16, d
// rows 16 mt + 4 (lane / 16) + v), the maximum (in units of log 2) in m_run, the sum in l_run.
// With MODS the scores are worked on (score_mods.h) and the chunks are counted in places (kappai_key_at):
// the kept first keys stand in front of the window's, whose places are their positions.  Without, for
// the block kernel at head size 256, which has no registers for the page ids of attn_decode_wave.
template <bool MODS>
__device__ __forceinline__ void attn_decode_chunk_wave(
    const bf16_t* __restrict__ q, int q_stride, const bf16_t* __restrict__ k_pool,
    const bf16_t* __restrict__ vt_pool, const int* __restrict__ bt, int max_blocks, int t, int g,
    int H, int G, int ps, float scale, int lo, int hi, int first, int stride, int k_end,
    f32x4_t (&o)[D_MT], float& m_run, float& l_run, int pos, const kappai_score_mods* mods) {
  const int lane = threadIdx.x % WAVE;
  const int rep = H / G;
  const int col = lane % 16, kg = lane / 16;
  const bool head_ok = col < rep;
  const int h = g * rep + (head_ok ? col : 0);
  // the page ids of the first chunk of keys: asked for before anything else, so that the keys
  // can be asked for as soon as they are there, whatever else is still on its way
  const int keep = MODS ? mods->keep_first : 0;
  const int lo32 = (lo / 32) * 32;
  const int kept = MODS ? kappai_kept_places(keep, lo32) : 0;
  auto ask_pages = [&](int c0) {      // lane i: the page of the chunk's places 16 i .. 16 i + 15
    const int key = MODS ? kappai_key_at(c0 + 16 * lane, lo32, kept) : c0 + 16 * lane;
    return 16 * lane < D_KPW && key / ps < max_blocks && (key <= hi || (MODS && key < keep)) ? bt[key / ps] : -1;
  };
  int pages_first = first < k_end ? ask_pages(first) : -1;
  bf16x8_t qf[D_KS];
  {
    const bf16_t* qr = q + (size_t)t * q_stride + (size_t)h * HEAD_DIM;
#pragma unroll
    for (int ks = 0; ks < D_KS; ++ks) {
      u32x4_t v = {0u, 0u, 0u, 0u};
      const int d0 = 32 * ks + 8 * kg;
      if (head_ok && d0 < HEAD_DIM) v = *reinterpret_cast<const u32x4_t*>(qr + d0);
      qf[ks] = as_frag(v);
    }
  }
#pragma unroll
  for (int mt = 0; mt < D_MT; ++mt) o[mt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  m_run = -INFINITY;
  l_run = 0.f;

  // A wave takes its keys in chunks of D_KPW: first the chunk's page ids (one load, handed
  // round by shuffles), then every key and value load of the chunk at once (16 bytes a lane
  // each), then the matrix products and the softmax: two memory round trips a chunk, whatever
  // its length.  (Two chunks' loads in flight at once were measured: the registers they take
  // halve the waves a SIMD holds, and 64 requests at 4096 keys took 140 us instead of 100.)
  constexpr int NCH = D_KPW / 32;
  struct Chunk {
    u32x4_t kf[NCH][2][D_KS];
    u32x4_t vv[NCH][D_MT];
    float bias[MODS ? NCH : 1][8];     // of the lane's eight keys, the last key first
  };
  const float* bias_row = MODS && mods->dist_bias != nullptr ? kappai_bias_row(*mods, h) : nullptr;
  auto ask = [&](int c0, int my_page, Chunk& ch) {
    // Row r of the key tile tt (of the 32 keys from kb) is key kb + 8 (r / 4) + 4 tt + r % 4:
    // the lane that holds rows 4 kg .. 4 kg + 3 of both tiles' scores then holds the keys
    // kb + 8 kg .. + 7 in order, and their values are ONE 16-byte piece of a V^T row.
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int kb = MODS ? kappai_key_at(c0 + 32 * c, lo32, kept) : c0 + 32 * c;
      // (what the row does not see reads as zero)
      const int f_lo = MODS && kb < keep ? kb : lo, f_hi = MODS && kb < lo32 ? keep - 1 : hi;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const int key = kb + 8 * (col / 4) + 4 * tt + col % 4;
        const int page = __shfl(my_page, 2 * c + (key - kb) / 16, WAVE);
#pragma unroll
        for (int ks = 0; ks < D_KS; ++ks)
          ch.kf[c][tt][ks] = load_k8_pg(k_pool, page, G, g, ps, key, 32 * ks + 8 * kg, f_lo, f_hi);
      }
      const int pv = __shfl(my_page, 2 * c + kg / 2, WAVE);
#pragma unroll
      for (int mt = 0; mt < D_MT; ++mt)
        ch.vv[c][mt] = load_vt8_pg(vt_pool, pv, G, g, ps, 16 * mt + col, kb + 8 * kg,
                                    f_lo, f_hi);
      if constexpr (MODS) {
        if (bias_row != nullptr) {     // distances base .. base + 7, by the row's edges at most
          const int base = max(-KAPPAI_BIAS_PAD, min(pos - kb - 8 * kg - 7, mods->dist_cols - 1));
          const f32x4_any_t b0 = *reinterpret_cast<const f32x4_any_t*>(bias_row + base);
          const f32x4_any_t b1 = *reinterpret_cast<const f32x4_any_t*>(bias_row + base + 4);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            ch.bias[c][i] = b0[i];
            ch.bias[c][4 + i] = b1[i];
          }
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) ch.bias[c][i] = 0.f;
        }
      }
    }
  };
  auto work = [&](int c0, const Chunk& ch) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      if (c0 + 32 * c >= k_end) break;
      const int kb = MODS ? kappai_key_at(c0 + 32 * c, lo32, kept) : c0 + 32 * c;
      f32x4_t s[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        s[tt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < D_KS; ++ks)
          s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(ch.kf[c][tt][ks]), qf[ks], s[tt],
                                                          0, 0, 0);
      }
      // lane holds, for head `col`, keys kb + 8*kg + 4*tt + v
      float mloc = -INFINITY;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int key = kb + 8 * kg + 4 * tt + v;
          const bool ok = (key >= lo || (MODS && key < keep)) && key <= hi;
          float x = s[tt][v] * scale;
          if constexpr (MODS) {
            if (mods->softcap > 0.f) x = kappai_fast_cap(x, mods->softcap);
            x += ch.bias[c][7 - (4 * tt + v)];
          }
          s[tt][v] = ok ? x * LOG2E : -INFINITY;
          mloc = fmaxf(mloc, s[tt][v]);
        }
      mloc = fmaxf(mloc, __shfl_xor(mloc, 16, WAVE));
      mloc = fmaxf(mloc, other_half(mloc));
      const float m_new = fmaxf(m_run, mloc);
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;
      const float corr = fast_exp2(m_run - m_safe);
      float lsum = 0.f;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          s[tt][v] = fast_exp2(s[tt][v] - m_safe);
          lsum += s[tt][v];
        }
      lsum += __shfl_xor(lsum, 16, WAVE);
      lsum += other_half(lsum);
      l_run = l_run * corr + lsum;
      m_run = m_new;
      const u32x4_t pw = {pack_bf16(s[0][0], s[0][1]), pack_bf16(s[0][2], s[0][3]),
                          pack_bf16(s[1][0], s[1][1]), pack_bf16(s[1][2], s[1][3])};
      const bf16x8_t pf = as_frag(pw);
#pragma unroll
      for (int mt = 0; mt < D_MT; ++mt) {
        o[mt] = o[mt] * corr;
        o[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(ch.vv[c][mt]), pf, o[mt], 0, 0, 0);
      }
    }
  };
  for (int c0 = first; c0 < k_end; c0 += stride) {
    Chunk ca;
    ask(c0, c0 == first ? pages_first : ask_pages(c0), ca);
    work(c0, ca);
  }
}

// How many keys a split takes in this step.  The host sizes the grid for up to n_splits splits of
// at least kps_min keys from the step's longest context; what the rows really hold decides here:
// as many keys a split that the rows' keys together give D_TARGET_WAVES waves work (requests of
// mixed lengths then get shorter splits than their longest context alone would give them, and
// no wave walks a long row's keys by itself while the rest of the chip has nothing to do), and
// no fewer than the longest row needs to fit into n_splits, in whole numbers of `unit` (the scored wave walks
// chunks of D_KPW).  Every wave of the step computes the same number from the same table; splits past a row's
// keys do nothing and are not merged.
#define D_TARGET_WAVES 2048
__device__ __forceinline__ int keys_of_row(int pos, int window, int keep) {
  const int lo32 = kappai_first_key(pos, window) / 32 * 32;
  return pos + 1 - lo32 + kappai_kept_places(keep, lo32);
}
__device__ __forceinline__ int step_keys_per_split(const int* __restrict__ row_pos,
                                                   const int* __restrict__ row_ids, int n_rows,
                                                   int window, int keep, int G, int kps_min,
                                                   int n_splits, int unit) {
  const int lane = threadIdx.x % WAVE;
  int total32 = 0, longest = 0;                  // the sum in units of 32 keys, rounded up by row
  for (int i = lane; i < n_rows; i += WAVE) {
    const int n = keys_of_row(row_pos[row_ids ? row_ids[i] : i], window, keep);
    total32 += (n + 31) / 32;
    longest = max(longest, n);
  }
  total32 = wave_sum(total32);
  longest = wave_max(longest);
  const long long want = ((long long)total32 * G * 32 + D_TARGET_WAVES - 1) / D_TARGET_WAVES;
  int kps = want > (1 << 30) ? (1 << 30) : (int)want;
  kps = max(kps, (longest + n_splits - 1) / n_splits);
  kps = max(kps, kps_min);
  return __builtin_amdgcn_readfirstlane((kps + unit - 1) / unit * unit);
}

// The keys of a row split over blocks: block (t, g, split) is one wave that takes the keys
// k_begin + split * kps .. (kps: step_keys_per_split, at least the caller's keys_per_split) and
// writes its partial result; attn_merge adds up those of the splits that had keys.
// (FUSED: with the prologue of QkFuse; a kernel of its own, because the prologue's registers would
// halve the waves a SIMD holds for the steps that do not use it)
// (PLAN: the keys per split come from step_keys_per_split, else they are the caller's: a kernel of
// its own, because the rule's code costs half a microsecond even where it is skipped)
// (The arguments of this kernel and of the two that do a row in one block stand in the order in which they are
// needed: the first fourteen words come in registers, and they are those on the way to the row's pages, which
// are three dependent reads ahead of the first key.  The pools' addresses are asked for beside the position.
// One row of 16 heads at 200 to 1,000 keys, whole pass of 22 layers with 6 of these: 7,280 -> 7,260 us for 64
// tokens, 16 rows at 4,000 keys 1,318 -> 1,303 us a step.)
template <bool FUSED, bool PLAN, bool MODS = false>
__global__ __launch_bounds__(64, (FUSED && HEAD_DIM != 64) || MODS || HEAD_DIM > 128 ? 1 : 2) void attn_decode_kernel(
    const int* __restrict__ row_pos, const int* __restrict__ row_seg,
    const int* __restrict__ block_tables, const int* __restrict__ row_ids, int max_blocks, int H, int G,
    int ps, int q_stride, int window, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_pool,
    const bf16_t* __restrict__ vt_pool, float* __restrict__ part_o, float* __restrict__ part_ml,
    float scale, int keys_per_split, int n_splits, QkFuse qk, kappai_score_mods mods) {
  // (the arguments on the way to the row's pages come first: those are handed over in registers)
  // (row_ids: the kernel's rows are these rows of the step, partial results are kept by their
  // place in the list)
  // Blocks go to the CUs in the order of their numbers, the row's number fastest: with a number
  // of rows that divides the number of CUs, a CU would get the same row in every (kv head,
  // split), and rows of different lengths would load the CUs unevenly.  Hence the rows are
  // taken in an order that turns with the kv head and the split.
  const int g = blockIdx.y, split = blockIdx.z, lane = threadIdx.x;
  const int ti = (int)((blockIdx.x + 7u * (blockIdx.y + gridDim.y * blockIdx.z)) % gridDim.x);
  const int t = row_ids ? row_ids[ti] : ti;
  const int rep = H / G;
  const int col = lane % 16, kg = lane / 16;
  const int pos = row_pos[t];
  const int seg = row_seg[t];
  const int keep = MODS ? mods.keep_first : 0;
  const int kps = PLAN ? step_keys_per_split(row_pos, row_ids, (int)gridDim.x, window, keep, G,
                                             keys_per_split, n_splits, MODS ? D_KPW : D_SPLIT_SHARE)
                       : keys_per_split;
  const int* bt = block_tables + (size_t)seg * max_blocks;
  const int lo = kappai_first_key(pos, window);
  const int lo32 = (lo / 32) * 32;
  const int k_begin = lo32 - (MODS ? kappai_kept_places(keep, lo32) : 0) + split * kps;
  if (k_begin > pos) return;                                   // a split past the row's keys
  const int k_end = min(k_begin + kps, pos + 1);                // exclusive
  const bool head_ok = col < rep;
  const int h = g * rep + (head_ok ? col : 0);
  const size_t pbase = ((size_t)ti * H + h) * n_splits + split;
  f32x4_t o[D_MT];
  float m_run, l_run;
  if constexpr (MODS)
    attn_decode_chunk_wave<true>(q, q_stride, k_pool, vt_pool, bt, max_blocks, t, g, H, G, ps, scale, lo,
                                 k_end - 1, k_begin, D_KPW, k_end, o, m_run, l_run, pos, &mods);
  else
    attn_decode_wave<FUSED>(q, q_stride, k_pool, vt_pool, bt, max_blocks, t, g, H, G, ps, scale, lo,
                            k_begin, k_end, o, m_run, l_run, qk, pos);
  if (!head_ok) return;
  if (kg == 0) {
    part_ml[2 * pbase] = m_run;
    part_ml[2 * pbase + 1] = l_run;
  }
  float* po = part_o + pbase * HEAD_DIM;
#pragma unroll
  for (int mt = 0; mt < D_MT; ++mt)
    *reinterpret_cast<f32x4_t*>(po + 16 * mt + 4 * kg) = o[mt];
}

// (eight waves at most: a wave keeps a whole chunk's loads in registers, which 16 waves a block
// would not leave room for)
#define D_BLOCK_MAX_WAVES 8
// The keys of a row split over the waves of one block (t, g): equal shares (with MODS wave w
// takes the chunks w, w + NW, ... of D_KPW keys), the waves' results meet in LDS and are added up there in
// the order of the waves, so that nothing goes through memory and no second kernel is needed.  The split of
// a row's keys depends on the row's own position and on the number of waves only.  For batches with
// (rows x kv heads) enough to fill the chip, or contexts short enough for one block.
// LDS: sh_o [NW][rep][HEAD_DIM], then sh_m [NW][16], sh_l [NW][16] (floats).
template <bool MODS, bool FUSED, int SHARE>
__device__ __forceinline__ void attn_one_row(const bf16_t* q, int q_stride, const bf16_t* k_pool,
                                             const bf16_t* vt_pool, bf16_t* out, int out_stride,
                                             const int* bt, int max_blocks, int t, int pos, int g, int H,
                                             int G, int ps, int window, float scale,
                                             const kappai_score_mods& mods, float* sh, int NW,
                                             const QkFuse* qk) {
  const int lane = threadIdx.x % WAVE;
  // (in scalar registers: the walk over the wave's keys is then scalar work)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int rep = H / G;
  const int col = lane % 16, kg = lane / 16;
  const int lo = kappai_first_key(pos, window);
  const int lo32 = (lo / 32) * 32;
  const int k_begin = lo32 - (MODS ? kappai_kept_places(mods.keep_first, lo32) : 0);
  const int k_end = pos + 1;
  f32x4_t o[D_MT];
  float m_run, l_run;
  if constexpr (MODS || (HEAD_DIM == 256 && !FUSED)) {
    attn_decode_chunk_wave<MODS>(q, q_stride, k_pool, vt_pool, bt, max_blocks, t, g, H, G, ps, scale, lo, pos,
                                 k_begin + wave * D_KPW, NW * D_KPW, k_end, o, m_run, l_run, pos, &mods);
  } else {
    const int per = ((k_end - k_begin + SHARE - 1) / SHARE + NW - 1) / NW * SHARE;
    const int from = k_begin + wave * per;
    if (FUSED && from >= k_end) {              // (no keys: no prologue either)
#pragma unroll
      for (int mt = 0; mt < D_MT; ++mt) o[mt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      m_run = -INFINITY;
      l_run = 0.f;
    } else {
      attn_decode_wave<FUSED>(q, q_stride, k_pool, vt_pool, bt, max_blocks, t, g, H, G, ps, scale, lo,
                              from, min(from + per, k_end), o, m_run, l_run,
                              FUSED ? *qk : QkFuse{}, pos);
    }
  }
  float* sh_o = sh;
  float* sh_m = sh + (size_t)NW * rep * HEAD_DIM;
  float* sh_l = sh_m + NW * 16;
  if (col < rep) {
    float* po = sh_o + ((size_t)wave * rep + col) * HEAD_DIM;
#pragma unroll
    for (int mt = 0; mt < D_MT; ++mt)
      *reinterpret_cast<f32x4_t*>(po + 16 * mt + 4 * kg) = o[mt];
    if (kg == 0) {
      sh_m[wave * 16 + col] = m_run;
      sh_l[wave * 16 + col] = l_run;
    }
  }
  __syncthreads();
  // out[t, g rep + c, e] for (c, e) in turn over the block's threads
  for (int i = threadIdx.x; i < rep * HEAD_DIM; i += NW * WAVE) {
    const int c = i / HEAD_DIM, e = i % HEAD_DIM;
    float M = -INFINITY;
    for (int w = 0; w < NW; ++w) M = fmaxf(M, sh_m[w * 16 + c]);
    float L = 0.f, acc = 0.f;
    for (int w = 0; w < NW; ++w) {
      const float m = sh_m[w * 16 + c];
      const float wgt = m == -INFINITY ? 0.f : fast_exp2(m - M);
      L += sh_l[w * 16 + c] * wgt;
      acc = fmaf(sh_o[((size_t)w * rep + c) * HEAD_DIM + e], wgt, acc);
    }
    if (mods.sink != nullptr && M != -INFINITY)
      L += fast_exp2(mods.sink[g * rep + c] * LOG2E - M);
    const float inv = L > 0.f ? 1.0f / L : 0.f;
    out[(size_t)t * out_stride + (size_t)(g * rep + c) * HEAD_DIM + e] = f32_to_bf16(acc * inv);
  }
}

template <bool MODS>
__global__ __launch_bounds__(D_BLOCK_MAX_WAVES * WAVE) void attn_decode_block_kernel(
    const int* __restrict__ row_pos, const int* __restrict__ row_seg,
    const int* __restrict__ block_tables, int max_blocks, int H, int G, int ps, int q_stride, int window,
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ vt_pool,
    bf16_t* __restrict__ out, int out_stride, float scale, kappai_score_mods mods) {
  extern __shared__ float sh_dec[];
  const int t = blockIdx.x;
  attn_one_row<MODS, false, D_BLOCK_SHARE>(q, q_stride, k_pool, vt_pool, out, out_stride,
                                           block_tables + (size_t)row_seg[t] * max_blocks, max_blocks, t,
                                           row_pos[t], blockIdx.y, H, G, ps, window, scale, mods, sh_dec,
                                           blockDim.x / WAVE);
}

// attn_decode_block_kernel with the prologue of QkFuse in the waves that have keys (see
// D_QK_BLOCK_MAX_KEYS).
#if HEAD_DIM == 64
__global__ __launch_bounds__(D_BLOCK_MAX_WAVES * WAVE) void attn_decode_block_qk_kernel(
    const int* __restrict__ row_pos, const int* __restrict__ row_seg,
    const int* __restrict__ block_tables, int max_blocks, int H, int G, int ps, int row_stride, int window,
    const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ vt_pool,
    bf16_t* __restrict__ out, int out_stride, float scale, QkFuse qk) {
  extern __shared__ float sh_dec[];
  const int t = blockIdx.x;
  attn_one_row<false, true, D_BLOCK_SHARE>(qkv, row_stride, k_pool, vt_pool, out, out_stride,
                            block_tables + (size_t)row_seg[t] * max_blocks, max_blocks, t, row_pos[t],
                            blockIdx.y, H, G, ps, window, scale,
                            kappai_score_mods{0.f, nullptr, 0, nullptr, 0}, sh_dec,
                            blockDim.x / WAVE, &qk);
}
#endif

// out[t, h, :] = sum_s o_s 2^(m_s - M) / sum_s l_s 2^(m_s - M).  Four waves share the splits
// (wave w takes s = w, w+4, ...); each computes its splits' weights one per lane.  The partial
// outputs of MERGE_AHEAD splits are asked for before the maxima, so that with up to 32 splits
// the kernel waits for memory once.  (Loads without conditions: of loads in branches of their own the compiler
// puts a wait between.)
#define MERGE_WAVES 4
#define MERGE_AHEAD 8
__global__ __launch_bounds__(MERGE_WAVES * WAVE) void attn_merge_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml,
    const int* __restrict__ row_pos, const int* __restrict__ row_ids, int H, int splits_stride, int window,
    int keep, int kps_min, int plan_unit, int G, bf16_t* __restrict__ out, int out_stride,
    const float* __restrict__ sink) {
  constexpr int NPL = (HEAD_DIM + WAVE - 1) / WAVE;
  __shared__ float sh_acc[MERGE_WAVES][NPL * WAVE];
  __shared__ float sh_l[MERGE_WAVES];
  const int t = row_ids ? row_ids[blockIdx.x] : blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const size_t base = ((size_t)blockIdx.x * H + h) * splits_stride;
  // the partial outputs of this wave's splits number j .. j + MERGE_AHEAD - 1, of the first
  // `bound` splits
  float o[MERGE_AHEAD][NPL];
#if defined(__HIP_DEVICE_COMPILE__)
  const __amdgpu_buffer_rsrc_t parts = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(part_o + base * HEAD_DIM), 0, splits_stride * HEAD_DIM * 4, 0x00020000);
  auto part_at = [&](int e, int sk, int bound) {
    const int at = e < HEAD_DIM && sk < bound ? (sk * HEAD_DIM + e) * 4 : 0x7FFFFF00;
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(parts, at, 0, 0));
  };
#else
  auto part_at = [&](int, int, int) { return 0.f; };
#endif
  auto ask = [&](int j, int bound) {
#pragma unroll
    for (int k = 0; k < MERGE_AHEAD; ++k) {
      const int sk = wave + MERGE_WAVES * (j + k);
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        // (splits behind the last and places behind the head: outside the buffer, zeros, nothing read)
        o[k][i] = part_at(lane + i * WAVE, sk, bound);
      }
    }
  };
  // The first partial outputs and maxima are asked for before the number of splits that had keys
  // is known (it takes the row's position): whatever the grid has room for is loaded, and what
  // lies past the row's splits (never written, or by an earlier step) is dropped afterwards.
  ask(0, splits_stride);
  const float m_first = lane < splits_stride ? part_ml[2 * (base + lane)] : -INFINITY;
  float2 ml_first = make_float2(-INFINITY, 0.f);        // of the split wave + MERGE_WAVES * lane
  if (wave + MERGE_WAVES * lane < splits_stride)
    ml_first = *reinterpret_cast<const float2*>(part_ml + 2 * (base + wave + MERGE_WAVES * lane));
  // the splits of this row that had keys (the decode kernel's own rule)
  const int kps = plan_unit ? step_keys_per_split(row_pos, row_ids, (int)gridDim.x, window, keep, G,
                                                  kps_min, splits_stride, plan_unit)
                            : kps_min;
  const int n_splits = (keys_of_row(row_pos[t], window, keep) + kps - 1) / kps;
#pragma unroll
  for (int k = 0; k < MERGE_AHEAD; ++k)
#pragma unroll
    for (int i = 0; i < NPL; ++i)
      if (wave + MERGE_WAVES * k >= n_splits) o[k][i] = 0.f;
  float M = lane < n_splits ? m_first : -INFINITY;
  for (int s = lane + WAVE; s < n_splits; s += WAVE) M = fmaxf(M, part_ml[2 * (base + s)]);
  M = wave_max(M);
  float L = 0.f;
  float acc[NPL];
#pragma unroll
  for (int i = 0; i < NPL; ++i) acc[i] = 0.f;
  // this wave's splits, 64 at a time: split index s = wave + MERGE_WAVES * j
  for (int j0 = 0; wave + MERGE_WAVES * j0 < n_splits; j0 += WAVE) {
    const int s = wave + MERGE_WAVES * (j0 + lane);
    float wgt = 0.f, l = 0.f;
    if (s < n_splits) {
      const float2 ml = j0 == 0 ? ml_first
                                : *reinterpret_cast<const float2*>(part_ml + 2 * (base + s));
      wgt = ml.x == -INFINITY ? 0.f : fast_exp2(ml.x - M);
      l = ml.y * wgt;
    }
    L += wave_sum(l);
    for (int k0 = 0; k0 < WAVE; k0 += MERGE_AHEAD) {
      if (wave + MERGE_WAVES * (j0 + k0) >= n_splits) break;
      if (j0 + k0 > 0) ask(j0 + k0, n_splits);
#pragma unroll
      for (int k = 0; k < MERGE_AHEAD; ++k) {
        // a split past the end has the weight 0 and the partial output 0
        const float wk = __shfl(wgt, k0 + k, WAVE);
#pragma unroll
        for (int i = 0; i < NPL; ++i) acc[i] = fmaf(o[k][i], wk, acc[i]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NPL; ++i) sh_acc[wave][i * WAVE + lane] = acc[i];
  if (lane == 0) sh_l[wave] = L;
  __syncthreads();
  if (wave != 0) return;
  L = (sh_l[0] + sh_l[1]) + (sh_l[2] + sh_l[3]);
  if (sink != nullptr && M != -INFINITY) L += fast_exp2(sink[h] * LOG2E - M);   // (sink: a logit)
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  bf16_t* dst = out + (size_t)t * out_stride + (size_t)h * HEAD_DIM;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int e = lane + i * WAVE;
    const float v = (sh_acc[0][i * WAVE + lane] + sh_acc[1][i * WAVE + lane]) +
                    (sh_acc[2][i * WAVE + lane] + sh_acc[3][i * WAVE + lane]);
    if (e < HEAD_DIM) dst[e] = f32_to_bf16(v * inv);
  }
}

extern "C" int kappai_attn_keys_per_wave(void) { return D_KPW; }

// Waves of a block of the decode kernel that merges in LDS, for `rep` query heads a kv head:
// as many as 64 KB of LDS hold partial results for (D_BLOCK_MAX_WAVES at most), 0 if not even two.
extern "C" int kappai_attn_decode_block_waves(int rep) {
  if (rep < 1 || rep > 16) return 0;
  const int per_wave = (rep * HEAD_DIM + 32) * (int)sizeof(float);
  int nw = (64 * 1024) / per_wave;
  nw = nw > D_BLOCK_MAX_WAVES ? D_BLOCK_MAX_WAVES : nw;
  return nw >= 2 ? nw : 0;
}

// Decode attention with the keys of a row split over the `n_waves` waves of one block per (row, kv
// head); no workspace, no second kernel.
// `mods` (may be null): a cap on the scores, a bias by distance, a sink (score_mods.h).
extern "C" int kappai_attn_decode_block_scored(const void* q, int q_stride, const void* k_pool,
                                               const void* vt_pool, void* out, int out_stride,
                                               const int* row_pos, const int* row_seg,
                                               const int* block_tables, int max_blocks, int T,
                                               int H, int G, int ps, int window, float scale,
                                               int n_waves, const kappai_score_mods* mods,
                                               hipStream_t stream) {
  if (T <= 0) return 0;
  if (ps % 16 || G < 1 || H % G || H / G > 16 || G > 65535 || (q_stride % 8) || n_waves < 1 ||
      n_waves > kappai_attn_decode_block_waves(H / G))
    return (int)hipErrorInvalidValue;
  if (kappai_mods_change_scores(mods) &&
      (mods->keep_first < 0 || (mods->dist_bias != nullptr && mods->dist_cols < 1)))
    return (int)hipErrorInvalidValue;
  const int rep = H / G;
  const size_t lds = (size_t)n_waves * (rep * HEAD_DIM + 32) * sizeof(float);
  if (kappai_mods_change_scores(mods))
    hipLaunchKernelGGL(attn_decode_block_kernel<true>, dim3(T, G), dim3(n_waves * WAVE), lds,
                       stream, row_pos, row_seg, block_tables, max_blocks, H, G, ps, q_stride, window,
                       (const bf16_t*)q, (const bf16_t*)k_pool, (const bf16_t*)vt_pool, (bf16_t*)out,
                       out_stride, scale, *mods);
  else
    hipLaunchKernelGGL(attn_decode_block_kernel<false>, dim3(T, G), dim3(n_waves * WAVE), lds,
                       stream, row_pos, row_seg, block_tables, max_blocks, H, G, ps, q_stride, window,
                       (const bf16_t*)q, (const bf16_t*)k_pool, (const bf16_t*)vt_pool, (bf16_t*)out,
                       out_stride, scale,
                       kappai_score_mods{0.f, nullptr, 0, mods != nullptr ? mods->sink : nullptr, 0});
  KAPPAI_RETURN_LAUNCH_STATUS();
}

extern "C" int kappai_attn_decode_block(const void* q, int q_stride, const void* k_pool,
                                        const void* vt_pool, void* out, int out_stride,
                                        const int* row_pos, const int* row_seg,
                                        const int* block_tables, int max_blocks, int T, int H,
                                        int G, int ps, int window, float scale, int n_waves,
                                        hipStream_t stream) {
  return kappai_attn_decode_block_scored(q, q_stride, k_pool, vt_pool, out, out_stride, row_pos,
                                         row_seg, block_tables, max_blocks, T, H, G, ps, window,
                                         scale, n_waves, nullptr, stream);
}

// The most rows for which a step does better with kappai_attn_decode_qk than with a kernel for norm, rotation
// and store ahead of the decode kernels (0: this head size does not take it).  Every wave of a row and kv head
// does the prologue again.  us, two kernels / one, 32 heads of 64 on 8: 200 keys 5 rows 7.4 / 7.1, 16 rows 7.9 /
// 7.2; 1,500 keys 8 rows 11.9 / 10.8, 16 rows 17.6 / 15.9; 4,000 keys 8 rows 19.7 / 17.9, 16 rows 30.0 / 28.6;
// 16 rows of 100 to 7,100 keys 26.6 / 23.2 (more rows come as partial sums, which it does not take).  Heads of 128 have
// registers for one such wave a SIMD: 5 rows of 4,000 keys 24.1 / 27.3, 8 rows of 1,500 18.0 / 21.1.
#define D_QK_ROWS (!D_QK_FUSABLE ? 0 : HEAD_DIM == 64 ? 16 : 4)
extern "C" int kappai_attn_decode_takes_qk(void) { return D_QK_ROWS; }

// The most keys with which kappai_attn_decode_qk keeps a row's keys in one block (0: never at this head
// size).  One kernel in the place of two, but a CU takes in no more than about 50 GB/s of keys.  1 to 4 rows
// of 8 kv heads, us against split and merge: 40 keys 5.7 / 7.8, 300 keys 7.5 / 8.2, 500 keys 8.4 to 8.9 / 8.7 to
// 9.3, and beyond the split wins; a captured step knows its contexts as powers of two only, so the line is at
// 512.  Head size 128 has no registers for prologue and keys at two waves a SIMD (when it was tried 40 keys
// 9.9 / 10.6, 307 keys 15.2 / 10.6).
#define D_QK_BLOCK_MAX_KEYS (HEAD_DIM == 64 ? 512 : 0)
extern "C" int kappai_attn_decode_block_qk_keys(void) { return D_QK_BLOCK_MAX_KEYS; }

// The arguments that kappai_attn_decode_qk adds: qkv [T, row_stride] is the projection as it
// comes out of its product (q heads, then with store_kv the k heads and the v heads); q_norm_w /
// k_norm_w [d] float or null; cos_tab / sin_tab [positions, d / 2] float (rotate-half over the
// whole head) or both null; the pools are written at each row's own position when store_kv.
static bool qk_args_ok(const void* qkv, int row_stride, const float* q_norm_w,
                       const float* k_norm_w, const float* cos_tab, const float* sin_tab,
                       const void* k_pool, const void* vt_pool) {
  return D_QK_FUSABLE && row_stride % 8 == 0 && ((uintptr_t)qkv % 16) == 0 &&
         ((uintptr_t)q_norm_w % 16) == 0 && ((uintptr_t)k_norm_w % 16) == 0 &&
         ((uintptr_t)cos_tab % 16) == 0 && ((uintptr_t)sin_tab % 16) == 0 &&
         (cos_tab == nullptr) == (sin_tab == nullptr) && ((uintptr_t)k_pool % 16) == 0 &&
         vt_pool != nullptr;
}

extern "C" int kappai_attn_head_dim(void) { return HEAD_DIM; }

// variant: 0 = chosen by shape, 1 = one block per (tile, head), 2 = key tiles shared by four
// query heads of a kv head (head sizes 64 and 128, a multiple of four heads per kv head).
// `mods` (may be null; score_mods.h): with them the kernel of one block a (tile, head) runs.
extern "C" int kappai_attn_prefill_scored(const void* q, int q_stride, const void* k_pool,
                                          const void* vt_pool, void* out, int out_stride,
                                          const int* q_tiles, int n_tiles, const int* row_pos,
                                          const int* block_tables, int max_blocks, int H, int G,
                                          int ps, int window, float scale, int variant,
                                          const kappai_score_mods* mods, hipStream_t stream) {
  if (n_tiles <= 0) return 0;
  const float* sink = mods != nullptr ? mods->sink : nullptr;
  if (kappai_mods_change_scores(mods)) {
    if (ps % 16 || G < 1 || H % G || H > 65535 || (q_stride % 8) || (out_stride % 4) ||
        variant == 2 || mods->keep_first < 0 ||
        (mods->dist_bias != nullptr && mods->dist_cols < 1))
      return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(attn_prefill_kernel<true>, dim3(n_tiles, H), dim3(P_NW * WAVE), 0, stream,
                       q_tiles, row_pos, block_tables, max_blocks, H, G, ps, q_stride, window,
                       (const bf16_t*)q, (const bf16_t*)k_pool, (const bf16_t*)vt_pool, (bf16_t*)out,
                       out_stride, scale, *mods);
    KAPPAI_RETURN_LAUNCH_STATUS();
  }
  if (ps % 16 || G < 1 || H % G || H > 65535 || (q_stride % 8) || (out_stride % 4))
    return (int)hipErrorInvalidValue;
  const int rep = H / G;
  const bool shared_ok = PG_OK && rep % 4 == 0;
  if (variant == 2 && !shared_ok) return (int)hipErrorInvalidValue;
  // (the kernels over shared key tiles keep offsets of 31 bits within a kv head's part of a page)
  const bool near = (size_t)ps * HEAD_DIM * sizeof(bf16_t) < 0x7FFFFF00u;
  // sharing pays when there are blocks enough to fill the chip without splitting the keys of
  // a q tile over waves
  const bool shared = near && (variant == 2 || (variant == 0 && shared_ok && n_tiles * (H / 4) >= 256));
#if PG_OK
  if (shared) {
    hipLaunchKernelGGL(attn_prefill_shared_kernel, dim3(n_tiles, H / 4), dim3(8 * WAVE), 0, stream,
                       q_tiles, row_pos, block_tables, max_blocks, H, G, ps, q_stride, window,
                       (const bf16_t*)q, (const bf16_t*)k_pool, (const bf16_t*)vt_pool, (bf16_t*)out,
                       out_stride, scale, sink);
    KAPPAI_RETURN_LAUNCH_STATUS();
  }
#endif
#if HEAD_DIM == 256
  // (from the first tile on.  us with / without, 16 heads on one kv head: one portion of 5 rows 6.9 /
  // 8.7, of 32 rows 11.1 / 10.1 (the worst there is: a key tile or two that are full, on an empty chip), of
  // 32 rows behind 2,000 keys 131 / 165; 64 lone rows of 32 keys 6.9 / 10.0, 63 of 800 keys 64 / 126)
  if (near && variant == 0 && rep % 4 == 0) {
    hipLaunchKernelGGL(attn_prefill_heads_kernel, dim3(n_tiles, H / 4), dim3(8 * WAVE), 0, stream,
                       q_tiles, row_pos, block_tables, max_blocks, H, G, ps, q_stride, window,
                       (const bf16_t*)q, (const bf16_t*)k_pool, (const bf16_t*)vt_pool, (bf16_t*)out,
                       out_stride, scale, sink);
    KAPPAI_RETURN_LAUNCH_STATUS();
  }
#endif
  hipLaunchKernelGGL(attn_prefill_kernel<false>, dim3(n_tiles, H), dim3(P_NW * WAVE), 0, stream,
                     q_tiles, row_pos, block_tables, max_blocks, H, G, ps, q_stride, window,
                     (const bf16_t*)q, (const bf16_t*)k_pool, (const bf16_t*)vt_pool, (bf16_t*)out,
                     out_stride, scale, kappai_score_mods{0.f, nullptr, 0, sink, 0});
  KAPPAI_RETURN_LAUNCH_STATUS();
}

extern "C" int kappai_attn_prefill(const void* q, int q_stride, const void* k_pool,
                                   const void* vt_pool, void* out, int out_stride,
                                   const int* q_tiles, int n_tiles, const int* row_pos,
                                   const int* block_tables, int max_blocks, int H, int G, int ps,
                                   int window, float scale, int variant, hipStream_t stream) {
  return kappai_attn_prefill_scored(q, q_stride, k_pool, vt_pool, out, out_stride, q_tiles,
                                    n_tiles, row_pos, block_tables, max_blocks, H, G, ps, window,
                                    scale, variant, nullptr, stream);
}

static int launch_decode(const void* q, int q_stride, const void* k_pool, const void* vt_pool,
                         void* out, int out_stride, float* part_o, float* part_ml,
                         const int* row_pos, const int* row_seg, const int* block_tables,
                         int max_blocks, int T, int H, int G, int ps, int window, float scale,
                         int keys_per_split, int n_splits, const QkFuse& qk, const int* row_ids,
                         hipStream_t stream, const kappai_score_mods* mods = nullptr) {
  if (T <= 0) return 0;
  const bool scored = kappai_mods_change_scores(mods);
  if (scored && (qk.on || mods->keep_first < 0 ||
                 (mods->dist_bias != nullptr && mods->dist_cols < 1)))
    return (int)hipErrorInvalidValue;
  const kappai_score_mods m =
      scored ? *mods : kappai_score_mods{0.f, nullptr, 0, mods != nullptr ? mods->sink : nullptr, 0};
  if (ps % 16 || G < 1 || H % G || H / G > 16 || G > 65535 || n_splits < 1 || n_splits > 65535 ||
      keys_per_split < D_KPW || keys_per_split % D_KPW || (q_stride % 8))
    return (int)hipErrorInvalidValue;
  // The rows' own lengths decide the keys per split when the grid has more blocks than the waves
  // aimed at (else they could not ask for longer splits than the grid's own), and not in the form
  // with the prologue, which has no registers to spare: up to 16 rows of lengths that differ do better
  // without the rule but with the prologue (16 rows of 100 to 7,100 keys, 32 heads of 64 on 8 and 16 on 8: 35.8 and
  // 34.4 us with a kernel for norm, rotation and store and the rule, 32.5 and 33.0 so; one of 8,000 keys among 15 of
  // 200: 20.4 and 19.9, 17.5 and 17.4).
  const bool plan = !qk.on && (long long)T * G * n_splits > D_TARGET_WAVES;
#define KAPPAI_DECODE(FUSED, PLAN, MODS)                                                         \
  hipLaunchKernelGGL((attn_decode_kernel<FUSED, PLAN, MODS>), dim3(T, G, n_splits), dim3(WAVE),  \
                     0, stream, row_pos, row_seg, block_tables, row_ids, max_blocks, H, G, ps,   \
                     q_stride, window, (const bf16_t*)q, (const bf16_t*)k_pool,                  \
                     (const bf16_t*)vt_pool, part_o, part_ml, scale, keys_per_split, n_splits,   \
                     qk, m)
  if (qk.on) KAPPAI_DECODE(true, false, false);
  else if (scored && plan) KAPPAI_DECODE(false, true, true);
  else if (scored) KAPPAI_DECODE(false, false, true);
  else if (plan) KAPPAI_DECODE(false, true, false);
  else KAPPAI_DECODE(false, false, false);
#undef KAPPAI_DECODE
  hipLaunchKernelGGL(attn_merge_kernel, dim3(T, H), dim3(MERGE_WAVES * WAVE), 0, stream,
                     (const float*)part_o, (const float*)part_ml, row_pos, row_ids, H, n_splits, window,
                     m.keep_first, keys_per_split, plan ? (scored ? D_KPW : D_SPLIT_SHARE) : 0, G,
                     (bf16_t*)out, out_stride, m.sink);
  KAPPAI_RETURN_LAUNCH_STATUS();
}

extern "C" int kappai_attn_decode(const void* q, int q_stride, const void* k_pool,
                                  const void* vt_pool, void* out, int out_stride, float* part_o,
                                  float* part_ml, const int* row_pos, const int* row_seg,
                                  const int* block_tables, int max_blocks, int T, int H, int G,
                                  int ps, int window, float scale, int keys_per_split,
                                  int n_splits, hipStream_t stream) {
  return launch_decode(q, q_stride, k_pool, vt_pool, out, out_stride, part_o, part_ml, row_pos,
                       row_seg, block_tables, max_blocks, T, H, G, ps, window, scale,
                       keys_per_split, n_splits, QkFuse{}, nullptr, stream);
}

// kappai_attn_decode (row_ids null) or kappai_attn_decode_rows with `mods` (score_mods.h).
extern "C" int kappai_attn_decode_scored(const void* q, int q_stride, const void* k_pool,
                                         const void* vt_pool, void* out, int out_stride,
                                         float* part_o, float* part_ml, const int* row_ids,
                                         const int* row_pos, const int* row_seg,
                                         const int* block_tables, int max_blocks, int T, int H,
                                         int G, int ps, int window, float scale,
                                         int keys_per_split, int n_splits,
                                         const kappai_score_mods* mods, hipStream_t stream) {
  return launch_decode(q, q_stride, k_pool, vt_pool, out, out_stride, part_o, part_ml, row_pos,
                       row_seg, block_tables, max_blocks, T, H, G, ps, window, scale,
                       keys_per_split, n_splits, QkFuse{}, row_ids, stream, mods);
}

// kappai_attn_decode for some rows of a step: row_ids [T] names them (rows of q, row_pos, row_seg
// and out), part_o / part_ml hold T rows.  For the single decoded tokens of a step that also
// holds prompt portions: a row that stands alone over a long context is one tile for the tiled
// kernel, whose block then walks all its keys by itself.
extern "C" int kappai_attn_decode_rows(const void* q, int q_stride, const void* k_pool,
                                       const void* vt_pool, void* out, int out_stride,
                                       float* part_o, float* part_ml, const int* row_ids,
                                       const int* row_pos, const int* row_seg,
                                       const int* block_tables, int max_blocks, int T, int H,
                                       int G, int ps, int window, float scale, int keys_per_split,
                                       int n_splits, hipStream_t stream) {
  if (row_ids == nullptr) return (int)hipErrorInvalidValue;
  return launch_decode(q, q_stride, k_pool, vt_pool, out, out_stride, part_o, part_ml, row_pos,
                       row_seg, block_tables, max_blocks, T, H, G, ps, window, scale,
                       keys_per_split, n_splits, QkFuse{}, row_ids, stream);
}

// kappai_attn_decode with the norm, the rotation and the store of the rows' own keys and values in
// the kernel's prologue (see qk_args_ok for the added arguments).  Every split of
// a row must find the row's position inside the keys the splits cover: the caller's n_splits *
// keys_per_split reach beyond the longest context, as for kappai_attn_decode.
extern "C" int kappai_attn_decode_qk(const void* qkv, int row_stride, void* k_pool, void* vt_pool,
                                     void* out, int out_stride, float* part_o, float* part_ml,
                                     const int* row_pos, const int* row_seg,
                                     const int* block_tables, int max_blocks, int T, int H, int G,
                                     int ps, int window, float scale, int keys_per_split,
                                     int n_splits, const float* q_norm_w, const float* k_norm_w,
                                     float eps, const float* cos_tab, const float* sin_tab,
                                     int store_kv, hipStream_t stream) {
  if (!qk_args_ok(qkv, row_stride, q_norm_w, k_norm_w, cos_tab, sin_tab, k_pool, vt_pool))
    return (int)hipErrorInvalidValue;
  const QkFuse qk{1, store_kv ? 1 : 0, q_norm_w, k_norm_w, eps, cos_tab, sin_tab, (bf16_t*)k_pool,
                  (bf16_t*)vt_pool};
#if HEAD_DIM == 64
  const int n_waves = G > 0 && H % G == 0 ? kappai_attn_decode_block_waves(H / G) : 0;
  if (T > 0 && n_waves > 0 && keys_per_split > 0 && n_splits > 0 &&
      (long long)keys_per_split * n_splits <= D_QK_BLOCK_MAX_KEYS) {
    if (ps % 16 || G > 65535) return (int)hipErrorInvalidValue;
    const size_t lds = (size_t)n_waves * (H / G * HEAD_DIM + 32) * sizeof(float);
    hipLaunchKernelGGL(attn_decode_block_qk_kernel, dim3(T, G), dim3(n_waves * WAVE), lds, stream,
                       row_pos, row_seg, block_tables, max_blocks, H, G, ps, row_stride, window,
                       (const bf16_t*)qkv, (const bf16_t*)k_pool, (const bf16_t*)vt_pool, (bf16_t*)out,
                       out_stride, scale, qk);
    KAPPAI_RETURN_LAUNCH_STATUS();
  }
#endif
  return launch_decode(qkv, row_stride, k_pool, vt_pool, out, out_stride, part_o, part_ml, row_pos,
                       row_seg, block_tables, max_blocks, T, H, G, ps, window, scale,
                       keys_per_split, n_splits, qk, nullptr, stream);
}

// ---------------------------------------------------------------------------------------
// the decode attention for callers that cannot allocate: partial results in a device array
// of the library's own
// ---------------------------------------------------------------------------------------
static __device__ __align__(256) float scratch[KAPPAI_ATTN_STATIC_SCRATCH_FLOATS];

#define KAPPAI_MAX_DEVICES 64
// the address of each device's copy of `scratch`; in host code the array's name is only a
// stand-in for the symbol, never an address that a kernel could use
static float* g_scratch_ptr[KAPPAI_MAX_DEVICES];
static thread_local char g_static_error[256];

extern "C" int kappai_attn_decode_static_capacity(void) { return KAPPAI_ATTN_STATIC_SCRATCH_FLOATS; }

extern "C" const char* kappai_attn_decode_static_error(void) { return g_static_error; }

static int static_scratch_of_current_device(float** ptr) {
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return (int)err;
  if (dev < 0 || dev >= KAPPAI_MAX_DEVICES) {
    snprintf(g_static_error, sizeof g_static_error,
             "kappai_attn_decode_static: device %d is beyond the %d this library keeps track of",
             dev, KAPPAI_MAX_DEVICES);
    return (int)hipErrorInvalidDevice;
  }
  float* p = __atomic_load_n(&g_scratch_ptr[dev], __ATOMIC_ACQUIRE);
  if (p == nullptr) {
    void* sym = nullptr;
    err = hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch));
    if (err != hipSuccess || sym == nullptr) {
      snprintf(g_static_error, sizeof g_static_error,
               "kappai_attn_decode_static: hipGetSymbolAddress failed on device %d: %s", dev,
               hipGetErrorString(err));
      return (int)(err != hipSuccess ? err : hipErrorInvalidSymbol);
    }
    p = static_cast<float*>(sym);
    __atomic_store_n(&g_scratch_ptr[dev], p, __ATOMIC_RELEASE);   // the same value from any thread
  }
  *ptr = p;
  return 0;
}

extern "C" int kappai_attn_decode_static_init(void) {
  float* p = nullptr;
  return static_scratch_of_current_device(&p);
}

extern "C" int kappai_attn_decode_static(const void* q, int q_stride, const void* k_pool,
                                         const void* vt_pool, void* out, int out_stride,
                                         const int* row_pos, const int* row_seg,
                                         const int* block_tables, int max_blocks, int T, int H,
                                         int G, int ps, int window, float scale,
                                         int keys_per_split, int n_splits, hipStream_t stream) {
  g_static_error[0] = 0;
  if (T <= 0) return 0;
  if (H < 1 || n_splits < 1) {
    snprintf(g_static_error, sizeof g_static_error,
             "kappai_attn_decode_static: H = %d heads and n_splits = %d must be positive", H,
             n_splits);
    return (int)hipErrorInvalidValue;
  }
  const long long entries = (long long)T * H * n_splits;
  const long long need = entries * (HEAD_DIM + 2);
  if (need > KAPPAI_ATTN_STATIC_SCRATCH_FLOATS) {
    snprintf(g_static_error, sizeof g_static_error,
             "kappai_attn_decode_static: %d rows x %d heads x %d splits need %lld floats of partial "
             "results (head size %d); the library's array holds %d: use fewer splits or rows, or "
             "kappai_attn_decode with a workspace of the caller's",
             T, H, n_splits, need, HEAD_DIM, KAPPAI_ATTN_STATIC_SCRATCH_FLOATS);
    return (int)hipErrorInvalidValue;
  }
  float* base = nullptr;
  const int rc = static_scratch_of_current_device(&base);
  if (rc != 0) return rc;
  // part_o first (a multiple of 16 floats, so part_ml stays 16-byte aligned as well)
  float* part_o = base;
  float* part_ml = base + entries * HEAD_DIM;
  const int status = kappai_attn_decode(q, q_stride, k_pool, vt_pool, out, out_stride, part_o,
                                        part_ml, row_pos, row_seg, block_tables, max_blocks, T, H,
                                        G, ps, window, scale, keys_per_split, n_splits, stream);
  if (status == (int)hipErrorInvalidValue)
    snprintf(g_static_error, sizeof g_static_error,
             "kappai_attn_decode_static: an argument that kappai_attn_decode refuses (page size "
             "%d, %d heads over %d kv heads, %d keys a split, q stride %d)",
             ps, H, G, keys_per_split, q_stride);
  return status;
}
