// Attention over the paged cache.
//
//   qk_norm_rope_store  per-head RMSNorm of q and k (src/backend/cpu/scalar/quants.c:1521-1531),
//                       rotation at the row's absolute position
//                       (src/backend/cpu/quants.h:395-438: rotate-half or interleaved pairs),
//                       q rewritten in place, k and v stored into their pages
//                       (src/backend/cpu/common.c:1603-1622).  The projection may also arrive
//                       as float partial sums of a product split over its input dimension.
//   paged_attention_rows  one wave per (row, head): causal softmax(q.k/sqrt(d)) v over the keys
//                       lo..pos of the row's request, read through its block table
//                       (src/backend/cpu/scalar/core.c:383-433, 623-666), online softmax in float.
//   paged_attention_f32  the same for float32 heads of whole 16s, sixteen (row, head) places a
//                       block on the matrix cores.
//
// The key pool is [page][kv_head][page_size][head_dim]; the value pool is stored transposed,
// [page][kv_head][head_dim][page_size], which is what the matrix-core kernels want.  Token p of
// a request lives in page block_table[p / page_size] at offset p % page_size.
#include "common.h"
#include "score_mods.h"

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

#define MAX_HEAD_DIM 512

// rot_mode: 0 none, 1 rotate-half pairs (j, j+rot/2), 2 interleaved pairs (2j, 2j+1)
// A block of QKS_WAVES waves takes QKS_SLOTS heads (q, k or v) of one row, a wave a head at a
// time, each wave with its own piece of LDS.
#define QKS_WAVES 4
#define QKS_SLOTS 16
template <typename T>
__global__ __launch_bounds__(QKS_WAVES * WAVE) void qk_norm_rope_store_kernel(
    T* __restrict__ qkv, int row_stride, const float* __restrict__ q_norm_w,
    const float* __restrict__ k_norm_w, float eps, const float* __restrict__ cos_tab,
    const float* __restrict__ sin_tab, int rot_dim, int rot_mode, T* __restrict__ k_pool,
    T* __restrict__ v_pool, const int* __restrict__ row_pos, const int* __restrict__ row_seg,
    const int* __restrict__ block_tables, int max_blocks, int H, int G, int d, int ps,
    int n_slots, const float* __restrict__ parts, int n_parts, T* __restrict__ q_out,
    int q_stride) {
  __shared__ float bufs[QKS_WAVES][MAX_HEAD_DIM];
  const int t = blockIdx.x, lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  float* buf = bufs[wave];
  const int pos = row_pos[t];
  if (rot_mode == 0) rot_dim = 0;
  const int half = rot_dim / 2;
  const float* ct = cos_tab + (size_t)pos * half;
  const float* st = sin_tab + (size_t)pos * half;
  const int* bt = block_tables + (size_t)row_seg[t] * max_blocks;
  const int slot_end = min(n_slots, (int)(blockIdx.y + 1) * QKS_SLOTS);
  for (int slot = blockIdx.y * QKS_SLOTS + wave; slot < slot_end; slot += QKS_WAVES) {
    const size_t at = (size_t)t * row_stride + (size_t)slot * d;
    // with `parts` the row arrives as float sums over n_parts ranges of the projection's input
    // dimension, [n_parts][rows][row_stride]; added in order and rounded to T they are what the
    // unsplit projection would have stored, and q goes to a buffer of its own
    const size_t plane = (size_t)gridDim.x * row_stride;
    auto value = [&](int e) -> float {
      if (!parts) return to_f32(qkv[at + e]);
      float sum = parts[at + e];
      for (int k = 1; k < n_parts; ++k) sum += parts[k * plane + at + e];
      T rounded;
      from_f32(&rounded, sum);
      return to_f32(rounded);
    };
    T* dst = parts ? q_out + (size_t)t * q_stride + (size_t)slot * d : qkv + at;
    if (slot >= H) {
      const int g = (slot - H) % G;
      const size_t pg = (size_t)bt[pos / ps] * G + g;
      if (slot >= H + G) {  // v: copied into its page, transposed
        T* vdst = v_pool + pg * d * ps + pos % ps;
        for (int e = lane; e < d; e += WAVE) from_f32(vdst + (size_t)e * ps, value(e));
        continue;
      }
      dst = k_pool + (pg * ps + pos % ps) * d;
    }
    const float* nw = slot < H ? q_norm_w : k_norm_w;
    float ss = 0.f;
    for (int e = lane; e < d; e += WAVE) {
      const float v = value(e);
      buf[e] = v;
      ss += v * v;
    }
    if (nw) {
      ss = wave_sum(ss);
      const float sc = 1.0f / sqrtf(ss / (float)d + eps);
      for (int e = lane; e < d; e += WAVE) buf[e] = buf[e] * sc * nw[e];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int j = lane; j < half; j += WAVE) {
      const int i0 = rot_mode == 1 ? j : 2 * j;
      const int i1 = rot_mode == 1 ? j + half : 2 * j + 1;
      const float c = ct[j], s = st[j];
      const float v0 = buf[i0], v1 = buf[i1];
      from_f32(dst + i0, v0 * c - v1 * s);
      from_f32(dst + i1, v0 * s + v1 * c);
    }
    for (int e = rot_dim + lane; e < d; e += WAVE) from_f32(dst + e, buf[e]);
    // the next head overwrites the wave's piece of LDS
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// bfloat16, the whole head rotated in halves (or not at all), d / 8 a power of two up to 64:
// a lane takes 8 consecutive elements of a head, so that a wave works on 512 / d heads at once
// without LDS; the sum of squares and the rotation's partner (the lane d / 16 away) come by
// shuffles.  The blocks from qk_blocks on store the values: a wave takes 8 rows of 64 value columns and turns
// them over in LDS, so that where the rows are 8 neighbouring positions of a page a lane stores the 16 bytes
// of one column (else 8 values of two bytes as they come).
// Bound by a chain of reads in small steps, by its stores in large ones: everything that hangs on nothing is
// asked for first, then what the position and the segment name, before any arithmetic.  One after
// another, 32 heads of 64 on 8: 2,048 rows 11.6 -> 7.5 us, eight portions of 100 rows 6.6 -> 4.4, single rows 2.9
// as before (64 of them from three sums 3.5 -> 3.4); 16 on 8, 512 rows 4.7 -> 3.1.
typedef __attribute__((ext_vector_type(4))) uint32_t qks_u32x4_t;
template <int LPH, bool PARTS>
__global__ __launch_bounds__(256) void qk_norm_rope_store_vec_kernel(
    const int* __restrict__ row_pos, const int* __restrict__ row_seg, bf16_t* __restrict__ qkv,
    const float* __restrict__ parts, int row_stride, int T, int n_slots, int H, int qk_blocks, int n_parts,
    const float* __restrict__ q_norm_w, const float* __restrict__ k_norm_w, const float* __restrict__ cos_tab,
    const float* __restrict__ sin_tab, const int* __restrict__ block_tables, int max_blocks, int G, int ps,
    int rotate, float eps, int v_wide, bf16_t* __restrict__ k_pool, bf16_t* __restrict__ v_pool,
    bf16_t* __restrict__ q_out, int q_stride) {
  constexpr int d = LPH * 8, half = d / 2;
  // 8 values of the projection, rounded to bfloat16: what the unsplit product would have stored where they
  // come as float sums over n_parts ranges of its input dimension (added in order)
  auto eight = [&](size_t at) -> qks_u32x4_t {
    if (!PARTS) return *reinterpret_cast<const qks_u32x4_t*>(qkv + at);
    const size_t plane = (size_t)T * row_stride;
    float4 lo = *reinterpret_cast<const float4*>(parts + at);
    float4 hi = *reinterpret_cast<const float4*>(parts + at + 4);
#pragma unroll 4
    for (int k = 1; k < n_parts; ++k) {
      const float4 a = *reinterpret_cast<const float4*>(parts + k * plane + at);
      const float4 b = *reinterpret_cast<const float4*>(parts + k * plane + at + 4);
      lo.x += a.x; lo.y += a.y; lo.z += a.z; lo.w += a.w;
      hi.x += b.x; hi.y += b.y; hi.z += b.z; hi.w += b.w;
    }
    qks_u32x4_t raw;
    raw[0] = pack_bf16x2(lo.x, lo.y);
    raw[1] = pack_bf16x2(lo.z, lo.w);
    raw[2] = pack_bf16x2(hi.x, hi.y);
    raw[3] = pack_bf16x2(hi.z, hi.w);
    return raw;
  };
  if ((int)blockIdx.x >= qk_blocks) {
    __shared__ __attribute__((aligned(16))) bf16_t turn[256 / WAVE][8][64];
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int groups = (G * LPH + 7) / 8;                        // of 64 value columns
    const unsigned unit = (blockIdx.x - qk_blocks) * (256 / WAVE) + wave;
    const int t0 = (int)(unit / groups) * 8, col0 = (int)(unit % groups) * 8;
    if (t0 >= T) return;
    const int i = lane / 8, c = col0 + lane % 8;                 // this lane's row and eight columns
    const bool in = t0 + i < T && c < G * LPH;
    const int t = min(t0 + i, T - 1), g = min(c, G * LPH - 1) / LPH, e0 = 8 * (c % LPH);
    const int pos = row_pos[t], seg = row_seg[t];
    const qks_u32x4_t raw = eight((size_t)t * row_stride + (size_t)H * d + (size_t)G * d +
                                  8 * (size_t)min(c, G * LPH - 1));
    const int page = block_tables[(size_t)seg * max_blocks + pos / ps];
    // (lane 0 has row t0, and a page takes 8 positions from a multiple of 8 on)
    const int pos0 = __builtin_amdgcn_readfirstlane(pos), seg0 = __builtin_amdgcn_readfirstlane(seg);
    const bool fits = t0 + 8 <= T && pos0 % 8 == 0 && pos == pos0 + i && seg == seg0;
    if (v_wide && __builtin_amdgcn_ballot_w64(!fits) == 0) {
      *reinterpret_cast<qks_u32x4_t*>(&turn[wave][i][8 * (lane % 8)]) = raw;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      qks_u32x4_t col;                                           // column e0 + i of rows t0 .. t0 + 7
#pragma unroll
      for (int j = 0; j < 4; ++j)
        col[j] = (uint32_t)turn[wave][2 * j][8 * (lane % 8) + i] |
                 (uint32_t)turn[wave][2 * j + 1][8 * (lane % 8) + i] << 16;
      if (in)
        *reinterpret_cast<qks_u32x4_t*>(v_pool + (((size_t)page * G + g) * d + e0 + i) * ps + pos0 % ps) = col;
      return;
    }
    if (!in) return;
    bf16_t* vdst = v_pool + (((size_t)page * G + g) * d + e0) * ps + pos % ps;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      vdst[(size_t)(2 * j) * ps] = (bf16_t)(raw[j] & 0xffffu);
      vdst[(size_t)(2 * j + 1) * ps] = (bf16_t)(raw[j] >> 16);
    }
    return;
  }
  // n_slots: the query heads and, where keys are stored, the kv heads; T * n_slots * LPH < 2^31
  const unsigned total = (unsigned)T * n_slots * LPH, gid = blockIdx.x * 256u + threadIdx.x;
  const bool active = gid < total;
  const unsigned idx = active ? gid : total - 1;
  const int part = (int)(idx % LPH);
  const unsigned head = idx / LPH;
  const int t = (int)(head / (unsigned)n_slots), slot = (int)(head - (unsigned)t * n_slots);
  const bool stores_k = n_slots > H;
  const int pos = row_pos[t], seg = stores_k ? row_seg[t] : 0;
  const int e0 = 8 * part;
  const size_t at = (size_t)t * row_stride + (size_t)slot * d + e0;
  const qks_u32x4_t raw = eight(at);
  // (the rest of the arguments in one wait, while those loads are under way)
  asm volatile("" : "+s"(q_norm_w), "+s"(k_norm_w), "+s"(cos_tab), "+s"(sin_tab), "+s"(block_tables),
                    "+s"(max_blocks), "+s"(ps), "+s"(rotate), "+s"(k_pool), "+s"(q_out));
  const float* nw = slot < H ? q_norm_w : k_norm_w;
  float4 w0 = make_float4(1.f, 1.f, 1.f, 1.f), w1 = w0;
  if (nw) {
    w0 = *reinterpret_cast<const float4*>(nw + e0);
    w1 = *reinterpret_cast<const float4*>(nw + e0 + 4);
  }
  const int page = stores_k ? block_tables[(size_t)seg * max_blocks + pos / ps] : 0;
  const bool low = e0 < half;
  float4 c0, c1, s0, s1;
  if (rotate) {
    const size_t turn_at = (size_t)pos * half + (low ? e0 : e0 - half);
    c0 = *reinterpret_cast<const float4*>(cos_tab + turn_at);
    c1 = *reinterpret_cast<const float4*>(cos_tab + turn_at + 4);
    s0 = *reinterpret_cast<const float4*>(sin_tab + turn_at);
    s1 = *reinterpret_cast<const float4*>(sin_tab + turn_at + 4);
  }
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __uint_as_float(raw[i] << 16);
    v[2 * i + 1] = __uint_as_float(raw[i] & 0xffff0000u);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
#pragma unroll
  for (int m = LPH / 2; m >= 1; m /= 2) ss += __shfl_xor(ss, m, WAVE);
  if (nw) {
    const float sc = 1.0f / sqrtf(ss / (float)d + eps);
    const float wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = v[i] * sc * wv[i];
  }
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = v[i];
  if (LPH >= 2) {
    // partner element e +- d/2 lives in the lane LPH/2 away, same place
    float other[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) other[i] = __shfl_xor(v[i], LPH / 2 > 0 ? LPH / 2 : 1, WAVE);
    if (rotate) {
      const float cv[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
      const float sv[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
      for (int i = 0; i < 8; ++i)
        r[i] = low ? v[i] * cv[i] - other[i] * sv[i] : other[i] * sv[i] + v[i] * cv[i];
    }
  }
  if (!active) return;
  qks_u32x4_t o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = pack_bf16x2(r[2 * i], r[2 * i + 1]);
  bf16_t* dst = slot >= H ? k_pool + (((size_t)page * G + (slot - H)) * ps + pos % ps) * d + e0
                : PARTS   ? q_out + (size_t)t * q_stride + (size_t)slot * d + e0
                          : qkv + at;
  *reinterpret_cast<qks_u32x4_t*>(dst) = o;
}

extern "C" int kappai_qk_norm_rope_store(void* qkv, int row_stride, const float* q_norm_w,
                                         const float* k_norm_w, float eps, const float* cos_tab,
                                         const float* sin_tab, int rot_dim, int rot_mode,
                                         void* k_pool, void* v_pool, const int* row_pos,
                                         const int* row_seg, const int* block_tables,
                                         int max_blocks, int T, int H, int G, int d, int ps,
                                         int store_kv, int is_bf16, const float* parts,
                                         int n_parts, void* q_out, int q_stride,
                                         hipStream_t stream) {
  // parts != null: the projection as [n_parts][T][row_stride] float partial sums instead of
  // qkv; q is then written to q_out [T][q_stride] (bfloat16 only)
  if (T <= 0) return 0;
  if (d > MAX_HEAD_DIM || d < 1 || rot_dim > d || (rot_dim & 1)) return (int)hipErrorInvalidValue;
  if (parts && (!is_bf16 || n_parts < 1 || !q_out)) return (int)hipErrorInvalidValue;
  const int n_slots = store_kv ? H + 2 * G : H, qk_slots = store_kv ? H + G : H;
  const bool whole_rot = rot_mode == 0 || rot_dim == 0 || (rot_mode == 1 && rot_dim == d);
  const int lph = d / 8;
  if (is_bf16 && whole_rot && d % 8 == 0 && lph >= 2 && lph <= 64 && (lph & (lph - 1)) == 0 &&
      row_stride % 8 == 0 && ((uintptr_t)qkv % 16) == 0 && ((uintptr_t)k_pool % 16) == 0 &&
      ((uintptr_t)parts % 16) == 0 && ((uintptr_t)q_out % 16) == 0 && q_stride % 8 == 0 &&
      ((uintptr_t)cos_tab % 16) == 0 && ((uintptr_t)sin_tab % 16) == 0 &&
      (!q_norm_w || ((uintptr_t)q_norm_w % 16) == 0) &&
      (!k_norm_w || ((uintptr_t)k_norm_w % 16) == 0) && (long long)T * qk_slots * lph < (1LL << 31)) {
    const int rotate = rot_mode == 1 && rot_dim == d;
    const int qk_blocks = (int)(((long long)T * qk_slots * lph + 255) / 256);
    const long long v_units = store_kv ? ((long long)T + 7) / 8 * ((G * lph + 7) / 8) : 0;
    const dim3 gv((unsigned)(qk_blocks + (v_units + 3) / 4));
    const int v_wide = ps % 8 == 0 && ((uintptr_t)v_pool % 16) == 0;
#define QKS_LAUNCH_AS(N, P)                                                                      \
  hipLaunchKernelGGL((qk_norm_rope_store_vec_kernel<N, P>), gv, dim3(256), 0, stream, row_pos, row_seg, \
                     (bf16_t*)qkv, parts, row_stride, T, qk_slots, H, qk_blocks, n_parts, q_norm_w,     \
                     k_norm_w, cos_tab, sin_tab, block_tables, max_blocks, G, ps, rotate, eps, v_wide,  \
                     (bf16_t*)k_pool, (bf16_t*)v_pool, (bf16_t*)q_out, q_stride)
#define QKS_LAUNCH(N)                                                                            \
  if (parts) QKS_LAUNCH_AS(N, true);                                                             \
  else QKS_LAUNCH_AS(N, false)
    switch (lph) {
      case 2: QKS_LAUNCH(2); break;
      case 4: QKS_LAUNCH(4); break;
      case 8: QKS_LAUNCH(8); break;
      case 16: QKS_LAUNCH(16); break;
      case 32: QKS_LAUNCH(32); break;
      default: QKS_LAUNCH(64); break;
    }
#undef QKS_LAUNCH
#undef QKS_LAUNCH_AS
    KAPPAI_RETURN_LAUNCH_STATUS();
  }
  dim3 grid(T, (n_slots + QKS_SLOTS - 1) / QKS_SLOTS);
  if (is_bf16)
    hipLaunchKernelGGL(qk_norm_rope_store_kernel<bf16_t>, grid, dim3(QKS_WAVES * WAVE), 0, stream,
                       (bf16_t*)qkv, row_stride, q_norm_w, k_norm_w, eps, cos_tab, sin_tab,
                       rot_dim, rot_mode, (bf16_t*)k_pool, (bf16_t*)v_pool, row_pos, row_seg,
                       block_tables, max_blocks, H, G, d, ps, n_slots, parts, n_parts,
                       (bf16_t*)q_out, q_stride);
  else
    hipLaunchKernelGGL(qk_norm_rope_store_kernel<float>, grid, dim3(QKS_WAVES * WAVE), 0, stream, (float*)qkv,
                       row_stride, q_norm_w, k_norm_w, eps, cos_tab, sin_tab, rot_dim, rot_mode,
                       (float*)k_pool, (float*)v_pool, row_pos, row_seg, block_tables, max_blocks,
                       H, G, d, ps, n_slots, nullptr, 0, nullptr, 0);
  KAPPAI_RETURN_LAUNCH_STATUS();
}

// ---------------------------------------------------------------------------------------
__device__ __forceinline__ float dot_row(const float* __restrict__ qs, const float* __restrict__ k,
                                         int d) {
  float s = 0.f;
  for (int e = 0; e < d; e += 4) {
    const float4 kv = *reinterpret_cast<const float4*>(k + e);
    s = fmaf(qs[e], kv.x, s);
    s = fmaf(qs[e + 1], kv.y, s);
    s = fmaf(qs[e + 2], kv.z, s);
    s = fmaf(qs[e + 3], kv.w, s);
  }
  return s;
}

__device__ __forceinline__ float dot_row(const float* __restrict__ qs,
                                         const bf16_t* __restrict__ k, int d) {
  float s = 0.f;
  for (int e = 0; e < d; e += 8) {
    const uint4 kv = *reinterpret_cast<const uint4*>(k + e);
    const uint32_t w[4] = {kv.x, kv.y, kv.z, kv.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s = fmaf(qs[e + 2 * i], __uint_as_float(w[i] << 16), s);
      s = fmaf(qs[e + 2 * i + 1], __uint_as_float(w[i] & 0xffff0000u), s);
    }
  }
  return s;
}

#define ATT_NPL (MAX_HEAD_DIM / WAVE)

template <typename T, bool MODS>
__global__ __launch_bounds__(64) void paged_attention_rows_kernel(
    const T* __restrict__ q, int q_stride, const T* __restrict__ k_pool,
    const T* __restrict__ v_pool, T* __restrict__ out, int out_stride,
    const int* __restrict__ row_pos, const int* __restrict__ row_seg,
    const int* __restrict__ block_tables, int max_blocks, int H, int G, int d, int ps, int window,
    float scale, kappai_score_mods mods) {
  __shared__ float qs[MAX_HEAD_DIM];
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int g = h / (H / G);
  const int pos = row_pos[t];
  const int* bt = block_tables + (size_t)row_seg[t] * max_blocks;
  const int lo = kappai_first_key(pos, window);
  const T* qr = q + (size_t)t * q_stride + (size_t)h * d;
  for (int e = lane; e < d; e += WAVE) qs[e] = to_f32(qr[e]);
  __syncthreads();

  float m = -INFINITY, l = 0.f;
  float acc[ATT_NPL];
#pragma unroll
  for (int i = 0; i < ATT_NPL; ++i) acc[i] = 0.f;

  // the kept first positions that lie before the window, then the window: one row of places
  const int kept = MODS ? min(mods.keep_first, lo) : 0;
  const int n_keys = kept + pos - lo + 1;
  for (int base = 0; base < n_keys; base += WAVE) {
    const int place = base + lane;
    const int tk = place < kept ? place : lo + place - kept;
    const bool valid = place < n_keys;
    float s = -INFINITY;
    unsigned long long voff = 0;
    if (valid) {
      const size_t pg = (size_t)bt[tk / ps] * G + g;
      s = dot_row(qs, k_pool + (pg * ps + tk % ps) * d, d) * scale;
      if (MODS) s = kappai_modified_score(mods, s, h, pos - tk);
      voff = (unsigned long long)(pg * d * ps + tk % ps);
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float p = valid ? expf(s - m_new) : 0.f;
    const float corr = expf(m - m_new);
    l = l * corr + wave_sum(p);
#pragma unroll
    for (int i = 0; i < ATT_NPL; ++i) acc[i] *= corr;
    const int nk = min(WAVE, n_keys - base);
    for (int kk = 0; kk < nk; ++kk) {
      const float pk = __shfl(p, kk, WAVE);
      const unsigned lo32 = __shfl((unsigned)(voff & 0xffffffffull), kk, WAVE);
      const unsigned hi32 = __shfl((unsigned)(voff >> 32), kk, WAVE);
      const T* vr = v_pool + (((unsigned long long)hi32 << 32) | lo32);
#pragma unroll
      for (int i = 0; i < ATT_NPL; ++i) {
        const int e = lane + i * WAVE;
        if (e < d) acc[i] = fmaf(pk, to_f32(vr[(size_t)e * ps]), acc[i]);
      }
    }
    m = m_new;
  }
  if (MODS && mods.sink != nullptr) l += expf(mods.sink[h] - m);
  const float inv = 1.0f / l;
  T* o = out + (size_t)t * out_stride + (size_t)h * d;
#pragma unroll
  for (int i = 0; i < ATT_NPL; ++i) {
    const int e = lane + i * WAVE;
    if (e < d) from_f32(o + e, acc[i] * inv);
  }
}

// ---------------------------------------------------------------------------------------
// float32 attention on the matrix cores (v_mfma_f32_16x16x4_f32: float products and sums).
//
// A block takes one kv head and sixteen places (row, head of the kv head's): as many rows of one
// segment, at positions that follow one another, as fit beside each other, so a prompt's rows share every key and value they read, and a
// decoded row has its heads in one block.  Its waves take steps of 16 keys in turns (step s
// belongs to wave s % NW wherever a row's keys begin and end) and meet in LDS at the end, so a row's
// result does not depend on the rows it is computed with.  Scores are made keys x places, which
// is the layout in which the weights enter the product with the transposed values: nothing moves
// between lanes but the maximum and the sum of a place.  Bound by the latency of a step's loads and the chain of
// products and exponentials behind them, so the next step's loads are under way while one is worked on and the
// pages they hang on a step before that; the rows' tables are read once, side by side.  One after another, 16
// heads of 64 on 8 kv heads, with pages looked up on the way to the loads / ahead of them: a prompt step of 150, 275
// and 400 tokens 41.2 / 39.6 us, of 1,000 443 / 415, three decoded rows at 150 to 400 keys 11.8 / 10.9, four at
// 4,000 78 / 67; the same bits.  (A wave a (row, head) took 126 us on average over the first and the third.)
template <int NT>
__global__ __launch_bounds__((NT <= 4 ? 8 : 4) * WAVE) void paged_attention_f32_kernel(
    const int* __restrict__ row_pos, const int* __restrict__ row_seg, int T, int H, int G, int ps,
    const int* __restrict__ block_tables, int max_blocks, int q_stride, const float* __restrict__ q,
    const float* __restrict__ k_pool, const float* __restrict__ v_pool, float* __restrict__ out,
    int out_stride, int window, float scale) {
  constexpr int D = 16 * NT, NW = NT <= 4 ? 8 : 4;
  __shared__ float part[NW][16][D + 1];
  __shared__ float part_m[NW][16], part_l[NW][16];
  const int per = H / G, heads = min(per, 16), R = 16 / heads, pieces = (per + heads - 1) / heads;
  const int g = blockIdx.y / pieces, h0 = g * per + blockIdx.y % pieces * heads;
  // Rows beside each other are one block's only while their positions follow one another: of the keys
  // from the first row's first to the last row's own each is then seen by some row, and no page is
  // read that no row needs.  The lanes look at the rows side by side (1,000 rows of one prompt 443 us,
  // 466 with one row after the other).
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int t0 = blockIdx.x, seen_row = min(max(t0 - 1 + lane, 0), T - 1);     // (lane 0: the row before)
  const int pos_of = row_pos[seen_row], seg_of = row_seg[seen_row];
  const int seg = __builtin_amdgcn_readlane(seg_of, 1), pos0 = __builtin_amdgcn_readlane(pos_of, 1);
  if (t0 % R != 0 && __builtin_amdgcn_readlane(seg_of, 0) == seg &&
      __builtin_amdgcn_readlane(pos_of, 0) == pos0 - 1)
    return;                                                 // the block of an earlier row has it
  const bool beside = lane >= 1 && lane - 1 < R - t0 % R && t0 - 1 + lane < T && seg_of == seg &&
                      pos_of == pos0 + lane - 1;
  const int t1 = t0 + __builtin_ctzll(~(__builtin_amdgcn_ballot_w64(beside) >> 1));
  const int r = lane % 16, quad = lane / 16;
  int row = t0 + r / heads, head = h0 + r % heads;
  if (row >= t1 || head >= (g + 1) * per) row = t0, head = h0;    // a place without work of its own
  const int pos = pos0 + (row - t0), lo = kappai_first_key(pos, window);
  const int pos_max = __builtin_amdgcn_readfirstlane(wave_max(pos));
  const int lo_min = __builtin_amdgcn_readfirstlane(-wave_max(-lo));
  const int* bt = block_tables + (size_t)seg * max_blocks;

  f32x4_t qv[NT], acc[NT], kv[NT], vv[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    qv[j] = *reinterpret_cast<const f32x4_t*>(q + (size_t)row * q_stride + (size_t)head * D +
                                              16 * j + 4 * quad);
    acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  // keys outside lo_min .. pos_max are read from the nearest one inside (their pages may be gone); a step's
  // pages are looked up a step ahead of its loads, which hang on them
  const auto key_of = [&](int st) { return min(max(16 * st + r, lo_min), pos_max); };
  const auto four_of = [&](int st) { return min(max(16 * st + 4 * quad, lo_min / 4 * 4), pos_max / 4 * 4); };
  struct Pages { int k, v; };
  const auto look_up = [&](int st) { return Pages{bt[key_of(st) / ps], bt[four_of(st) / ps]}; };
  const auto fetch = [&](int st, const Pages& at, f32x4_t (&kf)[NT], f32x4_t (&vf)[NT]) {
    const float* kp = k_pool + (((size_t)at.k * G + g) * ps + key_of(st) % ps) * D + 4 * quad;
    const float* vp = v_pool + (((size_t)at.v * G + g) * D + r) * ps + four_of(st) % ps;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      kf[j] = *reinterpret_cast<const f32x4_t*>(kp + 16 * j);
      vf[j] = *reinterpret_cast<const f32x4_t*>(vp + (size_t)16 * j * ps);
    }
  };
  float m = -INFINITY, l = 0.f;
  const int first = lo_min / 16, last = pos_max < 0 ? -1 : pos_max / 16;
  int st = first + ((wave - first) % NW + NW) % NW;
  Pages now{0, 0}, next{0, 0};
  if (st <= last) {
    now = look_up(st);
    next = look_up(st + NW);
    fetch(st, now, kv, vv);
  }
  const auto work = [&](const f32x4_t (&kv)[NT], f32x4_t (&vv)[NT]) {
    // (four chains: a product waits 50 clocks for the one before it in its own)
    f32x4_t part_s[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) part_s[e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        part_s[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[j][e], qv[j][e], part_s[e], 0, 0, 0);
    f32x4_t s = (part_s[0] + part_s[1]) + (part_s[2] + part_s[3]);
    const int key0 = 16 * st + 4 * quad;       // this lane's scores: keys key0 .. key0 + 3, place r
    bool seen[4], odd = false;
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      seen[i] = key0 + i <= pos && key0 + i >= lo;
      s[i] = seen[i] ? s[i] * scale : -INFINITY;
      top = fmaxf(top, s[i]);
      const bool inside = key0 + i <= pos_max && key0 + i >= lo_min;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (!inside) vv[j][i] = 0.f;           // (nobody's: what lies there is anything)
        odd |= !(fabsf(vv[j][i]) < INFINITY);
      }
    }
    top = fmaxf(top, lane_xor16(top));
    top = fmaxf(top, lane_xor32(top));
    const float m_new = fmaxf(m, top);
    const float ref = m_new == -INFINITY ? 0.f : m_new;
    const float corr = expf(m - ref);
    f32x4_t p;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = seen[i] ? expf(s[i] - ref) : 0.f;
      sum += p[i];
    }
    sum += lane_xor16(sum);
    sum += lane_xor32(sum);
    l = l * corr + sum;
    m = m_new;
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] *= corr;
    if (!__any(odd)) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[j][e], p[e], acc[j], 0, 0, 0);
    } else {
      // a value that is no finite number must not meet the weight 0 of a place that does not see
      // its key: place by place, with the keys that the place sees
      for (int c = 0; c < 16; ++c) {
        const int pos_c = __shfl(pos, c, WAVE), lo_c = __shfl(lo, c, WAVE);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool sees = key0 + e <= pos_c && key0 + e >= lo_c;
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            const f32x4_t got = __builtin_amdgcn_mfma_f32_16x16x4f32(
                sees ? vv[j][e] : 0.f, p[e], acc[j], 0, 0, 0);
            if (r == c) acc[j] = got;
          }
        }
      }
    }
  };
  // two sets of registers in turn (copied from one to the other, a step's loads would be waited for at the end
  // of the step before).  Fetched behind the last step too, where every key is the last row's own: behind a
  // condition the products of this step would wait for the next one's loads.
  const auto step = [&](const f32x4_t (&kv)[NT], f32x4_t (&vv)[NT], f32x4_t (&kn)[NT], f32x4_t (&vn)[NT]) {
    now = next;
    next = look_up(st + 2 * NW);
    fetch(st + NW, now, kn, vn);
    __builtin_amdgcn_sched_barrier(0);
    work(kv, vv);
    st += NW;
  };
  f32x4_t kn[NT], vn[NT];
  while (st <= last) {
    step(kv, vv, kn, vn);
    if (st > last) break;
    step(kn, vn, kv, vv);
  }
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) part[wave][r][16 * j + 4 * quad + i] = acc[j][i];
  if (quad == 0) {
    part_m[wave][r] = m;
    part_l[wave][r] = l;
  }
  __syncthreads();
  for (int at = threadIdx.x; at < 16 * D; at += NW * WAVE) {
    const int place = at / D, e = at % D;
    const int to = t0 + place / heads, hd = h0 + place % heads;
    if (place >= R * heads || to >= t1 || hd >= (g + 1) * per) continue;
    float top = part_m[0][place];
#pragma unroll
    for (int w = 1; w < NW; ++w) top = fmaxf(top, part_m[w][place]);
    float sum = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      // (a wave without a key for this place holds nothing)
      const float f = part_m[w][place] == -INFINITY && part_l[w][place] == 0.f
                          ? 0.f : expf(part_m[w][place] - top);
      sum += part_l[w][place] * f;
      o += part[w][place][e] * f;
    }
    out[(size_t)to * out_stride + (size_t)hd * D + e] = o * (1.0f / sum);
  }
}

template <typename T, bool MODS>
static void rows_launch(const void* q, int q_stride, const void* k_pool, const void* v_pool,
                        void* out, int out_stride, const int* row_pos, const int* row_seg,
                        const int* block_tables, int max_blocks, int T_, int H, int G, int d,
                        int ps, int window, float scale, kappai_score_mods mods,
                        hipStream_t stream) {
  hipLaunchKernelGGL((paged_attention_rows_kernel<T, MODS>), dim3(T_, H), dim3(WAVE), 0, stream,
                     (const T*)q, q_stride, (const T*)k_pool, (const T*)v_pool, (T*)out,
                     out_stride, row_pos, row_seg, block_tables, max_blocks, H, G, d, ps, window,
                     scale, mods);
}

// `mods` (may be null): see score_mods.h
extern "C" int kappai_paged_attention_rows_scored(
    const void* q, int q_stride, const void* k_pool, const void* v_pool, void* out,
    int out_stride, const int* row_pos, const int* row_seg, const int* block_tables,
    int max_blocks, int T, int H, int G, int d, int ps, int window, float scale, int is_bf16,
    const kappai_score_mods* mods, hipStream_t stream) {
  if (T <= 0) return 0;
  if (d > MAX_HEAD_DIM || d % 8 || G < 1 || H % G || H > 65535) return (int)hipErrorInvalidValue;
  const bool on = kappai_mods_on(mods);
  if (on && ((mods->dist_bias && mods->dist_cols < 1) || mods->keep_first < 0))
    return (int)hipErrorInvalidValue;
  const kappai_score_mods m = on ? *mods : kappai_score_mods{0.f, nullptr, 0, nullptr, 0};
  // Plain float32 scores over heads of whole 16s: the matrix cores.  What they do not take (worked-on
  // scores, other head sizes, rows or pages that are not aligned to 16 bytes) and bfloat16 shapes
  // that no tiled kernel takes go row by row.
  if (!is_bf16 && !on && d % 16 == 0 && d <= 128 && ps % 4 == 0 && q_stride % 4 == 0 &&
      (uintptr_t)q % 16 == 0 && (uintptr_t)k_pool % 16 == 0 && (uintptr_t)v_pool % 16 == 0) {
    const int per = H / G, heads = per < 16 ? per : 16;
    const dim3 grid(T, G * ((per + heads - 1) / heads));
#define F32_ATT(NT)                                                                             \
  case NT:                                                                                      \
    hipLaunchKernelGGL(paged_attention_f32_kernel<NT>, grid, dim3((NT <= 4 ? 8 : 4) * WAVE), 0,  \
                       stream, row_pos, row_seg, T, H, G, ps, block_tables, max_blocks, q_stride, \
                       (const float*)q, (const float*)k_pool, (const float*)v_pool, (float*)out, \
                       out_stride, window, scale);                   \
    break;
    switch (d / 16) {
      F32_ATT(1) F32_ATT(2) F32_ATT(3) F32_ATT(4) F32_ATT(5) F32_ATT(6) F32_ATT(7) F32_ATT(8)
    }
#undef F32_ATT
    KAPPAI_RETURN_LAUNCH_STATUS();
  }
#define ROWS_ARGS q, q_stride, k_pool, v_pool, out, out_stride, row_pos, row_seg, block_tables, \
                  max_blocks, T, H, G, d, ps, window, scale, m, stream
  if (is_bf16) {
    if (on) rows_launch<bf16_t, true>(ROWS_ARGS); else rows_launch<bf16_t, false>(ROWS_ARGS);
  } else {
    if (on) rows_launch<float, true>(ROWS_ARGS); else rows_launch<float, false>(ROWS_ARGS);
  }
#undef ROWS_ARGS
  KAPPAI_RETURN_LAUNCH_STATUS();
}

extern "C" int kappai_paged_attention_rows(const void* q, int q_stride, const void* k_pool,
                                           const void* v_pool, void* out, int out_stride,
                                           const int* row_pos, const int* row_seg,
                                           const int* block_tables, int max_blocks, int T, int H,
                                           int G, int d, int ps, int window, float scale,
                                           int is_bf16, hipStream_t stream) {
  return kappai_paged_attention_rows_scored(q, q_stride, k_pool, v_pool, out, out_stride, row_pos,
                                            row_seg, block_tables, max_blocks, T, H, G, d, ps,
                                            window, scale, is_bf16, nullptr, stream);
}
