// Read-side kernels on the reference's flat tensor layouts: query rotation /
// sketch, the asymmetric score estimator, and key / value de-quantisation.

#include <algorithm>
#include "tq_common.h"
#include "tq_cache_append.h"
#include "tq_prep.h"
#include "tq_options.h"
#include "tq_decode_mfma.h"

namespace tq {
bool prep_tile_per_workgroup(int n_tiles, int d);

// q_rot = q Pi^T, q_sk = q S^T for `rows` query vectors (triton_kernels.py:527-528), fp32.
// A workgroup handles R consecutive rows (the query heads of one KV head when
// called from the decode path) and a slice of ROT_COLS output columns with
// ROT_COLS x ROT_SLICES threads: thread (j, s) sums slice s of the contraction for
// its column of every row, so each matrix element is read once per workgroup; the
// slices meet in LDS.
constexpr int ROT_SLICES = 8;      // (ROT_COLS = 32 output columns per workgroup: tq_prep.h)

// sq[0 .. tot) = the first `have` elements of row row0 of q and those behind it as fp32, zeros behind them (have and tot multiples of 8):
// 16-byte loads, all of a thread's in flight together, when q allows them.  fp32 rows of d may lie q_row > d elements apart (a word at a time,
// 8 rows of 128 took four loads behind one another: the rotation 6.5 us, now 5.5).
template <bool APART>
__device__ __forceinline__ void rows_to_lds(const void* __restrict__ q, int dtype, int64_t row0, int have, int tot,
                                            float* __restrict__ sq, int tid, int n_threads, int d, int64_t q_row) {
  const int64_t off = row0 * d;
  if (APART && ((uintptr_t)q & 15) == 0 && q_row % 4 == 0) {
    const float* src = (const float*)q + row0 * q_row;
    const unsigned per = (unsigned)d / 4;
#pragma unroll 2
    for (int c = tid; c < tot / 4; c += n_threads)
      *(float4*)(sq + 4 * c) = 4 * c < have ? *(const float4*)(src + (unsigned)c / per * q_row + (unsigned)c % per * 4) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  } else if (APART) {
    const float* src = (const float*)q + row0 * q_row;
    for (int o = tid; o < tot; o += n_threads) sq[o] = o < have ? src[o / d * q_row + o % d] : 0.0f;
  } else if ((((uintptr_t)q) & 15) == 0 && dtype != TQ_F32) {
    const uint4* src = (const uint4*)((const uint16_t*)q + off);
    const bool bf = dtype == TQ_BF16;
#pragma unroll 4
    for (int c = tid; c < tot / 8; c += n_threads) {
      const uint4 w = 8 * c < have ? src[c] : make_uint4(0u, 0u, 0u, 0u);
      const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
      float v[8];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[2 * k] = bf ? __uint_as_float(ws[k] << 16) : f16_bits_to_f32((uint16_t)(ws[k] & 0xffffu));
        v[2 * k + 1] = bf ? __uint_as_float(ws[k] & 0xffff0000u) : f16_bits_to_f32((uint16_t)(ws[k] >> 16));
      }
      *(float4*)(sq + 8 * c) = make_float4(v[0], v[1], v[2], v[3]);
      *(float4*)(sq + 8 * c + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
  } else if ((((uintptr_t)q) & 15) == 0) {
    const float4* src = (const float4*)((const float*)q + off);
#pragma unroll 4
    for (int c = tid; c < tot / 4; c += n_threads)
      *(float4*)(sq + 4 * c) = 4 * c < have ? src[c] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  } else {
    for (int o = tid; o < tot; o += n_threads) sq[o] = o < have ? load_as_f32(q, off + o, dtype) : 0.0f;
  }
}

// BATCH: matrix rows of both matrices requested before the first is used (8, 16 or 24, a divisor of the d / 8 rows a
// thread contracts): the kernel is a chain of memory latencies, one per batch (head_dim 576: 9 -> 3; the sums add in
// the same order whatever the batch).
// HALVES (1 or 2): a workgroup of HALVES x 256 threads takes HALVES x 8 rows; the halves run the same loads a
// moment apart, so the second finds the matrix lines in the compute unit's cache: with many rows half the traffic
// from L2 for the same work per thread (128 rows at head_dim 576: 42 -> 21 MB).
// PACK (a decode step at a head size of the wide-head page kernel): the workgroup also turns its 32 columns - one
// plane word - of every row into the kernel's fp6 query operands (four terms per value, as prep_query_body packs them
// for the other head sizes) and writes them where the page-kernel workgroups of the row's head group fetch them,
// and the workgroups of the first word write the rows' statistics.  The operands are normalised by bounds every
// workgroup can compute from the raw query: |q_rot_j| <= ||q|| (Pi is orthogonal) and |q_sk_j| <= ||q|| max_j ||S_j||;
// the sums over all coordinates the scores need are q . colsum(Pi), q . colsum(S).
// APART: rows of q that are not one behind another (an instance of its own: 45 rows of 64 took 4.6 us without the branch and 5.0 with it)
template <int BATCH, int HALVES, bool PACK, bool APART>
__global__ void __launch_bounds__(ROT_COLS * ROT_SLICES * HALVES)
rotate_query_kernel(const void* __restrict__ q, int dtype, int64_t rows, int R, tq_layer ly, float* __restrict__ q_rot,
                    float* __restrict__ q_sk, WidePack wp, int64_t q_row) {
  extern __shared__ __align__(16) float sm[];
  constexpr int T1 = ROT_COLS * ROT_SLICES;
  const int d = ly.d, tid = threadIdx.x, half = tid / T1, t1 = tid - half * T1, jl = t1 % ROT_COLS, sl = t1 / ROT_COLS;
  const int j = blockIdx.y * ROT_COLS + jl;
  float* sq = sm;                                  // [R][d] inputs (R rows per workgroup: up to 8 per half)
  float* pa = sq + R * d;                          // [ROT_SLICES][R][ROT_COLS] partial sums
  float* pb = pa + ROT_SLICES * R * ROT_COLS;
  const int64_t row0 = (int64_t)blockIdx.x * R;
  const int nr = (int)((rows - row0) < R ? (rows - row0) : R);
  // the first batch of matrix rows (and, below, the column sums) is requested before the queries: neither depends on them
  const int per = d / ROT_SLICES, i0 = sl * per;
  float mp[BATCH], ms[BATCH];
#pragma unroll
  for (int k = 0; k < BATCH; ++k) {
    mp[k] = ly.PiT[(int64_t)(i0 + k) * d + j];
    ms[k] = ly.ST[(int64_t)(i0 + k) * d + j];
  }
  constexpr int CS = PACK ? 12 : 1;                // column sums of a lane (PACK; d <= 768)
  float cs1[CS], cs2[CS];
  if constexpr (PACK) {
#pragma unroll
    for (int k = 0; k < CS; ++k) {
      const int c = min((tid & 63) + 64 * k, d - 1);
      cs1[k] = ly.Pi_colsum[c];
      cs2[k] = ly.S_colsum[c];
    }
  }
  rows_to_lds<APART>(q, dtype, row0, nr * d, R * d, sq, tid, (int)blockDim.x, d, q_row);
  __syncthreads();
  float* s_rot = pb + ROT_SLICES * R * ROT_COLS;   // PACK: [R][ROT_COLS] this word's rotated values, then the sketched ones
  float* s_sk = s_rot + R * ROT_COLS;
  float* s_rs = s_sk + R * ROT_COLS;               // PACK: [R][2] multipliers of q_rot / q_sk
  float* s_cf = s_rs + 2 * R;                      // PACK: [16] coefficient of each term plane
  if constexpr (PACK) {
    // row statistics, a wavefront per row (every workgroup of the rows computes the same ones)
    const int lane = tid & 63, wv = tid >> 6, n_wv = (int)blockDim.x >> 6;
    const float cmax = wide_coef_bound(ly, wp);
    for (int r = wv; r < nr; r += n_wv) {
      float ss = 0.0f, s1 = 0.0f, s2 = 0.0f;
#pragma unroll
      for (int k = 0; k < CS; ++k) {
        const int c = lane + 64 * k;
        const float x = c < d ? sq[r * d + c] : 0.0f;
        ss = fmaf(x, x, ss);
        s1 = fmaf(x, cs1[k], s1);
        s2 = fmaf(x, cs2[k], s2);
      }
      ss = wave_sum_fast(ss); s1 = wave_sum_fast(s1); s2 = wave_sum_fast(s2);
      if (lane == 0) {
        const float nq = sqrtf(ss), k = wp.sm_scale * 1.4426950408889634f;
        // bound < 2^e: e = exponent field - 126, kept within +-100
        const int e1 = min(max((int)((__float_as_uint(fabsf(k) * nq * cmax) >> 23) & 255u) - 126, -100), 100);
        const int e2 = min(max((int)((__float_as_uint(2.0f * fabsf(k * ly.qjl_scale) * nq * ly.S_rownorm_max) >> 23) & 255u) - 126, -100), 100);
        s_rs[2 * r] = k * __uint_as_float((uint32_t)(127 - e1) << 23);
        s_rs[2 * r + 1] = 2.0f * k * ly.qjl_scale * __uint_as_float((uint32_t)(127 - e2) << 23);
        if (blockIdx.y == 0) {
          float* st = wp.q_stat + (row0 + r) * 4;
          st[0] = (float)e1; st[1] = (float)e2; st[2] = k * ly.term_const * s1; st[3] = -k * ly.qjl_scale * s2;
        }
      }
    }
    if (tid < 16) s_cf[tid] = wide_term_plane_coef(ly, wp, tid);
  }
  const int r0 = half * ROT_MAX_ROWS, RH = min(R - r0, ROT_MAX_ROWS);      // this half's rows: r0 .. r0 + RH - 1
  float a[ROT_MAX_ROWS], b[ROT_MAX_ROWS];
#pragma unroll
  for (int r = 0; r < ROT_MAX_ROWS; ++r) a[r] = b[r] = 0.0f;
  // BATCH matrix rows at a time: all their loads are in flight before the first use
  for (int ib = i0; ib < i0 + per; ib += BATCH) {
    if (ib > i0) {                                         // (the same for every thread)
#pragma unroll
      for (int k = 0; k < BATCH; ++k) {
        mp[k] = ly.PiT[(int64_t)(ib + k) * d + j];
        ms[k] = ly.ST[(int64_t)(ib + k) * d + j];
      }
    }
#pragma unroll
    for (int r = 0; r < ROT_MAX_ROWS; ++r) {
      if (r < RH) {
#pragma unroll
        for (int k4 = 0; k4 < BATCH / 4; ++k4) {
          const float4 x4 = *(const float4*)(sq + (r0 + r) * d + ib + 4 * k4);      // (ib and d are multiples of 8)
          const float xs[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            a[r] = fmaf(xs[k], mp[4 * k4 + k], a[r]);
            b[r] = fmaf(xs[k], ms[4 * k4 + k], b[r]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < ROT_MAX_ROWS; ++r) {
    if (r < RH) {
      pa[(sl * R + r0 + r) * ROT_COLS + jl] = a[r];
      pb[(sl * R + r0 + r) * ROT_COLS + jl] = b[r];
    }
  }
  __syncthreads();
  for (int o = tid; o < nr * ROT_COLS; o += blockDim.x) {
    const int r = o / ROT_COLS, c = o - r * ROT_COLS;
    float ra = 0.0f, rb = 0.0f;
    for (int k = 0; k < ROT_SLICES; ++k) { ra += pa[(k * R + r) * ROT_COLS + c]; rb += pb[(k * R + r) * ROT_COLS + c]; }
    q_rot[(row0 + r) * d + blockIdx.y * ROT_COLS + c] = ra;
    q_sk[(row0 + r) * d + blockIdx.y * ROT_COLS + c] = rb;
    if constexpr (PACK) {
      s_rot[o] = ra;
      s_sk[o] = rb;
    }
  }
  if constexpr (PACK) {
    __syncthreads();
    wide_pack_word(wp, d, nr, (int)row0, (int)blockIdx.y, s_rot, s_sk, s_rs, s_cf, tid, (int)blockDim.x, 0, wp.ntp);
  }
}

// the rotation on the matrix cores (rotate_mfma_body, tq_prep.h) as a launch of its own
template <int KPW, bool F16Q>
__global__ void __launch_bounds__(ROTM_THREADS)
rotate_mfma_kernel(const uint16_t* __restrict__ q, int64_t rows, int n_tiles, tq_layer ly, float* __restrict__ q_rot,
                   float* __restrict__ q_sk, WidePack wp) {
  extern __shared__ __align__(16) float sm[];
  rotate_mfma_body<KPW, F16Q>(q, rows, n_tiles, ly, q_rot, q_sk, wp, (int)blockIdx.x, sm);
}

template <int KPW, bool F16Q, int NT>
__global__ void __launch_bounds__(64 * ROTR_WAVES, 2)
rotate_rows_kernel(const uint16_t* __restrict__ q, int64_t rows, int n_tiles, int n_groups, tq_layer ly,
                   float* __restrict__ q_rot, float* __restrict__ q_sk, WidePack wp) {
  extern __shared__ __align__(16) unsigned char rows_smem[];
  rotate_rows_body<KPW, F16Q, NT>(q, rows, n_tiles, n_groups, ly, q_rot, q_sk, wp, (int)blockIdx.x, rows_smem);
}

template <int PER, int DT, bool PACKED>
__global__ void __launch_bounds__(PREP_COLS * PREP_SLICES)
prep_query_kernel(const void* __restrict__ q, int G, int gpw, int64_t n_rows, int g_tot, tq_layer ly, float sm_scale,
                  float* __restrict__ q_rot, float* __restrict__ q_sk, float* __restrict__ q_stat,
                  uint32_t* __restrict__ qa_pack, unsigned long long* __restrict__ arrivals, int head_rows, int n_units,
                  int n_prep, PagePrefetch pf, SplitPlan sp) {
  extern __shared__ __align__(16) float sm[];
  // the schedule of the page kernel's workgroups in front
  if (sp.items && blockIdx.x < SCHED_FRONT) {
    if (blockIdx.x == 0) schedule_splits_body<PREP_COLS * PREP_SLICES>(sp, threadIdx.x, (int*)sm);
    return;
  }
  // the preparation workgroups first (unit fastest, as a two-dimensional grid would order them), then the
  // workgroups that read the page kernel's first pages ahead of it
  const int id = blockIdx.x - (sp.items ? SCHED_FRONT : 0);
  if (id < n_prep)
    prep_query_body<PER, DT, PACKED>(q, G, gpw, n_rows, g_tot, ly, sm_scale, q_rot, q_sk, q_stat, qa_pack, arrivals, head_rows,
                                     id % n_units, id / n_units, sm);
  else
    prefetch_pages_body<PREP_COLS * PREP_SLICES>(pf, id - n_prep);
}

// The preparation on the matrix cores (bf16 queries, head_dim 128 / 256; fp16 queries, 128): a workgroup per (tile of up to 16 query
// rows, plane word), then the page-prefetch workgroups.
// WW: a workgroup per tile, its wavefronts each taking a plane word at a time.
template <int D, bool WW, bool F16Q>
__global__ void __launch_bounds__(PREP_MFMA_THREADS)
prep_mfma_kernel(const uint16_t* __restrict__ q, int G, int64_t n_rows, tq_layer ly, float sm_scale,
                 float* __restrict__ q_stat, uint32_t* __restrict__ qa_pack, unsigned long long* __restrict__ arrivals,
                 int head_rows, int n_tiles, int n_prep, PagePrefetch pf, SplitPlan sp) {
  extern __shared__ __align__(16) float sm[];
  if (sp.items && blockIdx.x < SCHED_FRONT) {
    if (blockIdx.x == 0) schedule_splits_body<PREP_MFMA_THREADS>(sp, threadIdx.x, (int*)sm);
    return;
  }
  const int id = blockIdx.x - (sp.items ? SCHED_FRONT : 0);
  if (id < n_prep)
    prep_mfma_body<D, WW, F16Q>(q, G, n_rows, ly, sm_scale, q_stat, qa_pack, arrivals, head_rows, id % n_tiles, id / n_tiles, sm);
  else
    prefetch_pages_body<PREP_MFMA_THREADS>(pf, id - n_prep);
}

// The exact tokens of a cache object: fp32 rows (batch, H, n, d) with element strides, and the queries they meet.
struct CacheTail {
  const float* q;
  int64_t q_row;             // elements from a query to the next
  const float* k;
  int64_t s_b, s_h, s_r;
  int H, n;
  float scale;
};

// scores[b, i, k] on the matrix cores: v_mfma_f32_16x16x4_f32 with sixteen rotated / sketched queries as rows, sixteen keys as columns
// and fp32 operands on both sides (a centroid or a sign is an fp32 number), so nothing is split or rounded.  Of every sixteen
// coordinates a lane holds four of its key and the same four of its query, which it reads straight from the rotation's rows: the four lanes
// of a row take 64 consecutive bytes (a quarter of the coordinates in a row per lane touched 64 lines per load: 215 us where the kernel
// that this replaces took 180).  NT tiles of sixteen queries share one expansion of the codes.
// Bound by latency in small calls, else by the fp32 matrix rate (two MFMAs of 32 cycles per 4 coordinates of a 16 x 16 tile).  One key per
// thread with the queries as LDS broadcasts, which this replaces, read 64 bytes of LDS per key and coordinate: 32 queries x 4096 keys of
// 128 18.0 -> 5.1 us; the call with its rotation, 8 heads x 16384 keys x 128 queries of 128 166 -> 130 us, of 256 308 -> 251, 1000 keys of 576
// and 33 queries 78 -> 25.
// CACHE: the workgroups behind those of the compressed keys take the exact ones, a wavefront per row at a time
// key0: first key of the launch (a grid dimension counts fewer than 2^32 threads: 2^28 keys at a time)
constexpr int SCORE_KEYS = 64;     // keys per workgroup: sixteen for each of four wavefronts
constexpr int64_t SCORE_LAUNCH_KEYS = 1 << 28;
constexpr int SCORE_ROWS = 4;      // exact rows per workgroup: one per wavefront (eight behind one another, 4000 keys and 128 rows of 8 heads: 9.7 us, now 7.8)

// Word w of a row of codes; BYTES: rows that are not 4-byte aligned
template <bool BYTES>
__device__ __forceinline__ uint32_t code_word(const uint8_t* __restrict__ row, int w) {
  if constexpr (!BYTES) return ((const uint32_t*)row)[w];
  const uint8_t* p = row + 4 * w;
  return p[0] | (uint32_t)p[1] << 8 | (uint32_t)p[2] << 16 | (uint32_t)p[3] << 24;
}

template <int EFF, int NT, bool BYTES>
__device__ __forceinline__ void score_tiles(const float* __restrict__ rot, const float* __restrict__ sk, const int64_t (&row)[NT],
                                            const float* s_cent, int d, int kb, const uint8_t* __restrict__ ip,
                                            const uint8_t* __restrict__ sp, prep_f32x4 (&am)[NT], prep_f32x4 (&aq)[NT]) {
  typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));        // (the caller's scratch: any float address)
  constexpr unsigned mask = (1u << EFF) - 1u;
  for (int c0 = 0; c0 < d; c0 += 64) {
    uint32_t sb[2], iw[4];                                      // shifted to this lane's four coordinates of each sixteen
#pragma unroll
    for (int j = 0; j < 2; ++j) sb[j] = code_word<BYTES>(sp, (c0 >> 5) + j) >> (4 * kb);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (EFF == 1) iw[j] = code_word<BYTES>(ip, (c0 >> 5) + (j >> 1)) >> (16 * (j & 1) + 4 * kb);
      if (EFF == 2) iw[j] = code_word<BYTES>(ip, (c0 >> 4) + j) >> (8 * kb);
      if (EFF == 4) iw[j] = code_word<BYTES>(ip, (c0 >> 3) + 2 * j + (kb >> 1)) >> (16 * (kb & 1));
    }
    f32x4_u r[NT][4], k[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        r[t][j] = *(const f32x4_u*)(rot + row[t] + c0 + 16 * j + 4 * kb);
        k[t][j] = *(const f32x4_u*)(sk + row[t] + c0 + 16 * j + 4 * kb);
      }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float cv = s_cent[(iw[j] >> (EFF * e)) & mask];
        const float sg = __uint_as_float(0xbf800000u ^ (sb[j >> 1] << (31 - 16 * (j & 1) - e) & 0x80000000u));   // bit set: +1
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          am[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(r[t][j][e], cv, am[t], 0, 0, 0);
          aq[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[t][j][e], sg, aq[t], 0, 0, 0);
        }
      }
  }
}

template <bool CACHE, int NT, bool BYTES = false>
__global__ void __launch_bounds__(256)
score_kernel(const float* __restrict__ q_rot, const float* __restrict__ q_sk, int64_t n_q,
             const uint8_t* __restrict__ idx, const uint8_t* __restrict__ signs, const void* __restrict__ norms,
             int norm_dtype, const float* __restrict__ rnorms, int64_t n_k, int64_t key0, tq_layer ly, float* __restrict__ scores,
             CacheTail tail) {
  __shared__ float s_cent[16];
  const int d = ly.d, mb = ly.mse_bits;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t b = blockIdx.z, q0 = (int64_t)blockIdx.y * (16 * NT);
  if constexpr (CACHE) {
    const int64_t nkb = (n_k + SCORE_KEYS - 1) / SCORE_KEYS;
    if ((int64_t)blockIdx.x >= nkb) {
      const int ni = (int)((n_q - q0) < 16 * NT ? (n_q - q0) : 16 * NT);
      for (int r = ((int)blockIdx.x - (int)nkb) * SCORE_ROWS + wave, e = min(r - wave + SCORE_ROWS, tail.n); r < e; r += 4) {
        const float* row = tail.k + b / tail.H * tail.s_b + b % tail.H * tail.s_h + r * tail.s_r;
        for (int i = 0; i < ni; ++i) {
          const float* qr = tail.q + (b * n_q + q0 + i) * tail.q_row;
          float a = 0.0f;
          for (int c = lane; c < d; c += 64) a = fmaf(qr[c], row[c], a);
          a = wave_sum_fast(a);
          if (lane == 0) scores[(b * n_q + q0 + i) * (n_k + tail.n) + n_k + r] = __fmul_rn(a, tail.scale);
        }
      }
      return;
    }
  }
  if (threadIdx.x < (1 << mb)) s_cent[threadIdx.x] = ly.centroids[threadIdx.x];
  __syncthreads();
  const int64_t k0 = key0 + (int64_t)blockIdx.x * SCORE_KEYS + wave * 16;
  if (k0 >= n_k) return;
  const int n = lane & 15, kb = lane >> 4;
  const int64_t key = k0 + n < n_k ? k0 + n : n_k - 1;          // (keys and queries that do not exist: the last one, not stored)
  const int eff = eff_bits(mb);
  const uint8_t* ip = idx + (b * n_k + key) * idx_row_bytes(d, mb);
  const uint8_t* sp = signs + (b * n_k + key) * (d >> 3);
  int64_t row[NT];
  prep_f32x4 am[NT], aq[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int64_t i = q0 + 16 * t + n;
    row[t] = (b * n_q + (i < n_q ? i : n_q - 1)) * d;
    am[t] = aq[t] = prep_f32x4{0, 0, 0, 0};
  }
  const float nk = load_as_f32(norms, b * n_k + key, norm_dtype);
  const float rk = __fmul_rn(ly.qjl_scale, rnorms[b * n_k + key]);
  if (eff == 1) score_tiles<1, NT, BYTES>(q_rot, q_sk, row, s_cent, d, kb, ip, sp, am, aq);
  else if (eff == 2) score_tiles<2, NT, BYTES>(q_rot, q_sk, row, s_cent, d, kb, ip, sp, am, aq);
  else score_tiles<4, NT, BYTES>(q_rot, q_sk, row, s_cent, d, kb, ip, sp, am, aq);
  if (k0 + n >= n_k) return;
  // (CACHE: the rows of scores go on with those of the exact tokens, and all of them are scaled)
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t qi = q0 + 16 * t + 4 * kb + i;
      if (qi >= n_q) continue;
      const float s = __fadd_rn(__fmul_rn(am[t][i], nk), __fmul_rn(aq[t][i], rk));
      if constexpr (CACHE) scores[(b * n_q + qi) * (n_k + tail.n) + key] = __fmul_rn(s, tail.scale);
      else scores[(b * n_q + qi) * n_k + key] = s;
    }
}

// Tiles of sixteen queries per wavefront: two where that still leaves two workgroups per compute unit (the call, 8 heads x 16384 keys x 128
// queries of 128 / 256: 133 / 254 us with two, 137 / 265 with one; fewer queries or keys: the same)
__host__ static int score_query_tiles(int64_t batch, int64_t n_q, int64_t n_k) {
  if (n_q <= 16) return 1;
  return batch * ((n_q + 31) / 32) * ((n_k + SCORE_KEYS - 1) / SCORE_KEYS) >= 2 * (int64_t)device_compute_units() ? 2 : 1;
}

// x_hat for a tile of TILE vectors: (c[idx] Pi) * norm + (sigma S) * (qjl_scale * rnorm)
// (quantizer.py:151-165, 259-272).  d threads, thread i owns output coordinate i and
// sums over j in ascending order.  The tile's centroid and sign values sit in LDS as
// [j][TILE] rows (padded by 4 floats) so one 16-byte broadcast read feeds four FMAs.
template <int TILE, bool QJL>
__global__ void __launch_bounds__(1024)
dequant_keys_kernel(const uint8_t* __restrict__ idx, const uint8_t* __restrict__ signs, const void* __restrict__ norms,
                    int norm_dtype, const float* __restrict__ rnorms, int64_t n_vec, tq_layer ly,
                    float* __restrict__ out) {
  constexpr int LD = TILE + 4;
  extern __shared__ float sm[];
  const int d = ly.d, mb = ly.mse_bits, i = threadIdx.x;
  float* sc = sm;             // [d][LD] centroid values
  float* ss = sm + LD * d;    // [d][LD] +-1
  const int eff = eff_bits(mb), per = 8 / eff, row = idx_row_bytes(d, mb), srow = d >> 3;
  const unsigned mask = (1u << eff) - 1u;
  const int64_t v0 = (int64_t)blockIdx.x * TILE;
  for (int t = 0; t < TILE; ++t) {
    int64_t v = v0 + t;
    float cv = 0.0f, sg = 0.0f;
    if (v < n_vec) {
      unsigned byte = idx[v * row + i / per];
      cv = ly.centroids[(byte >> (eff * (i % per))) & mask];
      if (QJL) sg = ((signs[v * srow + (i >> 3)] >> (i & 7)) & 1u) ? 1.0f : -1.0f;
    }
    sc[i * LD + t] = cv;
    if (QJL) ss[i * LD + t] = sg;
  }
  __syncthreads();
  float a[TILE], b[QJL ? TILE : 1];
#pragma unroll
  for (int t = 0; t < TILE; ++t) a[t] = 0.0f;
#pragma unroll
  for (int t = 0; t < (QJL ? TILE : 1); ++t) b[t] = 0.0f;
#pragma unroll 2
  for (int j = 0; j < d; ++j) {
    const float pv = ly.Pi[(int64_t)j * d + i];
    const float sv = QJL ? ly.S[(int64_t)j * d + i] : 0.0f;
#pragma unroll
    for (int t4 = 0; t4 < TILE / 4; ++t4) {
      const float4 c = *reinterpret_cast<const float4*>(sc + j * LD + 4 * t4);
      a[4 * t4 + 0] = fmaf(c.x, pv, a[4 * t4 + 0]);
      a[4 * t4 + 1] = fmaf(c.y, pv, a[4 * t4 + 1]);
      a[4 * t4 + 2] = fmaf(c.z, pv, a[4 * t4 + 2]);
      a[4 * t4 + 3] = fmaf(c.w, pv, a[4 * t4 + 3]);
      if (QJL) {
        const float4 g = *reinterpret_cast<const float4*>(ss + j * LD + 4 * t4);
        b[4 * t4 + 0] = fmaf(g.x, sv, b[4 * t4 + 0]);
        b[4 * t4 + 1] = fmaf(g.y, sv, b[4 * t4 + 1]);
        b[4 * t4 + 2] = fmaf(g.z, sv, b[4 * t4 + 2]);
        b[4 * t4 + 3] = fmaf(g.w, sv, b[4 * t4 + 3]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < TILE; ++t) {
    int64_t v = v0 + t;
    if (v < n_vec) {
      float r = __fmul_rn(a[t], load_as_f32(norms, v, norm_dtype));
      if (QJL) r = __fadd_rn(r, __fmul_rn(b[t], __fmul_rn(ly.qjl_scale, rnorms[v])));
      out[v * d + i] = r;
    }
  }
}

template <int TILE, bool QJL>
static int launch_dequant_keys(const uint8_t* idx, const uint8_t* signs, const void* norms, int norm_dtype,
                               const float* rnorms, int64_t n_vec, const tq_layer* layer, float* out, hipStream_t st) {
  const int d = layer->d;
  const size_t smem = (size_t)(QJL ? 2 : 1) * (TILE + 4) * d * sizeof(float);
  auto kern = dequant_keys_kernel<TILE, QJL>;
  if (smem > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return (int)e;
  }
  kern<<<dim3((unsigned)((n_vec + TILE - 1) / TILE)), dim3(d), smem, st>>>(idx, signs, norms, norm_dtype, rnorms, n_vec,
                                                                            *layer, out);
  TQ_CHECK_LAUNCH();
  return TQ_OK;
}

// fp32(code) * scale + zero with separately rounded multiply and add (kv_cache.py:101-116)
__global__ void dequant_values_kernel(const uint8_t* __restrict__ data, const void* __restrict__ scales,
                                      const void* __restrict__ zeros, int dtype, int64_t n_vec, int d, int gs, int bits,
                                      float* __restrict__ out) {
  int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (gid >= n_vec * d) return;
  int64_t v = gid / d;
  int c = (int)(gid - v * d);
  const int per = 8 / bits, ng = d / gs;
  unsigned byte = data[v * (d / per) + c / per];
  float code = (float)((byte >> (bits * (c % per))) & ((1u << bits) - 1u));
  float s = load_as_f32(scales, v * ng + c / gs, dtype);
  float z = load_as_f32(zeros, v * ng + c / gs, dtype);
  out[gid] = __fadd_rn(__fmul_rn(code, s), z);
}

// The same arithmetic, a thread per 8 consecutive channels (they share a group when the group size is a
// multiple of 8): one load of the packed codes, scale and zero read once, two 16-byte stores.
template <int BITS>
__global__ void dequant_values8_kernel(const uint8_t* __restrict__ data, const void* __restrict__ scales,
                                       const void* __restrict__ zeros, int dtype, int64_t n_vec, int d, int gs,
                                       float* __restrict__ out) {
  const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;      // chunk of 8 channels
  const int cpv = d >> 3;
  if (gid >= n_vec * cpv) return;
  const int64_t v = gid / cpv;
  const int c0 = (int)(gid - v * cpv) * 8;
  const int ng = d / gs;
  const uint8_t* src = data + v * (d * BITS / 8) + c0 * BITS / 8;
  uint64_t bits64;
  if (BITS == 2) bits64 = *(const uint16_t*)src;
  else if (BITS == 4) bits64 = *(const uint32_t*)src;
  else bits64 = *(const uint64_t*)src;
  const float sc = load_as_f32(scales, v * ng + c0 / gs, dtype);
  const float z = load_as_f32(zeros, v * ng + c0 / gs, dtype);
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float code = (float)(uint32_t)((bits64 >> (BITS * i)) & ((1u << BITS) - 1u));
    r[i] = __fadd_rn(__fmul_rn(code, sc), z);
  }
  float4* dst = (float4*)(out + v * d + c0);
  dst[0] = make_float4(r[0], r[1], r[2], r[3]);
  dst[1] = make_float4(r[4], r[5], r[6], r[7]);
}

}  // namespace tq

using namespace tq;

static int check_layer_rd(const tq_layer* ly, bool need_sketch) {
  if (!ly) return TQ_ENULL;
  if (ly->d < 64 || ly->d > 768 || (ly->d & 63)) return TQ_EUNSUPPORTED;
  if (ly->mse_bits < 1 || ly->mse_bits > 4) return TQ_EUNSUPPORTED;
  if (!ly->Pi || !ly->PiT || !ly->centroids) return TQ_ENULL;
  if (need_sketch && (!ly->S || !ly->ST)) return TQ_ENULL;
  return TQ_OK;
}

namespace tq {
// matrix-core de-quantiser (tq_quantize_mfma.hip); TQ_EUNSUPPORTED = use the vector-ALU kernel
int launch_dequant_mfma(const uint8_t* idx, const uint8_t* signs, const void* norms, int norm_dtype, const float* rnorms,
                        int64_t n_vec, const tq_layer& ly, float* out, hipStream_t st);

// Whether launch_rotate_query prepares these rows on the matrix cores (bf16 queries at head_dim 128 / 256, fp16 queries at 128, with
// the split matrices at hand; whole groups of G heads; operands only).
// (head_dim 256 with few rows keeps the vector-ALU kernel: 64 rows - 32 workgroups here, each pulling 96 KB of
// matrix terms - measured 1 us slower per step; from 64 workgroups on the two are level or this one ahead:
// 16 x 8192 at 32 q heads 35.0 -> 34.5 us per step, 64 x 2048 40.2 -> 36.4, 256 x 1024 107.6 -> 86.2)
bool prep_on_matrix_cores(const void* q, int dtype, int64_t rows, const tq_layer* layer, int G, int g_tot) {
  const int d = layer->d;
  if (g_tot > 0 && g_tot % G == 0) g_tot = 0;
  const int rows_tile = (16 / G) * G;
  const int64_t n_mprep = ((rows + rows_tile - 1) / rows_tile) * (d / 32);
  const int mfma_opt = opt_prep_mfma.load(std::memory_order_relaxed);
  // (fp16 queries, as two bf16 terms, at head_dim 128: 96 sequences of 40 heads 29.4 us on the vector ALU, 16 here)
  return ((dtype == TQ_BF16 && (d == 128 || d == 256)) || (dtype == TQ_F16 && d == 128)) && layer->Pi_split && layer->S_split && layer->Pi_colsum &&
         layer->S_colsum && g_tot == 0 && G <= ROT_MAX_ROWS && rows % G == 0 && (((uintptr_t)q) & 15) == 0 &&
         mfma_opt != 0 && (d == 128 || n_mprep >= 64 || mfma_opt > 1);
}

// Matrix-core preparation: a workgroup per tile of query rows (its wavefronts a plane word each) instead of one per (tile, word)
bool prep_tile_per_workgroup(int n_tiles, int d) {
  const int opt_ww = opt_prep_words.load(std::memory_order_relaxed);
  return opt_ww < 0 ? d == 128 && (int64_t)n_tiles * (d / 32) > (int64_t)4 * device_compute_units() : opt_ww != 0;
}

// Whether the rotation launch of a decode step also packs the wide-head page kernel's query operands ...
static bool rotate_packs(int64_t rows, const tq_layer* layer, const WidePack* wide) {
  return wide != nullptr && wide->qa != nullptr && wide->q_stat != nullptr && layer->Pi_colsum && layer->S_colsum &&
         wide->ntp >= 2 && wide->ntp <= 9 && rows % wide->Hq == 0 && rows < (1 << 30) && layer->d <= 768;
}
// Row tiles from which a rotation keeps a (plane word, product) pair's matrix terms in LDS and passes over the tiles
// (rotate_rows_body) instead of running a workgroup per (tile, word, product): when the latter are more than the card holds
// at once, two per compute unit.
bool rotate_by_rows(int64_t rows, int d) {
  return ((rows + 15) / 16) * 8 * ((2 * (d / ROT_COLS) + 7) / 8) > 2 * (int64_t)device_compute_units();
}
// ... and whether the launch that packs does so on the matrix cores (with the layer's split matrices: bf16 queries, fp16 queries as
// two bf16 terms)
bool rotate_on_matrix_cores(const void* q, int dtype, int64_t rows, const tq_layer* layer, const WidePack* wide) {
  const int d = layer->d;
  return rotate_packs(rows, layer, wide) && layer->Pi_split && layer->S_split &&
         (((uintptr_t)q) & 15) == 0 && d % 64 == 0 && d >= 320 && d <= 704 &&
         (dtype == TQ_BF16 || dtype == TQ_F16) &&
         opt_prep_mfma.load(std::memory_order_relaxed) != 0;
}

// q_rot_unused: the caller only needs the packed operands and statistics (the page kernel on the matrix
// cores), not the fp32 rotated / sketched queries
int launch_rotate_query(const void* q, int dtype, int64_t rows, const tq_layer* layer, float* q_rot, float* q_sk,
                        float* q_stat, uint32_t* qa_pack, int G, float sm_scale, hipStream_t st, bool q_rot_unused,
                        unsigned long long* arrivals, const PagePrefetch* prefetch, int g_tot, const WidePack* wide,
                        const SplitPlan& plan, int64_t q_row) {
  const int d = layer->d;
  if (qa_pack) {       // operands of the matrix-core decode kernel wanted
    // g_tot: query heads per KV head when its groups of G are unequal (0: the rows are whole groups of G)
    if (g_tot > 0 && g_tot % G == 0) g_tot = 0;
    if (!q_stat || !layer->Pi_colsum || !layer->S_colsum || G > ROT_MAX_ROWS || (g_tot > 0 ? rows % g_tot : rows % G) ||
        (d != 64 && d != 128 && d != 256))
      return TQ_EUNSUPPORTED;
    const int head_rows = decode_mfma_head_rows(d, G);      // rows of a group's operands the page kernel reads
    if (q_rot_unused && prep_on_matrix_cores(q, dtype, rows, layer, G, g_tot)) {
      const int rows_tile = (16 / G) * G;
      const int n_tiles = (int)((rows + rows_tile - 1) / rows_tile);
      // (several tiles per workgroup - in turn, or their products first and then all four wavefronts packing - measured
      // slower at every size: 256 x 1024 tokens 83.0 -> 83.9 us per step with four, 64 x 2048 33.8 -> 38.6)
      // Head_dim 128 with more (tile, word) pairs than the card holds workgroups of this kernel at once (four per compute
      // unit): a workgroup per tile, its wavefronts taking a plane word each (256 x 1024 tokens, 32 q / 8 KV heads:
      // preparation 16.5 -> 12.3 us; smaller ones lose 1 - 2 us, and at head_dim 256, where a wavefront takes two words in
      // turn, 128 x 2048 at 16 q / 2 KV heads goes from 44.6 to 54.5 us per step).
      const bool ww = prep_tile_per_workgroup(n_tiles, d);
      const int n_mprep = ww ? n_tiles : n_tiles * (d / 32);
      PagePrefetch pf;
      if (prefetch && prefetch->blocks > 0 && prefetch->n_wg > 0 && n_mprep <= 2 * device_compute_units()) pf = *prefetch;
      const int n_sched = plan.items ? SCHED_FRONT : 0;
      pf.front = n_mprep + n_sched;
      const dim3 grid((unsigned)(n_sched + n_mprep + (pf.blocks > 0 ? pf.n_wg : 0))), block(PREP_MFMA_THREADS);
      size_t smem = (size_t)prep_mfma_smem_floats() * sizeof(float) * (ww ? 4 : 1);
      if (n_sched && smem < SCHED_SMEM_INTS * sizeof(int)) smem = SCHED_SMEM_INTS * sizeof(int);
#define TQ_PREP_MFMA(D, WW)                                                                                            \
  {                                                                                                                    \
    auto kern = dtype == TQ_F16 ? prep_mfma_kernel<128, WW, true> : prep_mfma_kernel<D, WW, false>;                    \
    kern<<<grid, block, smem, st>>>((const uint16_t*)q, G, rows, *layer, sm_scale, q_stat, qa_pack, arrivals, head_rows, \
                                    n_tiles, n_mprep, pf, plan);                                                       \
  }
      if (d == 128 && ww) TQ_PREP_MFMA(128, true)
      else if (d == 128) TQ_PREP_MFMA(128, false)
      else if (ww) TQ_PREP_MFMA(256, true)
      else TQ_PREP_MFMA(256, false)
#undef TQ_PREP_MFMA
      hipError_t e = hipGetLastError();
      return e == hipSuccess ? TQ_OK : (int)e;
    }
    // one group of heads per workgroup while the card holds all of them at once (three workgroups of 74 registers
    // per lane on each compute unit); beyond that, as many whole groups as fit a workgroup's eight rows
    // (64 x 2048 tokens at 32 q / 8 KV heads: 45.9 -> 42.2 us per step, 256 x 1024: 134 -> 121)
    const int gpw = g_tot > 0 ? 1 : prep_groups_per_workgroup(G, (rows / G) * (d / PREP_COLS), 3 * (int64_t)device_compute_units());
    const int64_t rows_per_wg = (int64_t)G * gpw;
    size_t smem = prep_smem_bytes(G * gpw, d);
    const int n_units = g_tot > 0 ? (int)(rows / g_tot) * ((g_tot + G - 1) / G) : (int)((rows + rows_per_wg - 1) / rows_per_wg);
    const int n_prep = n_units * (d / PREP_COLS);
    PagePrefetch pf;
    // (a preparation that already fills the card - hundreds of sequences - gains nothing from more workgroups:
    // 64 x 2048 tokens at 32 q / 8 KV heads measured 44.6 -> 46.3 us per step with them)
    if (prefetch && prefetch->blocks > 0 && prefetch->n_wg > 0 && n_prep <= 2 * device_compute_units()) pf = *prefetch;
    const int n_sched = plan.items ? SCHED_FRONT : 0;
    if (n_sched && smem < SCHED_SMEM_INTS * sizeof(int)) smem = SCHED_SMEM_INTS * sizeof(int);
    pf.front = n_prep + n_sched;
    const dim3 grid((unsigned)(n_sched + n_prep + (pf.blocks > 0 ? pf.n_wg : 0))), block(PREP_COLS * PREP_SLICES);
#define TQ_PREP(PER, DT)                                                                                               \
  {                                                                                                                    \
    if (gpw > 1)                                                                                                       \
      prep_query_kernel<PER, DT, true><<<grid, block, smem, st>>>(q, G, gpw, rows, g_tot, *layer, sm_scale, q_rot, q_sk, q_stat, \
                                                                  qa_pack, arrivals, head_rows, n_units, n_prep, pf, plan);              \
    else                                                                                                               \
      prep_query_kernel<PER, DT, false><<<grid, block, smem, st>>>(q, G, gpw, rows, g_tot, *layer, sm_scale, q_rot, q_sk, q_stat, \
                                                                   qa_pack, arrivals, head_rows, n_units, n_prep, pf, plan);             \
  }
#define TQ_PREP_DT(PER)                              \
  {                                                  \
    if (dtype == TQ_BF16) TQ_PREP(PER, TQ_BF16)      \
    else if (dtype == TQ_F16) TQ_PREP(PER, TQ_F16)   \
    else if (dtype == TQ_F32) TQ_PREP(PER, TQ_F32)   \
    else return TQ_EINVAL;                           \
  }
    if (d == 64) TQ_PREP_DT(4)
    else if (d == 128) TQ_PREP_DT(8)
    else TQ_PREP_DT(16)
#undef TQ_PREP_DT
#undef TQ_PREP
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? TQ_OK : (int)e;
  }
  // rows per workgroup: 8, or 16 (two halves of 256 threads) when that still leaves a workgroup for half the compute units
  const bool wide_rows = rows >= 32 && ((rows + 15) / 16) * (d / ROT_COLS) >= device_compute_units() / 2;
  const int max_r = wide_rows ? 16 : ROT_MAX_ROWS;
  const int R = (int)(rows < max_r ? rows : max_r);
  if (R < 1 || d % ROT_COLS || d % (8 * ROT_SLICES)) return TQ_EUNSUPPORTED;
  const bool pack = rotate_packs(rows, layer, wide);
  const WidePack wp = pack ? *wide : WidePack{};
  // bf16 and fp16 queries with the layer's split matrices: rotation and packing on the matrix cores
  if (rotate_on_matrix_cores(q, dtype, rows, layer, wide)) {
    const int n_tiles = (int)((rows + 15) / 16), pair_rounds = (2 * (d / ROT_COLS) + 7) / 8;
    if (rotate_by_rows(rows, d)) {
      // shares of the tiles: one workgroup per compute unit (the terms fill its LDS), at least a tile each
      const int slots = device_compute_units() / (8 * pair_rounds);
      const int n_groups = slots < 1 ? 1 : (slots > n_tiles ? n_tiles : slots);
      // row tiles a wavefront takes at a time: a workgroup's share in one pass where three each are enough
      const int per = (n_tiles + n_groups - 1) / n_groups, nt = per <= ROTR_WAVES ? 1 : (per <= 2 * ROTR_WAVES ? 2 : 3);
      const dim3 rgrid((unsigned)(8 * pair_rounds * n_groups));
      const size_t rsm = (size_t)rotate_rows_smem_bytes(d);
#define TQ_ROTR(KPW)                                                                                                   \
  case KPW: {                                                                                                          \
    auto kern = dtype == TQ_F16 ? (nt == 1 ? rotate_rows_kernel<KPW, true, 1> : nt == 2 ? rotate_rows_kernel<KPW, true, 2> : rotate_rows_kernel<KPW, true, 3>) \
                                : (nt == 1 ? rotate_rows_kernel<KPW, false, 1> : nt == 2 ? rotate_rows_kernel<KPW, false, 2> : rotate_rows_kernel<KPW, false, 3>); \
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)rsm);       \
    if (e != hipSuccess) return (int)e;                                                                                \
    kern<<<rgrid, dim3(64 * ROTR_WAVES), rsm, st>>>((const uint16_t*)q, rows, n_tiles, n_groups, *layer, q_rot, q_sk, wp); \
  } break;
      switch (d / 64) {
        TQ_ROTR(5) TQ_ROTR(6) TQ_ROTR(7) TQ_ROTR(8) TQ_ROTR(9) TQ_ROTR(10) TQ_ROTR(11)
      }
#undef TQ_ROTR
      hipError_t e = hipGetLastError();
      return e == hipSuccess ? TQ_OK : (int)e;
    }
    const dim3 mgrid((unsigned)(8 * pair_rounds * n_tiles)), mblock(ROTM_THREADS);
    const size_t msm = (size_t)rotate_mfma_smem_floats() * sizeof(float);
#define TQ_ROTM(KPW) \
  case KPW:                                                                                                            \
    if (dtype == TQ_F16) rotate_mfma_kernel<KPW, true><<<mgrid, mblock, msm, st>>>((const uint16_t*)q, rows, n_tiles, *layer, q_rot, q_sk, wp); \
    else rotate_mfma_kernel<KPW, false><<<mgrid, mblock, msm, st>>>((const uint16_t*)q, rows, n_tiles, *layer, q_rot, q_sk, wp);               \
    break;
    switch (d / 64) {
      TQ_ROTM(5) TQ_ROTM(6) TQ_ROTM(7) TQ_ROTM(8) TQ_ROTM(9) TQ_ROTM(10) TQ_ROTM(11)
    }
#undef TQ_ROTM
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? TQ_OK : (int)e;
  }
  size_t smem = (size_t)(R * d + 2 * ROT_SLICES * R * ROT_COLS + (pack ? 2 * R * ROT_COLS + 2 * R + 16 : 0)) * sizeof(float);
  const dim3 rgrid((unsigned)((rows + R - 1) / R), d / ROT_COLS), rblock(ROT_COLS * ROT_SLICES * (wide_rows ? 2 : 1));
  const int per = d / ROT_SLICES;
#define TQ_ROTATE(BATCH, MAXR)                                                                                         \
  {                                                                                                                    \
    auto kern = pack ? rotate_query_kernel<BATCH, MAXR, true, false> : rotate_query_kernel<BATCH, MAXR, false, false>; \
    if (q_row != layer->d) kern = rotate_query_kernel<BATCH, MAXR, false, true>;                                       \
    if (smem > 48 * 1024) {                                                                                            \
      hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);    \
      if (e != hipSuccess) return (int)e;                                                                              \
    }                                                                                                                  \
    kern<<<rgrid, rblock, smem, st>>>(q, dtype, rows, R, *layer, q_rot, q_sk, wp, q_row);                              \
  }
#define TQ_ROTATE_R(BATCH)                 \
  {                                        \
    if (wide_rows) TQ_ROTATE(BATCH, 2)     \
    else TQ_ROTATE(BATCH, 1)               \
  }
  if (per % 24 == 0) TQ_ROTATE_R(24)
  else if (per % 16 == 0) TQ_ROTATE_R(16)
  else TQ_ROTATE_R(8)
#undef TQ_ROTATE_R
#undef TQ_ROTATE
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  return TQ_OK;
}
}  // namespace tq

extern "C" int tq_rotate_query(const void* q, int dtype, int64_t rows, const tq_layer* layer, float* q_rot,
                               float* q_sk, void* stream) {
  int rc = check_layer_rd(layer, true);
  if (rc) return rc;
  if (!q || !q_rot || !q_sk) return TQ_ENULL;
  if (rows < 0 || dtype < TQ_F32 || dtype > TQ_BF16) return TQ_EINVAL;
  if (rows == 0) return TQ_OK;
  return launch_rotate_query(q, dtype, rows, layer, q_rot, q_sk, nullptr, nullptr, 1, 0.0f, (hipStream_t)stream, false, nullptr, nullptr, 0, nullptr, SplitPlan{}, layer->d);
}

extern "C" int tq_score(const void* q, int dtype, int64_t batch, int64_t n_q, const uint8_t* idx, const uint8_t* signs,
                        const void* norms, int norm_dtype, const float* rnorms, int64_t n_k, const tq_layer* layer,
                        float* scores, float* work, void* stream) {
  int rc = check_layer_rd(layer, true);
  if (rc) return rc;
  if (!q || !idx || !signs || !norms || !rnorms || !scores || !work) return TQ_ENULL;
  if (batch < 0 || n_q < 0 || n_k < 0 || norm_dtype < TQ_F32 || norm_dtype > TQ_BF16) return TQ_EINVAL;
  if (batch > 65535) return TQ_EUNSUPPORTED;
  if (batch == 0 || n_q == 0 || n_k == 0) return TQ_OK;
  const int d = layer->d;
  float* q_rot = work;
  float* q_sk = work + batch * n_q * d;
  rc = tq_rotate_query(q, dtype, batch * n_q, layer, q_rot, q_sk, stream);
  if (rc) return rc;
  const int nt = score_query_tiles(batch, n_q, n_k);
  const bool words = (uintptr_t)idx % 4 == 0 && (uintptr_t)signs % 4 == 0;
  auto kern = words ? (nt == 2 ? score_kernel<false, 2> : score_kernel<false, 1>)
                    : (nt == 2 ? score_kernel<false, 2, true> : score_kernel<false, 1, true>);
  for (int64_t key0 = 0; key0 < n_k; key0 += SCORE_LAUNCH_KEYS) {
    const int64_t keys = std::min(n_k - key0, SCORE_LAUNCH_KEYS);
    const dim3 grid((unsigned)((keys + SCORE_KEYS - 1) / SCORE_KEYS), (unsigned)((n_q + 16 * nt - 1) / (16 * nt)), (unsigned)batch);
    kern<<<grid, dim3(256), 0, (hipStream_t)stream>>>(q_rot, q_sk, n_q, idx, signs, norms, norm_dtype, rnorms, n_k, key0, *layer, scores,
                                                      CacheTail{});
    TQ_CHECK_LAUNCH();
  }
  return TQ_OK;
}

extern "C" int tq_dequant_keys(const uint8_t* idx, const uint8_t* signs, const void* norms, int norm_dtype,
                               const float* rnorms, int64_t n_vec, const tq_layer* layer, float* out, void* stream) {
  int rc = check_layer_rd(layer, signs != nullptr);
  if (rc) return rc;
  if (!idx || !norms || !out) return TQ_ENULL;
  if (signs && !rnorms) return TQ_ENULL;
  if (n_vec < 0 || norm_dtype < TQ_F32 || norm_dtype > TQ_BF16) return TQ_EINVAL;
  if (n_vec == 0) return TQ_OK;
  hipStream_t st = (hipStream_t)stream;
  rc = tq::launch_dequant_mfma(idx, signs, norms, norm_dtype, rnorms, n_vec, *layer, out, st);
  if (rc != TQ_EUNSUPPORTED) return rc;
  // vector-ALU kernel: 32 vectors per workgroup while both LDS tiles fit (d <= 512), else 16
  const bool wide = layer->d <= 512;
  if (signs)
    return wide ? launch_dequant_keys<32, true>(idx, signs, norms, norm_dtype, rnorms, n_vec, layer, out, st)
                : launch_dequant_keys<16, true>(idx, signs, norms, norm_dtype, rnorms, n_vec, layer, out, st);
  return wide ? launch_dequant_keys<32, false>(idx, signs, norms, norm_dtype, rnorms, n_vec, layer, out, st)
              : launch_dequant_keys<16, false>(idx, signs, norms, norm_dtype, rnorms, n_vec, layer, out, st);
}

extern "C" int tq_dequant_values(const uint8_t* data, const void* scales, const void* zeros, int dtype, int64_t n_vec,
                                 int d, int group_size, int bits, float* out, void* stream) {
  if (!data || !scales || !zeros || !out) return TQ_ENULL;
  if (bits != 2 && bits != 4 && bits != 8) return TQ_EUNSUPPORTED;
  if (d <= 0 || group_size <= 0 || d % group_size || (d * bits) % 8 || n_vec < 0) return TQ_EINVAL;
  if (dtype < TQ_F32 || dtype > TQ_BF16) return TQ_EINVAL;
  if (n_vec == 0) return TQ_OK;
  hipStream_t st = (hipStream_t)stream;
  // chunks of 8 channels when they stay inside a group and the accesses are aligned
  const int cb = bits;                                          // bytes of codes per chunk
  if (d % 8 == 0 && group_size % 8 == 0 && (uintptr_t)data % cb == 0 && (uintptr_t)out % 16 == 0) {
    const int64_t chunks = n_vec * (d / 8);
    const dim3 grid((unsigned)((chunks + 255) / 256)), block(256);
    if (bits == 2) dequant_values8_kernel<2><<<grid, block, 0, st>>>(data, scales, zeros, dtype, n_vec, d, group_size, out);
    else if (bits == 4) dequant_values8_kernel<4><<<grid, block, 0, st>>>(data, scales, zeros, dtype, n_vec, d, group_size, out);
    else dequant_values8_kernel<8><<<grid, block, 0, st>>>(data, scales, zeros, dtype, n_vec, d, group_size, out);
    TQ_CHECK_LAUNCH();
    return TQ_OK;
  }
  int64_t total = n_vec * d;
  dequant_values_kernel<<<dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>(
      data, scales, zeros, dtype, n_vec, d, group_size, bits, out);
  TQ_CHECK_LAUNCH();
  return TQ_OK;
}

// ---- a step of the self-contained cache object (kv_cache.py:119-349): fp32 rows, one flat tensor per section --------
namespace tq {

// (values and copies of a token, behind the key quantiser's launch: one launch where a concatenation per section, and its host time, stood)
__global__ void __launch_bounds__(256) cache_rest_kernel(CacheRest A) { cache_rest_body(A, (int)blockIdx.x); }

int launch_cache_append(const float* keys, int64_t stride, int64_t rows, const tq_layer& ly, const KeyRowsSink& ks, const CacheRest& rest, hipStream_t st);

// Weighted sum of the values: a share of the compressed tokens, or 32 exact rows, per workgroup.  A thread owns one word of
// codes (32 / VB channels of one group) of every 256 / words-th token of the share; code * scale + zero rounds twice, as
// dequantize_values does, and meets its weight in fp32.  Bound by latency (32,768 tokens of 128: 2.4 MB): shares of 128 tokens.
constexpr int ATT_TOKENS = 128, ATT_ROWS = 32;
template <int VB>
__global__ void __launch_bounds__(256)
cache_attend_kernel(const float* __restrict__ w, int64_t n_q, const uint32_t* __restrict__ data, const float* __restrict__ scales,
                    const float* __restrict__ zeros, int n_c, int d, int gs, const float* __restrict__ v, int64_t s_b, int64_t s_h,
                    int64_t s_r, int H, int n_buf, int n_shares, float* __restrict__ part) {
  constexpr int CPW = 32 / VB;
  __shared__ float s_acc[256 * (CPW + 1)];
  const int tid = threadIdx.x, share = blockIdx.x;
  const int64_t bh = blockIdx.z, row = bh * n_q + blockIdx.y;
  const float* wr = w + row * (n_c + n_buf);
  float* out = part + (row * gridDim.x + share) * d;
  if (share < n_shares) {
    const int WR = d / CPW, ng = d / gs, col = tid % WR, t_in = tid / WR, RP = 256 / WR, g = col * CPW / gs;
    const int t1 = min((share + 1) * ATT_TOKENS, n_c);
    float acc[CPW];
#pragma unroll
    for (int e = 0; e < CPW; ++e) acc[e] = 0.0f;
#pragma unroll 4
    for (int t = share * ATT_TOKENS + t_in; t < t1; t += RP) {
      const int64_t tok = bh * n_c + t;
      const uint32_t x = data[tok * WR + col];
      const float sc = scales[tok * ng + g], z = zeros[tok * ng + g], wt = wr[t];
#pragma unroll
      for (int e = 0; e < CPW; ++e)
        acc[e] = fmaf(wt, __fadd_rn(__fmul_rn((float)((x >> (VB * e)) & ((1u << VB) - 1u)), sc), z), acc[e]);
    }
#pragma unroll
    for (int e = 0; e < CPW; ++e) s_acc[tid * (CPW + 1) + e] = acc[e];
    __syncthreads();
    if (tid < d) {
      float a = 0.0f;
      for (int r = 0; r < RP; ++r) a += s_acc[(r * WR + tid / CPW) * (CPW + 1) + tid % CPW];
      out[tid] = a;
    }
  } else {
    const int r0 = (share - n_shares) * ATT_ROWS, r1 = min(r0 + ATT_ROWS, n_buf), c = tid % d, sub = tid / d, RS = 256 / d;
    const float* vb = v + bh / H * s_b + bh % H * s_h + c;
    float a = 0.0f;
#pragma unroll 8
    for (int r = r0 + sub; r < r1; r += RS) a = fmaf(wr[n_c + r], vb[r * s_r], a);
    s_acc[tid] = a;
    __syncthreads();
    if (tid < d) {
      for (int k = 1; k < RS; ++k) a += s_acc[k * d + tid];
      out[tid] = a;
    }
  }
}

// (the shares of a row in order, sixteen requested at a time, also the last ones: 36 shares 4.0 -> 3.5 us)
constexpr int SUM_AHEAD = 16;
__global__ void cache_attend_sum_kernel(const float* __restrict__ part, int n, int d, float* __restrict__ out) {
  const int64_t row = blockIdx.x;
  const int c = threadIdx.x;
  float a = 0.0f;
  for (int s0 = 0; s0 < n; s0 += SUM_AHEAD) {
    float x[SUM_AHEAD];
#pragma unroll
    for (int k = 0; k < SUM_AHEAD; ++k) x[k] = part[(row * n + min(s0 + k, n - 1)) * d + c];
#pragma unroll
    for (int k = 0; k < SUM_AHEAD; ++k) a += s0 + k < n ? x[k] : 0.0f;      // (a is never -0)
  }
  out[row * d + c] = a;
}

static bool cache_dims(int64_t batch, int H, int d) { return batch > 0 && batch <= 65535 && H > 0 && batch % H == 0 && (d == 64 || d == 128 || d == 256); }

}  // namespace tq

extern "C" size_t tq_cache_append_bytes(int64_t batch, int d, int mse_bits, int value_bits, int group_size) {
  if (batch <= 0 || d <= 0 || mse_bits < 1 || mse_bits > 4 || value_bits <= 0 || group_size <= 0) return 0;
  // (the key's codes and norms, where two launches hand them on; a value's go straight to their place)
  return batch * ((size_t)idx_row_bytes(d, mse_bits) + d / 8 + 8) + 5 * 16;
}

extern "C" int tq_cache_append(const float* key, const float* value, int64_t key_stride, int64_t value_stride, const float* key_buf,
                               const float* value_buf, int64_t ks_b, int64_t ks_h, int64_t ks_r, int64_t vs_b, int64_t vs_h, int64_t vs_r, int64_t batch,
                               int H, int n_buf, const tq_layer* layer, int value_bits, int group_size, int64_t n_c,
                               const uint8_t* idx, const uint8_t* signs, const float* norms, const float* rnorms,
                               const uint8_t* data, const float* scales, const float* zeros, uint8_t* idx_out,
                               uint8_t* signs_out, float* norms_out, float* rnorms_out, uint8_t* data_out, float* scales_out,
                               float* zeros_out, float* key_buf_out, float* value_buf_out, void* work, void* stream) {
  if (!key || !value || !key_buf || !value_buf || !layer || !idx_out || !signs_out || !norms_out || !rnorms_out || !data_out ||
      !scales_out || !zeros_out || !key_buf_out || !value_buf_out || !work)
    return TQ_ENULL;
  const int d = layer->d;
  if (!cache_dims(batch, H, d) || n_buf < 1 || n_c < 0 || group_size < 16 || d % group_size || key_stride < d || value_stride < d) return TQ_EINVAL;
  if (value_bits != 2 && value_bits != 4 && value_bits != 8) return TQ_EUNSUPPORTED;
  // (lengths in bytes of a section's row are ints)
  if (n_c > (1 << 20) || n_buf > (1 << 20)) return TQ_EUNSUPPORTED;
  if (ks_r != d || vs_r != d || ks_h < d || vs_h < d) return TQ_EUNSUPPORTED;      // a buffer's rows lie one behind another
  if (batch != H && (ks_b != H * ks_h || vs_b != H * vs_h)) return TQ_EUNSUPPORTED;
  if (n_c > 0 && (!idx || !signs || !norms || !rnorms || !data || !scales || !zeros)) return TQ_ENULL;
  // (sections are copied in words; keys and values arrive as fp32)
  if (n_c > 0 && (((uintptr_t)idx | (uintptr_t)signs | (uintptr_t)norms | (uintptr_t)rnorms | (uintptr_t)data | (uintptr_t)scales | (uintptr_t)zeros) & 3))
    return TQ_EUNSUPPORTED;
  const int ng = d / group_size, ib = idx_row_bytes(d, layer->mse_bits), sb = d / 8, db = d * value_bits / 8;
  // the codes of the rows that leave the buffer
  uintptr_t at = ((uintptr_t)work + 15) & ~(uintptr_t)15;
  auto take = [&](size_t n) { const uintptr_t p = at; at += (n + 15) & ~(size_t)15; return p; };
  uint8_t* n_idx = (uint8_t*)take(batch * ib);
  uint8_t* n_sgn = (uint8_t*)take(batch * sb);
  float* n_nrm = (float*)take(batch * 4);
  float* n_rn = (float*)take(batch * 4);
  const int n = (int)n_c;
  CacheRest A;
  A.rows = (int)batch;
  A.v = value_buf; A.v_stride = vs_h;
  A.data = data_out + (size_t)n * db; A.scales = scales_out + (size_t)n * ng; A.zeros = zeros_out + (size_t)n * ng;
  A.step = n + 1;
  A.d = d; A.gs = group_size; A.bits = value_bits;
  auto section = [&](int i, const void* a, int64_t a_stride, int a_bytes, const void* b, int64_t b_stride, int b_bytes, void* dst, int64_t dst_stride) {
    A.s[i] = CopySection{(const uint8_t*)a, (const uint8_t*)b, (uint8_t*)dst, a_stride, b_stride, dst_stride, a_bytes, b_bytes, 0};
  };
  section(0, data, (int64_t)n * db, n * db, nullptr, 0, 0, data_out, (int64_t)(n + 1) * db);
  section(1, scales, (int64_t)n * ng * 4, n * ng * 4, nullptr, 0, 0, scales_out, (int64_t)(n + 1) * ng * 4);
  section(2, zeros, (int64_t)n * ng * 4, n * ng * 4, nullptr, 0, 0, zeros_out, (int64_t)(n + 1) * ng * 4);
  section(3, key_buf + d, ks_h * 4, (n_buf - 1) * d * 4, key, key_stride * 4, d * 4, key_buf_out, (int64_t)n_buf * d * 4);
  section(4, value_buf + d, vs_h * 4, (n_buf - 1) * d * 4, value, value_stride * 4, d * 4, value_buf_out, (int64_t)n_buf * d * 4);
  // the key's sections, with the codes from `work` behind them or (alone) without
  auto key_sections = [&](bool with_codes) {
    section(5, idx, (int64_t)n * ib, n * ib, with_codes ? n_idx : nullptr, ib, with_codes ? ib : 0, idx_out, (int64_t)(n + 1) * ib);
    section(6, signs, (int64_t)n * sb, n * sb, with_codes ? n_sgn : nullptr, sb, with_codes ? sb : 0, signs_out, (int64_t)(n + 1) * sb);
    section(7, norms, (int64_t)n * 4, n * 4, with_codes ? n_nrm : nullptr, 4, with_codes ? 4 : 0, norms_out, (int64_t)(n + 1) * 4);
    section(8, rnorms, (int64_t)n * 4, n * 4, with_codes ? n_rn : nullptr, 4, with_codes ? 4 : 0, rnorms_out, (int64_t)(n + 1) * 4);
    A.copies = 0;
    for (auto& c : A.s) {
      c.first = A.copies;
      A.copies += copy_workgroups(c, batch);
    }
    return A.copies <= 1 << 23;                  // (a grid counts fewer than 2^32 threads)
  };
  int rc = check_layer_rd(layer, true);
  if (rc) return rc;
  if (!layer->thresholds) return TQ_ENULL;
  if (!key_sections(false)) return TQ_EUNSUPPORTED;
  const KeyRowsSink ks{{idx_out + (size_t)n * ib, signs_out + (size_t)n * sb, norms_out + n, rnorms_out + n, nullptr, nullptr}, (int64_t)n + 1};
  rc = launch_cache_append(key_buf, ks_h, batch, *layer, ks, A, (hipStream_t)stream);
  if (rc != TQ_EUNSUPPORTED) return rc;
  if (!key_sections(true)) return TQ_EUNSUPPORTED;
  rc = tq_quantize_keys(key_buf, TQ_F32, batch, ks_h, layer, n_idx, n_sgn, n_nrm, n_rn, nullptr, nullptr, 0, stream);
  if (rc) return rc;
  cache_rest_kernel<<<dim3((unsigned)(A.rows + A.copies)), dim3(256), 0, (hipStream_t)stream>>>(A);
  TQ_CHECK_LAUNCH();
  return TQ_OK;
}

extern "C" int tq_cache_scores_rows(const float* q, int64_t q_row, int64_t batch, int H, int64_t n_q, const uint8_t* idx, const uint8_t* signs,
                               const float* norms, const float* rnorms, int64_t n_c, const tq_layer* layer, const float* key_buf,
                               int64_t s_b, int64_t s_h, int64_t s_r, int n_buf, float scale, float* scores, float* work,
                               void* stream) {
  int rc = check_layer_rd(layer, true);
  if (rc) return rc;
  if (!q || !idx || !signs || !norms || !rnorms || !key_buf || !scores || !work) return TQ_ENULL;
  const int d = layer->d;
  if (!cache_dims(batch, H, d) || n_q <= 0 || n_c <= 0 || n_buf <= 0) return TQ_EINVAL;
  if (((uintptr_t)idx | (uintptr_t)signs) & 3 || n_c > SCORE_LAUNCH_KEYS || n_q > (1 << 18) || n_buf > (1 << 24)) return TQ_EUNSUPPORTED;
  if (q_row < d) return TQ_EINVAL;
  float* q_rot = work;
  float* q_sk = work + batch * n_q * d;
  rc = launch_rotate_query(q, TQ_F32, batch * n_q, layer, q_rot, q_sk, nullptr, nullptr, 1, 0.0f, (hipStream_t)stream, false, nullptr, nullptr, 0,
                           nullptr, SplitPlan{}, q_row);
  if (rc) return rc;
  const CacheTail tail{q, q_row, key_buf, s_b, s_h, s_r, H, n_buf, scale};
  const int nt = score_query_tiles(batch, n_q, n_c);
  const dim3 grid((unsigned)((n_c + SCORE_KEYS - 1) / SCORE_KEYS + (n_buf + SCORE_ROWS - 1) / SCORE_ROWS), (unsigned)((n_q + 16 * nt - 1) / (16 * nt)),
                  (unsigned)batch);
  auto kern = nt == 2 ? score_kernel<true, 2> : score_kernel<true, 1>;
  kern<<<grid, dim3(256), 0, (hipStream_t)stream>>>(
      q_rot, q_sk, n_q, idx, signs, norms, TQ_F32, rnorms, n_c, 0, *layer, scores, tail);
  TQ_CHECK_LAUNCH();
  return TQ_OK;
}

extern "C" int tq_cache_scores(const float* q, int64_t batch, int H, int64_t n_q, const uint8_t* idx, const uint8_t* signs,
                               const float* norms, const float* rnorms, int64_t n_c, const tq_layer* layer, const float* key_buf,
                               int64_t s_b, int64_t s_h, int64_t s_r, int n_buf, float scale, float* scores, float* work,
                               void* stream) {
  return tq_cache_scores_rows(q, layer ? layer->d : 0, batch, H, n_q, idx, signs, norms, rnorms, n_c, layer, key_buf, s_b, s_h, s_r, n_buf, scale,
                              scores, work, stream);
}

extern "C" size_t tq_cache_attend_bytes(int64_t batch, int64_t n_q, int d, int64_t n_c, int n_buf) {
  if (batch <= 0 || n_q <= 0 || d <= 0 || n_c < 0 || n_buf < 0) return 0;
  return (size_t)batch * n_q * d * sizeof(float) * ((n_c + ATT_TOKENS - 1) / ATT_TOKENS + (n_buf + ATT_ROWS - 1) / ATT_ROWS);
}

extern "C" int tq_cache_attend(const float* weights, int64_t batch, int H, int64_t n_q, const uint8_t* data, const float* scales,
                               const float* zeros, int64_t n_c, int d, int group_size, int value_bits, const float* value_buf,
                               int64_t s_b, int64_t s_h, int64_t s_r, int n_buf, float* out, float* work, void* stream) {
  if (!weights || !data || !scales || !zeros || !value_buf || !out || !work) return TQ_ENULL;
  if (!cache_dims(batch, H, d) || n_q <= 0 || n_c <= 0 || n_buf <= 0 || group_size < 16 || d % group_size) return TQ_EINVAL;
  if (group_size % 16 || ((uintptr_t)data & 3) || n_c > (1 << 28) || n_q > 65535 || n_buf > (1 << 24)) return TQ_EUNSUPPORTED;
  const int shares = (int)((n_c + ATT_TOKENS - 1) / ATT_TOKENS), all = shares + (n_buf + ATT_ROWS - 1) / ATT_ROWS;
  const dim3 grid((unsigned)all, (unsigned)n_q, (unsigned)batch);
#define TQ_ATTEND(VB)                                                                                                   \
  cache_attend_kernel<VB><<<grid, dim3(256), 0, (hipStream_t)stream>>>(weights, n_q, (const uint32_t*)data, scales, zeros, \
                                                                       (int)n_c, d, group_size, value_buf, s_b, s_h, s_r, H, n_buf, \
                                                                       shares, work)
  if (value_bits == 2) TQ_ATTEND(2);
  else if (value_bits == 4) TQ_ATTEND(4);
  else if (value_bits == 8) TQ_ATTEND(8);
  else return TQ_EUNSUPPORTED;
#undef TQ_ATTEND
  TQ_CHECK_LAUNCH();
  cache_attend_sum_kernel<<<dim3((unsigned)(batch * n_q)), dim3(d), 0, (hipStream_t)stream>>>(work, all, d, out);
  TQ_CHECK_LAUNCH();
  return TQ_OK;
}
