// Key quantiser on the matrix cores (gfx950, bf16 MFMA 16x16x32) for the head sizes that tq_quantize_mfma.hip has no
// instantiation for: any multiple of 64 up to 768 whose terms fit the LDS, the size being a run-time number.
//
// Arithmetic as there: every fp32 number is the exact sum of three bf16 terms, the three d x d contractions of the
// reference (quantizer.py:141,160,248) are assembled from bf16 products with fp32 accumulation, and the pairs of terms
// (a, b) with a + b > 2, which are below fp32 resolution, are left out.
//
// What bounds it: nothing alone.  A workgroup reads all three matrices - three terms each, 6.8 MB at d = 576 with what it
// reads twice - for every group of vectors, at the 64 bytes per clock that a compute unit takes from L2 (44 us), beside 32 us of
// MFMA and about 26 us of vector instructions for 32 vectors; these overlap within a contraction and not across its ends, where
// all wavefronts meet, and the contractions are three fifths of the kernel's time.  Hence the widest group whose terms fit the LDS
// (32 vectors: 3 x 32 x 1168 bytes at d = 576), one workgroup of up to 12 wavefronts per compute unit, each of which
// owns NPW column tiles for all vectors, and a ring of two slices per wavefront (2 x NPW x 3 KB) that is refilled while the
// other slice is multiplied - from the second contraction into the third across its end, so that the first slices of S are
// there when it begins; behind the first and the third, where single coordinates may be summed again, it is filled anew (kept
// through those sums it spills: 116 - 130 us where 88 were measured without them).
// The codes are those of the vector-ALU kernel, byte for byte: what rounding could decide is summed again in its order (see
// KW_NEAR_Y).
// Appends of 8192 vectors of 576, bf16, 4-bit keys: 404 us on the vector-ALU kernel, 118 us here; one token of each of 32
// sequences 181 -> 74 us; 8192 x 320: 129 -> 48, x 704: 515 -> 172.

#include <atomic>

#include "tq_key_mfma.h"
#include "tq_decode_mfma.h"
#include "tq_options.h"
#include <hip/hip_ext.h>

namespace tq {

constexpr int KW_MAX_WAVES = 12;

// LDS of a workgroup, in bytes from its start
struct WideSmem {
  int rs;                                  // row stride of a term tile in bf16: 4 banks (mod 64) from row to row
  int off_planes, off_off, off_small, bytes;
  __host__ __device__ WideSmem(int d, int mb, int tt, int waves) {
    rs = d + 8;
    off_planes = 3 * tt * rs * 2;                              // term tiles [3][tt][rs]
    off_off = off_planes + (mb + 1) * tt * (d / 32) * 4;       // bit planes [plane][tt][d / 32]
    off_small = off_off + tt * 8;                              // element offset of every vector
    // norm[tt], residual norm[tt], partial sums[waves][tt], validity[tt], thresholds between -inf and +inf[18], centroid
    // terms[16] (8 bytes each), vectors with a projection near zero[2]
    bytes = off_small + tt * (3 + waves) * 4 + 18 * 4 + 16 * 8 + 2 * 4;
  }
};

template <int NPW>
struct WideRing { u32x4 b[2][NPW][3]; };

// One slice of 32 contraction indices of a matrix for the wavefront's column tiles (term matrices in MFMA operand
// order: a wavefront's load of one operand is one contiguous kilobyte).
template <int NPW>
__device__ __forceinline__ void load_wide_slice(const uint16_t* m_terms, int ct0, int tiles, int kb_n, int kblk, uint32_t lane_off,
                                                u32x4 (&dst)[NPW][3]) {
#pragma unroll
  for (int c = 0; c < NPW; ++c)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      const char* base = (const char*)m_terms + ((size_t)(b * tiles + ct0 + c) * kb_n + kblk) * 1024;
      dst[c][b] = *(const u32x4*)(base + lane_off);
    }
}

template <int NPW>
__device__ __forceinline__ void fill_ring(const uint16_t* m_terms, int ct0, int tiles, int kb_n, int lane, WideRing<NPW>& ring) {
  load_wide_slice<NPW>(m_terms, ct0, tiles, kb_n, 0, lane * 16, ring.b[0]);
  load_wide_slice<NPW>(m_terms, ct0, tiles, kb_n, 1, lane * 16, ring.b[1]);
}

// One slice of a contraction for the wavefront's column tiles
template <int NPW, int MT, int NA>
__device__ __forceinline__ void multiply_slice(const uint16_t* a_lane, int rs, int kblk, const u32x4 (&b)[NPW][3], f32x4 (&acc)[MT][NPW]) {
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    u32x4 av[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) av[m] = *(const u32x4*)(a_lane + (a * 16 * MT + 16 * m) * rs + 32 * kblk);
#pragma unroll
    for (int t = 0; t < 3; ++t)
      if (a + t <= 2) {
#pragma unroll
        for (int c = 0; c < NPW; ++c)                           // consecutive MFMAs go to different accumulators
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m][c] = mfma_bf16(b[c][t], av[m], acc[m][c]);
      }
  }
}

// out[t][n] = sum_k A[t][k] M[n][k] for the wavefront's column tiles; the ring holds slices 0 and 1 of M on entry and, if
// NEXT, of m_next on return.  acc[m][c][i] = out[16 m + (lane & 15)][16 (ct0 + c) + 4 (lane >> 4) + i].
template <int NPW, int MT, int NA, bool NEXT>
__device__ __forceinline__ void contract_wide(const uint16_t* a_terms, int rs, const uint16_t* m_terms, const uint16_t* m_next,
                                              int ct0, int tiles, int kb_n, int lane, WideRing<NPW>& ring, f32x4 (&acc)[MT][NPW]) {
  const uint16_t* a_lane = a_terms + (lane & 15) * rs + 8 * (lane >> 4);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int c = 0; c < NPW; ++c) acc[m][c] = f32x4{0, 0, 0, 0};
#pragma unroll 1
  for (int k2 = 0; k2 < kb_n - (NEXT ? 0 : 2); k2 += 2) {       // (d is a multiple of 64: an even number of slices)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      multiply_slice<NPW, MT, NA>(a_lane, rs, k2 + h, ring.b[h], acc);
      const int next = k2 + h + 2;
      const bool over = NEXT && next >= kb_n;
      load_wide_slice<NPW>(over ? m_next : m_terms, ct0, tiles, kb_n, over ? next - kb_n : next, lane * 16, ring.b[h]);
    }
  }
  if constexpr (!NEXT) {
#pragma unroll
    for (int h = 0; h < 2; ++h) multiply_slice<NPW, MT, NA>(a_lane, rs, kb_n - 2 + h, ring.b[h], acc);
  }
}

// ---- sums in the order of the vector-ALU kernel ---------------------------------------------------------------------------

// 16 consecutive numbers of a vector in the LDS: NA bf16 terms, term_stride apart (their sum, smallest first, is exact) ...
template <int NA>
struct TermRow {
  const uint16_t* p;
  int term_stride;
  __device__ __forceinline__ void get(int j, float (&u)[16]) const {
#pragma unroll
    for (int a = NA - 1; a >= 0; --a)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4 v = *(const u32x4*)(p + a * term_stride + j + 8 * h);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float f = __uint_as_float((e & 1) ? v[e >> 1] & 0xffff0000u : v[e >> 1] << 16);
          u[8 * h + e] = a == NA - 1 ? f : u[8 * h + e] + f;
        }
      }
  }
};
// ... or fp32
struct FloatRow {
  const float* p;
  __device__ __forceinline__ void get(int j, float (&u)[16]) const {
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      const f32x4 v = *(const f32x4*)(p + j + e);
      u[e] = v.x; u[e + 1] = v.y; u[e + 2] = v.z; u[e + 3] = v.w;
    }
  }
};

// sum = fma(u[e], m of element 16 Q + e, sum) for e = 0 .. 15 in turn; lane i of a DPP row holds elements 4 i .. 4 i + 3 and its
// row's lanes read them through the row broadcast.  (A register that a VALU instruction wrote may be read through DPP
// two instructions later, which the compiler does not see inside assembly: hence the s_nop.)
template <int Q>
__device__ __forceinline__ void ordered_steps(const float (&u)[16], const f32x4& m, float& sum) {
#define TQ_STEP(M, U, L) "\n\tv_fmac_f32_dpp %0, %" #M ", %" #U " row_newbcast:%" #L " row_mask:0xf bank_mask:0xf"
  asm("s_nop 1"
      TQ_STEP(1, 5, 21) TQ_STEP(2, 6, 21) TQ_STEP(3, 7, 21) TQ_STEP(4, 8, 21)
      TQ_STEP(1, 9, 22) TQ_STEP(2, 10, 22) TQ_STEP(3, 11, 22) TQ_STEP(4, 12, 22)
      TQ_STEP(1, 13, 23) TQ_STEP(2, 14, 23) TQ_STEP(3, 15, 23) TQ_STEP(4, 16, 23)
      TQ_STEP(1, 17, 24) TQ_STEP(2, 18, 24) TQ_STEP(3, 19, 24) TQ_STEP(4, 20, 24)
      : "+v"(sum)
      : "v"(m.x), "v"(m.y), "v"(m.z), "v"(m.w), "v"(u[0]), "v"(u[1]), "v"(u[2]), "v"(u[3]), "v"(u[4]), "v"(u[5]), "v"(u[6]),
        "v"(u[7]), "v"(u[8]), "v"(u[9]), "v"(u[10]), "v"(u[11]), "v"(u[12]), "v"(u[13]), "v"(u[14]), "v"(u[15]),
        "n"(4 * Q), "n"(4 * Q + 1), "n"(4 * Q + 2), "n"(4 * Q + 3));
#undef TQ_STEP
}
// sum_j u[j] row[j], the products added one by one in ascending order: the bits of the vector-ALU kernel.  The 16 lanes of a DPP
// row share one matrix row, requested three times 64 elements ahead (the fp32 matrices are in no cache), and every lane
// has a vector of its own.  All lanes of the wavefront have to be active.
template <class U>
__device__ __forceinline__ float ordered_dot(const U& vec, const float* __restrict__ row, int d, int n) {
  const f32x4* run = (const f32x4*)row + n;
  f32x4 ahead[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) ahead[q] = run[min(64 * q, d - 64) / 4];
  float sum = 0.0f;
#pragma unroll 1
  for (int j0 = 0; j0 < d; j0 += 64) {
    const f32x4 cur = ahead[0];
    ahead[0] = ahead[1];
    ahead[1] = ahead[2];
    ahead[2] = run[min(j0 + 192, d - 64) / 4];
    float u[16];
    vec.get(j0, u); ordered_steps<0>(u, cur, sum);
    vec.get(j0 + 16, u); ordered_steps<1>(u, cur, sum);
    vec.get(j0 + 32, u); ordered_steps<2>(u, cur, sum);
    vec.get(j0 + 48, u); ordered_steps<3>(u, cur, sum);
  }
  return sum;
}

// `bits` of the first lane of this lane's DPP row that has any (`open`: the lanes that do); 0 if none has.
__device__ __forceinline__ uint32_t leader_bits(uint32_t bits, uint64_t open, int lane) {
  const uint32_t row = (uint32_t)(open >> (lane & 48)) & 0xffffu;
  const uint32_t got = __shfl(bits, (lane & 48) + (row ? __builtin_ctz(row) : 0), 64);
  return row ? got : 0u;
}

// How near to a threshold a coordinate of the unit vector, and how near to zero a projection of the residual, is decided by the
// sums in the order of the vector-ALU kernel, so that a row gets that kernel's codes whatever its alignment and its batch: an
// index that falls the other way takes a quarter of the vector's signs with it, and what is attended to changes.  The two orders
// come apart by 2.1e-8 in the root mean square (coordinates; relative to the vector's length) and by 2.4e-8 (projections; relative to
// sqrt(d) times it); the margins are eleven and five times that.  Over 65536 vectors of each of eight sizes 64 .. 768,
// three types and four distributions (Gaussian, ten-fold channels, one spike, off-centre) no code differs, where without
// them one index in about 3000 vectors of 576 did.  Residual norms agree to 1e-6.
// What it costs, 8192 vectors of 576: 85.8 -> 112 us (nothing near anything 94, indices 95: a pass over fp32 Pi, 16 us, by the
// workgroups that have a projection near zero - one group of 32 in five).
constexpr float KW_NEAR_Y = 0x1p-22f, KW_NEAR_P = 0x1p-23f;
constexpr int KW_REDO = 2;                 // vectors whose residual is computed again at a time (more: bound by the LDS reads)

template <int DT, int NPW, int MT, class Source, class Sink>
__global__ void __launch_bounds__(KW_MAX_WAVES * 64, NPW == 1 ? 4 : 3)       // (head_dim 64: four workgroups of four wavefronts)
key_wide_kernel(const void* __restrict__ x, Source src, tq_layer ly, Sink sink, int64_t n_tiles, int mse_only) {
  using E = Elem<DT>;
  using S = typename E::storage;
  constexpr int TT = 16 * MT, NA1 = InTerms<DT>::N;
  constexpr int JX = 3 * NPW;                                   // chunks of 4 x 16 coordinates: d <= 12 * 16 * NPW
  constexpr bool paged = std::is_same<Sink, KeyPagedSink>::value;
  const int d = ly.d, mb = ly.mse_bits, n_thr = (1 << mb) - 1;
  const int W = d >> 5, tiles = d >> 4, kb_n = d >> 5;
  const int tid0 = threadIdx.x, wave0 = __builtin_amdgcn_readfirstlane(tid0 >> 6);
  const int waves = blockDim.x >> 6, nthreads = blockDim.x;
  WideRing<NPW> ring;
  fill_ring<NPW>(ly.Pi_split, wave0 * NPW, tiles, kb_n, tid0 & 63, ring);

  extern __shared__ __align__(16) unsigned char smem[];
  const WideSmem sm(d, mb, TT, waves);
  const int rs = sm.rs;
  uint16_t* terms = (uint16_t*)smem;                            // unit vector, then centroids, then residual
  uint32_t* spl = (uint32_t*)(smem + sm.off_planes);
  int64_t* soff = (int64_t*)(smem + sm.off_off);
  float* snorm = (float*)(smem + sm.off_small);
  float* srn = snorm + TT;
  float* spart = srn + TT;
  int* svalid = (int*)(spart + waves * TT);
  float* sthr = (float*)(svalid + TT);
  u32x2* slut = (u32x2*)(sthr + 18);                            // bf16 terms of a centroid: {t0 | t1 << 16, t2}
  if (tid0 < n_thr) sthr[tid0 + 1] = ly.thresholds[tid0];       // (index i lies between sthr[i] and sthr[i + 1])
  if (tid0 < 2) sthr[tid0 * (n_thr + 1)] = tid0 ? INFINITY : -INFINITY;
  uint32_t* sopen = (uint32_t*)(slut + 16);
  if (tid0 < (1 << mb)) {
    uint32_t t[3];
    split3_pk(ly.centroids[tid0], 0.0f, t);
    slut[tid0] = u32x2{(t[0] & 0xffffu) | (t[1] << 16), t[2] & 0xffffu};
  }
  // runs of different lengths: only the pages that they touch are numbered (index behind the fixed part of the LDS)
  int* cum = (int*)(smem + sm.bytes);
  if constexpr (paged) {
    if (src.compact) {
      RaggedSource rg;
      static_cast<PagedSource&>(rg) = src;
      rg.template page_index<256>(cum, cum + src.B + 1, tid0);
      n_tiles = (int64_t)__builtin_amdgcn_readfirstlane(cum[src.B]) * src.H;
    }
  }
  // where a tile's rows are, and (pages) which logical page and head it is; the tile number is uniform over a wavefront
  auto look_up = [&](int64_t tile, TileAddr& ta, int& b, int& lpage, int& h) {
    if constexpr (paged) {
      PagedSource::Coord c[1];
      if (src.compact) {
        RaggedSource rg;
        static_cast<PagedSource&>(rg) = src;
        c[0] = rg.coord(tile, cum, tid0 & 63);
      } else {
        c[0] = src.coord(tile);
      }
      TileAddr t1[1];
      int lp[1];
      src.template tile_addrs<1>(c, t1, lp);
      ta = t1[0];
      b = c[0].b;
      lpage = lp[0];
      h = c[0].h;
    } else {
      ta = src.tile_addr(tile);
      b = lpage = h = 0;
    }
  };

  const int64_t n_groups = (n_tiles + MT - 1) / MT;
  for (int64_t g = blockIdx.x; g < n_groups; g += gridDim.x) {
    const int64_t tile0 = g * MT;
    // (re-read through an opaque copy in every pass: otherwise the per-thread address arithmetic is hoisted and spilled)
    int tid = tid0, wave = wave0;
    asm volatile("" : "+v"(tid), "+s"(wave));
    const int lane = tid & 63, n = lane & 15, kb = lane >> 4, ct0 = wave * NPW;
    if (tid < 2) sopen[tid] = 0;
    // (1) norm, unit vector in the input dtype (quantizer.py:136-138) and its bf16 terms: 16 lanes per vector, which
    //     hold all of it, four coordinates per lane and chunk
#pragma unroll 1
    for (int t4 = wave; t4 < TT / 4; t4 += waves) {
      const int64_t tile = tile0 + (t4 >> 2);
      TileAddr ta;
      int b, lpage, h;
      look_up(tile < n_tiles ? tile : n_tiles - 1, ta, b, lpage, h);
      const int t = 4 * t4 + kb, slot = t & 15;
      const bool ok = tile < n_tiles && slot >= ta.lo && slot < ta.hi;
      const int64_t off = ok ? ta.base + slot * src.slot_stride() : 0;       // (absent slots read the first vector)
      float xs[JX][4];
#pragma unroll
      for (int j = 0; j < JX; ++j)
        if (j < kb_n / 2) {
          load_run<DT, 4>((const S*)x + off + 64 * j + 4 * n, xs[j]);
#pragma unroll
          for (int i = 0; i < 4; ++i) xs[j][i] = ok ? xs[j][i] : 0.0f;
        }
      // The squares are added in the order of the vector-ALU kernel (coordinates 64 apart in turn, then a butterfly over the
      // 64 sums): a 16-bit norm that meets a rounding tie would else come out a step apart, and the unit vector, a handful of
      // indices and a quarter of the signs with it.  (Rotations by 8, 4, 2, 1 lanes are the butterfly's exchanges.)
      float sq[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < JX; ++j)
        if (j < kb_n / 2) {
#pragma unroll
          for (int i = 0; i < 4; ++i) sq[i] += xs[j][i] * xs[j][i];
        }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sq[i] += dpp_mov<0x128>(sq[i]);
        sq[i] += dpp_mov<0x124>(sq[i]);
        sq[i] += dpp_mov<0x122>(sq[i]);
        sq[i] += dpp_mov<0x121>(sq[i]);
      }
      const float ss = (sq[0] + sq[2]) + (sq[1] + sq[3]);
      const float nrm = E::round(sqrtf(ss));
      const float den = E::round(nrm + 1e-10f);
      if (n == 0) {
        snorm[t] = nrm;
        svalid[t] = ok;
        soff[t] = off;
      }
      // (quotients of bf16 numbers: a product with the reciprocal and one residual correction rounds like the division
      // inside this range; see the kernel of head_dim 128 / 256)
      const bool fast = DT == TQ_BF16 && den > 0x1p-60f && den < 0x1p60f;
      const float rden = __builtin_amdgcn_rcpf(den);
#pragma unroll
      for (int j = 0; j < JX; ++j)
        if (j < kb_n / 2) {
          float u[4];
          if (fast) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float q0 = xs[j][i] * rden;
              u[i] = fmaf(fmaf(-q0, den, xs[j][i]), rden, q0);
            }
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] = xs[j][i] / den;
          }
          uint16_t* dst = terms + t * rs + 64 * j + 4 * n;
          if constexpr (DT == TQ_BF16) {
            *(u32x2*)dst = u32x2{cvt_pk_bf16(u[0], u[1]), cvt_pk_bf16(u[2], u[3])};
          } else {
            uint32_t lo[3], hi[3];
            split3_pk(E::round(u[0]), E::round(u[1]), lo);
            split3_pk(E::round(u[2]), E::round(u[3]), hi);
#pragma unroll
            for (int a = 0; a < NA1; ++a) *(u32x2*)(dst + a * TT * rs) = u32x2{lo[a], hi[a]};
          }
        }
    }
    __syncthreads();

    f32x4 acc[MT][NPW];
    // (2) y = u Pi^T, bucketise: index bit planes and the centroids' bf16 terms
    // (the next matrix is asked for when the indices are settled: what that takes would push its operands out of the registers)
    contract_wide<NPW, MT, NA1, false>(terms, rs, ly.Pi_split, nullptr, ct0, tiles, kb_n, lane, ring, acc);
    uint32_t codes[MT][NPW];                                    // four indices, a byte each
    uint32_t near = 0;                                          // coordinates that lie on a threshold within rounding
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const float nrm = snorm[16 * m + n];
      const float margin = svalid[16 * m + n] ? KW_NEAR_Y * (nrm / E::round(nrm + 1e-10f)) : 0.0f;
#pragma unroll
      for (int c = 0; c < NPW; ++c) {
        int idx[4] = {0, 0, 0, 0};
#pragma unroll 1
        for (int k = 1; k <= n_thr; ++k) {                      // searchsorted: count thresholds below y (NaN counts all)
          const float th = sthr[k];
#pragma unroll
          for (int i = 0; i < 4; ++i) idx[i] += !(acc[m][c][i] <= th);
        }
        codes[m][c] = idx[0] | idx[1] << 8 | idx[2] << 16 | idx[3] << 24;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float y = acc[m][c][i], lo = sthr[idx[i]], hi = sthr[idx[i] + 1];
          near |= (uint32_t)(fminf(y - lo, hi - y) < margin) << ((m * NPW + c) * 4 + i);
        }
      }
    }
    // Those coordinates (one vector in a hundred has one): a DPP row of lanes works on one matrix row at a time, for all of
    // its 16 vectors.
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(near != 0) != 0, 0))
    while (const uint64_t open = __builtin_amdgcn_ballot_w64(near != 0)) {
      const uint32_t first = leader_bits(near, open, lane);
      const int bit = first ? __builtin_ctz(first) : 0, i = bit & 3, mc = bit >> 2, m = mc / NPW, c = mc % NPW;
      const float y = ordered_dot(TermRow<NA1>{terms + (16 * m + n) * rs, TT * rs},
                                  ly.Pi + (size_t)(16 * (ct0 + c) + 4 * kb + i) * d, d, n);
      uint32_t code = 0;
#pragma unroll 1
      for (int k = 1; k <= n_thr; ++k) code += !(y <= sthr[k]);
      const bool mine = near >> bit & 1;
      near &= ~((uint32_t)mine << bit);
#pragma unroll
      for (int o = 0; o < MT * NPW; ++o) {
        const bool here = mine && o == mc;
        const uint32_t old = codes[o / NPW][o % NPW];
        codes[o / NPW][o % NPW] = here ? (old & ~(0xffu << 8 * i)) | code << 8 * i : old;
        if constexpr (!paged) {
#pragma unroll
          for (int i2 = 0; i2 < 4; ++i2) acc[o / NPW][o % NPW][i2] = here && i2 == i ? y : acc[o / NPW][o % NPW][i2];
        }
      }
    }
    fill_ring<NPW>(mse_only ? ly.Pi_split : ly.PiT_split, ct0, tiles, kb_n, lane, ring);
    __syncthreads();                                            // every wavefront has read the unit-vector terms
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int t = 16 * m + n;
#pragma unroll
      for (int c = 0; c < NPW; ++c) {
        const int ct = ct0 + c, col0 = 16 * ct + 4 * kb;
        if constexpr (!paged) {
          if (sink.y_dbg && svalid[t]) *(f32x4*)(sink.y_dbg + (tile0 * TILE + t) * d + col0) = acc[m][c];
        }
        int idx[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) idx[i] = codes[m][c] >> 8 * i & 0xff;
        // a column tile is half a plane word
#pragma unroll 1
        for (int p = 0; p < mb; ++p) {
          uint32_t v = 0;
#pragma unroll
          for (int i = 0; i < 4; ++i) v |= (uint32_t)((idx[i] >> (mb - 1 - p)) & 1) << (4 * kb + i);
          v = or_over_kb(v);
          if (kb == 0) ((uint16_t*)spl)[(p * TT + t) * (2 * W) + ct] = (uint16_t)v;
        }
        u32x2 e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = slut[idx[i]];
        uint16_t* dst = terms + t * rs + col0;
        *(u32x2*)dst = u32x2{(e[0].x & 0xffffu) | (e[1].x << 16), (e[2].x & 0xffffu) | (e[3].x << 16)};
        *(u32x2*)(dst + TT * rs) = u32x2{(e[0].x >> 16) | (e[1].x & 0xffff0000u), (e[2].x >> 16) | (e[3].x & 0xffff0000u)};
        *(u32x2*)(dst + 2 * TT * rs) = u32x2{e[0].y | (e[1].y << 16), e[2].y | (e[3].y << 16)};
      }
    }
    __syncthreads();
    if (!mse_only) {
      // (3) x_hat = (c Pi) * norm ; r = x - x_hat ; ||r||^2 ; r as bf16 terms (quantizer.py:241-245)
      contract_wide<NPW, MT, 3, true>(terms, rs, ly.PiT_split, ly.S_split, ct0, tiles, kb_n, lane, ring, acc);
      __syncthreads();                                          // every wavefront has read the centroid terms
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int t = 16 * m + n;
        const float nrm = snorm[t];
        const S* xrow = (const S*)x + soff[t];
        const bool ok = svalid[t];
        float sq = 0.0f;
#pragma unroll
        for (int c = 0; c < NPW; ++c) {
          const int col0 = 16 * (ct0 + c) + 4 * kb;
          float r[4], xv[4];
          load_run<DT, 4>(xrow + col0, xv);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float xh = acc[m][c][i] * nrm;
            r[i] = (ok ? xv[i] : 0.0f) - xh;
            sq += r[i] * r[i];
          }
          uint32_t lo[3], hi[3];
          split3_pk(r[0], r[1], lo);
          split3_pk(r[2], r[3], hi);
#pragma unroll
          for (int a = 0; a < 3; ++a) *(u32x2*)(terms + (a * TT + t) * rs + col0) = u32x2{lo[a], hi[a]};
        }
        sq = sum_over_kb(sq);
        if (kb == 0) spart[wave * TT + t] = sq;
      }
      __syncthreads();
      if (tid < TT) {
        float v = 0.0f;
        for (int w = 0; w < waves; ++w) v += spart[w * TT + tid];
        srn[tid] = sqrtf(v);
      }
      // (4) p = r S^T ; sign bits (quantizer.py:248-249)
      contract_wide<NPW, MT, 3, false>(terms, rs, ly.S_split, nullptr, ct0, tiles, kb_n, lane, ring, acc);
      uint32_t near_p = 0;
      const float near_scale = KW_NEAR_P * sqrtf((float)d);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int t = 16 * m + n;
        const float margin = svalid[t] ? near_scale * snorm[t] : 0.0f;
        const uint32_t before = near_p;
#pragma unroll
        for (int c = 0; c < NPW; ++c) {
          const int ct = ct0 + c;
          uint32_t v = 0;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v |= (uint32_t)(acc[m][c][i] > 0.0f) << (4 * kb + i);
            near_p |= (uint32_t)(fabsf(acc[m][c][i]) < margin) << ((m * NPW + c) * 4 + i);
          }
          v = or_over_kb(v);
          if (kb == 0) ((uint16_t*)spl)[(mb * TT + t) * (2 * W) + ct] = (uint16_t)v;
          if constexpr (!paged) {
            if (sink.p_dbg && svalid[t]) *(f32x4*)(sink.p_dbg + (tile0 * TILE + t) * d + 16 * ct + 4 * kb) = acc[m][c];
          }
        }
        if (near_p != before) atomicOr(sopen + (t >> 5), 1u << (t & 31));
      }
      __syncthreads();
      // Projections that are zero within rounding: the vector's residual is computed again in the vector-ALU kernel's order,
      // a thread per coordinate, KW_REDO vectors over one pass of Pi, then the sums over the rows of S in question.
      // The terms are no longer needed: the numbers take their place.
      uint64_t redo = sopen[0] | (MT > 2 ? (uint64_t)sopen[1] << 32 : 0);
      if (__builtin_expect(redo != 0, 0))
      do {
        float* cbuf = (float*)smem;                             // [KW_REDO][d] centroids
        float* rbuf = cbuf + KW_REDO * d;                       // [KW_REDO][d] residuals
        const int t0 = __builtin_amdgcn_readfirstlane(__builtin_ctzll(redo));
        redo &= redo - 1;
        const int t1 = redo ? __builtin_amdgcn_readfirstlane(__builtin_ctzll(redo)) : t0;
        redo &= redo - 1;
        for (int j = tid; j < d; j += nthreads) {
          int i0 = 0, i1 = 0;
#pragma unroll 1
          for (int p = 0; p < mb; ++p) {
            i0 = 2 * i0 + (int)(spl[(p * TT + t0) * W + (j >> 5)] >> (j & 31) & 1);
            i1 = 2 * i1 + (int)(spl[(p * TT + t1) * W + (j >> 5)] >> (j & 31) & 1);
          }
          const u32x2 e0 = slut[i0], e1 = slut[i1];             // (the terms add up exactly)
          cbuf[j] = (__uint_as_float(e0.y << 16) + __uint_as_float(e0.x & 0xffff0000u)) + __uint_as_float(e0.x << 16);
          cbuf[d + j] = (__uint_as_float(e1.y << 16) + __uint_as_float(e1.x & 0xffff0000u)) + __uint_as_float(e1.x << 16);
        }
        __syncthreads();
        for (int j = tid; j < d; j += nthreads) {
          float xh0 = 0.0f, xh1 = 0.0f;
          constexpr int U = NPW == 1 ? 32 : 64;                 // rows of Pi in flight: no cache holds it
#pragma unroll 1
          for (int i0 = 0; i0 < d; i0 += U) {
            float m[U];
#pragma unroll
            for (int i = 0; i < U; ++i) m[i] = ly.Pi[(size_t)(i0 + i) * d + j];
#pragma unroll
            for (int i = 0; i < U; i += 4) {
              const f32x4 u0 = *(const f32x4*)(cbuf + i0 + i), u1 = *(const f32x4*)(cbuf + d + i0 + i);
#pragma unroll
              for (int k = 0; k < 4; ++k) {
                xh0 = fmaf(u0[k], m[i + k], xh0);
                xh1 = fmaf(u1[k], m[i + k], xh1);
              }
            }
          }
          rbuf[j] = E::load(x, soff[t0] + j) - xh0 * snorm[t0];
          rbuf[d + j] = E::load(x, soff[t1] + j) - xh1 * snorm[t1];
        }
        __syncthreads();
        uint32_t open_now = 0, second = 0;                      // this lane's open signs of these vectors, of t1
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const uint32_t own = near_p & (((1u << (4 * NPW - 1)) * 2 - 1) << (m * NPW * 4));
          if (16 * m + n == t0) open_now |= own;
          else if (16 * m + n == t1) { open_now |= own; second |= own; }
        }
        while (const uint64_t open = __builtin_amdgcn_ballot_w64(open_now != 0)) {
          const uint32_t first = leader_bits(open_now, open, lane);
          const int bit = first ? __builtin_ctz(first) : 0, i = bit & 3, mc = bit >> 2, m = mc / NPW, c = mc % NPW;
          const int col = 16 * (ct0 + c) + 4 * kb + i, t = 16 * m + n;
          const float p = ordered_dot(FloatRow{rbuf + ((second >> bit & 1) ? d : 0)}, ly.S + (size_t)col * d, d, n);
          if (open_now >> bit & 1) {
            uint32_t* word = spl + (mb * TT + t) * W + (col >> 5);
            if (p > 0.0f) atomicOr(word, 1u << (col & 31));
            else atomicAnd(word, ~(1u << (col & 31)));
            if constexpr (!paged) {
              if (sink.p_dbg) sink.p_dbg[(tile0 * TILE + t) * d + col] = p;
            }
            open_now &= ~(1u << bit);
          }
        }
        __syncthreads();                                        // the next vectors overwrite the numbers
      } while (redo);
      fill_ring<NPW>(ly.Pi_split, ct0, tiles, kb_n, lane, ring);
    }
    __syncthreads();
    // (5) write
    if constexpr (!paged) {
      // flat format of the reference (quantizer.py:38-69): a dword of a row is 32 / eff codes, code s at bit eff * s
      const int eff = eff_bits(mb), n_per = 32 / eff, row_dw = idx_row_bytes(d, mb) >> 2;
      for (int o = tid; o < TT * row_dw; o += nthreads) {
        const int t = o / row_dw, k = o - t * row_dw;
        if (!svalid[t]) continue;
        const int c0 = k * n_per;
        uint32_t dw = 0;
        for (int p = 0; p < mb; ++p) {
          uint32_t w = spl[(p * TT + t) * W + (c0 >> 5)] >> (c0 & 31);
          if (eff == 2) {
            w &= 0xffffu;
            w = (w | (w << 8)) & 0x00ff00ffu;
            w = (w | (w << 4)) & 0x0f0f0f0fu;
            w = (w | (w << 2)) & 0x33333333u;
            w = (w | (w << 1)) & 0x55555555u;
          } else if (eff == 4) {
            w &= 0xffu;
            w = (w | (w << 12)) & 0x000f000fu;
            w = (w | (w << 6)) & 0x03030303u;
            w = (w | (w << 3)) & 0x11111111u;
          }
          dw |= w << (mb - 1 - p);
        }
        ((uint32_t*)sink.idx)[(tile0 * TILE + t) * row_dw + k] = dw;
      }
      if (!mse_only) {
        for (int o = tid; o < TT * W; o += nthreads) {
          const int t = o / W, w = o - t * W;
          if (svalid[t]) ((uint32_t*)sink.sign)[(tile0 * TILE + t) * W + w] = spl[(mb * TT + t) * W + w];
        }
      }
      if (tid < TT && svalid[tid]) {
        const int64_t v = tile0 * TILE + tid;
        E::store(sink.norm, v, snorm[tid]);
        if (!mse_only) sink.rnorm[v] = srn[tid];
      }
    } else {
      // pages: wavefronts m, m + MT, .. write tile m, so the page look-up is uniform; words in page order
      const tq_page_layout& L = sink.L;
      const int planes = mb + 1, m = wave % MT, nsub = (waves - m + MT - 1) / MT;
      const int64_t tile = tile0 + m;
      if (tile < n_tiles && __builtin_amdgcn_ballot_w64(lane < TILE && svalid[16 * m + n]) != 0) {
        TileAddr ta;
        int b, lpage, h;
        look_up(tile, ta, b, lpage, h);
        const int64_t page = checked_page(sink.block_table, sink.max_pages, sink.num_pages, b, lpage);
        if (page >= 0) {
          uint8_t* pg = sink.pool + (page * src.H + h) * (int64_t)L.page_bytes;
          const int w4 = W >= 4 ? W >> 2 : 1;
          for (int o = (wave / MT) * 64 + lane; o < planes * W * TILE; o += nsub * 64) {
            int p, w, nn;
            if (L.key_lane_major) {
              p = o % planes;
              const int r = o / planes, jh = r % w4, q = r / w4;
              nn = q % TILE;
              w = jh * 4 + q / TILE;
            } else {
              nn = o % TILE;
              w = o / TILE % W;
              p = o / TILE / W;
            }
            if (svalid[16 * m + nn]) *(uint32_t*)(pg + L.off_keys + 4 * o) = spl[(p * TT + 16 * m + nn) * W + w];
          }
          if (wave / MT == 0 && lane < TILE && svalid[16 * m + lane]) {
            float* meta = (float*)(pg + L.off_meta);
            meta[2 * lane] = snorm[16 * m + lane];
            meta[2 * lane + 1] = srn[16 * m + lane];
          }
        }
      }
    }
    __syncthreads();                                            // the next group overwrites what the writers read
  }
}

// a lane loads four elements at once
__host__ static bool aligned_for_fours(const void* x, int dtype, const FlatSource& s) {
  return (uintptr_t)x % (4 * elem_bytes(dtype)) == 0 && s.row_stride % 4 == 0;
}
__host__ static bool aligned_for_fours(const void* x, int dtype, const PagedSource& s) {
  return (uintptr_t)x % (4 * elem_bytes(dtype)) == 0 && s.stride_b % 4 == 0 && s.stride_t % 4 == 0 && s.stride_h % 4 == 0 &&
         s.stride_blk % 4 == 0;
}
__host__ static bool wide_sink_ok(const KeyFlatSink& s, int mse_only) {
  return (uintptr_t)s.y_dbg % 16 == 0 && (uintptr_t)s.p_dbg % 16 == 0 && (uintptr_t)s.idx % 4 == 0 &&
         (mse_only || (uintptr_t)s.sign % 4 == 0);
}
__host__ static bool wide_sink_ok(const KeyPagedSink&, int) { return true; }
__host__ static int index_entries(const FlatSource&) { return 0; }
__host__ static int index_entries(const PagedSource& s) { return s.compact ? s.B + 1 + KW_MAX_WAVES : 0; }

template <int DT, int NPW, int MT, class Source, class Sink>
static int launch_wide(const void* x, const Source& src, const tq_layer& ly, const Sink& sink, int mse_only, int64_t tiles,
                       int cus, hipStream_t st) {
  constexpr int LDS = 160 * 1024;
  auto kern = key_wide_kernel<DT, NPW, MT, Source, Sink>;
  const int waves = ly.d / 16 / NPW;
  const int smem = WideSmem(ly.d, ly.mse_bits, 16 * MT, waves).bytes + index_entries(src) * 4;
  if (smem > LDS) return TQ_EUNSUPPORTED;
  static std::atomic<uint64_t> configured{0};           // per instantiation, one bit per device; the attribute is sticky
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return TQ_EINVAL;
  if (dev >= 64 || !(configured.load() >> dev & 1)) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return (int)e;
    if (dev < 64) configured.fetch_or(1ull << dev);
  }
  const int64_t groups = (tiles + MT - 1) / MT;
  const int per_cu = std::max(1, std::min(LDS / smem, 16 / waves));
  const unsigned grid = (unsigned)std::min<int64_t>(groups, (int64_t)cus * per_cu);
  hipEvent_t ev_start = nullptr, ev_stop = nullptr;
  if (std::is_same<Sink, KeyPagedSink>::value && take_time_hook(1, ev_start, ev_stop))
    hipExtLaunchKernelGGL(kern, dim3(grid), dim3(waves * 64), smem, st, ev_start, ev_stop, 0, x, src, ly, sink, tiles, mse_only);
  else
    kern<<<dim3(grid), dim3(waves * 64), smem, st>>>(x, src, ly, sink, tiles, mse_only);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? TQ_OK : (int)e;
}

// TQ_EUNSUPPORTED when this kernel does not take the call (no split matrices, a head size or an alignment that it does
// not serve): the caller falls back to the vector-ALU kernel.
template <class Source, class Sink>
int launch_key_wide(const void* x, int dtype, const Source& src, const tq_layer& ly, const Sink& sink, int mse_only,
                    int64_t tiles, hipStream_t st) {
  if (!ly.Pi_split || (!mse_only && (!ly.PiT_split || !ly.S_split))) return TQ_EUNSUPPORTED;
  if (ly.mse_bits < 1 || ly.mse_bits > 4 || ly.d % 64 != 0) return TQ_EUNSUPPORTED;
  if (!aligned_for_fours(x, dtype, src) || !wide_sink_ok(sink, mse_only)) return TQ_EUNSUPPORTED;
  // column tiles per wavefront: the fewest that leave at most KW_MAX_WAVES wavefronts
  int npw = 1;
  while (npw <= 4 && (ly.d / 16 % npw != 0 || ly.d / 16 / npw > KW_MAX_WAVES)) ++npw;
  if (npw > 4) return TQ_EUNSUPPORTED;
  const int cus = device_compute_units();
  // one 16-vector tile per workgroup while every tile has a compute unit to itself: half of the MFMAs behind one another; and
  // where more do not fit the LDS (head_dim 768: 4-bit keys with the index of more than 35 ragged runs, 5-bit keys)
  const bool small = tiles <= cus;
#define TQ_KW(DT_, NPW_, MT_)                                                                                             \
  if (dtype == DT_ && npw == NPW_) {                                                                                       \
    const int rc = small ? TQ_EUNSUPPORTED : launch_wide<DT_, NPW_, MT_, Source, Sink>(x, src, ly, sink, mse_only, tiles, cus, st); \
    if (rc != TQ_EUNSUPPORTED) return rc;                                                                                  \
    return launch_wide<DT_, NPW_, 1, Source, Sink>(x, src, ly, sink, mse_only, tiles, cus, st);                            \
  }
#define TQ_KW_ALL(DT_) TQ_KW(DT_, 1, 4) TQ_KW(DT_, 2, 2) TQ_KW(DT_, 3, 2) TQ_KW(DT_, 4, 2)
  TQ_KW_ALL(TQ_BF16) TQ_KW_ALL(TQ_F16) TQ_KW_ALL(TQ_F32)
#undef TQ_KW_ALL
#undef TQ_KW
  return TQ_EUNSUPPORTED;
}

template int launch_key_wide<FlatSource, KeyFlatSink>(const void*, int, const FlatSource&, const tq_layer&,
                                                      const KeyFlatSink&, int, int64_t, hipStream_t);
template int launch_key_wide<PagedSource, KeyPagedSink>(const void*, int, const PagedSource&, const tq_layer&,
                                                        const KeyPagedSink&, int, int64_t, hipStream_t);

}  // namespace tq
