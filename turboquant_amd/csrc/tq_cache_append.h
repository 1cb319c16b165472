// What a token of the cache object (kv_cache.py:203-245) is besides the codes of the key that leaves the buffer: every section and both
// buffers written anew, and the codes of the value.  Shared by the launch that quantises the key as well (tq_quantize_mfma.hip) and by the
// one behind the other key quantisers (tq_score.hip).
#pragma once

#include "tq_quantize.h"

namespace tq {

// Row r of a section becomes its `a` bytes followed by its `b` bytes, at r * dst_stride.
struct CopySection {
  const uint8_t *a, *b;
  uint8_t* dst;
  int64_t a_stride, b_stride, dst_stride;
  int a_bytes, b_bytes;
  int first;                                     // workgroup of the copies that it begins with
};
constexpr int CACHE_SECTIONS = 9, CACHE_CHUNKS = 4;      // pieces of a copy that a thread has in flight
struct CacheRest {
  CopySection s[CACHE_SECTIONS];                 // in the order of their workgroups
  int rows, copies;                              // value rows (a workgroup each, first), workgroups of the copies
  const float* v;                                // rows of values, v_stride elements apart
  int64_t v_stride;
  uint8_t* data;                                 // where row 0's codes, scales and zeros go; row r's are `step` rows further on each time
  float *scales, *zeros;
  int64_t step;
  int d, gs, bits;
};

// bytes of a piece: 16 where a section's rows and both its parts allow them, else a word
__host__ __device__ __forceinline__ int copy_piece(const CopySection& c) {
  const uintptr_t all = (uintptr_t)c.a | (uintptr_t)c.b | (uintptr_t)c.dst | (uintptr_t)(c.a_stride | c.b_stride | c.dst_stride) |
                        (uintptr_t)(c.a_bytes | c.b_bytes);
  return all & 15 ? 4 : 16;
}
__host__ inline int copy_workgroups(const CopySection& c, int64_t rows) {
  const int64_t pieces = rows * (c.a_bytes + c.b_bytes) / copy_piece(c);
  return (int)((pieces + 256 * CACHE_CHUNKS - 1) / (256 * CACHE_CHUNKS));
}

typedef uint32_t U4 __attribute__((ext_vector_type(4)));

template <class Piece>
__device__ __forceinline__ void copy_rows(const CopySection& c, int64_t rows, int64_t wg) {
  const uint32_t per = (uint32_t)(c.a_bytes + c.b_bytes) / sizeof(Piece), a_per = (uint32_t)c.a_bytes / sizeof(Piece);
  const int64_t o0 = wg * (CACHE_CHUNKS * 256), r0 = o0 / per;      // (uniform; the lanes go on in 32 bits)
  const uint32_t e0 = (uint32_t)(o0 - r0 * per);
  // (every load unconditional, all in flight together: one under a branch is waited for at once; pieces behind the last row read its last)
  Piece x[CACHE_CHUNKS];
  Piece* to[CACHE_CHUNKS];
  bool in[CACHE_CHUNKS];
#pragma unroll
  for (int k = 0; k < CACHE_CHUNKS; ++k) {
    const uint32_t o = e0 + k * 256 + threadIdx.x, rr = o / per;
    in[k] = r0 + rr < rows;
    const int64_t r = in[k] ? r0 + rr : rows - 1;
    const uint32_t e = in[k] ? o - rr * per : per - 1;
    const Piece* a = (const Piece*)(c.a + r * c.a_stride) + e;
    const Piece* b = (const Piece*)(c.b + r * c.b_stride) + (e - a_per);
    x[k] = *(e < a_per ? a : b);
    to[k] = (Piece*)(c.dst + r * c.dst_stride) + e;
  }
  // (written past the L2, whose dirty lines a launch's end waits for: 15 MB of copies behind a key's own launch 18.9 -> 6.4 us, though the
  // scores that read them next take 15.6 us for 13.9)
#pragma unroll
  for (int k = 0; k < CACHE_CHUNKS; ++k)
    if (in[k]) __builtin_nontemporal_store(x[k], to[k]);
}

// Workgroup `id` of rows + copies, 256 threads; d <= 256.
__device__ __forceinline__ void cache_rest_body(const CacheRest& A, int id) {
  __shared__ float sx[256], s_sc[16], s_z[16];
  __shared__ uint8_t s_code[256];
  if (id >= A.rows) {
    id -= A.rows;
    int k = 0;
#pragma unroll
    for (int i = 1; i < CACHE_SECTIONS; ++i) k += id >= A.s[i].first;
    const CopySection c = A.s[k];
    if (copy_piece(c) == 16) copy_rows<U4>(c, A.rows, id - c.first);
    else copy_rows<uint32_t>(c, A.rows, id - c.first);
    return;
  }
  const int tid = threadIdx.x, d = A.d, gs = A.gs, ng = d / gs;
  const float levels = (float)((1 << A.bits) - 1);
  if (tid < d) sx[tid] = A.v[id * A.v_stride + tid];
  __syncthreads();
  if (tid < ng) {
    float sc, lo;
    value_group<TQ_F32>(sx + tid * gs, gs, tid, levels, sc, lo);
    s_sc[tid] = sc;
    s_z[tid] = lo;
    const int64_t at = id * A.step * ng + tid;
    A.scales[at] = sc;
    A.zeros[at] = lo;
  }
  __syncthreads();
  if (tid < d) s_code[tid] = value_code<TQ_F32>(sx[tid], s_z[tid / gs], s_sc[tid / gs], levels);
  __syncthreads();
  const int per = 32 / A.bits, words = d / per;
  if (tid < words) {
    uint32_t w = 0;
    for (int s = 0; s < per; ++s) w |= (uint32_t)s_code[tid * per + s] << (A.bits * s);
    ((uint32_t*)(A.data + id * A.step * (d * A.bits / 8)))[tid] = w;
  }
}

}  // namespace tq
