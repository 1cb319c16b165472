// Value quantiser for 16-bit inputs and 2/4-bit codes, a tile of 16 tokens at a time: the body that the value kernel
// (tq_quantize.hip) and the small page write (tq_quantize_mfma.hip) share.
#pragma once

#include <type_traits>

#include "tq_common.h"
#include "tq_quantize.h"

namespace tq {

struct ValFlatSink {
  uint8_t* data;
  void* scale;
  void* zero;
};
struct ValPagedSink {
  uint8_t* pool;
  const int32_t* block_table;
  int max_pages;
  int num_pages;           // pages of the pool (see checked_page)
  tq_page_layout L;
};

__host__ inline size_t value_chunk_smem(int slab, int bits) {
  return (size_t)(slab / 8) * (TILE * (bits == 2 ? 2 : 4) + 16) + TILE * sizeof(int);
}
// inputs that the body takes: group sizes that are a power of two of 16 .. 128 and do not cross a slab
__host__ inline bool value_chunk_takes(int dtype, int bits, int gs, int slab) {
  return dtype != TQ_F32 && (bits == 2 || bits == 4) && gs >= 16 && gs <= 128 && slab % gs == 0 && (gs & (gs - 1)) == 0;
}
// ... and rows whose 16-byte chunks are aligned
__host__ inline bool value_chunks_aligned(const void* v, const FlatSource& s) {
  return (uintptr_t)v % 16 == 0 && s.row_stride % 8 == 0;
}
__host__ inline bool value_chunks_aligned(const void* v, const PagedSource& s) {
  return (uintptr_t)v % 16 == 0 && s.stride_b % 8 == 0 && s.stride_t % 8 == 0 && s.stride_h % 8 == 0 &&
         s.stride_blk % 8 == 0;
}

// round to the input dtype and back with the hardware conversions (v_cvt_pk_bf16_f32 / v_cvt_f16_f32,
// round to nearest even; NaN stays NaN)
template <int DT>
__device__ __forceinline__ float round_hw(float v) {
  if constexpr (DT == TQ_BF16) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    const f32x2_t f = {v, 0.0f};
    const bf16x2_t r = __builtin_convertvector(f, bf16x2_t);
    uint32_t u;
    __builtin_memcpy(&u, &r, 4);
    return __uint_as_float(u << 16);
  } else {
    return Elem<DT>::round(v);
  }
}

// out[i] = in[i] - sub rounded to the input dtype, i < 8; bf16 rounds two numbers per conversion instruction
template <int DT>
__device__ __forceinline__ void round_pairs(const float (&in)[8], float sub, float (&out)[8]) {
  if constexpr (DT == TQ_BF16) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x2_t f = {in[2 * i] - sub, in[2 * i + 1] - sub};
      const bf16x2_t r = __builtin_convertvector(f, bf16x2_t);
      uint32_t u;
      __builtin_memcpy(&u, &r, 4);
      out[2 * i] = __uint_as_float(u << 16);
      out[2 * i + 1] = __uint_as_float(u & 0xffff0000u);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = round_hw<DT>(in[i] - sub);
  }
}

// Value quantiser for 16-bit inputs and 2/4-bit codes: a thread owns 8 consecutive channels of one token (one
// 16-byte load), a group's minimum / maximum meet through cross-lane exchanges, and the codes pass through LDS only to
// be transposed into the page's per-channel fields.  Arithmetic and rounding are those of value_tile_kernel.
// A workgroup takes one tile's `slab` channels (64, 128 or 256: whole tokens in a row of 16 lanes); head sizes that are
// not one of these are slabs side by side in the grid's second dimension (a group never crosses a slab).
// Bound by memory: 8192 vectors of 576, 4-bit codes, 9.4 MB in: value_tile_kernel 17.5 us, nine slabs of 64 7.8 us.
// A workgroup of 2 * slab threads; c0: its first channel; smem: value_chunk_smem(slab, VB) bytes.
template <int DT, int VB, class Source, class Sink>
__device__ __forceinline__ void value_chunk_body(const void* __restrict__ v, const Source& src, int d, int slab, int gs, const Sink& sink,
                                                 int tile, int c0, unsigned char* smem) {
  using E = Elem<DT>;
  static_assert(DT != TQ_F32, "16-bit inputs");
  const int tid = threadIdx.x;
  const int cpt = slab >> 3;                       // chunks (threads) per token
  const int t = tid >> (31 - __builtin_clz(cpt)), ck = tid & (cpt - 1);     // token slot, chunk
  const int tpg = gs >> 3;                         // threads per group (power of two, <= 16)
  // a thread's 8 codes are one word of 8 * VB bits; the words of a chunk's 16 tokens lie together
  // (rows padded by 16 bytes), so that the thread that assembles half a channel field reads the
  // words of its 8 tokens with one or two 16-byte loads
  using CodeWord = typename std::conditional<VB == 2, uint16_t, uint32_t>::type;
  constexpr int CROW = TILE * (int)sizeof(CodeWord) + 16;      // bytes per chunk row
  unsigned char* scode = smem;                     // [slab / 8] rows of CROW bytes
  int* svalid = (int*)(smem + (size_t)cpt * CROW); // [TILE]

  // where the tile's rows are and which of its slots exist: uniform, looked up through the scalar cache
  TileAddr ta;
  // page lookup issued together with the input load (clamped into the table: a tile without a
  // single existing slot may lie beyond it, and then nothing is stored anyway)
  int64_t page = 0;
  int head = 0;
  if constexpr (std::is_base_of<PagedSource, Source>::value) {
    PagedSource::Coord c[1] = {src.coord(tile)};
    TileAddr ta1[1];
    int lpage[1];
    src.template tile_addrs<1>(c, ta1, lpage);
    ta = ta1[0];
    head = c[0].h;
    if constexpr (!std::is_same<Sink, ValFlatSink>::value)
      page = checked_page(sink.block_table, sink.max_pages, sink.num_pages, c[0].b, lpage[0]);
  } else {
    ta = src.tile_addr(tile);
  }
  if (ta.hi <= 0) return;                          // (uniform) a page behind the end of a ragged run
  const bool ok = t >= ta.lo && t < ta.hi;
  const int64_t off = ta.base + (int64_t)t * src.slot_stride();
  const bool page_ok = page >= 0;                    // uniform over the workgroup; false: nothing is stored
  // unconditional load (slots that do not exist read the first vector)
  const uint4 raw = *(const uint4*)((const uint16_t*)v + (ok ? off : 0) + c0 + ck * 8);
  if (ck == 0) svalid[t] = ok;
  // a tile none of whose slots exists may lie beyond the block table: leave before looking it up
  const int n_ok = __syncthreads_count(ok);
  if (n_ok == 0) return;
  const bool full_tile = n_ok == 2 * slab;
  float x[8];
  {
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = DT == TQ_BF16 ? __uint_as_float(w[i] << 16) : f16_bits_to_f32((uint16_t)(w[i] & 0xffffu));
      x[2 * i + 1] = DT == TQ_BF16 ? __uint_as_float(w[i] & 0xffff0000u) : f16_bits_to_f32((uint16_t)(w[i] >> 16));
    }
  }
  float lo = x[0], hi = x[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) {
    lo = fminf(lo, x[i]);
    hi = fmaxf(hi, x[i]);
  }
  // a NaN among the 8 inputs, on the packed 16-bit patterns: magnitude bits above those of infinity
  int has_nan;
  {
    typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
    u16x2_t m = __builtin_bit_cast(u16x2_t, raw.x & 0x7fff7fffu);
    m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2_t, raw.y & 0x7fff7fffu));
    m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2_t, raw.z & 0x7fff7fffu));
    m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2_t, raw.w & 0x7fff7fffu));
    constexpr uint16_t inf_bits = DT == TQ_BF16 ? 0x7f80 : 0x7c00;
    has_nan = (m[0] > inf_bits) | (m[1] > inf_bits);
  }
  // the threads of a group are neighbouring lanes inside a row of 16: DPP moves (quad swaps, then half-row and
  // row mirrors, which pair quads that already agree) instead of shuffles through the LDS
  auto reduce_step = [&](auto ctrl_c) {
    constexpr int CTRL = decltype(ctrl_c)::value;
    lo = fminf(lo, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, lo), CTRL, 0xF, 0xF, true)));
    hi = fmaxf(hi, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, hi), CTRL, 0xF, 0xF, true)));
    has_nan |= __builtin_amdgcn_update_dpp(0, has_nan, CTRL, 0xF, 0xF, true);
  };
  if (tpg >= 2) reduce_step(std::integral_constant<int, 0xB1>{});
  if (tpg >= 4) reduce_step(std::integral_constant<int, 0x4E>{});
  if (tpg >= 8) reduce_step(std::integral_constant<int, 0x141>{});
  if (tpg >= 16) reduce_step(std::integral_constant<int, 0x140>{});
  if (has_nan) lo = hi = __uint_as_float(0x7fc00000u);       // torch min/max propagate NaN
  const float levels = (float)((1 << VB) - 1);
  // (hi - lo) / levels as a product: both are numbers of at most 8 significant bits, so is the divisor of every
  // quotient below, and such a quotient is never a rounding tie of the 16-bit format and at least 2^-17
  // (relative) away from one: a product with a reciprocal good to an ulp rounds like the division (checked
  // over all pairs of significands and the three nearest reciprocals).  fp16 keeps the division.
  const float range = round_hw<DT>(hi - lo);
  float sc = round_hw<DT>(DT == TQ_BF16 ? range * (1.0f / levels) : range / levels);
  const float floor_v = round_hw<DT>(1e-10f);
  sc = (sc != sc) ? sc : fmaxf(sc, floor_v);
  const float z = lo;
  // Quotients of bf16 numbers, rounded to bf16: a * (1/s) with any reciprocal good to an ulp (see above).
  // Used when the scale is an ordinary number; everything else takes the division.
  const bool fast_div = DT == TQ_BF16 && sc > 0x1p-60f && sc < 0x1p60f;
  const float rsc = __builtin_amdgcn_rcpf(sc);
  float quo[8];
  if (fast_div) {                // every a of the group is finite and at most (levels + 1) * sc < 2^64 then
    float a[8];
    round_pairs<DT>(x, z, a);
#pragma unroll
    for (int i = 0; i < 8; ++i) quo[i] = a[i] * rsc;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) quo[i] = round_hw<DT>(x[i] - z) / sc;
  }
  // 8 codes, VB bits each, channel order.  The codes are small integers held in floats: 16 bits' worth of
  // them are put together with exact multiply-adds and converted once.
  float qr[8];
  round_pairs<DT>(quo, 0.0f, qr);
  uint32_t codes = 0;
#pragma unroll
  for (int hw = 0; hw < (VB == 2 ? 1 : 2); ++hw) {
    constexpr int PER = 16 / VB;                   // codes per 16 bits
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      // clamp to [0, levels]; a NaN becomes code 0 (the median-of-three instruction returns the minimum of
      // its operands when one of them is a NaN)
      const float q = __builtin_amdgcn_fmed3f(rintf(qr[hw * PER + i]), 0.0f, levels);
      acc = fmaf(q, (float)(1 << (VB * i)), acc);
    }
    codes |= (uint32_t)acc << (16 * hw);
  }
  if constexpr (!std::is_same<Sink, ValFlatSink>::value) *(CodeWord*)(scode + ck * CROW + t * sizeof(CodeWord)) = (CodeWord)codes;
  const int ng = d / gs, g = (c0 + ck * 8) / gs;
  const bool leader = (ck & (tpg - 1)) == 0;

  if constexpr (std::is_same<Sink, ValFlatSink>::value) {
    if (ok) {
      const int64_t vec = (int64_t)tile * TILE + t;
      uint8_t* dst = sink.data + vec * (d * VB / 8) + (c0 / 8 + ck) * VB;           // 8 codes = VB bytes, little-end first
      if (VB == 2) *(uint16_t*)dst = (uint16_t)codes;
      else *(uint32_t*)dst = codes;
      if (leader) {
        E::store(sink.scale, vec * ng + g, sc);
        E::store(sink.zero, vec * ng + g, z);
      }
    }
  } else {
    const tq_page_layout& L = sink.L;
    uint8_t* pg = sink.pool + (page * src.H + head) * (int64_t)L.page_bytes;
    if (ok && leader && page_ok) {
      E::store(pg + L.off_vscale, g * TILE + t, sc);
      E::store(pg + L.off_vzero, g * TILE + t, z);
    }
    __syncthreads();
    // channel c: a field of 16*VB bits, token n at bit VB*n; read-modify-write keeps the codes of
    // slots this call does not touch
    // every thread assembles half a field: 8 tokens of one channel (16 bits of 2-bit codes, 32 of 4-bit)
    {
      const int c = tid >> 1, half = tid & 1;
      uint8_t* fbytes = pg + vfield_off(L, c0 + c) + half * VB;
      const unsigned char* row = scode + (c >> 3) * CROW + half * 8 * sizeof(CodeWord);
      const int sh = (c & 7) * VB;                   // the channel's code inside a word
      uint32_t neu = 0, mask = VB == 2 ? 0xffffu : 0xffffffffu;
      if constexpr (VB == 2) {
        const uint4 w = *(const uint4*)row;          // 8 tokens, two to a dword
        const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t pr = (ww[k] >> sh) & 0x00030003u;
          neu |= ((pr | (pr >> 14)) & 0xfu) << (4 * k);
        }
      } else {
        const uint4 w0 = *(const uint4*)row, w1 = *(const uint4*)(row + 16);
        const uint32_t ww[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
        for (int k = 0; k < 8; ++k) neu |= ((ww[k] >> sh) & 0xfu) << (4 * k);
      }
      if (!full_tile) {                              // uniform over the workgroup
        mask = 0;
#pragma unroll
        for (int s2 = 0; s2 < 8; ++s2) mask |= (svalid[half * 8 + s2] ? (1u << VB) - 1u : 0u) << (VB * s2);
        neu &= mask;
      }
      if (mask != 0 && page_ok) {
        if (VB == 2) {
          uint16_t* f16p = (uint16_t*)fbytes;
          const uint32_t old = (mask == 0xffffu) ? 0u : *f16p;
          *f16p = (uint16_t)((old & ~mask) | neu);
        } else {
          uint32_t* f32p = (uint32_t*)fbytes;
          const uint32_t old = (mask == 0xffffffffu) ? 0u : *f32p;
          *f32p = (old & ~mask) | neu;
        }
      }
    }
  }
}

}  // namespace tq
