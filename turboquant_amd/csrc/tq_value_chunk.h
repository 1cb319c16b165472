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
  return (size_t)(slab / 8) * (TILE * (bits == 2 ? 2 : 4) + 16);
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

// bits of a number that a rounding to the input dtype has left (or one of the input's): nothing is left to round
template <int DT>
__device__ __forceinline__ uint16_t stored_bits(float v) {
  return DT == TQ_BF16 ? (uint16_t)(__float_as_uint(v) >> 16) : f32_to_f16_bits(v);
}

// Value quantiser for 16-bit inputs and 2/4-bit codes: a thread owns 8 consecutive channels of one token (one
// 16-byte load), a group's minimum / maximum meet through cross-lane exchanges, and the codes pass through LDS only to
// be transposed into the page's per-channel fields.  Arithmetic and rounding are those of value_tile_kernel.
// A workgroup takes one tile's `slab` channels (64, 128 or 256: whole tokens in a row of 16 lanes); head sizes that are
// not one of these are slabs side by side in the grid's second dimension (a group never crosses a slab).
// Bound by vector instructions: about 185 per wavefront of 512 values, and the kernel takes the time that a SIMD needs to issue them (262,144
// vectors of 128 in bf16, 67 MB in: 25.5 us; reading them takes 10).  What exists of a tile follows from two numbers and not from flags in
// LDS counted over the workgroup, the minimum and maximum are the bare instructions, a NaN is looked for by wavefront, groups are shifts,
// fp16 quotients are products: bf16 31.2 -> 25.5 us, 120,000 vectors in fp16 21.1 -> 15.5, 262,144 of 256 33 -> 27.
// 8192 vectors of 576, 4-bit codes, 9.4 MB in: value_tile_kernel 17.5 us, nine slabs of 64 7.8 us.
// A workgroup of 2 * slab threads; c0: its first channel; smem: value_chunk_smem(slab, VB) bytes.
template <int DT, int VB, class Source, class Sink>
__device__ __forceinline__ void value_chunk_body(const void* __restrict__ v, const Source& src, int d, int slab, int gs, const Sink& sink,
                                                 int tile, int c0, unsigned char* smem) {
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

  // where the tile's rows are and which of its slots exist: uniform, looked up through the scalar cache
  TileAddr ta;
  int head = 0, b = 0, lpage = 0;
  if constexpr (std::is_base_of<PagedSource, Source>::value) {
    PagedSource::Coord c[1] = {src.coord(tile)};
    TileAddr ta1[1];
    int lp[1];
    src.template tile_addrs<1>(c, ta1, lp);
    ta = ta1[0];
    head = c[0].h;
    b = c[0].b;
    lpage = lp[0];
  } else {
    ta = src.tile_addr(tile);
  }
  // (a tile none of whose slots exists may lie beyond the block table, or behind the end of a ragged run: leave before looking it up)
  const int first = max(ta.lo, 0), last = min(ta.hi, TILE);      // its existing slots
  if (last <= first) return;
  const bool full_tile = last - first == TILE, ok = t >= first && t < last;
  // the page is looked up while the input is on its way
  int64_t page = 0;
  if constexpr (!std::is_same<Sink, ValFlatSink>::value) page = checked_page(sink.block_table, sink.max_pages, sink.num_pages, b, lpage);
  const bool page_ok = page >= 0;                    // uniform over the workgroup; false: nothing is stored
  // unconditional load (slots that do not exist read the nearest one that does); a lane's part of the address in 24-bit numbers where
  // the strides are, which they are but for exotic views
  const int tr = min(max(t, first), last - 1);
  const uint16_t* rows = (const uint16_t*)v + ta.base + c0;
  const int64_t stride = src.slot_stride();
  uint4 raw;
  if ((uint64_t)stride < (1u << 24)) raw = *(const uint4*)(rows + (__umul24(tr, (uint32_t)stride) + (uint32_t)(ck * 8)));
  else raw = *(const uint4*)(rows + tr * stride + ck * 8);
  float x[8];
  {
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = DT == TQ_BF16 ? __uint_as_float(w[i] << 16) : f16_bits_to_f32((uint16_t)(w[i] & 0xffffu));
      x[2 * i + 1] = DT == TQ_BF16 ? __uint_as_float(w[i] & 0xffff0000u) : f16_bits_to_f32((uint16_t)(w[i] >> 16));
    }
  }
  // (the instructions themselves: fminf / fmaxf first make every operand canonical, an instruction each; the comparisons below see a NaN)
  auto min2 = [](float p, float q) { float r; asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(p), "v"(q)); return r; };
  auto max2 = [](float p, float q) { float r; asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(p), "v"(q)); return r; };
  auto min3 = [](float p, float q, float s) { float r; asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(p), "v"(q), "v"(s)); return r; };
  auto max3 = [](float p, float q, float s) { float r; asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(p), "v"(q), "v"(s)); return r; };
  float lo = min2(min3(min3(min3(x[0], x[1], x[2]), x[3], x[4]), x[5], x[6]), x[7]);
  float hi = max2(max3(max3(max3(x[0], x[1], x[2]), x[3], x[4]), x[5], x[6]), x[7]);
  // the threads of a group are neighbouring lanes inside a row of 16: DPP moves (quad swaps, then half-row and
  // row mirrors, which pair quads that already agree) instead of shuffles through the LDS
  auto over_group = [&](auto step) {
    step(std::integral_constant<int, 0xB1>{});                   // (a group has at least 16 channels)
    if (tpg >= 4) step(std::integral_constant<int, 0x4E>{});
    if (tpg >= 8) step(std::integral_constant<int, 0x141>{});
    if (tpg >= 16) step(std::integral_constant<int, 0x140>{});
  };
  over_group([&](auto ctrl_c) {
    constexpr int CTRL = decltype(ctrl_c)::value;
    lo = min2(lo, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, lo), CTRL, 0xF, 0xF, true)));
    hi = max2(hi, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, hi), CTRL, 0xF, 0xF, true)));
  });
  // torch min / max propagate NaN, the instructions do not: a wavefront that holds one looks for its group
  const bool nan = __builtin_isunordered(x[0], x[1]) || __builtin_isunordered(x[2], x[3]) || __builtin_isunordered(x[4], x[5]) || __builtin_isunordered(x[6], x[7]);
  if (__builtin_amdgcn_ballot_w64(nan) != 0) {
    int has_nan = nan;
    over_group([&](auto ctrl_c) { has_nan |= __builtin_amdgcn_update_dpp(0, has_nan, decltype(ctrl_c)::value, 0xF, 0xF, true); });
    if (has_nan) lo = hi = __uint_as_float(0x7fc00000u);
  }
  const float levels = (float)((1 << VB) - 1);
  // (hi - lo) / levels as a product: both are numbers of at most 8 significant bits, so is the divisor of every
  // quotient below, and such a quotient is never a rounding tie of the 16-bit format and at least 2^-17
  // (relative) away from one: a product with a reciprocal good to an ulp rounds like the division (checked
  // over all pairs of significands and the three nearest reciprocals).  fp16 keeps the division here.
  const float range = round_hw<DT>(hi - lo);
  float sc = round_hw<DT>(DT == TQ_BF16 ? range * (1.0f / levels) : range / levels);
  const float floor_v = round_hw<DT>(1e-10f);
  sc = (sc != sc) ? sc : fmaxf(sc, floor_v);
  const float z = lo;
  // Quotients of bf16 numbers, rounded to bf16: a * (1/s) with any reciprocal good to an ulp (see above).  Quotients of fp16 numbers: the
  // product and one correction by its remainder are the fp32 quotient itself, to the bit (11 significant bits on either side, the three
  // nearest reciprocals, all pairs).  Used when the scale is an ordinary number; everything else takes the division.
  const bool fast_div = DT == TQ_BF16 ? sc > 0x1p-60f && sc < 0x1p60f : sc >= 0x1p-24f && sc < 0x1p16f;
  const float rsc = __builtin_amdgcn_rcpf(sc);
  float quo[8];
  if (fast_div) {                // every a of the group is finite and at most (levels + 1) * sc < 2^64 then
    float a[8];
    round_pairs<DT>(x, z, a);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      quo[i] = a[i] * rsc;
      if constexpr (DT == TQ_F16) quo[i] = fmaf(fmaf(-quo[i], sc, a[i]), rsc, quo[i]);
    }
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
    float acc;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      // clamp to [0, levels]; a NaN becomes code 0 (the median-of-three instruction returns the minimum of
      // its operands when one of them is a NaN)
      const float q = __builtin_amdgcn_fmed3f(rintf(qr[hw * PER + i]), 0.0f, levels);
      acc = i == 0 ? q : fmaf(q, (float)(1 << (VB * i)), acc);
    }
    codes |= (uint32_t)acc << (16 * hw);
  }
  if constexpr (!std::is_same<Sink, ValFlatSink>::value) *(CodeWord*)(scode + ck * CROW + t * sizeof(CodeWord)) = (CodeWord)codes;
  const int g_bits = __builtin_ctz((unsigned)gs), ng = d >> g_bits, g = (c0 + ck * 8) >> g_bits;      // (groups are powers of two)
  const bool leader = (ck & (tpg - 1)) == 0;

  if constexpr (std::is_same<Sink, ValFlatSink>::value) {
    if (ok) {
      const int64_t vec = (int64_t)tile * TILE + t;
      uint8_t* dst = sink.data + vec * (d * VB / 8) + (c0 / 8 + ck) * VB;           // 8 codes = VB bytes, little-end first
      if (VB == 2) *(uint16_t*)dst = (uint16_t)codes;
      else *(uint32_t*)dst = codes;
      if (leader) {
        ((uint16_t*)sink.scale)[vec * ng + g] = stored_bits<DT>(sc);
        ((uint16_t*)sink.zero)[vec * ng + g] = stored_bits<DT>(z);
      }
    }
  } else {
    const tq_page_layout& L = sink.L;
    uint8_t* pg = sink.pool + (page * src.H + head) * (int64_t)L.page_bytes;
    if (ok && leader && page_ok) {
      *(uint16_t*)(pg + (uint32_t)(L.off_vscale + (g * TILE + t) * 2)) = stored_bits<DT>(sc);
      *(uint16_t*)(pg + (uint32_t)(L.off_vzero + (g * TILE + t) * 2)) = stored_bits<DT>(z);
    }
    __syncthreads();
    // channel c: a field of 16*VB bits, token n at bit VB*n; read-modify-write keeps the codes of
    // slots this call does not touch
    // every thread assembles half a field: 8 tokens of one channel (16 bits of 2-bit codes, 32 of 4-bit)
    {
      const int c = tid >> 1, half = tid & 1;
      const int cc = c0 + c;                         // (vfield_off, with 24-bit products)
      uint8_t* fbytes = pg + (uint32_t)(L.off_vdata + (__umul24(cc & 15, d >> 4) + (cc >> 4)) * (VB * 2) + half * VB);
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
        // the bits of tokens first .. last - 1, those of this half
        const int f = min(max(first - half * 8, 0), 8), l = min(max(last - half * 8, 0), 8);
        const uint64_t below = ((uint64_t)1 << (VB * l)) - 1, before = ((uint64_t)1 << (VB * f)) - 1;
        mask = (uint32_t)(below & ~before);
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
