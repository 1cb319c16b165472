// Page kernel on the matrix cores for dozens of query heads on one wide KV head (head_dim 512 / 576 with more than 8 query
// heads per KV head: latent attention, where all of a layer's query heads share one latent).  Same partials (m, l, acc[d])
// per context split as the other page kernels (score.py:114-173 over compressed pages).
//
// The kernel of tq_decode_wide.hip takes 8 heads per workgroup and unpacks every page once per group of 8: 128 heads are
// sixteen passes of unpacking, and its value MFMAs carry 8 heads in 16 rows.  Here a PAIR of wavefronts owns sixteen heads for the
// whole step, one for the scores and the softmax, one for the values, a block of 32 tokens apart:
//   * queries stay put.  The fp6 query operands carry no codebook coefficient - a plane's products are summed
//     first and then weighted -, so the index planes share one set: 16 heads x 4 terms are 12 registers per 64 coordinates, 108 at
//     head_dim 576, loaded once; the sketched queries, which one plane uses, lie in LDS.
//   * scores: v_mfma_scale_f32_32x32x64_f8f6f4 with 32 tokens as rows (their bit planes are the fp4 operand, masked
//     in place) and 16 heads x 2 terms as columns, two of them for the four terms.  The sums of a head's two columns
//     meet with one register swap between neighbouring rows of lanes, which also deals the 32 tokens to the four rows of lanes
//     as the value product wants them: the weights go to the same lane of the partner.
//   * values: channels as rows, heads as columns; codes masked in place are bf16 denormals (row operand),
//     weight x group scale is the column operand, one product for the two channel tiles of a group.  Zero points: one more
//     product with the groups as rows.  Where head tiles stand side by side a value wavefront sums two of them over half the channels:
//     codes are unpacked and scales widened once for both, 400 vector instructions a block instead of 580.
//   * softmax: a lane holds 8 scores of ONE head, every accumulator of a lane belongs to that head, so the running reference
//     and its rare moves are per-lane scalars.
// A workgroup of HW x TW pairs walks a range of tokens: HW head tiles side by side on the same pages (four: 64 heads
// per pass over the pages), and with fewer tiles TW blocks of 32 tokens side by side.  The pages lie in LDS, two turns of keys and
// two of values, filled by LDS-direct loads that the value wavefronts spread over their turn (one occupies the
// compute unit's address path for about 64 clocks, and a wavefront that issues several in a row waits for that).
//
// Bound: instruction issue.  A block costs a SIMD 90 score and 38 value MFMAs (3,500 clocks of its matrix unit) and 860 vector
// instructions; an MFMA holds a wavefront's issue for about 13 clocks and a vector instruction for 4, so the two roles
// together issue for about 5,100 clocks, and take 6,700 - 7,700 (at 1.8 - 2.1 GHz, where the fp4 x fp6 products leave the card).  Without the
// value wavefronts' work the kernel takes 113 us of its 137, without the scores' 87; the page requests and the masks of the bit
// planes cost nothing.  A lone wavefront issues once in five clocks at best: with both roles
// in one wavefront of 512 registers a block took 10,000.  16 x 8192 tokens of 576, 4-bit keys and values, page kernel of 128 heads, average of sixty
// steps: 411 us with the kernel of 8 heads, 150 - 157 with a head tile per value wavefront and one sum per plane (its registers spilled), 138 now.
// Steps: 128 heads 172 -> 165 (166 -> 157 on another card), 64 heads 105 -> 102, 32 heads 72 -> 66, 16 heads (one tile, as before) 60.
// Measured and not kept: a plane's words read a pair of planes ahead 138, requests in the first half of a turn 137 - 141, the scores' wavefronts
// first at issue 141 - 145.

#include "tq_decode_mfma_impl.h"

namespace tq {

constexpr int HD_BLK = 32;                 // tokens of a wavefront's block (two pages)
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x6 __attribute__((ext_vector_type(6)));

// Page geometry tq_page_layout_init gives 16-bit pages with groups of 32 (checked at the launch)
struct HeadsGeom { int off_meta, off_vdata, off_vscale, off_vzero, page_bytes, lane_major, kslot, vslot; };
__host__ __device__ constexpr int heads_odd_lines(int bytes) { return (bytes / 128) % 2 ? bytes : bytes + 128; }
__host__ __device__ constexpr HeadsGeom heads_geom(int d, int mb, int vb) {
  HeadsGeom g{};
  int off = (mb + 1) * (d / 8) * TQ_PAGE_TOKENS;
  g.off_meta = off;   off += 8 * TQ_PAGE_TOKENS;
  g.off_vdata = off;  off += d * vb * 2;
  g.off_vscale = off; off += (d / 32) * TQ_PAGE_TOKENS * 2;
  g.off_vzero = off;  off += (d / 32) * TQ_PAGE_TOKENS * 2;
  g.page_bytes = (off + 127) & ~127;
  g.lane_major = d % 128 == 0 ? 1 : 0;
  // the parts of a page in LDS: odd multiples of 128 bytes, so that the two pages of a block start 32 banks apart
  g.kslot = heads_odd_lines(g.off_vdata);
  g.vslot = heads_odd_lines(g.page_bytes - g.off_vdata);
  return g;
}
// pairs of wavefronts of a workgroup: head tiles side by side x blocks side by side
constexpr int heads_hw(int tiles) { return tiles >= 3 ? 4 : tiles; }
constexpr int heads_tw(int hw) { return hw == 4 ? 1 : 4 - hw; }
// head tiles that a value wavefront sums (it takes as small a part of the channels)
constexpr int heads_vt(int hw) { return hw >= 2 ? 2 : 1; }
// LDS: sketched queries of the head tiles, two turns of key and of value parts, the weights a pair hands over
constexpr int heads_qs_bytes(int d, int hw) { return hw * 2 * (d / 64) * HQ_OP * 4; }
constexpr int HD_HAND = 9 * 64;            // floats of a pair's hand-over: 8 weights and the reference's move per lane
constexpr size_t heads_smem(int d, int mb, int vb, int hw) {
  const HeadsGeom g = heads_geom(d, mb, vb);
  const int tw = heads_tw(hw);
  return (size_t)heads_qs_bytes(d, hw) + (size_t)4 * tw * (g.kslot + g.vslot) + (size_t)hw * tw * HD_HAND * sizeof(float);
}

template <int SEL>
__device__ __forceinline__ f32x16 mfma_keys(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3, const i32x6& q, f32x16 c, int scale_q) {
  const i32x8 av = {(int)a0, (int)a1, (int)a2, (int)a3, 0, 0, 0, 0};
  const i32x8 bv = {q[0], q[1], q[2], q[3], q[4], q[5], 0, 0};
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, c, 4 /*A: fp4*/, 2 /*B: fp6 e2m3*/, 0, 128, SEL, scale_q);
}

template <int D, int MB, int VB, bool F16P, int HW>
__global__ void __launch_bounds__(128 * HW * heads_tw(HW), 2)
decode_heads_kernel(const uint32_t* __restrict__ qa, const float* __restrict__ q_stat, int Hq, int Hkv, int n_tiles,
                    const uint8_t* __restrict__ pool, const int32_t* __restrict__ block_table, int bt_stride,
                    const int32_t* __restrict__ seq_lens, tq_layer ly, float* __restrict__ parts, int n_parts, int n_split,
                    int len_sub, int max_pages, int num_pages) {
  constexpr int TW = heads_tw(HW), NP = HW * TW;                   // pairs of wavefronts
  constexpr int NX = MB == 3 ? 1 : 0, NC = D / 64, W = D / 32, NG = D / 32;
  constexpr HeadsGeom GC = heads_geom(D, MB, VB);
  static_assert(VB == 2 || VB == 4, "2- and 4-bit values");
  static_assert(MB == 2 || MB == 3, "3- and 4-bit keys: an even number of index planes and multi-bit terms");
  static_assert(heads_smem(D, MB, VB, HW) <= 160 * 1024, "LDS");
  static_assert(heads_smem(D, MB, VB, HW) >= sizeof(float) * (NP * (NG * 16 + 128) + HW * (TW - 1) * 2 * NG * 256), "room for the sums handed over at the end");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, kb = lane >> 4;
  // (wavefronts go to the SIMDs in turn: with four pairs a SIMD gets one of each role)
  const bool scorer = wave < NP;
  const int pair = scorer ? wave : wave - NP, hw = pair % HW, tw = pair / HW;
  // Workgroups go to the card's eight dies in turn, each with an L2 of its own: a die takes consecutive work items, so that the head
  // groups of a range of tokens (the same pages) and the ranges of a sequence (the same queries) share it.
  const int hgroups = (n_tiles + HW - 1) / HW;
  int item = (int)blockIdx.x;
  {
    const int total = (int)gridDim.x, die = item & 7, rest = total & 7;
    item = die * (total >> 3) + min(die, rest) + (item >> 3);
  }
  const int hg = item % hgroups, split = (item / hgroups) % n_split, bk = item / (hgroups * n_split);
  const int b = bk / Hkv, kvh = bk - b * Hkv, tile = hg * HW + hw;
  const bool live = tile < n_tiles;                                // (a pair without heads fetches pages and keeps the barriers)
  const int g_tot = Hq / Hkv;
  const int qbase = kvh * g_tot + tile * 16;                       // query head of column 0
  const int G = live ? min(16, g_tot - tile * 16) : 0;

  extern __shared__ __align__(16) unsigned char smem_raw[];
  unsigned char* qs = smem_raw;                                    // [HW][term pair][64 coordinates] sketched-query operands
  unsigned char* kring = qs + heads_qs_bytes(D, HW);               // [2][TW][2 pages][GC.kslot]
  unsigned char* vring = kring + 4 * TW * GC.kslot;                // [2][TW][2 pages][GC.vslot]
  float* hand = (float*)(vring + 4 * TW * GC.vslot) + pair * HD_HAND;      // [2][64][4] weights, [64] the reference's move

  const int seq_len = max(min(seq_lens[b], max_pages * TQ_PAGE_TOKENS) - len_sub, 0);
  const int n_pages = (seq_len + TQ_PAGE_TOKENS - 1) / TQ_PAGE_TOKENS;
  const int n_blocks = (seq_len + HD_BLK - 1) / HD_BLK;
  const int per_split = (n_blocks + n_split - 1) / n_split;
  const int blk_begin = split * per_split, blk_end = min(blk_begin + per_split, n_blocks);
  if (blk_begin >= blk_end) {                                      // nothing to read: an empty partial (the same for the whole workgroup)
    if (tw == 0 && scorer)
      for (int o = lane; o < G * (D + 2); o += 64) {
        const int g = o / (D + 2), e = o - g * (D + 2);
        parts[(((int64_t)b * Hq + qbase + g) * n_parts + split) * (D + 2) + e] = e == 0 ? MF_NEG * 0.6931471805599453f : 0.0f;
      }
    return;
  }
  const int n_iter = (blk_end - blk_begin + TW - 1) / TW;
  const int32_t* bt = block_table + (int64_t)b * bt_stride;
  const uint8_t* pool_h = pool + (int64_t)kvh * GC.page_bytes;
  const uint32_t page_stride = (uint32_t)((int64_t)Hkv * GC.page_bytes);

  // Page numbers: lane l of tbl_a holds the table entry of page pbase + l, tbl_b that of page pbase + 64 + l.  Entries past
  // the end of the sequence repeat the last one; an entry outside the pool becomes page 0 with the top bit set: its tokens
  // get no weight.
  int pbase = 2 * blk_begin;
  auto load_tbl = [&](int first) -> int {
    const int raw = bt[min(first + lane, n_pages - 1)];
    return (unsigned)raw < (unsigned)num_pages ? raw : (int)0x80000000;
  };
  bool has_bad;
  {
    bool bad = false;
    const int e1 = min(2 * blk_end, n_pages);
    for (int e = 2 * blk_begin + lane; e < e1; e += 64) bad |= (unsigned)bt[e] >= (unsigned)num_pages;
    has_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
  }
  int tbl_a = load_tbl(pbase), tbl_b = load_tbl(pbase + 64);
  // (used here, so that the compiler knows of no pending load of its own inside the loop)
  asm volatile("" : "+v"(tbl_a), "+v"(tbl_b));
  auto page_entry = [&](int page) -> int {
    const int rel = __builtin_amdgcn_readfirstlane(min(page, n_pages - 1) - pbase);
    const int ea = __builtin_amdgcn_readlane(tbl_a, rel & 63), eb = __builtin_amdgcn_readlane(tbl_b, rel & 63);
    return rel < 64 ? ea : eb;
  };
  // existing tokens of page pg of block blk: a prefix (none on a page outside the pool)
  auto tokens_of = [&](int blk, int pg) -> int {
    if (has_bad && page_entry(2 * blk + pg) < 0) return 0;
    return min(max(seq_len - blk * HD_BLK - 16 * pg, 0), 16);
  };
  auto partial = [&](int blk) -> bool { return has_bad || (blk + 1) * HD_BLK > seq_len; };

  // Request k of this value wavefront in turn t: a kilobyte of the keys of turn t + 2 or of the values of turn t + 1 (the last
  // piece of a part overlaps the one before it); behind the last block of the range the last block is read again.
  constexpr int VBYTES = GC.page_bytes - GC.off_vdata;
  constexpr int PK = (GC.off_vdata + 1023) / 1024, PV = (VBYTES + 1023) / 1024, PP = PK + PV, TOTAL = TW * 2 * PP, NR = (TOTAL + NP - 1) / NP;
  static_assert(GC.off_vdata >= 1024 && VBYTES >= 1024, "a part of a page is at least one request long");
  const uint32_t kring_lds = (uint32_t)(uintptr_t)kring, vring_lds = (uint32_t)(uintptr_t)vring;
  // (the page address is a scalar and the lane's part a constant register)
  const uint32_t lane16 = (uint32_t)lane * 16;
  auto request = [&](int k, int t) __attribute__((always_inline)) {
    const int q = pair + k * NP;
    if (q >= TOTAL) return;                                        // (the same for the whole wavefront)
    const int pgi = q / PP, pc = q - pgi * PP;
    const bool keys = pc < PK;
    const int turn = keys ? t + 2 : t + 1;
    if (turn >= n_iter || turn < 0) return;
    const int blk = min(blk_begin + turn * TW + (pgi >> 1), blk_end - 1);
    const uint32_t pid = (uint32_t)page_entry(2 * blk + (pgi & 1)) & 0x7fffffffu;
    const int at = keys ? min(pc * 1024, GC.off_vdata - 1024) : min((pc - PK) * 1024, VBYTES - 1024);
    const uint32_t slot = (uint32_t)((turn & 1) * TW * 2 + pgi);
    const uint32_t lds = keys ? kring_lds + slot * GC.kslot + at : vring_lds + slot * GC.vslot + at;
    dma_so<16>(lane16, pool_h + (uint64_t)pid * page_stride + (keys ? at : GC.off_vdata + at),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)lds));
  };
  const uint32_t* qsrc = qa + (((int64_t)b * Hkv + kvh) * n_tiles + (live ? tile : 0)) * (int64_t)(4 * NC * HQ_OP);

  if (scorer) {
    // ================================================================ scores and softmax, a turn ahead of the values
    i32x6 Q[2][NC];
    int sq;                                                        // E8M0 codes of this lane's column: (product, term pair) in bytes
    float c_idx, c_sgn;
    {
#pragma unroll
      for (int tp = 0; tp < 2; ++tp)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const uint32_t* op = qsrc + (tp * NC + c) * HQ_OP;
          const u32x4 lo = *(const u32x4*)(op + lane * 4);
          const uint2 hi = *(const uint2*)(op + 256 + lane * 2);
          Q[tp][c] = i32x6{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi.x, (int)hi.y};
        }
      const bool in = n < G;
      const f32x4 st = in ? *(const f32x4*)(q_stat + ((int64_t)b * Hq + qbase + n) * 4) : f32x4{0, 0, 0, 0};
      const int e1 = 127 + (int)st[0], e2 = 127 + (int)st[1];
      // column (head, t): term t of pair 0, t + 2 of pair 1; 4 v / 2^E is stored, so term t carries 2^(E - 2 - 5 t)
      const int t01 = (kb & 1) ? 7 : 2, t23 = t01 + 10;
      sq = (e1 - t01) | ((e1 - t23) << 8) | ((e2 - t01) << 16) | ((e2 - t23) << 24);
      c_idx = st[2]; c_sgn = st[3];
    }
    // the sketched queries of this head tile to LDS, the tile's scorers a share each
    {
      constexpr int BYTES = 2 * NC * HQ_OP * 4;                    // (a multiple of a kilobyte and a half)
      const uint8_t* src = (const uint8_t*)(qsrc + 2 * NC * HQ_OP);
      const uint32_t at0 = (uint32_t)(uintptr_t)qs + (uint32_t)(hw * BYTES);
      for (int pc = tw; pc < (BYTES + 1023) / 1024; pc += TW) {
        const int at = min(pc * 1024, BYTES - 1024);
        dma_so<16>(lane16, src + at, (uint32_t)__builtin_amdgcn_readfirstlane((int)(at0 + (uint32_t)at)));
      }
    }
    // coefficient of every index term plane: the bits from the highest down, then the multi-bit term
    float coef[MB + NX];
#pragma unroll
    for (int p = 0; p < MB + NX; ++p) coef[p] = 0.0f;
    int xpl = 0;
    for (int t = 0; t < ly.n_terms; ++t) {
#pragma unroll
      for (int p = 0; p < MB; ++p)
        if (ly.term_mask[t] == (1 << (MB - 1 - p))) coef[p] = ly.term_coef[t];
      if (NX && __builtin_popcount(ly.term_mask[t]) > 1) {
        coef[MB + NX - 1] = ly.term_coef[t];
#pragma unroll
        for (int p = 0; p < MB; ++p)
          if (ly.term_mask[t] & (1 << (MB - 1 - p))) xpl |= 1 << p;
      }
    }
    uint32_t xmask[MB];                                            // the stored planes the multi-bit term XORs
#pragma unroll
    for (int k = 0; k < MB; ++k) xmask[k] = (__builtin_amdgcn_readfirstlane(xpl) >> k) & 1 ? 0xffffffffu : 0u;
    float m_run = MF_NEG, l_run = 0.0f;
    const unsigned char* q_lds = qs + hw * (2 * NC * HQ_OP * 4) + lane * 16;
    const int half = lane >> 5;
    // everything has landed, said in a way the compiler counts (it would wait for the operands inside the loop)
    __builtin_amdgcn_s_waitcnt(0x0F70);
    for (int t = -1; t < n_iter; ++t) {
      __syncthreads();                                             // the keys of turn t + 1 have landed
      if (2 * (blk_begin + max(t, 0) * TW) >= pbase + 64) {        // the table registers move on (every wavefront alike)
        pbase += 64;
        tbl_a = tbl_b;
        tbl_b = load_tbl(pbase + 64);
        asm volatile("" : "+v"(tbl_b));
      }
      const int blk = blk_begin + (t + 1) * TW + tw;
      const bool work = live && t + 1 < n_iter && blk < blk_end;
      float sc[8], alpha = 1.0f;
      if (work) {
        // row operand of the scores: lane (token lane % 32, word 2 c + lane / 32)
        const unsigned char* kp = kring + (((t + 1) & 1) * TW * 2 + tw * 2 + (kb & 1)) * GC.kslot;
        auto word = [&](int p, int c) __attribute__((always_inline)) -> uint32_t {
          if (GC.lane_major) {
            constexpr int W4 = W / 4;
            return *(const uint32_t*)(kp + (((((2 * c + half) & 3) * 16 + n) * W4 + (c >> 1)) * (MB + 1) + p) * 4);
          }
          return *(const uint32_t*)(kp + ((p * W + 2 * c + half) * 16 + n) * 4);
        };
        f32x16 s_idx, u[2];
        uint32_t kx[NC];
        auto mfma2 = [&](auto sel_c, uint32_t x, const i32x6& qv, f32x16 c) __attribute__((always_inline)) {
          return mfma_keys<decltype(sel_c)::value>(x & 0x11111111u, x & 0x22222222u, x & 0x44444444u, (x >> 3) & 0x11111111u, qv, c, sq);
        };
        // Two sums at a time, their products in turn, so that a product need not wait for the one before it.
#pragma unroll
        for (int p = 0; p < MB + NX; p += 2) {                     // the index planes and the multi-bit term, in pairs
#pragma unroll
          for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int i = 0; i < 16; ++i) u[k][i] = 0.0f;
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            uint32_t x[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              if (p + k == MB) x[k] = kx[c];
              else {
                x[k] = word(p + k, c);
                if (NX) kx[c] = p + k == 0 ? x[k] & xmask[0] : kx[c] ^ (x[k] & xmask[p + k]);
              }
            }
            u[0] = mfma2(std::integral_constant<int, 0>{}, x[0], Q[0][c], u[0]);
            u[1] = mfma2(std::integral_constant<int, 0>{}, x[1], Q[0][c], u[1]);
            u[0] = mfma2(std::integral_constant<int, 1>{}, x[0], Q[1][c], u[0]);
            u[1] = mfma2(std::integral_constant<int, 1>{}, x[1], Q[1][c], u[1]);
          }
#pragma unroll
          for (int i = 0; i < 16; ++i) s_idx[i] = fmaf(coef[p + 1], u[1][i], p == 0 ? coef[0] * u[0][i] : fmaf(coef[p], u[0][i], s_idx[i]));
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int i = 0; i < 16; ++i) u[k][i] = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; ++c) {                             // the sign plane, a sum per term pair
          const uint32_t x = word(MB, c);
#pragma unroll
          for (int tp = 0; tp < 2; ++tp) {
            const unsigned char* op = q_lds + (tp * NC + c) * (HQ_OP * 4);
            const u32x4 lo = *(const u32x4*)op;
            const uint2 hi = *(const uint2*)(op + 1024 - lane * 8);
            const i32x6 qv = {(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi.x, (int)hi.y};
            if (tp) u[1] = mfma2(std::integral_constant<int, 3>{}, x, qv, u[1]);
            else u[0] = mfma2(std::integral_constant<int, 2>{}, x, qv, u[0]);
          }
        }
        f32x16 s_sgn;
#pragma unroll
        for (int i = 0; i < 16; ++i) s_sgn[i] = u[0][i] + u[1][i];
        // register i of lane (column head + 16 t, half h) is token 8 (i / 4) + 4 h + i % 4; a head's two columns are
        // neighbouring rows of lanes.  The swap of registers i and i + 8 between them leaves lane row kb with tokens
        // 4 (kb / 2) + i % 4 + 8 (i / 4) of page kb % 2, i = 0..7, and both columns' sums of them.
        const unsigned char* meta = kp + GC.off_meta + (kb >> 1) * 32;
        f32x4 m4[4];                                               // (norm, residual norm) of tokens i, i + 1
#pragma unroll
        for (int i = 0; i < 4; ++i) m4[i] = *(const f32x4*)(meta + (2 * (i & 1) + 8 * (i >> 1)) * 8);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const auto ri = __builtin_amdgcn_permlane16_swap(__float_as_uint(s_idx[i]), __float_as_uint(s_idx[i + 8]), false, false);
          const auto rs = __builtin_amdgcn_permlane16_swap(__float_as_uint(s_sgn[i]), __float_as_uint(s_sgn[i + 8]), false, false);
          const float dot = (__uint_as_float(ri[0]) + __uint_as_float(ri[1])) + c_idx;
          const float sgn = (__uint_as_float(rs[0]) + __uint_as_float(rs[1])) + c_sgn;
          sc[i] = fmaf(m4[i >> 1][2 * (i & 1)], dot, m4[i >> 1][2 * (i & 1) + 1] * sgn);
        }
        if (partial(blk)) {                                        // (the same for the whole wavefront)
          const int have = (kb & 1) ? tokens_of(blk, 1) : tokens_of(blk, 0);
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (4 * (kb >> 1) + (i & 3) + 8 * (i >> 2) >= have) sc[i] = -INFINITY;
        }
        float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
        // The reference of a head only moves when a score exceeds it by more than a small slack (weights are at most
        // 2^REF_SLACK), so the usual block rescales nothing.
        constexpr float REF_SLACK = 4.0f;
        if (__builtin_amdgcn_ballot_w64(mx > m_run + REF_SLACK) != 0) {
          mx = max_xor32(mx);
          mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
          const bool move = mx > m_run + REF_SLACK;
          const float m_new = move ? mx : m_run;
          alpha = move ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
          m_run = m_new;
          l_run *= alpha;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          sc[i] = __builtin_amdgcn_exp2f(sc[i] - m_run);
          l_run += sc[i];
        }
      }
      __syncthreads();                                             // the partner is done with the weights of turn t
      if (work) {
        *(f32x4*)(hand + lane * 4) = f32x4{sc[0], sc[1], sc[2], sc[3]};
        *(f32x4*)(hand + 256 + lane * 4) = f32x4{sc[4], sc[5], sc[6], sc[7]};
        hand[512 + lane] = alpha;
      }
    }
    l_run += __shfl_xor(l_run, 16, 64);
    l_run = sum_xor32(l_run);
    __syncthreads();                                               // LDS is free
    float* xm = (float*)smem_raw + pair * 128;
    xm[lane] = m_run;
    xm[64 + lane] = l_run;
    __syncthreads();
    if (TW > 1) __syncthreads();
    return;
  }

  // ================================================================== values
  // A value wavefront takes VT head tiles of its block and 1 / VT of the channels: codes are unpacked and scales widened once for both
  // tiles, with as many accumulators as one tile of all channels.
  constexpr int VT = heads_vt(HW), NGV = NG / VT, NZ = (NGV + 15) / 16;
  static_assert(NG % VT == 0, "whole groups of channels");
  const int part = hw % VT, vpair = pair - part;                   // channels; first pair whose weights are read
  const int g0 = part * NGV, vtile = tile - part;
  const bool vlive = vtile < n_tiles;                              // (the second tile may lack heads: its sums are dropped)
  const float* vhand = hand - part * HD_HAND;
  // (the longer of the two roles, and the younger wavefronts, which a SIMD serves last)
  __builtin_amdgcn_s_setprio(2);
  f32x4 acc[VT][2 * NGV], zacc[VT][NZ];
#pragma unroll
  for (int v = 0; v < VT; ++v) {
#pragma unroll
    for (int c = 0; c < 2 * NGV; ++c) acc[v][c] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < NZ; ++c) zacc[v][c] = f32x4{0, 0, 0, 0};
  }
  for (int k = 0; k < NR; ++k) request(k, -2);                     // the keys of turn 0
  const uint32_t sel = (kb & 2) ? 0x07060302u : 0x05040100u;       // 4-bit codes: this lane's sixteen bits of a channel's two words
  for (int t = -1; t < n_iter; ++t) {
    stage_wait<0>();                                               // the values of this turn and the keys of the next have landed
    __syncthreads();
    if (2 * (blk_begin + max(t, 0) * TW) >= pbase + 64) {
      pbase += 64;
      tbl_a = tbl_b;
      tbl_b = load_tbl(pbase + 64);
      asm volatile("" : "+v"(tbl_b));
    }
    const int blk = blk_begin + t * TW + tw;
    if (vlive && t >= 0 && blk < blk_end) {
      float p[VT][8];
#pragma unroll
      for (int v = 0; v < VT; ++v) {
        const float* hv = vhand + v * HD_HAND;
        const f32x4 h0 = *(const f32x4*)(hv + lane * 4), h1 = *(const f32x4*)(hv + 256 + lane * 4);
        const float alpha = vtile + v < n_tiles ? hv[512 + lane] : 1.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[v][i] = h0[i];
          p[v][4 + i] = h1[i];
        }
        if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
          for (int c = 0; c < 2 * NGV; ++c) acc[v][c] *= alpha;
#pragma unroll
          for (int c = 0; c < NZ; ++c) zacc[v][c] *= alpha;
        }
      }
      const unsigned char* vp = vring + ((t & 1) * TW * 2 + tw * 2 + (kb & 1)) * GC.vslot - GC.off_vdata;      // offsets are those of the page
      if (partial(blk)) {
        // Tokens that do not exist: their slots may hold anything, and zero times anything has to be zero: their scales and
        // zero points become zero in LDS (the value wavefronts of a block all write the same).
        unsigned char* page = vring + ((t & 1) * TW * 2 + tw * 2) * GC.vslot + (GC.off_vscale - GC.off_vdata);
        for (int o = lane; o < 4 * NG * 8; o += 64) {              // [2 pages][scales, zero points][NG][8 pairs of tokens]
          const int pg = o / (2 * NG * 8), r = o - pg * (2 * NG * 8), have = pg ? tokens_of(blk, 1) : tokens_of(blk, 0);
          uint32_t* w = (uint32_t*)(page + pg * GC.vslot) + r;
          const int tok = 2 * (r & 7);
          *w &= (tok < have ? 0x0000ffffu : 0u) | (tok + 1 < have ? 0xffff0000u : 0u);
        }
        stage_release();
      }
      // zero points: groups as rows, tokens in natural order
#pragma unroll
      for (int zt = 0; zt < NZ; ++zt) {
        const unsigned char* zr = vp + GC.off_vzero + ((g0 + min(16 * zt + n, NGV - 1)) * 16 + 4 * (kb >> 1)) * 2;
        const uint2 z0 = *(const uint2*)zr, z1 = *(const uint2*)(zr + 16);
        const u32x4 az = {z0.x, z0.y, z1.x, z1.y};
#pragma unroll
        for (int v = 0; v < VT; ++v) {
          u32x4 pz;
#pragma unroll
          for (int r = 0; r < 4; ++r) pz[r] = F16P ? pack_f16(p[v][2 * r], p[v][2 * r + 1]) : pack_bf16(p[v][2 * r], p[v][2 * r + 1]);
          zacc[v][zt] = F16P ? mfma_f16(az, pz, zacc[v][zt]) : mfma(az, pz, zacc[v][zt]);
        }
      }
      // the code of register r's tokens sits at bit s of its 16-bit half, where it is the bf16 number code x 2^(s - 133): the
      // weight carries 2^(80 - s)
#pragma unroll
      for (int v = 0; v < VT; ++v)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int r = i & 3;
          p[v][i] *= VB == 4 ? ((r & 1) ? 0x1p76f : 0x1p80f) : (r == 0 ? 0x1p80f : (r == 1 ? 0x1p78f : (r == 2 ? 0x1p76f : 0x1p74f)));
        }
      const unsigned char* srow = vp + GC.off_vscale + 8 * (kb >> 1) + g0 * 32;
      const unsigned char* vrow = vp + GC.off_vdata + n * (D / 16) * (VB * 2) + g0 * (VB * 4);
#pragma unroll
      for (int g = 0; g < NGV; ++g) {
#pragma unroll
        for (int k = 0; k < NR; ++k)
          if (k * NGV / NR == g) request(k, t);
        const uint2 f0 = *(const uint2*)(srow + g * 32), f1 = *(const uint2*)(srow + g * 32 + 16);      // scales of tokens 4 u .., 8 + 4 u ..
        auto lo = [&](uint32_t w) { return F16P ? f16_lo(w) : __uint_as_float(w << 16); };
        auto hi = [&](uint32_t w) { return F16P ? f16_hi(w) : __uint_as_float(w & 0xffff0000u); };
        const float sv[8] = {lo(f0.x), hi(f0.x), lo(f0.y), hi(f0.y), lo(f1.x), hi(f1.x), lo(f1.y), hi(f1.y)};
        u32x4 a0, a1;
        if (VB == 4) {
          const uint32_t m0 = 0x000F000Fu, m1 = 0x00F000F0u;
          const u32x4 f = *(const u32x4*)(vrow + g * 16);
          const uint32_t x = __builtin_amdgcn_perm(f[1], f[0], sel), y = __builtin_amdgcn_perm(f[3], f[2], sel);
          a0 = u32x4{x & m0, x & m1, (x >> 8) & m0, (x >> 8) & m1};
          a1 = u32x4{y & m0, y & m1, (y >> 8) & m0, (y >> 8) & m1};
        } else {
          const uint32_t m0 = 0x00030003u, m1 = 0x000C000Cu, m2 = 0x00300030u, m3 = 0x00C000C0u;
          const uint2 f = *(const uint2*)(vrow + g * 8);
          const uint32_t x = f.x >> (8 * (kb >> 1)), y = f.y >> (8 * (kb >> 1));
          a0 = u32x4{x & m0, x & m1, x & m2, x & m3};
          a1 = u32x4{y & m0, y & m1, y & m2, y & m3};
        }
#pragma unroll
        for (int v = 0; v < VT; ++v) {
          u32x4 wv;
#pragma unroll
          for (int r = 0; r < 4; ++r) wv[r] = pack_bf16(p[v][r] * sv[r], p[v][4 + r] * sv[4 + r]);
          acc[v][2 * g] = mfma(a0, wv, acc[v][2 * g]);
          acc[v][2 * g + 1] = mfma(a1, wv, acc[v][2 * g + 1]);
        }
      }
    } else {
      for (int k = 0; k < NR; ++k) request(k, t);
    }
    __syncthreads();                                               // (the scorers hand over the next weights)
  }

  // ---------------------------------------------------------------- the partial (m, l, acc[d]) of every head
  __syncthreads();                                                 // LDS is free
  float* s_ep = (float*)smem_raw;
  float* mine = s_ep + NP * 128 + pair * (NG * 16);                // zero-point sums [tile][group][head]: lane (head n, groups 4 kb ..) of tile zt
#pragma unroll
  for (int v = 0; v < VT; ++v)
#pragma unroll
    for (int zt = 0; zt < NZ; ++zt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (16 * zt + 4 * kb + i < NGV) mine[(v * NGV + 16 * zt + 4 * kb + i) * 16 + n] = zacc[v][zt][i];
  stage_release();                                                 // (read back by the same wavefront only)
#pragma unroll
  for (int v = 0; v < VT; ++v)
#pragma unroll
    for (int g = 0; g < NGV; ++g) {
      const float z = mine[(v * NGV + g) * 16 + n];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[v][2 * g][i] = fmaf(acc[v][2 * g][i], 0x1p53f, z);
        acc[v][2 * g + 1][i] = fmaf(acc[v][2 * g + 1][i], 0x1p53f, z);
      }
    }
  float* xa = s_ep + NP * (128 + NG * 16) + (hw * (TW - 1)) * (2 * NG * 256);      // [TW - 1][2 NG][64][4]
  if (TW > 1 && tw > 0) {
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
      for (int c = 0; c < 2 * NGV; ++c) *(f32x4*)(xa + (((tw - 1) * 2 * NG + v * 2 * NGV + c) * 64 + lane) * 4) = acc[v][c];
  }
  __syncthreads();
  if (TW > 1) __syncthreads();
  if (tw > 0) return;
#pragma unroll
  for (int v = 0; v < VT; ++v) {
    if (vtile + v >= n_tiles) return;
    const float* xm = s_ep + (vpair + v) * 128;                    // the scorer's (m, l)
    float m_run = xm[lane], l_run = xm[64 + lane];
    // the blocks side by side: the first wavefront of a head tile and channel part adds the others' sums
#pragma unroll 1
    for (int o = 1; o < TW; ++o) {
      const float m1 = xm[o * HW * 128 + lane], l1 = xm[o * HW * 128 + 64 + lane], m_new = fmaxf(m_run, m1);
      const float f0 = __builtin_amdgcn_exp2f(m_run - m_new), f1 = __builtin_amdgcn_exp2f(m1 - m_new);
      l_run = fmaf(l_run, f0, l1 * f1);
      m_run = m_new;
#pragma unroll
      for (int c = 0; c < 2 * NGV; ++c) {
        const f32x4 x = *(const f32x4*)(xa + (((o - 1) * 2 * NG + v * 2 * NGV + c) * 64 + lane) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[v][c][i] = fmaf(acc[v][c][i], f0, x[i] * f1);
      }
    }
    const int vbase = qbase + (v - part) * 16;                     // query head of column 0
    if (n < min(16, g_tot - (vtile + v) * 16)) {
      float* row = parts + (((int64_t)b * Hq + vbase + n) * n_parts + split) * (D + 2);
      if (part == 0 && kb == 0) *(f32x2*)row = f32x2{m_run * 0.6931471805599453f, l_run};      // natural-log domain
      row += 2 + 32 * g0 + 4 * kb;
#pragma unroll
      for (int c = 0; c < 2 * NGV; ++c) {
        *(f32x2*)(row + 16 * c) = f32x2{acc[v][c][0], acc[v][c][1]};
        *(f32x2*)(row + 16 * c + 2) = f32x2{acc[v][c][2], acc[v][c][3]};
      }
    }
  }
}

// Whether a step of this shape runs the kernel above: more than 8 query heads per KV head, head_dim 512 / 576, 3- or 4-bit
// keys, 2- or 4-bit values, the page layout the library makes.  Not one sequence on one KV head (pairs: their product) whose splits of 8 heads each
// the card holds at once: the other kernel's groups of 8 heads take a compute unit each then, and their turns are shorter
// (576, 4-bit, best split counts of either, there / here: 16 heads x 8192 32 / 40 us, x 32768 47 / 53; 64 heads x 300 22.5 / 27.3, x 8192
// 37 / 45, x 16384 49 / 55; two sequences fill the card here).
bool decode_heads_has_kernel(const tq_layer& ly, const tq_page_layout& L, int g_tot, int64_t pairs, int n_split) {
  if (opt_wide_heads.load(std::memory_order_relaxed) == 0 || g_tot <= 8 || g_tot > 128) return false;
  if (pairs <= 1 && (g_tot <= 16 || n_split * ((g_tot + 7) / 8) <= device_compute_units())) return false;
  if ((ly.d != 512 && ly.d != 576) || L.d != ly.d || (ly.mse_bits != 2 && ly.mse_bits != 3) || L.mse_bits != ly.mse_bits) return false;
  if ((L.value_bits != 2 && L.value_bits != 4) || L.group_size != 32 || (L.dtype != TQ_BF16 && L.dtype != TQ_F16)) return false;
  int nx = 0;
  for (int t = 0; t < ly.n_terms; ++t)
    if (__builtin_popcount(ly.term_mask[t]) > 1) ++nx;
  if (ly.n_terms <= 0 || nx != (ly.mse_bits == 3 ? 1 : 0)) return false;
  const HeadsGeom g = heads_geom(L.d, L.mse_bits, L.value_bits);
  return L.off_keys == 0 && L.off_meta == g.off_meta && L.off_vdata == g.off_vdata && L.off_vscale == g.off_vscale &&
         L.off_vzero == g.off_vzero && L.page_bytes == g.page_bytes && L.key_lane_major == g.lane_major;
}

int launch_decode_heads(int B, int Hq, int Hkv, const uint8_t* pool, const int32_t* block_table, int bt_stride,
                        const int32_t* seq_lens, const tq_layer& ly, const tq_page_layout& L, float* parts, int n_parts,
                        int n_split, int len_sub, int max_pages, int num_pages, const WidePack& pre, hipStream_t st) {
  const int n_tiles = (Hq / Hkv + 15) / 16, hw = heads_hw(n_tiles);
  const int64_t items = (int64_t)B * Hkv * n_split * ((n_tiles + hw - 1) / hw);
  if (items > 0x7fffffff) return TQ_EUNSUPPORTED;
  const dim3 grid((unsigned)items);
  hipEvent_t t_start = nullptr, t_stop = nullptr;
  const bool timed = take_time_hook(0, t_start, t_stop);
#define TQ_HEADS(D, MB, VB, F16P, HW)                                                                                  \
  {                                                                                                                    \
    auto kern = decode_heads_kernel<D, MB, VB, F16P, HW>;                                                              \
    constexpr size_t smem = heads_smem(D, MB, VB, HW);                                                                  \
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);      \
    if (e != hipSuccess) return (int)e;                                                                                \
    const dim3 block(128 * HW * heads_tw(HW));                                                                         \
    if (timed)                                                                                                         \
      hipExtLaunchKernelGGL(kern, grid, block, smem, st, t_start, t_stop, 0, pre.qa, pre.q_stat, Hq, Hkv, n_tiles,     \
                            pool, block_table, bt_stride, seq_lens, ly, parts, n_parts, n_split, len_sub, max_pages,   \
                            num_pages);                                                                                \
    else                                                                                                               \
      kern<<<grid, block, smem, st>>>(pre.qa, pre.q_stat, Hq, Hkv, n_tiles, pool, block_table, bt_stride, seq_lens,    \
                                      ly, parts, n_parts, n_split, len_sub, max_pages, num_pages);                     \
  }
#define TQ_HEADS_HW(D, MB, VB, F16P)               \
  {                                                \
    if (hw == 1) TQ_HEADS(D, MB, VB, F16P, 1)      \
    else if (hw == 2) TQ_HEADS(D, MB, VB, F16P, 2) \
    else TQ_HEADS(D, MB, VB, F16P, 4)              \
  }
#define TQ_HEADS_T(D, MB, VB)                              \
  {                                                        \
    if (L.dtype == TQ_F16) TQ_HEADS_HW(D, MB, VB, true)    \
    else TQ_HEADS_HW(D, MB, VB, false)                     \
  }
#define TQ_HEADS_V(D)                                              \
  {                                                                \
    if (ly.mse_bits == 3 && L.value_bits == 4) TQ_HEADS_T(D, 3, 4) \
    else if (ly.mse_bits == 3) TQ_HEADS_T(D, 3, 2)                 \
    else if (L.value_bits == 4) TQ_HEADS_T(D, 2, 4)                \
    else TQ_HEADS_T(D, 2, 2)                                       \
  }
  if (ly.d == 576) TQ_HEADS_V(576)
  else TQ_HEADS_V(512)
#undef TQ_HEADS_V
#undef TQ_HEADS_T
#undef TQ_HEADS_HW
#undef TQ_HEADS
  TQ_CHECK_LAUNCH();
  return TQ_OK;
}

}  // namespace tq
